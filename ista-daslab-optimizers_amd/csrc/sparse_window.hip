// Sparse M-FAC's kernels over the window of MicroAdam's layout (m rows of k block-relative int16
// indices and k values, k_block_size entries per top-k block of d_block_size coordinates):
//   scalar products of the rows with a dense vector
//     (ista_daslab_cuda_sparse_mfac.SP, sparse_mfac/sparse_core_mfac_w_ef.py:185-203),
//   linear combination of the rows into a dense vector
//     (ista_daslab_cuda_sparse_mfac.LCG, sparse_core_mfac_w_ef.py:205-221),
//   copy_values with fp32 window values (sparse_core_mfac_w_ef.py:105-124, use_bf16 = False).
// A workgroup works on one top-k block: the block of the dense vector lives in LDS, the window
// entries of the block stream past it once.  Part of libmicroadam_hip.so.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/microadam_hip.h"
#include "ma_device.hpp"

namespace ma {
namespace {

constexpr int kLdsBytes = 160 * 1024;
constexpr int kRingRows = 32;          // rows the linear combination requests ahead
constexpr int kShortRing = 16;        // the same for rows of one to three entries
constexpr int kCombineThreads = 256;  // of a workgroup in which one wave applies the rows
constexpr int kSmallBlock = 13653;    // coordinates: more than two such blocks fit a CU's LDS
constexpr int kDotUnroll = 4;          // entries a lane requests ahead in the scalar products

__device__ __forceinline__ float widen(float x) { return x; }
__device__ __forceinline__ float widen(uint16_t x) { return bf2f(x); }
__device__ __forceinline__ void narrow(float *p, float v) { *p = v; }
__device__ __forceinline__ void narrow(uint16_t *p, float v) { *p = (uint16_t)f2bf(v); }

struct BlockSpan {
    int64_t e0;    // first coordinate of the top-k block
    int64_t col0;  // first window column of the block
    int len;       // coordinates in the block
    int kb;        // window entries per row in the block
};

// Work item of this workgroup, of `total`: the hardware deals consecutive workgroups to the 8
// XCDs in turn, the items are dealt so that every XCD, with its own L2, walks one contiguous
// eighth.  Neighbouring blocks' stretches of a window row share cache lines (410 bytes of 205
// bf16 entries touch 4.2 lines of 128).
__device__ __forceinline__ int xcd_item(int total) {
    constexpr int kXcds = 8;
    const int x = (int)blockIdx.x % kXcds, j = (int)blockIdx.x / kXcds;
    const int q = total / kXcds, r = total % kXcds;
    return x * q + (x < r ? x : r) + j;
}

__device__ __forceinline__ BlockSpan block_span(int64_t d, int dbs, int kbs, int64_t k, int64_t b) {
    BlockSpan s;
    s.e0 = b * dbs;
    s.col0 = b * kbs;
    const int64_t len = d - s.e0, kb = k - s.col0;
    s.len = (int)(len < dbs ? len : dbs);
    s.kb = (int)(kb < kbs ? kb : kbs);
    return s;
}

// Four window entries as they lie in memory, from any boundary an entry can lie on (the hardware
// takes unaligned loads).
struct __attribute__((packed, aligned(2))) IndexQuad {
    uint32_t w[2];
    __device__ __forceinline__ uint32_t index(int e) const {
        return (e & 1) ? w[e >> 1] >> 16 : w[e >> 1] & 0xffffu;
    }
    // both halves: the larger of `top` and the indices in that half
    __device__ __forceinline__ uint32_t largest(uint32_t top) const {
        typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
        const u16x2 t = __builtin_bit_cast(u16x2, top), a = __builtin_bit_cast(u16x2, w[0]),
                    b = __builtin_bit_cast(u16x2, w[1]);
        return __builtin_bit_cast(
            uint32_t, __builtin_elementwise_max(__builtin_elementwise_max(t, a), b));
    }
};
// two 16-bit numbers, each at most the one in `most`
__device__ __forceinline__ uint32_t both_at_most(uint32_t w, uint32_t most) {
    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(
        uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2, w), __builtin_bit_cast(u16x2, most)));
}
template <typename TV>
struct ValueQuad;
template <>
struct __attribute__((packed, aligned(2))) ValueQuad<uint16_t> {
    uint32_t w[2];
    __device__ __forceinline__ float value(int e) const {
        return __uint_as_float((e & 1) ? w[e >> 1] & 0xffff0000u : w[e >> 1] << 16);
    }
};
template <>
struct __attribute__((packed, aligned(4))) ValueQuad<float> {
    float f[4];
    __device__ __forceinline__ float value(int e) const { return f[e]; }
};

// First of the four entries that lane l holds of a row of kb >= 4: every entry is some lane's and
// no lane reads past the row; the last lanes hold entries that others hold too.
__device__ __forceinline__ int quad_start(int kb, int l) { return min(4 * l, kb - 4); }
// lanes' worth of quads, in wavefronts, that rows of kbs entries take
inline int quad_groups(int64_t kbs) { return (int)((kbs + 255) / 256); }

// 16 bytes of the dense vector += as many accumulators
__device__ __forceinline__ void add_sixteen_bytes(float *dst, const float *acc) {
    float4 o = *reinterpret_cast<const float4 *>(dst);
    const float4 a = *reinterpret_cast<const float4 *>(acc);
    o.x = o.x + a.x; o.y = o.y + a.y; o.z = o.z + a.z; o.w = o.w + a.w;
    *reinterpret_cast<float4 *>(dst) = o;
}
__device__ __forceinline__ void add_sixteen_bytes(uint16_t *dst, const float *acc) {
    uint4 o = *reinterpret_cast<const uint4 *>(dst);
    uint32_t *w = &o.x;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        w[i] = f2bf_pair(__uint_as_float(w[i] << 16) + acc[2 * i],
                         __uint_as_float(w[i] & 0xffff0000u) + acc[2 * i + 1]);
    *reinterpret_cast<uint4 *>(dst) = o;
}

// ---- scalar products ------------------------------------------------------------------------
// partial[b][r] = sum over the entries of row r in block b of V * g.  The block of g is staged in
// LDS in its own type and is all the LDS the kernel uses, so that four workgroups with a
// 20480-element bf16 block share a CU.  The second kernel adds the blocks' partial sums in a
// fixed order.

// wavefronts of lanes that rows of up to kbs entries take, with one entry before the first
inline int dot_groups(int64_t kbs) { return (int)((kbs + 1 + 255) / 256); }

// sum over the 64 lanes, in lane 63
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ float add_from(float v) {
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK,
                                                          0xF, true));
}
__device__ __forceinline__ float wave_sum_to_last(float v) {
    v = add_from<0x111>(v);       // row_shr 1, 2, 4, 8: the last lane of every 16
    v = add_from<0x112>(v);
    v = add_from<0x114>(v);
    v = add_from<0x118>(v);
    v = add_from<0x142, 0xA>(v);  // the rows' sums into the rows behind them
    return add_from<0x143, 0xC>(v);
}

// A wave sums ROWS rows at a time, four entries a request, the next ROWS rows requested before.
// What bounds it is how the window's 1 GB (25.6 M coordinates, 1024 rows of 1 %, bf16) is asked for:
// 16 two-byte requests a lane took 309 us; eight bytes a request with the workgroups of a block
// and of its neighbours on one XCD 260; the same from 4-byte boundaries 223 (4.7 TB/s).  The
// gathers from LDS are hidden behind it; four rows at a time and more or fewer workgroups a
// block were no faster (225 to 237), a block of g staged with five requests under way slower.
// G: as dot_groups; 0: rows of any length, entry by entry.
template <typename TG, typename TV, int G>
__global__ __launch_bounds__(kWG, 8) void sparse_dot_kernel(int64_t d, int dbs, int kbs, int64_t k,
                                                         int m_rows, int nblocks, int shares,
                                                         const TG *g, const int16_t *I,
                                                         const TV *V, float *partial) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int item = xcd_item(nblocks * shares), block = item / shares;
    const BlockSpan S = block_span(d, dbs, kbs, k, block);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    TG *gl = (TG *)lds_raw;

    // `shares` workgroups share the rows of a block
    constexpr int kWaves = kWG / 64;
    const int per = (m_rows + shares - 1) / shares;
    const int row_lo = item % shares * per;
    const int row_hi = row_lo + per < m_rows ? row_lo + per : m_rows;
    float *dst = partial + (int64_t)block * m_rows;

    auto stage = [&]() {
        const TG *src = g + S.e0;
        constexpr int kPer16 = 16 / sizeof(TG);
        int staged = 0;
        if ((((uintptr_t)src) & 15) == 0) {
            const int n16 = S.len / kPer16;
            for (int i = tid; i < n16; i += kWG) ((uint4 *)gl)[i] = ((const uint4 *)src)[i];
            staged = n16 * kPer16;
        }
        for (int i = staged + tid; i < S.len; i += kWG) gl[i] = src[i];
        __syncthreads();
    };

    if (G > 0 && S.kb >= 4) {
        constexpr int GG = G > 0 ? G : 1;
        constexpr int ROWS = 2;
        // Lane l takes the entries 4l .. 4l + 3 of a row's stretch, all one less if the stretch
        // begins on an odd entry: every load is 4-byte aligned then, where unaligned ones kept the
        // kernel at 260 us.  The outermost loads reach up to four entries into the neighbouring
        // stretches (a lane may start at entry kb: it is needed when the stretch begins one entry
        // earlier), whose terms are dropped; where the array may end behind the block the lanes
        // load from the stretch's own boundaries, aligned or not.
        const bool exact = S.col0 + S.kb + 4 > k;
        uint32_t from[GG];     // entry the lane's loads start at, from the row's first one
        bool own[2][GG][4];    // by the row's parity: which of the four are this lane's
#pragma unroll
        for (int q = 0; q < GG; ++q) {
            const int l = lane + q * 64;
            from[q] = (uint32_t)(exact ? min(4 * l, S.kb - 4) : 4 * l < S.kb + 1 ? 4 * l : 0);
#pragma unroll
            for (int odd = 0; odd < 2; ++odd)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int at = (int)from[q] - odd + e, lo = 4 * l - odd;
                    own[odd][q][e] = at >= lo && at < lo + 4 && at >= 0 && at < S.kb;
                }
        }
        auto first_of = [&](int r, int u) {
            const int row = r + u * kWaves < row_hi ? r + u * kWaves : row_hi - 1;
            return (int64_t)row * k + S.col0;
        };
        IndexQuad nix[ROWS][GG];
        ValueQuad<TV> nv[ROWS][GG];
        auto request = [&](int r) {
#pragma unroll
            for (int u = 0; u < ROWS; ++u) {
                int64_t first = first_of(r, u);
                if (!exact) first &= ~(int64_t)1;
#pragma unroll
                for (int q = 0; q < GG; ++q) {
                    uint32_t at = from[q] * 2u;
                    asm volatile("" : "+v"(at));  // (kept a 32-bit offset from the scalar address)
                    nix[u][q] = *reinterpret_cast<const IndexQuad *>(
                        reinterpret_cast<const char *>(I + first) + at);
                    nv[u][q] = *reinterpret_cast<const ValueQuad<TV> *>(
                        reinterpret_cast<const char *>(V + first) +
                        at * (uint32_t)(sizeof(TV) / 2));
                }
            }
        };
        if (row_lo < row_hi) request(row_lo + wave);
        stage();
        for (int r = row_lo + wave; r < row_hi; r += ROWS * kWaves) {
            IndexQuad ix[ROWS][GG];
            ValueQuad<TV> v[ROWS][GG];
            uint32_t top = 0;
#pragma unroll
            for (int u = 0; u < ROWS; ++u)
#pragma unroll
                for (int q = 0; q < GG; ++q) {
                    ix[u][q] = nix[u][q];
                    v[u][q] = nv[u][q];
                    top = ix[u][q].largest(top);
                }
            request(r + ROWS * kWaves);
            const bool stray =
                (top & 0xffffu) >= (uint32_t)S.len || (top >> 16) >= (uint32_t)S.len;
            const bool in_block = __builtin_amdgcn_ballot_w64(stray) == 0;
            float sum[ROWS];
            if (in_block) {
#pragma unroll
                for (int u = 0; u < ROWS; ++u) {
                    const bool odd = !exact && (first_of(r, u) & 1) != 0;
                    sum[u] = 0.0f;
#pragma unroll
                    for (int q = 0; q < GG; ++q) {
                        float t[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            t[e] = v[u][q].value(e) * widen(gl[ix[u][q].index(e)]);
                            t[e] = (odd ? own[1][q][e] : own[0][q][e]) ? t[e] : 0.0f;
                        }
                        sum[u] += (t[0] + t[1]) + (t[2] + t[3]);
                    }
                }
            } else {  // an index outside the block contributes nothing
#pragma unroll
                for (int u = 0; u < ROWS; ++u) {
                    const int64_t first = first_of(r, u);
                    sum[u] = 0.0f;
                    for (int j = lane; j < S.kb; j += 64) {
                        const int i = I[first + j];
                        if ((unsigned)i < (unsigned)S.len)
                            sum[u] += widen(V[first + j]) * widen(gl[i]);
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < ROWS; ++u) {
                const float all = wave_sum_to_last(sum[u]);
                if (lane == 63 && r + u * kWaves < row_hi) dst[r + u * kWaves] = all;
            }
        }
    } else {
        stage();
        // Two rows at a time, their requests without conditions (entries clamped into the row): under
        // a condition the compiler widens a value right behind its load and waits for it there.
        // 1220 blocks of 20480, 512 rows of 512 bf16: 420 us with conditions, 240 without.
        for (int r = row_lo + wave; r < row_hi; r += 2 * kWaves) {
            const bool two = r + kWaves < row_hi;
            const int64_t first[2] = {(int64_t)r * k + S.col0,
                                      (int64_t)(two ? r + kWaves : r) * k + S.col0};
            float acc[2] = {0.0f, 0.0f};
            for (int j0 = 0; j0 < S.kb; j0 += 64 * kDotUnroll) {
                int ix[2][kDotUnroll];
                TV v[2][kDotUnroll];
#pragma unroll
                for (int u = 0; u < kDotUnroll; ++u) {
                    const int j = min(j0 + u * 64 + lane, S.kb - 1);
#pragma unroll
                    for (int w = 0; w < 2; ++w) {
                        ix[w][u] = I[first[w] + j];
                        v[w][u] = V[first[w] + j];
                    }
                }
#pragma unroll
                for (int u = 0; u < kDotUnroll; ++u)
#pragma unroll
                    for (int w = 0; w < 2; ++w) {
                        const bool counts = j0 + u * 64 + lane < S.kb &&
                                            (unsigned)ix[w][u] < (unsigned)S.len;
                        const float t = widen(v[w][u]) * widen(gl[counts ? ix[w][u] : 0]);
                        acc[w] += counts ? t : 0.0f;
                    }
            }
#pragma unroll
            for (int w = 0; w < 2; ++w) {
                acc[w] = wave_sum_to_last(acc[w]);
                if (lane == 63 && (w == 0 || two)) dst[r + w * kWaves] = acc[w];
            }
        }
    }
}

// out[r] += sum over blocks of partial[b][r]: 16 rows per workgroup (a read covers 64 contiguous
// bytes), thread (part, row) adds blocks part, part + 32, ..., then the parts in order.
constexpr int kReduceRows = 16, kReduceParts = kWG / kReduceRows;
__global__ __launch_bounds__(kWG) void sparse_dot_reduce_kernel(const float *partial,
                                                                int64_t nblocks, int m_rows,
                                                                float *out) {
    __shared__ float part[kReduceParts][kReduceRows];
    const int rl = threadIdx.x % kReduceRows, p = threadIdx.x / kReduceRows;
    const int r = (int)blockIdx.x * kReduceRows + rl;
    float acc = 0.0f;
    if (r < m_rows) {
#pragma unroll 8
        for (int64_t b = p; b < nblocks; b += kReduceParts) acc += partial[b * m_rows + r];
    }
    part[p][rl] = acc;
    __syncthreads();
    if (p == 0 && r < m_rows) {
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < kReduceParts; ++i) sum += part[i][rl];
        out[r] = out[r] + sum;
    }
}

// ---- linear combination ---------------------------------------------------------------------
// acc[c] (fp32, LDS) takes the terms coef[r] * V[r][j] of the block's coordinates row by row in
// increasing r; the entries of one row name distinct coordinates, so a row is applied without
// atomics.  The accumulators fill the LDS (two 20480-element blocks per CU), so what bounds the
// kernel is the chain of rows.  ONE wave applies all rows of a block: the LDS operations of a wave
// execute in program order, so a row needs no barrier behind it, only its own reads; the next
// row's addresses and terms are formed, and a row's next request is made, while those are under
// way.  The window comes in through a ring of registers, four entries a request.  25.6 M coordinates,
// 1024 rows of 1 %, bf16: 360 us with the requests behind every fourth row and a check of its
// indices there, 332 in rounds of 32 rows without a branch.  With the LDS left out it still takes
// 300: what is left is one wave's issue of some 35 instructions a row, 230 cycles.  (LDS float
// atomics: 193 cycles a wave instruction, where a read and a write of four bytes take 12.)
typedef __attribute__((address_space(3))) float LdsFloat;
// read only, at addresses that are the same in all lanes: scalar loads
typedef __attribute__((address_space(4))) float ConstantFloat;

// LDS address of cell `half` (16 bits) of w: one instruction, as the kernel's dynamic LDS, which
// the accumulators begin, is all the LDS it has and so begins at address 0
template <int HALF>
__device__ __forceinline__ uint32_t cell_address(uint32_t w, uint32_t two) {
    uint32_t a;
    if (HALF == 0)
        asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD "
            "src1_sel:WORD_0" : "=v"(a) : "v"(two), "v"(w));
    else
        asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD "
            "src1_sel:WORD_1" : "=v"(a) : "v"(two), "v"(w));
    return a;
}

template <typename TV, int G, int RING, bool LONG>
__device__ __forceinline__ void combine_rows(float *acc, const BlockSpan &S, int64_t k, int m_rows,
                                             const float *coef, const int16_t *I, const TV *V,
                                             int lane) {
    constexpr uint32_t kWide = sizeof(TV) / 2;
    constexpr int kStep = 4;  // rows taken together behind the last whole round
    static_assert(RING % kStep == 0, "the ring in groups of kStep rows");
    // byte offset in a row of the indices of this lane's entries
    uint32_t start[G];
#pragma unroll
    for (int g = 0; g < G; ++g) start[g] = 2u * (uint32_t)quad_start(S.kb, lane + g * 64);
    IndexQuad ix[RING][G];
    ValueQuad<TV> v[RING][G];
    // Requests are made in row order and at every round alike (the last row again and again
    // behind the window's end), so that at any time the same number of them is under way and
    // the compiler can wait for the oldest ones alone.  Rows of a round are addressed from its
    // first one in 32 bits, LONG ones (RING of them do not fit) row by row.
    const uint32_t row_bytes = LONG ? 0 : (uint32_t)k * 2u;
    const int16_t *Ir = I + S.col0;
    const TV *Vr = V + S.col0;
    uint32_t row_at = 0, last_at = 0;
    int next_row = 0;
    auto aim = [&](int first) {  // the next RING requests are for the rows from `first` on
        if (LONG) return;
        const int row = first < m_rows ? first : m_rows - 1;
        const int more = m_rows - 1 - row;
        Ir = I + ((int64_t)row * k + S.col0);
        Vr = V + ((int64_t)row * k + S.col0);
        row_at = 0;
        last_at = (uint32_t)(more < RING ? more : RING) * row_bytes;
    };
    auto request = [&](int slot) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
            uint32_t at = start[g] + row_at;
            asm volatile("" : "+v"(at));  // (kept a 32-bit offset from the scalar address)
            ix[slot][g] = *reinterpret_cast<const IndexQuad *>(
                reinterpret_cast<const char *>(Ir) + at);
            v[slot][g] = *reinterpret_cast<const ValueQuad<TV> *>(
                reinterpret_cast<const char *>(Vr) + (at * kWide));
        }
        if (LONG) {
            const int64_t on = ++next_row < m_rows ? k : 0;
            Ir += on;
            Vr += on;
        } else {
            row_at = min(row_at + row_bytes, last_at);
        }
    };
    uint32_t cell[2][G][4];  // LDS addresses
    float term[2][G][4];
    uint32_t two = 2;
    asm volatile("" : "+v"(two));
    uint32_t top = 0;                                         // both halves: largest index so far
    const uint32_t last = (uint32_t)(S.len - 1) * 0x10001u;  // both halves: largest of the block
    auto prepare = [&](int which, int slot, float c) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
            top = ix[slot][g].largest(top);
            const uint32_t w0 = both_at_most(ix[slot][g].w[0], last);
            const uint32_t w1 = both_at_most(ix[slot][g].w[1], last);
            cell[which][g][0] = cell_address<0>(w0, two);
            cell[which][g][1] = cell_address<1>(w0, two);
            cell[which][g][2] = cell_address<0>(w1, two);
            cell[which][g][3] = cell_address<1>(w1, two);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                term[which][g][e] = c * v[slot][g].value(e);
                // (formed here: left to itself the compiler moves it to where it is used,
                // behind the wait for the reads)
                asm volatile("" : "+v"(term[which][g][e]));
            }
        }
    };
    float x[G][4];
    auto read = [&](int which) {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e) x[g][e] = *(LdsFloat *)(uintptr_t)cell[which][g][e];
    };
    // (lanes that hold the same entry write the same sum)
    auto add_write = [&](int which) {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e) x[g][e] = x[g][e] + term[which][g][e];
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e) *(LdsFloat *)(uintptr_t)cell[which][g][e] = x[g][e];
    };
    aim(0);
#pragma unroll
    for (int u = 0; u < RING; ++u) {
        request(u);
        __builtin_amdgcn_sched_barrier(0);
    }
    // Rounds of RING rows without a branch: whether an index lay outside the block is asked once,
    // at the end (a branch to another way of taking a row joins this one again, and there the
    // compiler waits for the whole ring).
    int r0 = 0;
    for (; r0 + RING <= m_rows; r0 += RING) {
        const ConstantFloat *cr = (const ConstantFloat *)(uintptr_t)(coef + r0);
        aim(r0 + RING);
        __builtin_amdgcn_sched_barrier(0);
        prepare(0, 0, cr[0]);
#pragma unroll
        for (int u = 0; u < RING; ++u) {
            read(u & 1);
            __builtin_amdgcn_sched_barrier(0);
            if (u + 1 < RING) prepare((u + 1) & 1, u + 1, cr[u + 1]);
            // (the row's slot is free: its next request goes out behind the reads too)
            request(u);
            __builtin_amdgcn_sched_barrier(0);
            add_write(u & 1);
        }
    }
    // the window's last rows, fewer than the ring holds
    const ConstantFloat *cr = (const ConstantFloat *)(uintptr_t)(coef + r0);
#pragma unroll
    for (int u0 = 0; u0 < RING; u0 += kStep) {
        if (r0 + u0 + kStep <= m_rows) {
            prepare(0, u0, cr[u0]);
#pragma unroll
            for (int u = 0; u < kStep; ++u) {
                read(u & 1);
                __builtin_amdgcn_sched_barrier(0);
                if (u + 1 < kStep) prepare((u + 1) & 1, u0 + u + 1, cr[u0 + u + 1]);
                __builtin_amdgcn_sched_barrier(0);
                add_write(u & 1);
            }
        } else {
#pragma unroll
            for (int u = 0; u < kStep - 1; ++u) {
                if (r0 + u0 + u < m_rows) {
                    prepare(0, u0 + u, cr[u0 + u]);
                    read(0);
                    add_write(0);
                }
            }
        }
    }
    const bool stray = (top & 0xffffu) >= (uint32_t)S.len || (top >> 16) >= (uint32_t)S.len;
    if (__builtin_amdgcn_ballot_w64(stray) != 0) {
        // an index outside the block, which contributes nothing: all over again, entry by entry
        for (int i = lane; i < S.len; i += 64) acc[i] = 0.0f;
        for (int r = 0; r < m_rows; ++r) {
            const int64_t first = (int64_t)r * k + S.col0;
            for (int j = lane; j < S.kb; j += 64) {
                const int i = I[first + j];
                const float t = coef[r] * widen(V[first + j]);
                if ((unsigned)i < (unsigned)S.len) acc[i] = acc[i] + t;
            }
        }
    }
}

// The same for rows of one to three entries: a lane holds one of them, the lanes behind the last
// one hold it too and write the same sum.  A last block of at most 300 coordinates has such rows
// at 1 %; it must not take longer than the others (one dependent trip to memory per row: 706 us
// for 1249 blocks that took 362 so).
template <typename TV, int RING>
__device__ __forceinline__ void combine_short_rows(float *acc, const BlockSpan &S, int64_t k,
                                                   int m_rows, const float *coef,
                                                   const int16_t *I, const TV *V, int lane) {
    const int16_t *Ij = I + S.col0 + min(lane, S.kb - 1);
    const TV *Vj = V + S.col0 + min(lane, S.kb - 1);
    int16_t ix[RING];
    TV v[RING];
    auto request = [&](int slot, int row) {
        const int64_t at = (int64_t)(row < m_rows ? row : m_rows - 1) * k;
        ix[slot] = Ij[at];
        v[slot] = Vj[at];
    };
#pragma unroll
    for (int u = 0; u < RING; ++u) {
        ix[u] = 0;
        v[u] = (TV)0;
    }
    float next_coef = 0.0f;
    for (int r0 = -RING; r0 < m_rows; r0 += RING) {
        const float cs = next_coef;
        next_coef = coef[r0 + RING + lane < m_rows ? r0 + RING + lane : m_rows - 1];
#pragma unroll
        for (int u = 0; u < RING; ++u) {
            if (r0 >= 0 && r0 + u < m_rows) {
                const float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cs), u));
                const float term = c * widen(v[u]);
                if ((unsigned)(int)ix[u] < (unsigned)S.len) acc[ix[u]] = acc[ix[u]] + term;
            }
            request(u, r0 + RING + u);
        }
    }
}

// G == 0: rows of any length, all threads, a barrier behind every row
template <typename TO, typename TV, int G, int WG, bool LONG>
__global__ __launch_bounds__(WG) void sparse_combine_kernel(int64_t d, int dbs, int kbs,
                                                             int64_t k, int m_rows,
                                                             const float *__restrict__ coef,
                                                             const int16_t *__restrict__ I,
                                                             const TV *__restrict__ V,
                                                             TO *__restrict__ out) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    constexpr int kRing = WG == 64 ? kRingRows / 2 : kRingRows;
    float *acc = (float *)lds_raw;
    const BlockSpan S = block_span(d, dbs, kbs, k, xcd_item((int)gridDim.x));
    const int tid = threadIdx.x;
    for (int i = tid; i < S.len / 4; i += WG)
        ((float4 *)acc)[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (tid < (S.len & 3)) acc[(S.len & ~3) + tid] = 0.0f;
    __syncthreads();

    // (expected: with the short rows' code in front of it this path runs 2 % slower)
    if (G > 0 && __builtin_expect(S.kb >= 4, 1)) {
        if (tid < 64)
            combine_rows<TV, (G > 0 ? G : 1), kRing / (G > 0 ? G : 1), LONG>(acc, S, k, m_rows,
                                                                            coef, I, V, tid);
        __syncthreads();
    } else if (G > 0) {
        if (tid < 64) combine_short_rows<TV, kShortRing>(acc, S, k, m_rows, coef, I, V, tid);
        __syncthreads();
    } else {
        for (int r = 0; r < m_rows; ++r) {
            const float c = coef[r];
            const int64_t at = (int64_t)r * k + S.col0;
            for (int j = tid; j < S.kb; j += WG) {
                const int ix = I[at + j];
                const float term = c * widen(V[at + j]);
                if ((unsigned)ix < (unsigned)S.len) acc[ix] = acc[ix] + term;
            }
            __syncthreads();
        }
    }

    TO *dst = out + S.e0;
    int done = 0;
    if ((((uintptr_t)dst) & 15) == 0) {
        constexpr int kPer = 16 / sizeof(TO);
        const int n = S.len / kPer;
#pragma unroll 4
        for (int i = tid; i < n; i += WG) add_sixteen_bytes(dst + i * kPer, acc + i * kPer);
        done = n * kPer;
    }
    for (int i = done + tid; i < S.len; i += WG) narrow(dst + i, widen(dst[i]) + acc[i]);
}

// ---- copy_values with typed window values ---------------------------------------------------
template <typename TD, typename TV>
__global__ __launch_bounds__(kWG) void copy_values_typed_kernel(int64_t k, int64_t dbs,
                                                                int64_t kbs, const int16_t *idx,
                                                                const void *inp, void *out,
                                                                int direction) {
    const int64_t j = (int64_t)blockIdx.x * kWG + threadIdx.x;
    if (j >= k) return;
    const int64_t pos = (j / kbs) * dbs + idx[j];
    if (direction == 1)
        narrow((TV *)out + j, widen(((const TD *)inp)[pos]));
    else
        narrow((TD *)out + pos, widen(((const TV *)inp)[j]));
}

template <typename K>
int allow_lds(K kernel, int bytes) {
    if (bytes <= 64 * 1024) return 0;
    return (int)hipFuncSetAttribute((const void *)kernel,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

int window_check(int64_t d, int64_t m_rows, int64_t k, int64_t dbs, int64_t kbs,
                 int64_t *nblocks) {
    if (d <= 0 || k <= 0 || m_rows < 0 || dbs <= 0 || kbs <= 0 || kbs > dbs) return MA_ERR_ARG;
    if (dbs > MA_MAX_D_BLOCK) return MA_ERR_BLOCK_SIZE;
    if (m_rows > MA_MAX_SPARSE_ROWS) return MA_ERR_WINDOW;
    *nblocks = (k + kbs - 1) / kbs;
    // every block row must start inside the vector
    if ((*nblocks - 1) * dbs >= d || *nblocks >= (int64_t)1 << 31) return MA_ERR_GEOMETRY;
    return 0;
}

bool known(int dtype) { return dtype == MA_F32 || dtype == MA_BF16; }

}  // namespace
}  // namespace ma

using namespace ma;

#define MA_DISPATCH2(A, B, CALL)                                      \
    if ((A) == MA_F32 && (B) == MA_F32) { CALL(float, float) }        \
    else if ((A) == MA_F32) { CALL(float, uint16_t) }                 \
    else if ((B) == MA_F32) { CALL(uint16_t, float) }                 \
    else { CALL(uint16_t, uint16_t) }

extern "C" {

int ma_sparse_scalar_products_workspace(int64_t d, int64_t m_rows, int64_t k,
                                        int64_t d_block_size, int64_t k_block_size,
                                        int64_t *bytes) {
    int64_t nblocks = 0;
    if (!bytes) return MA_ERR_ARG;
    const int rc = window_check(d, m_rows, k, d_block_size, k_block_size, &nblocks);
    if (rc) return rc;
    *bytes = nblocks * m_rows * (int64_t)sizeof(float);
    return 0;
}

int ma_sparse_scalar_products(int64_t d, int64_t m_rows, int64_t k, int64_t d_block_size,
                              int64_t k_block_size, const void *g, int g_dtype,
                              const int16_t *indices, const void *values, int values_dtype,
                              float *out, void *workspace, int64_t workspace_bytes,
                              void *stream) {
    int64_t nblocks = 0;
    if (!g || !indices || !values || !out || !known(g_dtype) || !known(values_dtype))
        return MA_ERR_ARG;
    int rc = window_check(d, m_rows, k, d_block_size, k_block_size, &nblocks);
    if (rc) return rc;
    if (m_rows == 0) return 0;
    if (!workspace || ((uintptr_t)workspace & 3) ||
        workspace_bytes < nblocks * m_rows * (int64_t)sizeof(float))
        return MA_ERR_ARG;
    const int esize = g_dtype == MA_F32 ? 4 : 2;
    const int lds = (int)((d_block_size * esize + 15) & ~(int64_t)15);
    if (lds > kLdsBytes) return MA_ERR_LDS;
    hipStream_t s = (hipStream_t)stream;
    float *partial = (float *)workspace;
    // enough workgroups to fill the CUs several times over, at least 64 rows each
    int64_t gy = (4096 + nblocks - 1) / nblocks, gy_max = m_rows / 64;
    gy = gy > gy_max ? gy_max : gy;
    gy = gy < 1 ? 1 : gy;
    // (arrays of two-byte elements that do not begin on four bytes: entry by entry)
    const int groups =
        (((uintptr_t)indices | (uintptr_t)values) & 3) == 0 ? dot_groups(k_block_size) : 0;
#define CALL_G(TG, TV, G)                                                                       \
    if ((rc = allow_lds(sparse_dot_kernel<TG, TV, G>, lds))) return rc;                         \
    rc = launch_kernel(sparse_dot_kernel<TG, TV, G>, dim3((unsigned)(nblocks * gy)), kWG, lds,  \
                       s, d, (int)d_block_size, (int)k_block_size, k, (int)m_rows,              \
                       (int)nblocks, (int)gy, (const TG *)g, indices, (const TV *)values,       \
                       partial);
#define CALL(TG, TV)                                                                            \
    if (groups == 1) { CALL_G(TG, TV, 1) }                                                      \
    else if (groups == 2) { CALL_G(TG, TV, 2) }                                                 \
    else { CALL_G(TG, TV, 0) }
    MA_DISPATCH2(g_dtype, values_dtype, CALL)
#undef CALL
#undef CALL_G
    if (rc) return rc;
    const unsigned rgrid = (unsigned)((m_rows + kReduceRows - 1) / kReduceRows);
    return launch_kernel(sparse_dot_reduce_kernel, dim3(rgrid), kWG, 0, s, partial, nblocks,
                         (int)m_rows, out);
}

int ma_sparse_linear_combination(int64_t d, int64_t m_rows, int64_t k, int64_t d_block_size,
                                 int64_t k_block_size, const float *coef,
                                 const int16_t *indices, const void *values, int values_dtype,
                                 void *out, int out_dtype, void *stream) {
    int64_t nblocks = 0;
    if (!coef || !indices || !values || !out || !known(out_dtype) || !known(values_dtype))
        return MA_ERR_ARG;
    int rc = window_check(d, m_rows, k, d_block_size, k_block_size, &nblocks);
    if (rc) return rc;
    if (m_rows == 0) return 0;
    const int lds = (int)(d_block_size * 4);
    if (lds > kLdsBytes) return MA_ERR_LDS;
    hipStream_t s = (hipStream_t)stream;
    // Rows of up to 512 entries per block: one wave applies them, against four waves (eight above
    // 256 entries) and a barrier per row: 1248 blocks of 20480, 1024 rows of 205 bf16: 332 us, 598;
    // 512 rows of 410: 318, 381; of 512: 317, 395.  Longer rows give a barrier more to do.
    // Rows of more than 2^25 entries do not fit a round's 32-bit offsets; addressed row by row
    // the 1024 rows of 205 take 387 us.  Small blocks, of which the LDS would hold more than two,
    // are short of waves: one to a workgroup, with half the rows under way (blocks of 512, 256
    // rows of 5: 591 us; with three idle waves beside it, 833; four waves and barriers, 769).
    const int groups = quad_groups(k_block_size) <= 2 ? quad_groups(k_block_size) : 0;
    const bool is_long = k > (1 << 25), small = d_block_size <= kSmallBlock;
    const int threads = groups == 0 ? kWG : small && !is_long ? 64 : kCombineThreads;
#define CALL_G(TO, TV, ...)                                                                     \
    if ((rc = allow_lds(sparse_combine_kernel<TO, TV, __VA_ARGS__>, lds))) return rc;           \
    rc = launch_kernel(sparse_combine_kernel<TO, TV, __VA_ARGS__>, dim3((unsigned)nblocks),     \
                       threads, lds, s, d, (int)d_block_size, (int)k_block_size, k,             \
                       (int)m_rows, coef, indices, (const TV *)values, (TO *)out);
#define CALL(TO, TV)                                                                            \
    if (groups == 0) { CALL_G(TO, TV, 0, kWG, false) }                                          \
    else if (is_long && groups == 1) { CALL_G(TO, TV, 1, kCombineThreads, true) }               \
    else if (is_long) { CALL_G(TO, TV, 2, kCombineThreads, true) }                              \
    else if (small && groups == 1) { CALL_G(TO, TV, 1, 64, false) }                             \
    else if (small) { CALL_G(TO, TV, 2, 64, false) }                                            \
    else if (groups == 1) { CALL_G(TO, TV, 1, kCombineThreads, false) }                         \
    else { CALL_G(TO, TV, 2, kCombineThreads, false) }
    MA_DISPATCH2(out_dtype, values_dtype, CALL)
#undef CALL
#undef CALL_G
    return rc;
}

int ma_copy_values_typed(int64_t d, int64_t k, int64_t d_block_size, int64_t k_block_size,
                         const int16_t *indices, const void *inp, void *out, int direction,
                         int dtype, int values_dtype, void *stream) {
    if (!indices || !inp || !out || d <= 0 || k < 0 || d_block_size <= 0 || k_block_size <= 0)
        return MA_ERR_ARG;
    if ((direction != 0 && direction != 1) || !known(dtype) || !known(values_dtype))
        return MA_ERR_ARG;
    if (d_block_size > MA_MAX_D_BLOCK) return MA_ERR_BLOCK_SIZE;
    if (k > 0 && ((k + k_block_size - 1) / k_block_size - 1) * d_block_size >= d)
        return MA_ERR_GEOMETRY;
    if (k == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const unsigned grid = (unsigned)((k + kWG - 1) / kWG);
#define CALL(TD, TV)                                                                   \
    rc = launch_kernel(copy_values_typed_kernel<TD, TV>, dim3(grid), kWG, 0, s, k,     \
                       d_block_size, k_block_size, indices, inp, out, direction);
    int rc = 0;
    MA_DISPATCH2(dtype, values_dtype, CALL)
#undef CALL
    return rc;
}

}  // extern "C"
