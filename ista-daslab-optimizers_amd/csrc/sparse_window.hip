// Sparse M-FAC's kernels over the window of MicroAdam's layout (m rows of k block-relative int16
// indices and k values, k_block_size entries per top-k block of d_block_size coordinates):
//   scalar products of the rows with a dense vector
//     (ista_daslab_cuda_sparse_mfac.SP, sparse_mfac/sparse_core_mfac_w_ef.py:185-203),
//   linear combination of the rows into a dense vector
//     (ista_daslab_cuda_sparse_mfac.LCG, sparse_core_mfac_w_ef.py:205-221),
//   copy_values with fp32 window values (sparse_core_mfac_w_ef.py:105-124, use_bf16 = False).
// One 512-thread workgroup per top-k block: the block of the dense vector lives in LDS, the
// window entries of the block stream past it once.  Part of libmicroadam_hip.so.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/microadam_hip.h"
#include "ma_device.hpp"

namespace ma {
namespace {

constexpr int kLdsBytes = 160 * 1024;
constexpr int kRingRows = 32;          // rows the linear combination requests ahead
constexpr int kCombineThreads = 256;  // of a workgroup in which one wave applies the rows
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

__device__ __forceinline__ BlockSpan block_span(int64_t d, int dbs, int kbs, int64_t k) {
    BlockSpan s;
    const int64_t b = blockIdx.x;
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
// partial[b][r] = sum over the entries of row r in block b of V * g; a wave per row, the lanes'
// sums folded by a butterfly.  The second kernel adds the blocks' partial sums in a fixed order.
template <typename TG, typename TV>
__global__ __launch_bounds__(kWG) void sparse_dot_kernel(int64_t d, int dbs, int kbs, int64_t k,
                                                         int m_rows, const TG *g,
                                                         const int16_t *I, const TV *V,
                                                         float *partial) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const BlockSpan S = block_span(d, dbs, kbs, k);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    TG *gl = (TG *)lds_raw;

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

    // the workgroups of one block (gridDim.y of them) share its rows; a wave takes two rows at
    // a time so that both rows' entries are in flight together
    constexpr int kWaves = kWG / 64;
    const int per = (m_rows + (int)gridDim.y - 1) / (int)gridDim.y;
    const int row_lo = (int)blockIdx.y * per;
    const int row_hi = row_lo + per < m_rows ? row_lo + per : m_rows;
    for (int r = row_lo + wave; r < row_hi; r += 2 * kWaves) {
        const int r2 = r + kWaves;
        const bool two = r2 < row_hi;
        const int64_t atA = (int64_t)r * k + S.col0, atB = (int64_t)(two ? r2 : r) * k + S.col0;
        float accA = 0.0f, accB = 0.0f;
        for (int j0 = 0; j0 < S.kb; j0 += 64 * kDotUnroll) {
            int ixA[kDotUnroll], ixB[kDotUnroll];
            TV vA[kDotUnroll], vB[kDotUnroll];
#pragma unroll
            for (int u = 0; u < kDotUnroll; ++u) {
                const int j = j0 + u * 64 + lane;
                ixA[u] = ixB[u] = -1;
                vA[u] = vB[u] = (TV)0;
                if (j < S.kb) {
                    ixA[u] = I[atA + j];
                    vA[u] = V[atA + j];
                    if (two) {
                        ixB[u] = I[atB + j];
                        vB[u] = V[atB + j];
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < kDotUnroll; ++u) {
                if ((unsigned)ixA[u] < (unsigned)S.len) accA += widen(vA[u]) * widen(gl[ixA[u]]);
                if ((unsigned)ixB[u] < (unsigned)S.len) accB += widen(vB[u]) * widen(gl[ixB[u]]);
            }
        }
#pragma unroll
        for (int s = 32; s > 0; s >>= 1) {
            accA += __shfl_xor(accA, s, 64);
            accB += __shfl_xor(accB, s, 64);
        }
        // straight to the workspace: LDS holds the block of g and nothing else, so that four
        // workgroups with a 20480-element bf16 block share a CU
        if (lane == 0) {
            float *dst = partial + (int64_t)blockIdx.x * m_rows;
            dst[r] = accA;
            if (two) dst[r2] = accB;
        }
    }
}

// out[r] += sum over blocks of partial[b][r]: a wave per row, lane l adds blocks l, l + 64, ...
// in increasing order, then the butterfly
__global__ __launch_bounds__(kWG) void sparse_dot_reduce_kernel(const float *partial,
                                                                int64_t nblocks, int m_rows,
                                                                float *out) {
    const int lane = threadIdx.x & 63;
    const int r = blockIdx.x * (kWG / 64) + (threadIdx.x >> 6);
    if (r >= m_rows) return;
    float acc = 0.0f;
    for (int64_t b = lane; b < nblocks; b += 64) acc += partial[b * m_rows + r];
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) acc += __shfl_xor(acc, s, 64);
    if (lane == 0) out[r] = out[r] + acc;
}

// ---- linear combination ---------------------------------------------------------------------
// acc[c] (fp32, LDS) takes the terms coef[r] * V[r][j] of the block's coordinates row by row in
// increasing r; the entries of one row name distinct coordinates, so a row is applied without
// atomics.  The accumulators fill the LDS (two 20480-element blocks per CU), so what bounds the
// kernel is the chain of rows.  ONE wave applies all rows of a block: the LDS operations of a wave
// execute in program order, so a row needs no barrier behind it, only its own reads; the next
// row's addresses and terms are formed while those are under way.  The window comes in through a
// ring of registers, four entries a request.
typedef __attribute__((address_space(3))) float LdsFloat;

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

template <typename TV, int G, int RING>
__device__ __forceinline__ void combine_rows(float *acc, const BlockSpan &S, int64_t k, int m_rows,
                                             const float *coef, const int16_t *I, const TV *V,
                                             int lane) {
    static_assert(RING <= 64, "a lane holds one coefficient of the ring");
    constexpr int kStep = 4;  // rows whose indices are checked together
    constexpr uint32_t kWide = sizeof(TV) / 2;
    // byte offset in a row of the indices of this lane's entries
    uint32_t start[G];
#pragma unroll
    for (int g = 0; g < G; ++g) start[g] = 2u * (uint32_t)quad_start(S.kb, lane + g * 64);
    IndexQuad ix[RING][G];
    ValueQuad<TV> v[RING][G];
    // Requests are made in row order and at every round alike (the last row again and again
    // behind the window's end), so that at any time the same number of them is under way and
    // the compiler can wait for the oldest ones alone.  Rows of a round are addressed from its
    // first one in 32 bits (the host checks that RING rows fit).
    const uint32_t row_bytes = (uint32_t)k * 2u;
    const int16_t *Ir = I + S.col0;
    const TV *Vr = V + S.col0;
    uint32_t row_at = 0, last_at = 0;
    auto aim = [&](int first) {  // the next RING requests are for the rows from `first` on
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
        row_at = min(row_at + row_bytes, last_at);
    };
    uint32_t cell[2][G][4];  // LDS addresses
    float term[2][G][4];
    uint32_t two = 2;
    asm volatile("" : "+v"(two));
    auto prepare = [&](int which, int slot, float c) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
            cell[which][g][0] = cell_address<0>(ix[slot][g].w[0], two);
            cell[which][g][1] = cell_address<1>(ix[slot][g].w[0], two);
            cell[which][g][2] = cell_address<0>(ix[slot][g].w[1], two);
            cell[which][g][3] = cell_address<1>(ix[slot][g].w[1], two);
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
    // (the first round only requests: a request is made at one place of the code, in one order,
    // whatever the round)
#pragma unroll
    for (int u = 0; u < RING; ++u)
#pragma unroll
        for (int g = 0; g < G; ++g) {
            ix[u][g] = IndexQuad{};
            v[u][g] = ValueQuad<TV>{};
        }
    float next_coef = 0.0f;
    for (int r0 = -RING; r0 < m_rows; r0 += RING) {
        const float cs = next_coef;
        next_coef = coef[r0 + RING + lane < m_rows ? r0 + RING + lane : m_rows - 1];
        aim(r0 + RING);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s0 = 0; s0 < RING; s0 += kStep) {
            const int row = r0 + s0;
            uint32_t top = 0;
#pragma unroll
            for (int u = 0; u < kStep; ++u)
#pragma unroll
                for (int g = 0; g < G; ++g) top = ix[s0 + u][g].largest(top);
            const bool stray =
                (top & 0xffffu) >= (uint32_t)S.len || (top >> 16) >= (uint32_t)S.len;
            const bool in_block = __builtin_amdgcn_ballot_w64(stray) == 0;
            auto coef_of = [&](int u) {
                return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cs), s0 + u));
            };
            if (r0 >= 0 && in_block && row + kStep <= m_rows) {
                prepare(0, s0, coef_of(0));
#pragma unroll
                for (int u = 0; u < kStep; ++u) {
                    read(u & 1);
                    __builtin_amdgcn_sched_barrier(0);
                    if (u + 1 < kStep) prepare((u + 1) & 1, s0 + u + 1, coef_of(u + 1));
                    __builtin_amdgcn_sched_barrier(0);
                    add_write(u & 1);
                }
            } else if (r0 >= 0 && in_block) {  // the window's last rows
#pragma unroll
                for (int u = 0; u < kStep - 1; ++u) {
                    if (row + u < m_rows) {
                        prepare(0, s0 + u, coef_of(u));
                        read(0);
                        add_write(0);
                    }
                }
            } else if (r0 >= 0) {
                // an index outside the block, which is skipped: these rows entry by entry
                for (int r = row; r < row + kStep && r < m_rows; ++r) {
                    const int64_t first = (int64_t)r * k + S.col0;
                    for (int j = lane; j < S.kb; j += 64) {
                        const int i = I[first + j];
                        const float t = coef[r] * widen(V[first + j]);
                        if ((unsigned)i < (unsigned)S.len) acc[i] = acc[i] + t;
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < kStep; ++u) {
                request(s0 + u);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
}

// G == 0: rows of any length, all threads, a barrier behind every row
template <typename TO, typename TV, int G, int WG>
__global__ __launch_bounds__(WG) void sparse_combine_kernel(int64_t d, int dbs, int kbs,
                                                             int64_t k, int m_rows,
                                                             const float *__restrict__ coef,
                                                             const int16_t *__restrict__ I,
                                                             const TV *__restrict__ V,
                                                             TO *__restrict__ out) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    float *acc = (float *)lds_raw;
    const BlockSpan S = block_span(d, dbs, kbs, k);
    const int tid = threadIdx.x;
    for (int i = tid; i < S.len / 4; i += WG)
        ((float4 *)acc)[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (tid < (S.len & 3)) acc[(S.len & ~3) + tid] = 0.0f;
    __syncthreads();

    if (G > 0 && S.kb >= 4) {
        if (tid < 64)
            combine_rows<TV, (G > 0 ? G : 1), kRingRows / (G > 0 ? G : 1)>(acc, S, k, m_rows, coef,
                                                                          I, V, tid);
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
#define CALL(TG, TV)                                                                            \
    if ((rc = allow_lds(sparse_dot_kernel<TG, TV>, lds))) return rc;                            \
    rc = launch_kernel(sparse_dot_kernel<TG, TV>, dim3((unsigned)nblocks, (unsigned)gy), kWG,   \
                       lds, s, d, (int)d_block_size, (int)k_block_size, k, (int)m_rows,         \
                       (const TG *)g, indices, (const TV *)values, partial);
    MA_DISPATCH2(g_dtype, values_dtype, CALL)
#undef CALL
    if (rc) return rc;
    const unsigned rgrid = (unsigned)((m_rows + kWG / 64 - 1) / (kWG / 64));
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
    // Rows of up to 512 entries per block: one wave applies them.  1248 blocks of 20480, 1024 rows
    // of 205 bf16: 360 us against 590 with four waves and a barrier per row.  Longer rows give a
    // barrier more to do, and a row of more than 2^25 entries does not fit the wave's offsets.
    const int groups = k <= (1 << 25) ? quad_groups(k_block_size) : 0;
#define CALL_G(TO, TV, G, WG)                                                                   \
    if ((rc = allow_lds(sparse_combine_kernel<TO, TV, G, WG>, lds))) return rc;                 \
    rc = launch_kernel(sparse_combine_kernel<TO, TV, G, WG>, dim3((unsigned)nblocks), WG, lds,  \
                       s, d, (int)d_block_size, (int)k_block_size, k, (int)m_rows, coef,        \
                       indices, (const TV *)values, (TO *)out);
#define CALL(TO, TV)                                                                            \
    if (groups == 1) { CALL_G(TO, TV, 1, kCombineThreads) }                                     \
    else if (groups == 2) { CALL_G(TO, TV, 2, kCombineThreads) }                                \
    else { CALL_G(TO, TV, 0, kWG) }
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
