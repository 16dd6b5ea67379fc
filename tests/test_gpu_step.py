"""GPU parity of the whole optimizer step, through the MicroAdam class, against the oracle.

Both routes of the class (the fused kernel and the op-by-op sequence) must reproduce the
oracle's state bit for bit: window indices and values, 4-bit error-feedback codes, bf16
min/max statistics, and here also the parameters themselves (the kernels use the same
unfused fp32 arithmetic as the oracle, so the stated 1e-3 / 1e-5 tolerance is met with
zero difference; the tolerance check is kept as the documented bar).
"""
import functools

import numpy as np
import pytest
import torch

from gpu_util import assert_state_equal, to_np

pytestmark = pytest.mark.gpu

REL_TOL = {torch.bfloat16: 1e-3, torch.float32: 1e-5}


def _run(oracle, sizes, dtype, m, q, k_init, alpha, wd, DB, steps, use_fused, grad_scale=1e-2,
         zero_step=None, lr=1e-3, seed=0, expect_route=None):
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(seed)
    cpu_params = [(torch.randn(n, generator=gen) * 0.02).to(dtype) for n in sizes]
    oparams = [to_np(p) for p in cpu_params]
    oref = oracle.OracleMicroAdam(oparams, m, lr, q, k_init, alpha, weight_decay=wd, d_block_size=DB)
    gparams = [torch.nn.Parameter(p.clone().cuda()) for p in cpu_params]
    opt = MicroAdam(gparams, m=m, lr=lr, quant_block_size=q, k_init=k_init, alpha=alpha,
                    weight_decay=wd)
    opt.d_block_size = DB
    opt.use_fused = use_fused
    for s in range(steps):
        grads = [(torch.randn(n, generator=gen) * grad_scale).to(dtype) for n in sizes]
        if zero_step is not None and s == zero_step:
            grads[0].zero_()
        for p, g in zip(gparams, grads):
            p.grad = g.clone().cuda()
        opt.step()
        oref.step([to_np(g) for g in grads])
        for i, p in enumerate(gparams):
            ctx = f"step {s + 1} tensor {i} (d={sizes[i]})"
            assert_state_equal(opt.state[p], oref.state[i], ctx)
            if alpha == -2:  # st['quant_err'] = a - Qinv(e_new), rewritten by every step
                assert np.array_equal(to_np(opt.state[p]["quant_err"]).reshape(-1),
                                      oref.state[i]["quant_err"]), f"{ctx}: quant_err"
            got, want = to_np(p.data), oparams[i]
            if not np.array_equal(got, want):
                gf = oracle.bf16_to_f32(got) if got.dtype == np.uint16 else got
                wf = oracle.bf16_to_f32(want) if want.dtype == np.uint16 else want
                rel = np.abs(gf - wf).max() / max(np.abs(wf).max(), 1e-30)
                raise AssertionError(f"{ctx}: parameters differ at {(got != want).sum()} entries, "
                                     f"max rel {rel:.3e} (bar {REL_TOL[dtype]})")
    if expect_route is not None:
        fused_now = [opt._fusable(p, opt.state[p]) and use_fused for p in gparams
                     if p.grad is not None]
        assert all(fused_now) == expect_route, fused_now
    return opt


CASES = [
    # sizes, dtype, m, q, k_init, alpha, wd, DB, steps
    ([3000, 257, 64, 1024], torch.bfloat16, 4, 64, 0.01, 0.0, 0.0, 1024, 9),
    ([5000], torch.float32, 3, 64, 0.02, 0.0, 0.0, 2048, 7),
    ([2500, 130], torch.bfloat16, 5, 32, 0.05, 0.0, 0.1, 512, 8),
    ([20480 * 2 + 4096, 768, 4096], torch.bfloat16, 10, 64, 0.01, 0.0, 0.0, 20480, 12),
    ([20480 + 4096], torch.float32, 10, 64, 0.01, 0.0, 0.01, 20480, 12),
    ([32768 + 1000], torch.bfloat16, 3, 128, 0.01, 0.0, 0.0, 32768, 5),
    ([10240 * 2 + 8], torch.bfloat16, 3, 8, 0.01, 0.0, 0.0, 10240, 5),
    ([1001, 777], torch.bfloat16, 3, 64, 0.03, 0.0, 0.0, 20480, 5),   # odd d: partial chunks
    # windows too large for the one-pass stage (20 rows of 5 %): the step in two launches, the
    # rows' chunk cuts cached; with weight decay and a tensor of exactly one block; more rows;
    # fp32 data (the general selection, fp32 parameters in the window kernel)
    ([20480 * 2 + 8192], torch.bfloat16, 20, 32, 0.05, 0.0, 0.0, 20480, 23),
    ([20480 * 2 + 4096, 20480], torch.bfloat16, 20, 64, 0.05, 0.0, 0.01, 20480, 22),
    ([20480 + 8192], torch.bfloat16, 24, 32, 0.05, 0.0, 0.0, 20480, 26),
    ([20480 * 2 + 8192], torch.float32, 20, 32, 0.05, 0.0, 0.0, 20480, 22),
    # more rows than the one-pass stage takes, but short block rows (1 %): two launches, without a
    # cache of chunk cuts (rows out of order: test_window_kernel_over_rows_out_of_order)
    ([20480 * 2 + 8192, 4096], torch.bfloat16, 18, 64, 0.01, 0.0, 0.0, 20480, 21),
    # a fifth of every block selected: a row has about 100 entries per 512 coordinates, more
    # than the window kernel's 64 lanes take in one go
    ([20480 * 2 + 4096], torch.bfloat16, 4, 64, 0.2, 0.0, 0.0, 20480, 7),
    # quantisation blocks longer than the 512 elements a wave holds per chunk
    ([20480 * 2 + 4096, 3000, 12288], torch.bfloat16, 4, 1024, 0.01, 0.0, 0.0, 20480, 6),
    ([20480 + 5000], torch.bfloat16, 10, 4096, 0.01, 0.0, 0.01, 20480, 12),
    ([20480 + 2048 + 77, 4096], torch.float32, 3, 2048, 0.01, 0.0, 0.0, 20480, 5),
    ([32768 + 9000], torch.bfloat16, 3, 4096, 0.01, 0.0, 0.0, 32768, 5),
    # more tensors of one size class than one launch takes (160): two launches
    ([96 + 8 * (i % 5) for i in range(190)] + [3000], torch.bfloat16, 3, 8, 0.05, 0.0, 0.0, 1024, 4),
]


@pytest.mark.parametrize("use_fused", [True, False], ids=["fused", "opbyop"])
@pytest.mark.parametrize("sizes,dtype,m,q,k_init,alpha,wd,DB,steps", CASES)
def test_step_matches_oracle(oracle, sizes, dtype, m, q, k_init, alpha, wd, DB, steps, use_fused):
    _run(oracle, sizes, dtype, m, q, k_init, alpha, wd, DB, steps, use_fused, zero_step=2,
         expect_route=use_fused)


GENERAL_CASES = [
    # alpha > 0 or d < q with odd quantisation blocks: only the op-by-op route applies
    ([4100, 33], torch.bfloat16, 3, 1000, 0.01, 0.5, 0.0, 1024, 7),
    ([999], torch.float32, 2, 100, 0.03, 0.25, 0.01, 400, 5),
    ([20480 * 3 + 77], torch.bfloat16, 4, 100001, 0.01, 0.5, 0.0, 20480, 6),
    ([50, 20], torch.bfloat16, 3, 60, 0.1, 0.0, 0.0, 20480, 4),
    # alpha == -2 with quantisation blocks that the one-pass kernels do not take
    ([4100, 33], torch.bfloat16, 3, 1000, 0.01, -2, 0.0, 1024, 5),
]


@pytest.mark.parametrize("sizes,dtype,m,q,k_init,alpha,wd,DB,steps", GENERAL_CASES)
def test_step_general_route(oracle, sizes, dtype, m, q, k_init, alpha, wd, DB, steps):
    _run(oracle, sizes, dtype, m, q, k_init, alpha, wd, DB, steps, True, expect_route=False)


QUANT_ERR_CASES = [
    # alpha == -2: the quantisation error goes straight into the parameters
    # (micro_adam.py:238-273), inside the one-pass kernels
    ([20480 + 4096, 300], torch.bfloat16, 4, 64, 0.01, -2, 0.0, 20480, 6),
    ([3000], torch.float32, 3, 64, 0.02, -2, 0.05, 1024, 5),
    ([20480 * 3, 1001], torch.bfloat16, 10, 64, 0.01, -2, 0.01, 20480, 12),
    ([20480 * 2 + 8192], torch.bfloat16, 20, 32, 0.05, -2, 0.0, 20480, 22),
    ([20480 + 77], torch.float32, 5, 32, 0.01, -2, 0.0, 20480, 7),
    ([20480 * 2 + 1000], torch.bfloat16, 4, 2048, 0.01, -2, 0.0, 20480, 6),
]


@pytest.mark.parametrize("use_fused", [True, False], ids=["fused", "opbyop"])
@pytest.mark.parametrize("sizes,dtype,m,q,k_init,alpha,wd,DB,steps", QUANT_ERR_CASES)
def test_step_quant_err_route(oracle, sizes, dtype, m, q, k_init, alpha, wd, DB, steps, use_fused):
    opt = _run(oracle, sizes, dtype, m, q, k_init, alpha, wd, DB, steps, use_fused, zero_step=2,
               expect_route=use_fused)
    # micro_adam.py:67-68; _run has compared it with the oracle's after every step
    assert all(st["quant_err"].any() for st in opt.state.values())


SPANNING_CASES = [
    # quantisation blocks at least as long as the top-k blocks: spanning route
    ([20480 * 5 + 77], torch.bfloat16, 10, 100000, 0.01, 0.5, 0.0, 20480, 12),
    ([20480 * 12 + 4096, 4096, 1000], torch.bfloat16, 4, 24576, 0.01, 0.3, 0.01, 20480, 8),
    ([5000, 3000], torch.float32, 3, 2048, 0.02, 0.25, 0.0, 1024, 6),
    ([40000], torch.bfloat16, 3, 20480, 0.01, 0.9, 0.0, 20480, 5),
    ([512 * 9 + 100], torch.bfloat16, 3, 520, 0.02, 0.5, 0.0, 512, 6),
    # alpha == 0 with long quantisation blocks (the reference's documented quant_block_size)
    ([20480 * 5 + 77, 4096], torch.bfloat16, 10, 100000, 0.01, 0.0, 0.0, 20480, 12),
    ([5000, 3000], torch.float32, 3, 2048, 0.02, 0.0, 0.01, 1024, 6),
    ([50, 20], torch.bfloat16, 3, 64, 0.1, 0.0, 0.0, 20480, 4),       # d < q: the fused route
]


@pytest.mark.parametrize("use_fused", [True, False], ids=["spanning", "opbyop"])
@pytest.mark.parametrize("sizes,dtype,m,q,k_init,alpha,wd,DB,steps", SPANNING_CASES)
def test_step_spanning_route(oracle, sizes, dtype, m, q, k_init, alpha, wd, DB, steps, use_fused):
    _run(oracle, sizes, dtype, m, q, k_init, alpha, wd, DB, steps, use_fused, zero_step=2,
         expect_route=use_fused)


SEGMENTED_CASES = [
    # quantisation blocks shorter than the top-k blocks that do not divide them: edges at every
    # place of a wave's 512-element stretch (q = 520), more than forty of them (q = 512 with a top-k
    # block that it does not divide), powers of two above 4096, one element of the last block in
    # a quantisation block of its own, tensors shorter than one and tensors of one top-k block
    ([20480 * 2 + 4096, 768, 10000, 20480], torch.bfloat16, 10, 10000, 0.01, 0.0, 0.0, 20480, 12),
    ([20480 * 3 + 1, 1001], torch.bfloat16, 4, 1000, 0.01, 0.0, 0.01, 20480, 7),
    ([20480 * 2 + 77, 20480 + 20000], torch.float32, 4, 16384, 0.01, 0.0, 0.01, 20480, 6),
    ([20480 * 3 + 4096], torch.bfloat16, 4, 8192, 0.02, 0.0, 0.0, 20480, 6),
    ([20480 * 4], torch.bfloat16, 4, 520, 0.01, 0.0, 0.0, 20480, 6),
    ([20480 * 2 + 9], torch.float32, 3, 20472, 0.01, 0.0, 0.0, 20480, 5),
    ([1032 * 5 + 3, 700, 24], torch.bfloat16, 3, 1000, 0.03, 0.0, 0.0, 1032, 7),
    ([4096 * 3 + 11], torch.float32, 3, 520, 0.02, 0.0, 0.0, 4096, 6),
    ([12288 * 2 + 8], torch.bfloat16, 3, 5000, 0.01, 0.0, 0.0, 12288, 5),
    ([32768 * 2 + 520], torch.bfloat16, 3, 520, 0.01, 0.0, 0.0, 32768, 5),
    ([20480 + 8192], torch.bfloat16, 20, 10000, 0.05, 0.0, 0.0, 20480, 22),
    # powers of two up to 4096 that do not divide the top-k block
    ([10240 * 2 + 4104, 10240 * 3], torch.bfloat16, 3, 4096, 0.01, 0.0, 0.0, 10240, 5),
    ([1032 * 4 + 3], torch.float32, 3, 512, 0.02, 0.0, 0.0, 1032, 5),
]


@pytest.mark.parametrize("spin", [None, "0"], ids=["exchange", "deferred"])
@pytest.mark.parametrize("sizes,dtype,m,q,k_init,alpha,wd,DB,steps", SEGMENTED_CASES)
def test_step_segmented_route(oracle, monkeypatch, sizes, dtype, m, q, k_init, alpha, wd, DB, steps,
                              spin):
    """spin "0": no block waits for its neighbours, every block that has one takes the sweep."""
    if spin is not None:
        monkeypatch.setenv("MA_SPAN_SPIN_LIMIT", spin)
    opt = _run(oracle, sizes, dtype, m, q, k_init, alpha, wd, DB, steps, True, zero_step=2)
    for p in opt.param_groups[0]["params"]:
        assert opt._fusable(p, opt.state[p]) == 5


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_segmented_route_takes_what_the_op_by_op_route_takes(value):
    """Infinite and undefined gradients, more of them than a top-k block selects: the same state
    and parameters as the op-by-op sequence leaves, bit for bit."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(3)
    d = 20480 * 2 + 4096
    start = (torch.randn(d, generator=gen) * 0.02).to(torch.bfloat16)
    g = (torch.randn(d, generator=gen) * 0.01).to(torch.bfloat16)
    g[25000:25300] = value
    states = []
    for fused in (True, False):
        p = torch.nn.Parameter(start.clone().cuda())
        opt = MicroAdam([p], m=3, lr=1e-3, quant_block_size=10000)
        opt.use_fused = fused
        for _ in range(2):
            p.grad = g.clone().cuda()
            opt.step()
        st = opt.state[p]
        states.append([to_np(p.data)] + [to_np(st[key]) for key in ("error", "min_vals", "max_vals")])
    for got, want in zip(*states):
        assert np.array_equal(got, want)


FUSED_DENSIFIED_CASES = [
    # 0 < alpha < 1 with quantisation blocks inside the top-k blocks: one pass
    ([20480 * 2 + 4096, 768, 4096], torch.bfloat16, 10, 64, 0.01, 0.5, 0.0, 20480, 12),
    ([3000, 257, 64, 1024], torch.bfloat16, 4, 64, 0.01, 0.25, 0.1, 1024, 9),
    ([5000], torch.float32, 3, 64, 0.02, 0.7, 0.0, 2048, 7),
    ([20480 + 4096], torch.float32, 10, 32, 0.01, 0.1, 0.01, 20480, 12),
    ([1001, 777], torch.bfloat16, 3, 64, 0.03, 0.5, 0.0, 20480, 5),   # odd d: partial chunks
    # quantisation blocks longer than the 512 elements a wave holds per chunk
    ([20480 * 2 + 4096, 3000], torch.bfloat16, 3, 1024, 0.01, 0.5, 0.0, 20480, 4),
    ([20480 + 5000], torch.float32, 4, 4096, 0.01, 0.3, 0.01, 20480, 6),
    ([32768 + 9000], torch.bfloat16, 3, 2048, 0.01, 0.7, 0.0, 32768, 5),
]


@pytest.mark.parametrize("use_fused", [True, False], ids=["fused", "opbyop"])
@pytest.mark.parametrize("sizes,dtype,m,q,k_init,alpha,wd,DB,steps", FUSED_DENSIFIED_CASES)
def test_step_fused_densified_route(oracle, sizes, dtype, m, q, k_init, alpha, wd, DB, steps,
                                    use_fused):
    _run(oracle, sizes, dtype, m, q, k_init, alpha, wd, DB, steps, use_fused, zero_step=2,
         expect_route=use_fused)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("q,DB", [(16, 4096), (32, 20480), (64, 20480), (128, 20480), (1024, 20480)])
def test_densified_second_quantisation(oracle, q, DB, dtype):
    """Codes of (1 - alpha) * Qinv(code) where a code maps to itself and where it does not:
    quantisation blocks around zero, blocks at 3, 30 and 300 times their range from zero (the
    rounding of the kept share then moves codes) and blocks of zeros, side by side in a wave."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(23)
    d = DB + 5 * q + 24
    offset = torch.tensor([0.0, 0.03, 0.3, 3.0, 0.0])[torch.arange(d) // q % 5]
    params = [(torch.randn(d, generator=gen) * 0.02).to(dtype)]
    oparams = [to_np(params[0])]
    oref = oracle.OracleMicroAdam(oparams, 3, 1e-3, q, 0.01, 0.3, d_block_size=DB)
    gp = torch.nn.Parameter(params[0].clone().cuda())
    opt = MicroAdam([gp], m=3, lr=1e-3, quant_block_size=q, k_init=0.01, alpha=0.3)
    opt.d_block_size = DB
    for step in range(3):
        g = offset + torch.randn(d, generator=gen) * 0.003
        g[torch.arange(d) // q % 5 == 4] = 0.0
        gp.grad = g.to(dtype).cuda()
        opt.step()
        assert opt._fusable(gp, opt.state[gp]) == 3
        oref.step([to_np(g.to(dtype))])
        assert_state_equal(opt.state[gp], oref.state[0], f"step {step + 1}")
        assert np.array_equal(to_np(gp.data), oparams[0]), f"step {step + 1}: parameters"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("q", [32, 64, 128, 512, 1024])
def test_densified_second_quantisation_of_a_short_block(oracle, q, dtype):
    """A tensor's last quantisation block with 1 to q - 1 of its q elements, at 30 times its range
    from zero, where the second quantisation moves some of the 16 codes: which of them the block's
    few elements have must not matter.  The blocks in front of it lie around zero, where every code
    maps to itself, and hold the largest elements, so that the top-k leaves the short one alone."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(q)
    tails = sorted({1, 7, 8, 16, 24, q // 2, q - 8, q - 1}) * 6
    sizes = [(20480 if i % 2 else 0) + 2 * q + t for i, t in enumerate(tails)]
    params = [(torch.randn(n, generator=gen) * 0.02).to(dtype) for n in sizes]
    oparams = [to_np(p) for p in params]
    oref = oracle.OracleMicroAdam(oparams, 3, 1e-3, q, 0.01, 0.3, d_block_size=20480)
    gparams = [torch.nn.Parameter(p.clone().cuda()) for p in params]
    opt = MicroAdam(gparams, m=3, lr=1e-3, quant_block_size=q, k_init=0.01, alpha=0.3)
    for step in range(3):
        grads = []
        for n, t in zip(sizes, tails):
            g = torch.randn(n, generator=gen) * 0.3
            g[n - t:] = 0.1 + torch.randn(t, generator=gen) * 0.003
            grads.append(g.to(dtype))
        for p, g in zip(gparams, grads):
            p.grad = g.clone().cuda()
        opt.step()
        oref.step([to_np(g) for g in grads])
        for i, p in enumerate(gparams):
            assert opt._fusable(p, opt.state[p]) == 3
            assert_state_equal(opt.state[p], oref.state[i], f"step {step + 1} tail {tails[i]}")
            assert np.array_equal(to_np(p.data), oparams[i]), (step, tails[i])


@pytest.mark.parametrize("use_fused", [True, False], ids=["fused", "opbyop"])
@pytest.mark.parametrize("scale", [1e-36, 3e-38, 1e-39])
def test_denormal_scale_gradients(oracle, scale, use_fused):
    """Gradients so small that quantisation steps and window values are fp32 / bf16 denormals:
    no flush to zero anywhere, and codes stay inside [0, 15] when the step (max - min) / 15
    is rounded coarsely."""
    _run(oracle, [20480 + 4096], torch.bfloat16, 3, 64, 0.01, 0.0, 0.0, 20480, 5, use_fused,
         grad_scale=scale)


@pytest.mark.parametrize("use_fused", [True, False], ids=["fused", "opbyop"])
def test_config1_plumbing(oracle, use_fused):
    """The plumbing configuration: one flat fp32 parameter, d = 1,048,576, N(0,1) gradients,
    m=10, k=1 %, q=64, hardware block size; run on to 100 steps (the configuration asks for 20;
    the fp32 tolerance is stated after 100), state and parameters compared after every step."""
    opt = _run(oracle, [1048576], torch.float32, 10, 64, 0.01, 0.0, 0.0, 20480, 100, use_fused,
               grad_scale=1.0, expect_route=use_fused)
    assert opt.d_block_size == 20480 and opt.steps == 100


def test_outlier_gradients(oracle):
    """Heavy-tailed gradients with outlier rows (the stress configuration's recipe, small)."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(3)
    rows, cols = 64, 2048
    p0 = (torch.randn(rows * cols, generator=gen) * 0.02).to(torch.bfloat16)
    hot = torch.rand(rows, generator=gen) < 0.05
    oparams = [to_np(p0)]
    oref = oracle.OracleMicroAdam(oparams, 20, 1e-3, 32, 0.05, 0, d_block_size=20480)
    gp = torch.nn.Parameter(p0.clone().cuda())
    opt = MicroAdam([gp], m=20, lr=1e-3, quant_block_size=32, k_init=0.05)
    dist = torch.distributions.StudentT(3.0)
    for s in range(6):
        torch.manual_seed(100 + s)
        g = dist.sample((rows, cols)) * 1e-3
        g[hot] *= 100
        g = g.to(torch.bfloat16).view(-1)
        gp.grad = g.clone().cuda()
        opt.step()
        oref.step([to_np(g)])
        assert_state_equal(opt.state[gp], oref.state[0], f"step {s + 1}")
        assert np.array_equal(to_np(gp.data), oparams[0])


def test_lr_schedule_none_grads_and_closure(oracle):
    """group['lr'] is re-read every step, parameters without a gradient are skipped, and the
    closure's loss is returned (micro_adam.py:102-105, 121, 125-126)."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(5)
    sizes = [4096, 2048]
    cpu = [(torch.randn(n, generator=gen) * 0.02).to(torch.bfloat16) for n in sizes]
    oparams = [to_np(p) for p in cpu]
    oref = oracle.OracleMicroAdam(oparams, 4, 1e-3, 64, 0.01, 0, d_block_size=20480)
    gparams = [torch.nn.Parameter(p.clone().cuda()) for p in cpu]
    opt = MicroAdam(gparams, m=4, lr=1e-3, quant_block_size=64)
    for s in range(6):
        lr = 1e-3 * (s + 1)
        opt.param_groups[0]["lr"] = lr
        grads = [(torch.randn(n, generator=gen) * 1e-2).to(torch.bfloat16) for n in sizes]
        if s % 2:
            grads[1] = None
        for p, g in zip(gparams, grads):
            p.grad = None if g is None else g.clone().cuda()
        loss = opt.step(closure=lambda: torch.tensor(1.5 + s))
        assert float(loss) == 1.5 + s
        oref.step([None if g is None else to_np(g) for g in grads], lr=lr)
        for i, p in enumerate(gparams):
            if oref.state[i] is not None:
                assert_state_equal(opt.state[p], oref.state[i], f"step {s + 1} tensor {i}")
            assert np.array_equal(to_np(p.data), oparams[i])


def test_logging_with_mixed_types_and_missing_gradients(oracle):
    """One list holding bf16 and fp32 tensors of all block classes, and on some logging steps a
    tensor without a gradient: the step is then several library calls (one per route and element
    type), whose kernels add their shares to the same six sums (micro_adam.py:121, 125-136,
    328, 330)."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(21)
    spec = [(20480 * 2 + 300, torch.bfloat16), (768, torch.bfloat16), (20480 + 8, torch.float32),
            (3000, torch.float32), (10000, torch.bfloat16)]
    cpu = [(torch.randn(n, generator=gen) * 0.02).to(dt) for n, dt in spec]
    oparams = [to_np(p) for p in cpu]
    oref = oracle.OracleMicroAdam(oparams, 4, 1e-3, 64, 0.01, 0, weight_decay=0.01)
    gparams = [torch.nn.Parameter(p.clone().cuda()) for p in cpu]
    opt = MicroAdam(gparams, m=4, lr=1e-3, quant_block_size=64, weight_decay=0.01)
    opt.log_interval = 2
    opt._logging_active = lambda: True
    logged = []
    opt._log = lambda *a: logged.append([float(x) for x in a[:6]])
    calls = []
    inner = opt._fused_step
    opt._fused_step = lambda route, dtype, entries, sums=None: (
        calls.append((opt.steps, dtype, len(entries), sums is not None)),
        inner(route, dtype, entries, sums))
    wanted = []
    for s in range(6):
        grads = [(torch.randn(n, generator=gen) * 1e-2).to(dt) for n, dt in spec]
        if s in (1, 4):
            grads[2] = None     # step 2 is a logging step, step 5 is not
        for p, g in zip(gparams, grads):
            p.grad = None if g is None else g.clone().cuda()
        opt.step()
        out = oref.step([None if g is None else to_np(g) for g in grads], metrics=(s + 1) % 2 == 0)
        if out is not None:
            wanted.append(out)
        for i, p in enumerate(gparams):
            if oref.state[i] is not None:
                assert_state_equal(opt.state[p], oref.state[i], f"step {s + 1} tensor {i}")
            assert np.array_equal(to_np(p.data), oparams[i]), f"step {s + 1} tensor {i}"
    # two calls per step (bf16, fp32), with sums exactly on the logging steps
    assert [c for c in calls if c[0] == 2] == [(2, torch.bfloat16, 3, True), (2, torch.float32, 1, True)]
    assert [c for c in calls if c[0] == 3] == [(3, torch.bfloat16, 3, False), (3, torch.float32, 2, False)]
    assert len(logged) == 3 == len(wanted)
    keys = ("norm_qe", "norm_g", "norm_u", "norm_e", "sparsity_u", "sparsity_qe")
    for got, want in zip(logged, wanted):
        for key, value in zip(keys, got):
            if key.startswith("sparsity"):
                assert value == want[key], (key, value, want[key])
            else:
                assert value == pytest.approx(want[key], rel=1e-5, abs=0), (key, value, want[key])


def test_state_layout_and_checkpoint_roundtrip():
    """State keys, dtypes and shapes as micro_adam.py:61-94; state_dict round trip, including
    the re-typing load_state_dict applies to floating-point state."""
    from ista_daslab_optimizers import MicroAdam
    torch.manual_seed(0)
    p = torch.nn.Parameter(torch.randn(20480 + 4096, device="cuda") * 0.02)
    opt = MicroAdam([p], m=10, lr=1e-3, quant_block_size=64)
    for _ in range(3):
        p.grad = torch.randn_like(p) * 1e-2
        opt.step()
    st = opt.state[p]
    assert st["I"].dtype == torch.int16 and st["I"].shape == (10, 205 + 41)
    assert st["V"].dtype == torch.bfloat16 and st["V"].shape == (10, 246)
    assert st["error"].dtype == torch.uint8 and st["error"].numel() == (20480 + 4096) // 2
    assert st["min_vals"].dtype == torch.bfloat16 and st["min_vals"].numel() == 384 + 1
    assert (st["index"], st["k"], st["d_block_size"], st["k_block_size_many"],
            st["k_block_size_few"], st["d_index_topk"]) == (3, 246, 20480, 205, 41, 20480)
    sd = opt.state_dict()
    p2 = torch.nn.Parameter(p.detach().clone())
    opt2 = MicroAdam([p2], m=10, lr=1e-3, quant_block_size=64)
    opt2.load_state_dict(sd)
    assert opt2.steps == opt.steps  # the reference loses the counter on resume (micro_adam.py:35)
    g = torch.randn_like(p) * 1e-2
    p.grad, p2.grad = g.clone(), g.clone()
    opt.step()
    opt2.step()
    assert opt2.state[p2]["V"].dtype == torch.bfloat16
    assert torch.equal(p.data, p2.data)
    for key in ("I", "V", "error", "min_vals", "max_vals"):
        assert torch.equal(opt.state[p][key], opt2.state[p2][key]), key
    # a framework that re-types the state (every tensor cast to the parameter's dtype) is
    # repaired on the next step, as the reference does for st['I']
    st2 = opt2.state[p2]
    for key in ("I", "V", "error", "min_vals", "max_vals"):
        st2[key] = st2[key].to(torch.float32)
    p.grad, p2.grad = g.clone(), g.clone()
    opt.step()
    opt2.step()
    assert st2["I"].dtype == torch.int16 and st2["error"].dtype == torch.uint8
    assert torch.equal(p.data, p2.data)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
def test_checkpoint_through_a_file(oracle, tmp_path, dtype):
    """torch.save -> torch.load(weights_only=True) -> load_state_dict into a fresh optimizer,
    mid-run and after the ring has wrapped: the resumed run continues bit for bit like the
    uninterrupted one and like the oracle (which never stopped), on the fused route."""
    from ista_daslab_optimizers import MicroAdam
    sizes, m = [20480 * 2 + 4096, 768], 4
    gen = torch.Generator().manual_seed(5)
    cpu_params = [(torch.randn(n, generator=gen) * 0.02).to(dtype) for n in sizes]
    oparams = [to_np(p) for p in cpu_params]
    oref = oracle.OracleMicroAdam(oparams, m, 1e-3, 64, 0.01, 0, weight_decay=0.01)
    params = [torch.nn.Parameter(p.clone().cuda()) for p in cpu_params]
    opt = MicroAdam(params, m=m, lr=1e-3, quant_block_size=64, weight_decay=0.01)
    for s in range(11):
        if s in (2, 7):  # before and after the window is full
            path = tmp_path / f"ckpt{s}.pt"
            torch.save({"opt": opt.state_dict(), "params": [p.data for p in params]}, path)
            del opt, params
            blob = torch.load(path, map_location="cuda", weights_only=True)
            params = [torch.nn.Parameter(t.clone()) for t in blob["params"]]
            opt = MicroAdam(params, m=m, lr=1e-3, quant_block_size=64, weight_decay=0.01)
            opt.load_state_dict(blob["opt"])
            assert opt.steps == s
            for p in params:
                st = opt.state[p]
                assert st["I"].dtype == torch.int16 and st["error"].dtype == torch.uint8
                assert st["V"].dtype == st["min_vals"].dtype == torch.bfloat16
                assert st["index"] == s % m
        grads = [(torch.randn(n, generator=gen) * 1e-2).to(dtype) for n in sizes]
        for p, g in zip(params, grads):
            p.grad = g.clone().cuda()
        opt.step()
        assert all(opt._fusable(p, opt.state[p]) == 1 for p in params)
        oref.step([to_np(g) for g in grads])
        for i, p in enumerate(params):
            assert_state_equal(opt.state[p], oref.state[i], f"step {s + 1} tensor {i}")
            assert np.array_equal(to_np(p.data), oparams[i]), f"step {s + 1} tensor {i}"


def test_checkpoint_made_for_another_block_size(oracle):
    """State whose geometry was derived from another device's top-k block size (the reference
    sizes d_block_size from the shared memory of the GPU it runs on, micro_adam.py:43-44): the
    fused kernels would derive a different geometry from this optimizer's own, so such tensors
    take the op-by-op route, which reads the stored geometry, and still match an oracle that
    runs with the checkpoint's block size."""
    from ista_daslab_optimizers import MicroAdam
    n, m, foreign = 20480 * 2 + 4096, 4, 12288
    gen = torch.Generator().manual_seed(6)
    p0 = (torch.randn(n, generator=gen) * 0.02).to(torch.bfloat16)
    oparams = [to_np(p0)]
    oref = oracle.OracleMicroAdam(oparams, m, 1e-3, 64, 0.01, 0, d_block_size=foreign)
    p = torch.nn.Parameter(p0.clone().cuda())
    src = MicroAdam([p], m=m, lr=1e-3, quant_block_size=64)
    src.d_block_size = foreign
    grads = [(torch.randn(n, generator=gen) * 1e-2).to(torch.bfloat16) for _ in range(6)]
    for g in grads[:3]:
        p.grad = g.clone().cuda()
        src.step()
        oref.step([to_np(g)])
    assert src.state[p]["d_block_size"] == foreign
    p2 = torch.nn.Parameter(p.detach().clone())
    dst = MicroAdam([p2], m=m, lr=1e-3, quant_block_size=64)   # d_block_size 20480
    dst.load_state_dict(src.state_dict())
    for s, g in enumerate(grads[3:]):
        p2.grad = g.clone().cuda()
        dst.step()
        assert dst._fusable(p2, dst.state[p2]) == 0
        oref.step([to_np(g)])
        assert_state_equal(dst.state[p2], oref.state[0], f"resumed step {s + 1}")
        assert np.array_equal(to_np(p2.data), oparams[0]), f"resumed step {s + 1}"


def test_cpu_parameter_is_rejected():
    from ista_daslab_optimizers import MicroAdam
    p = torch.nn.Parameter(torch.zeros(100))
    opt = MicroAdam([p], m=3, lr=1e-3, quant_block_size=64)
    p.grad = torch.ones(100)
    with pytest.raises(RuntimeError):
        opt.step()


def test_unaligned_views_take_the_general_route(oracle):
    """Parameters and gradients that are views at an odd element offset (not 16-byte aligned)
    cannot use the vector paths of the fused kernels; the step must still match."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(11)
    n, m, q = 5000, 3, 64
    p0 = (torch.randn(n, generator=gen) * 0.02).to(torch.bfloat16)
    oparams = [to_np(p0)]
    oref = oracle.OracleMicroAdam(oparams, m, 1e-3, q, 0.02, 0, d_block_size=2048)
    pbuf = torch.zeros(n + 8, dtype=torch.bfloat16, device="cuda")
    pbuf[3:3 + n] = p0.cuda()
    gp = torch.nn.Parameter(pbuf[3:3 + n])
    assert gp.data_ptr() % 16 != 0
    opt = MicroAdam([gp], m=m, lr=1e-3, quant_block_size=q, k_init=0.02)
    opt.d_block_size = 2048
    for s in range(5):
        g = (torch.randn(n, generator=gen) * 1e-2).to(torch.bfloat16)
        gbuf = torch.zeros(n + 8, dtype=torch.bfloat16, device="cuda")
        gbuf[1:1 + n] = g.cuda()
        gp.grad = gbuf[1:1 + n]
        opt.step()
        oref.step([to_np(g)])
        assert opt._fusable(gp, opt.state[gp]) == 0
        assert_state_equal(opt.state[gp], oref.state[0], f"step {s + 1}")
        assert np.array_equal(to_np(gp.data), oparams[0])


@pytest.mark.parametrize("use_fused", [True, False], ids=["fused", "opbyop"])
def test_window_rows_that_name_the_same_coordinates(oracle, use_fused):
    """Gradients with the same dominant coordinates in every step: every window row names the
    same coordinates, so almost all window entries share their coordinate with other rows
    (the reserve path of the one-pass window stage, where the short list overflows)."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(21)
    n, m = 20480 * 2 + 4096, 10
    p0 = (torch.randn(n, generator=gen) * 0.02).to(torch.bfloat16)
    spikes = torch.randperm(n, generator=gen)[: n // 100]
    oparams = [to_np(p0)]
    oref = oracle.OracleMicroAdam(oparams, m, 1e-3, 64, 0.01, 0, d_block_size=20480)
    gp = torch.nn.Parameter(p0.clone().cuda())
    opt = MicroAdam([gp], m=m, lr=1e-3, quant_block_size=64, k_init=0.01)
    opt.use_fused = use_fused
    for s in range(13):
        g = torch.randn(n, generator=gen) * 1e-3
        g[spikes] += torch.sign(torch.randn(spikes.numel(), generator=gen)) * (1.0 + 0.01 * s)
        g = g.to(torch.bfloat16)
        gp.grad = g.clone().cuda()
        opt.step()
        oref.step([to_np(g)])
        assert_state_equal(opt.state[gp], oref.state[0], f"step {s + 1}")
        assert np.array_equal(to_np(gp.data), oparams[0]), f"step {s + 1}"
    # the window really is that repetitive: the rows of a block name nearly the same coordinates
    I = opt.state[gp]["I"][:, :205].long()
    common = sum(len(set(I[0].tolist()) & set(I[r].tolist())) for r in range(1, m)) / (205 * (m - 1))
    assert common > 0.8, common


LOGGING_CASES = [
    # sizes, dtype, m, q, alpha, wd, route
    ([20480 * 2 + 4096, 768, 1001], torch.bfloat16, 4, 64, 0.0, 0.01, "fused"),
    ([20480 + 300], torch.float32, 3, 32, 0.0, 0.0, "fused"),
    ([20480 * 2 + 4096, 768], torch.bfloat16, 4, 64, 0.5, 0.0, "densified"),
    ([5000], torch.float32, 3, 64, 0.25, 0.01, "densified"),
    ([20480 * 3 + 100], torch.bfloat16, 4, 24576, 0.0, 0.01, "spanning"),
    ([20480 * 5 + 77, 4096], torch.bfloat16, 4, 100000, 0.3, 0.0, "spanning"),
    ([20480 * 2 + 4096, 300], torch.bfloat16, 4, 64, -2, 0.01, "quant_err"),
    ([20480 + 77], torch.float32, 3, 32, -2, 0.0, "quant_err"),
    ([20480 * 2 + 8192], torch.bfloat16, 20, 32, 0.0, 0.0, "fused"),   # 5 %: no coordinate cells
    ([20480 * 2 + 3000], torch.bfloat16, 4, 2048, 0.0, 0.01, "fused"),  # long quantisation blocks
]


@pytest.mark.parametrize("use_fused", [True, False], ids=["fused", "opbyop"])
@pytest.mark.parametrize("sizes,dtype,m,q,alpha,wd,route", LOGGING_CASES)
def test_logged_sums_match_oracle(oracle, sizes, dtype, m, q, alpha, wd, route, use_fused):
    """Logging steps (micro_adam.py:155-156, :271-272, :306-308, :320-324, :330-350): the six
    sums handed to _log against the oracle's, which adds the same values in float64.  The
    fused routes form them inside their kernels, in fp32 per block (at most 40 terms per thread,
    then 512 threads pairwise) and in double across blocks: relative error far below the 1e-5
    asked here.  The op-by-op route takes torch's norm of the buffer, whose result has the
    buffer's type (as in the reference): bf16 results, squared and added in bf16, 3e-2.  The zero counts are exact on both, and the step's
    state is the oracle's on logging steps as on any other."""
    from ista_daslab_optimizers import MicroAdam
    k_init = 0.05 if m == 20 else 0.01
    gen = torch.Generator().manual_seed(11)
    cpu_params = [(torch.randn(n, generator=gen) * 0.02).to(dtype) for n in sizes]
    oparams = [to_np(p) for p in cpu_params]
    oref = oracle.OracleMicroAdam(oparams, m, 1e-3, q, k_init, alpha, weight_decay=wd,
                                  d_block_size=20480)
    params = [torch.nn.Parameter(p.clone().cuda()) for p in cpu_params]
    opt = MicroAdam(params, m=m, lr=1e-3, quant_block_size=q, k_init=k_init, alpha=alpha,
                    weight_decay=wd)
    opt.use_fused = use_fused
    opt.log_interval = 2
    opt._logging_active = lambda: True
    logged = []
    opt._log = lambda *a: logged.append([float(x) for x in a[:6]])
    kernel_steps = []
    inner = opt._fused_step
    opt._fused_step = lambda *a, **kw: (kernel_steps.append(opt.steps), inner(*a, **kw))
    wanted = []
    for s in range(6):
        grads = [(torch.randn(n, generator=gen) * 0.01).to(dtype) for n in sizes]
        if s == 3:
            grads[0][: sizes[0] // 2] = 0  # zeros in the gradient: exact zeros may reach u
        for p, g in zip(params, grads):
            p.grad = g.clone().cuda()
        opt.step()
        out = oref.step([to_np(g) for g in grads], metrics=(s + 1) % 2 == 0)
        if out is not None:
            wanted.append(out)
        for i, p in enumerate(params):
            assert_state_equal(opt.state[p], oref.state[i], f"step {s + 1} tensor {i}")
            assert np.array_equal(to_np(p.data), oparams[i]), f"step {s + 1} tensor {i}"
    # every step, logging or not, took the route under test
    assert sorted(set(kernel_steps)) == ([1, 2, 3, 4, 5, 6] if use_fused else [])
    assert len(logged) == 3 == len(wanted)
    rel = 1e-5 if use_fused else (3e-2 if dtype == torch.bfloat16 else 1e-4)
    keys = ("norm_qe", "norm_g", "norm_u", "norm_e", "sparsity_u", "sparsity_qe")
    for got, want in zip(logged, wanted):
        for key, value in zip(keys, got):
            if key.startswith("sparsity"):
                assert value == want[key], (key, value, want[key])
            else:
                assert value == pytest.approx(want[key], rel=rel, abs=0), (key, value, want[key])
        assert want["norm_g"] > 0 and want["norm_u"] > 0 and want["norm_e"] > 0
        assert (want["norm_qe"] > 0) == (alpha == -2)
        if alpha <= 0:
            assert want["sparsity_u"] > 0


@functools.lru_cache(maxsize=None)
def _boundary_gradient(dtype, q):
    """Quantisation blocks of q elements that hold 0, M and the values around the rounding
    boundaries (k + 1/2) M / 15, for M over bf16 significands x all binary exponents."""
    sig = [1.0, 1.0078125, 1.25, 1.5, 1.9921875, 1.328125, 1.7109375]
    if q > 4096:
        sig = [1.0, 1.5, 1.9921875]
    exps = list(range(-126, 127))
    gen = torch.Generator().manual_seed(17)
    per_block = min(15, (q - 6) // 3)       # boundaries one block has room for
    turns = [list(range(i, min(i + per_block, 15))) for i in range(0, 15, per_block)]
    blocks = []
    for e in exps:
        for s_ in sig:
            M = torch.tensor(s_ * 2.0 ** e, dtype=torch.float64).to(dtype)
            u = (M.float() - 0.0) / 15.0
            for ks in turns:
                vals = [torch.zeros((), dtype=dtype)] + [M] * (8 if q >= 64 else 5)
                for k in ks:
                    x = ((k + 0.5) * u.double()).to(dtype)
                    lo = torch.nextafter(x.float(), torch.tensor(0.0)).to(dtype) if dtype == torch.float32 \
                        else (x.view(torch.int16) - 1).view(torch.bfloat16)
                    hi = torch.nextafter(x.float(), torch.tensor(float("inf"))).to(dtype) if dtype == torch.float32 \
                        else (x.view(torch.int16) + 1).view(torch.bfloat16)
                    vals += [lo, x, hi]
                rnd = (torch.rand(q - len(vals), generator=gen).double() * M.double()).to(dtype)
                blk = torch.cat([torch.stack(vals), rnd])
                blocks.append(blk[torch.randperm(q, generator=gen)])
    return torch.cat(blocks)


BOUNDARY_CASES = [
    # DB, q, alpha, use_fused, route the tensor must take (0 op by op, 1 fused, 2 spanning,
    # 3 fused densified)
    (4096, 64, 0.0, True, 1),      # one-chunk kernel, quantisation group size at run time
    (4096, 64, 0.0, False, 0),
    (20480, 64, 0.0, True, 1),     # hardware block, group of 8 lanes compiled in, statistics
    (20480, 32, 0.0, True, 1),     # shared across lanes; group of 4 lanes
    (20480, 2048, 0.0, True, 1),   # quantisation blocks longer than a wave's stretch
    (20480, 1024, 0.0, True, 1),
    (20480, 64, 0.5, True, 3),     # both quantisations of the densified step
    (20480, 2048, 0.5, True, 3),
    (20480, 24576, 0.0, True, 2),  # two-pass route: statistics across top-k blocks
    (20480, 24576, 0.5, True, 2),  # ... and the 2 x 16 table of its second pass
]


@pytest.mark.parametrize("DB,q,alpha,use_fused,route", BOUNDARY_CASES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_quantisation_rounding_boundaries(oracle, dtype, DB, q, alpha, use_fused, route):
    """The 4-bit codes where they are hardest to get right: every quantisation block holds its
    minimum 0, its maximum M, and for the 15 rounding boundaries the value nearest to
    (k + 1/2) u and its two neighbours (u = (M - 0) / 15 as the kernels form it; blocks too short
    for all 15 take them in turns), with M running through bf16 significands and through every
    binary exponent from -126 to 126, so that steps u that are subnormal, tiny, ordinary and huge
    all occur.  The fused kernels divide by a shared reciprocal where the oracle divides; the
    codes must agree bit for bit all the same, in every kernel instance that forms statistics or
    codes in its own way.  A second step with a zero gradient dequantises and requantises them."""
    from ista_daslab_optimizers import MicroAdam
    g0 = _boundary_gradient(dtype, q)
    pad = (-g0.numel()) % DB
    if q <= DB:  # whole top-k blocks, so that the full-block kernel instances run
        g0 = torch.cat([g0, torch.zeros(pad, dtype=dtype)])
    assert torch.isfinite(g0.float()).all()
    d = g0.numel()
    p0 = (torch.randn(d, generator=torch.Generator().manual_seed(18)) * 0.02).to(dtype)
    oparams = [to_np(p0)]
    oref = oracle.OracleMicroAdam(oparams, 4, 1e-3, q, 0.001, alpha, d_block_size=DB)
    gp = torch.nn.Parameter(p0.clone().cuda())
    opt = MicroAdam([gp], m=4, lr=1e-3, quant_block_size=q, k_init=0.001, alpha=alpha)
    opt.d_block_size = DB
    opt.use_fused = use_fused
    for step, g in enumerate([g0, torch.zeros_like(g0), g0]):
        gp.grad = g.clone().cuda()
        opt.step()
        assert (opt._fusable(gp, opt.state[gp]) if use_fused else 0) == route
        oref.step([to_np(g)])
        assert_state_equal(opt.state[gp], oref.state[0], f"step {step + 1}")
        assert np.array_equal(to_np(gp.data), oparams[0]), f"step {step + 1}: parameters"
    codes = oracle.unpack_codes(to_np(opt.state[gp]["error"]), d)
    assert set(np.unique(codes)) == set(range(16))


@pytest.mark.parametrize("kind", ["ties", "jumps", "one_wave", "few"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_selection_from_the_previous_threshold(oracle, dtype, kind):
    """fp32 blocks and partial blocks, whose selection starts from the previous row's threshold:
    magnitudes that tie at the threshold and at every bin edge, thresholds that jump past the
    bins in either direction, all large elements in one wave's stretch (its list overflows), and
    fewer non-zero elements than are selected."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(17)
    sizes = [20480 * 2 + 4096, 12288 + 700, 768, 300, 67, 9]
    params = [(torch.randn(n, generator=gen) * 0.02).to(dtype) for n in sizes]
    oparams = [to_np(p) for p in params]
    oref = oracle.OracleMicroAdam(oparams, 4, 1e-3, 8, 0.01, 0.0, d_block_size=20480)
    gparams = [torch.nn.Parameter(p.clone().cuda()) for p in params]
    opt = MicroAdam(gparams, m=4, lr=1e-3, quant_block_size=8, k_init=0.01)
    for step in range(9):
        grads = []
        for n in sizes:
            g = torch.randn(n, generator=gen) * 0.01
            if kind == "ties":
                g = torch.randint(-4, 5, (n,), generator=gen) * 2.0 ** -8
            elif kind == "jumps":
                g = g * [1.0, 1.0, 3.0, 3.0, 0.3, 1.0, 1000.0, 1000.0, 1.0][step]
            elif kind == "one_wave":
                g[:min(n, 600)] *= 50.0
            else:
                g[torch.rand(n, generator=gen) > 0.005] = 0.0
            grads.append(g.to(dtype))
        for p, g in zip(gparams, grads):
            p.grad = g.clone().cuda()
        opt.step()
        oref.step([to_np(g) for g in grads])
        for i, p in enumerate(gparams):
            assert_state_equal(opt.state[p], oref.state[i], f"step {step + 1} tensor {i}")
            assert np.array_equal(to_np(p.data), oparams[i]), (step, i)


def test_steps_of_one_table_follow_what_changes_between_them(oracle):
    """Once all tensors of a list took one table, the next step refreshes it in whole columns;
    what may change between steps is followed all the same: new gradient tensors, lr and weight
    decay per group, a missing gradient, a gradient that is not 16-byte aligned, a parameter whose
    storage moved, state cast to another type, an op-by-op step in between."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(29)
    sizes = [20480 + 4096, 768, 4096, 1024]
    cpu = [(torch.randn(n, generator=gen) * 0.02).to(torch.bfloat16) for n in sizes]
    oparams = [to_np(p) for p in cpu]
    gparams = [torch.nn.Parameter(p.clone().cuda()) for p in cpu]
    opt = MicroAdam([dict(params=gparams[:2]), dict(params=gparams[2:], weight_decay=0.1)], m=3,
                    lr=1e-3, quant_block_size=64)
    orefs = [oracle.OracleMicroAdam(oparams[:2], 3, 1e-3, 64, 0.01, 0.0, d_block_size=20480),
             oracle.OracleMicroAdam(oparams[2:], 3, 1e-3, 64, 0.01, 0.0, weight_decay=0.1,
                                    d_block_size=20480)]
    for s in range(12):
        grads = [(torch.randn(n, generator=gen) * 1e-2).to(torch.bfloat16) for n in sizes]
        lrs = [1e-3 * (1 + s), 2e-3]
        for group, lr in zip(opt.param_groups, lrs):
            group['lr'] = lr
        if s == 3:
            grads[1] = None
        for i, (p, g) in enumerate(zip(gparams, grads)):
            if g is None:
                p.grad = None
                continue
            p.grad = g.clone().cuda()
            if s == 6 and i == 0:  # an address 2 bytes off
                buf = torch.zeros(sizes[0] + 1, dtype=torch.bfloat16, device="cuda")
                buf[1:] = p.grad
                p.grad = buf[1:]
        if s == 7:
            gparams[3].data = gparams[3].data.clone()
        if s == 8:
            opt.state[gparams[0]]['I'] = opt.state[gparams[0]]['I'].to(torch.int32)
        opt.use_fused = s != 9
        opt.step()
        want = [None if g is None else to_np(g) for g in grads]
        for ref, lo, hi, lr in ((orefs[0], 0, 2, lrs[0]), (orefs[1], 2, 4, lrs[1])):
            ref.step(want[lo:hi], lr=lr)
        for i, p in enumerate(gparams):
            ref = orefs[i // 2].state[i % 2]
            if ref is not None:
                assert_state_equal(opt.state[p], ref, f"step {s + 1} tensor {i}")
            assert np.array_equal(to_np(p.data), oparams[i]), (s, i)
        if s in (2, 4, 11):
            assert opt._uniform is not None


@pytest.mark.parametrize("alpha", [0.0, 0.5])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("q", [50000, 100000, 1 << 20])
def test_spanning_route_takes_short_vectors(oracle, q, dtype, alpha):
    """Tensors of a single top-k block under quantisation blocks more than 62 times as long: all
    the quantisation block covers is that one block (q = 2^20 with single-block tensors only)."""
    sizes = [768, 125, 80, 9, 20480] + ([20480 * 2 + 77] if q < 1 << 20 else [])
    _run(oracle, sizes, dtype, 3, q, 0.01, alpha, 0.01, 20480, 5, True, zero_step=2,
         expect_route=True)


@pytest.mark.parametrize("sizes,dtype,m,k_init", [
    ([20480 * 2 + 8192], torch.bfloat16, 20, 0.03),        # partial block: 246 entries
    ([20480 + 4096, 20480], torch.float32, 20, 0.025),     # 512 entries a block
    ([20480 * 2], torch.bfloat16, 20, 0.01),               # full blocks of 205 entries
])
def test_logging_steps_write_dense_windows_rows_by_coordinate(sizes, dtype, m, k_init):
    """Windows that the ordinary step takes in two launches: the second one counts on block rows
    in coordinate order, those of the logging steps among them."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(41)
    params = [torch.nn.Parameter((torch.randn(n, generator=gen) * 0.02).to(dtype).cuda())
              for n in sizes]
    opt = MicroAdam(params, m=m, lr=1e-3, quant_block_size=32, k_init=k_init)
    opt.log_interval = 2
    opt._logging_active = lambda: True
    opt._log = lambda *a: None
    for step in range(16):
        for p in params:
            p.grad = (torch.randn(p.numel(), generator=gen) * 0.01).to(dtype).cuda()
        opt.step()
        for p in params:
            st = opt.state[p]
            row, many = st["I"][step % m].long().cpu(), st["k_block_size_many"]
            for part in row.split(many):
                assert torch.all(part[1:] > part[:-1]), (step, len(part))


def test_logging_step_of_a_list_on_several_routes(oracle):
    """A tensor whose gradient is not 16-byte aligned goes op by op beside the others: its sums and
    the kernels' are added."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(47)
    sizes = [20480 + 4096, 768]
    cpu = [(torch.randn(n, generator=gen) * 0.02).to(torch.bfloat16) for n in sizes]
    oparams = [to_np(p) for p in cpu]
    oref = oracle.OracleMicroAdam(oparams, 3, 1e-3, 64, 0.01, 0.0, d_block_size=20480)
    params = [torch.nn.Parameter(p.clone().cuda()) for p in cpu]
    opt = MicroAdam(params, m=3, lr=1e-3, quant_block_size=64)
    opt.log_interval = 1
    opt._logging_active = lambda: True
    logged = []
    opt._log = lambda *a: logged.append([float(x) for x in a[:6]])
    for step in range(2):
        grads = [(torch.randn(n, generator=gen) * 0.01).to(torch.bfloat16) for n in sizes]
        buf = torch.zeros(sizes[1] + 1, dtype=torch.bfloat16, device="cuda")
        buf[1:] = grads[1].cuda()
        params[0].grad, params[1].grad = grads[0].cuda(), buf[1:]
        opt.step()
        want = oref.step([to_np(g) for g in grads], metrics=True)
        for key, value in zip(("norm_qe", "norm_g", "norm_u", "norm_e"), logged[step]):
            # (the op-by-op sums are bf16's: 2^-9 a rounding, a few of them)
            assert value == pytest.approx(want[key], rel=3e-2, abs=0), key
        assert logged[step][4:] == [want["sparsity_u"], want["sparsity_qe"]]
        for i, p in enumerate(params):
            assert_state_equal(opt.state[p], oref.state[i], f"step {step + 1} tensor {i}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_logging_steps_of_the_segmented_route(oracle, dtype):
    """Its kernels do not form the logged sums: on a logging step the tensors that the spanning
    route takes go there, only the others op by op, and the state stays the oracle's."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(43)
    sizes = [20480 + 4096, 768, 10000, 33, 12288]
    cpu = [(torch.randn(n, generator=gen) * 0.02).to(dtype) for n in sizes]
    oparams = [to_np(p) for p in cpu]
    oref = oracle.OracleMicroAdam(oparams, 3, 1e-3, 10000, 0.01, 0.0, d_block_size=20480)
    params = [torch.nn.Parameter(p.clone().cuda()) for p in cpu]
    opt = MicroAdam(params, m=3, lr=1e-3, quant_block_size=10000)
    opt.log_interval = 2
    opt._logging_active = lambda: True
    logged, wanted = [], []
    opt._log = lambda *a: logged.append([float(x) for x in a[:6]])
    one_by_one, inner = [], opt.update_step
    opt.update_step = lambda p, *a: (one_by_one.append((opt.steps, p.numel())), inner(p, *a))[1]
    for step in range(5):
        grads = [(torch.randn(n, generator=gen) * 0.01).to(dtype) for n in sizes]
        for p, g in zip(params, grads):
            p.grad = g.clone().cuda()
        opt.step()
        out = oref.step([to_np(g) for g in grads], metrics=step % 2 == 1)
        if out is not None:
            wanted.append(out)
        for i, p in enumerate(params):
            assert opt._fusable(p, opt.state[p]) == 5
            assert_state_equal(opt.state[p], oref.state[i], f"step {step + 1} tensor {i}")
            assert np.array_equal(to_np(p.data), oparams[i]), (step, i)
    assert one_by_one == [(s, n) for s in (2, 4) for n in (24576, 12288)]
    assert len(logged) == 2 == len(wanted)
    rel = 3e-2 if dtype == torch.bfloat16 else 1e-4  # as in test_logged_sums_match_oracle, op by op
    for got, want in zip(logged, wanted):
        for key, value in zip(("norm_qe", "norm_g", "norm_u", "norm_e"), got):
            assert value == pytest.approx(want[key], rel=rel, abs=0), key
        assert got[4:] == [want["sparsity_u"], want["sparsity_qe"]]


@pytest.mark.parametrize("alpha", [0.0, 0.5])
@pytest.mark.parametrize("spin", [None, "0"], ids=["exchange", "deferred"])
def test_spanning_route_above_the_hardware_block(oracle, monkeypatch, spin, alpha):
    """Top-k blocks of more than 20480 elements, which run in kernels of their own."""
    if spin is not None:
        monkeypatch.setenv("MA_SPAN_SPIN_LIMIT", spin)
    _run(oracle, [32768 * 3 + 520, 24576 + 77], torch.bfloat16, 3, 65536, 0.01, alpha, 0.01, 32768, 5,
         True, zero_step=2, expect_route=True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("DB", [4096, 12288, 32768])
@pytest.mark.parametrize("q", [8, 16, 32, 64])
def test_densified_second_quantisation_of_run_time_groups(oracle, q, DB, dtype):
    """The kernels of other block lengths take the quantisation group at run time: one to eight
    lanes, which try several codes each or requantise their elements; blocks around zero and at
    30 times their range from it side by side, the last one short."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(q + DB)
    sizes = [DB + 5 * q + 3, DB - 2 * q + 5, 3 * q + 1]
    params = [(torch.randn(n, generator=gen) * 0.02).to(dtype) for n in sizes]
    oparams = [to_np(p) for p in params]
    oref = oracle.OracleMicroAdam(oparams, 3, 1e-3, q, 0.01, 0.3, d_block_size=DB)
    gparams = [torch.nn.Parameter(p.clone().cuda()) for p in params]
    opt = MicroAdam(gparams, m=3, lr=1e-3, quant_block_size=q, k_init=0.01, alpha=0.3)
    opt.d_block_size = DB
    for step in range(3):
        grads = []
        for n in sizes:
            far = torch.arange(n) // q % 80 >= 40 if n > DB // 2 else torch.arange(n) >= 3 * q
            g = torch.where(far, 0.1 + torch.randn(n, generator=gen) * 0.003,
                            torch.randn(n, generator=gen) * 0.3)
            grads.append(g.to(dtype))
        for p, g in zip(gparams, grads):
            p.grad = g.clone().cuda()
        opt.step()
        oref.step([to_np(g) for g in grads])
        for i, p in enumerate(gparams):
            assert opt._fusable(p, opt.state[p]) == 3
            assert_state_equal(opt.state[p], oref.state[i], f"step {step + 1} tensor {i}")
            assert np.array_equal(to_np(p.data), oparams[i]), (step, i)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("q", [64, 128])
@pytest.mark.parametrize("alpha", [-2, 0.3])
def test_undefined_elements_leave_their_neighbours_alone(dtype, q, alpha):
    """Undefined gradients, more of them than a top-k block selects: state and parameters as the
    op-by-op sequence leaves them, those of the elements packed into the same words included."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(3)
    d = 20480 * 2 + 4096 + 40
    start = (torch.randn(d, generator=gen) * 0.02).to(dtype)
    g = (torch.randn(d, generator=gen) * 0.01).to(dtype)
    g[torch.randperm(d, generator=gen)[:d // 20]] = float("nan")
    states = []
    for fused in (True, False):
        p = torch.nn.Parameter(start.clone().cuda())
        opt = MicroAdam([p], m=3, lr=1e-3, quant_block_size=q, alpha=alpha)
        opt.use_fused = fused
        for _ in range(2):
            p.grad = g.clone().cuda()
            opt.step()
        st = opt.state[p]
        states.append([p.data.float().cpu()] + [st[key].float().cpu() for key in
                      ("error", "min_vals", "max_vals", "quant_err") if key in st])
    for got, want in zip(*states):
        assert np.array_equal(got.numpy(), want.numpy(), equal_nan=True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("q,DB", [(8, 4096), (32, 20480), (64, 20480), (512, 20480)])
def test_densified_second_quantisation_around_its_bound(oracle, q, DB, dtype):
    """Blocks from once to nine times their range from zero: the kernels take the second codes to be
    the first ones where the larger magnitude is below 4.1 times the range (of the rounded
    statistics), and form them element by element beyond."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(q)
    d = DB + 7 * q
    which = torch.arange(d) // q
    far = torch.linspace(1.0, 9.0, int(which.max()) + 1, dtype=torch.float64)[which].float()
    sign = torch.where(which % 3 == 0, -1.0, 1.0)
    width = 2.0 ** (which % 5 - 9).float()
    params = [(torch.randn(d, generator=gen) * 0.02).to(dtype)]
    oparams = [to_np(params[0])]
    oref = oracle.OracleMicroAdam(oparams, 3, 1e-3, q, 0.01, 0.3, d_block_size=DB)
    gp = torch.nn.Parameter(params[0].clone().cuda())
    opt = MicroAdam([gp], m=3, lr=1e-3, quant_block_size=q, k_init=0.01, alpha=0.3)
    opt.d_block_size = DB
    for step in range(2):
        g = (sign * width * (far + torch.rand(d, generator=gen) - 0.5)).to(dtype)
        gp.grad = g.cuda()
        opt.step()
        assert opt._fusable(gp, opt.state[gp]) == 3
        oref.step([to_np(g)])
        assert_state_equal(opt.state[gp], oref.state[0], f"step {step + 1}")
        assert np.array_equal(to_np(gp.data), oparams[0]), f"step {step + 1}: parameters"


@pytest.mark.parametrize("spin", [None, "0"], ids=["exchange", "deferred"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("q,DB", [(24576, 20480), (520, 512), (8192, 4096), (16384, 12288)])
def test_spanning_second_quantisation(oracle, monkeypatch, spin, q, DB, dtype):
    """alpha > 0 with long quantisation blocks: blocks around zero, at 3, 30 and 300 times their
    range from it (where the kept share's codes are not the first ones) and blocks of zeros, tensors
    with an odd last element; exchanged in one pass, and every block deferred to the sweep."""
    from ista_daslab_optimizers import MicroAdam
    if spin is not None:
        monkeypatch.setenv("MA_SPAN_SPIN_LIMIT", spin)
    gen = torch.Generator().manual_seed(q)
    sizes = [6 * q + 77, q // 2 + 1]
    params = [(torch.randn(n, generator=gen) * 0.02).to(dtype) for n in sizes]
    oparams = [to_np(p) for p in params]
    oref = oracle.OracleMicroAdam(oparams, 3, 1e-3, q, 0.01, 0.3, d_block_size=DB)
    gparams = [torch.nn.Parameter(p.clone().cuda()) for p in params]
    opt = MicroAdam(gparams, m=3, lr=1e-3, quant_block_size=q, k_init=0.01, alpha=0.3)
    opt.d_block_size = DB
    for step in range(4):
        grads = []
        for n in sizes:
            kind = (torch.arange(n) // q + step // 2) % 5
            g = torch.tensor([0.0, 0.03, 0.3, 3.0, 0.0])[kind] + torch.randn(n, generator=gen) * 0.003
            g[kind == 4] = 0.0
            grads.append(g.to(dtype))
        for p, g in zip(gparams, grads):
            p.grad = g.clone().cuda()
        opt.step()
        oref.step([to_np(g) for g in grads])
        for i, p in enumerate(gparams):
            assert opt._fusable(p, opt.state[p]) == 2
            assert_state_equal(opt.state[p], oref.state[i], f"step {step + 1} tensor {i}")
            assert np.array_equal(to_np(p.data), oparams[i]), (step, i)


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_spanning_route_takes_what_the_op_by_op_route_takes(dtype, value):
    """alpha > 0: infinite and undefined gradients, more of them than a top-k block selects."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(3)
    d = 20480 * 6 + 4096
    start = (torch.randn(d, generator=gen) * 0.02).to(dtype)
    g = (torch.randn(d, generator=gen) * 0.01).to(dtype)
    g[20480:20480 * 2][torch.randperm(20480, generator=gen)[:1000]] = value
    states = []
    for fused in (True, False):
        p = torch.nn.Parameter(start.clone().cuda())
        opt = MicroAdam([p], m=3, lr=1e-3, quant_block_size=40960, alpha=0.5)
        opt.use_fused = fused
        for _ in range(2):
            p.grad = g.clone().cuda()
            opt.step()
        st = opt.state[p]
        states.append([p.data.float().cpu()] + [st[key].float().cpu() for key in
                      ("error", "min_vals", "max_vals")])
    for got, want in zip(*states):
        assert np.array_equal(got.numpy(), want.numpy(), equal_nan=True)


@pytest.mark.parametrize("change", ["nothing", "gradient missing", "gradient strided",
                                    "gradient unaligned", "parameter replaced", "learning rates",
                                    "no weight decay", "odd kinds of numbers", "state retyped"])
def test_table_refresh_takes_what_the_walk_takes(change):
    """A list that goes through one table, refreshed natively, against the walk over its tensors:
    the same parameters and states whatever one of the steps brings."""
    from ista_daslab_optimizers import MicroAdam
    results = []
    for walked in (False, True):
        gen = torch.Generator().manual_seed(11)
        shapes = [(64, 40), (300,), (128, 96)]
        params = [torch.nn.Parameter((torch.randn(s, generator=gen) * 0.02).bfloat16().cuda())
                  for s in shapes]
        other = torch.nn.Parameter((torch.randn(shapes[1], generator=gen) * 0.02).bfloat16().cuda())
        opt = MicroAdam([{"params": params[:2]}, {"params": params[2:], "lr": 3e-4}], m=3, lr=1e-3,
                        quant_block_size=64, weight_decay=0.01)
        for step in range(5):
            for group in opt.param_groups:
                for p in group["params"]:
                    p.grad = (torch.randn(p.shape, generator=gen) * 0.01).bfloat16().cuda()
            if step == 3:
                p = params[2]
                if change == "gradient missing":
                    p.grad = None
                elif change == "gradient strided":
                    p.grad = p.grad.t().contiguous().t()
                elif change == "gradient unaligned":
                    flat = torch.empty(p.numel() + 1, dtype=p.dtype, device="cuda")
                    p.grad = flat[1:].view(p.shape).copy_(p.grad)
                elif change == "parameter replaced":
                    opt.param_groups[0]["params"][1] = other
                    other.grad = params[1].grad
                elif change == "learning rates":
                    opt.param_groups[0]["lr"], opt.param_groups[1]["lr"] = 5e-3, 0
                elif change == "no weight decay":
                    opt.param_groups[1]["weight_decay"] = 0
                    del opt.param_groups[0]["weight_decay"]
                elif change == "odd kinds of numbers":
                    opt.param_groups[0]["lr"] = np.float64(2e-3)
                    opt.param_groups[1]["lr"] = torch.tensor(2e-3)
                elif change == "state retyped":
                    st = opt.state[params[0]]
                    st["I"] = st["I"].to(torch.bfloat16)
            if walked:
                opt._uniform = None
            if change == "gradient strided" and step == 3:
                with pytest.raises(RuntimeError, match="view size"):  # neither takes it
                    opt.step()
                break
            opt.step()
        results.append([p.data.float().cpu() for p in params + [other]] +
                       [opt.state[p][key].float().cpu() for p in params
                        for key in ("error", "min_vals", "max_vals", "I", "V")] +
                       [opt.state[p]["index"] for p in params])
    for got, want in zip(*results):
        assert torch.equal(got, want) if torch.is_tensor(got) else got == want


LONG_WINDOW_CASES = [
    # windows above 2560 entries a block that the longer one-pass stage takes (bf16, up to 15 rows
    # with two loads of four entries a thread), its last row length that fits and the first that
    # does not; 16 rows, and rows of up to 512 entries, in the two-launch form; fp32
    ([20480 * 2 + 17100, 20480 + 9, 18001, 4096], torch.bfloat16, 15, 64, 0.01, 0.01, 20480, 18),
    ([20480 * 2 + 12000], torch.bfloat16, 10, 32, 0.02, 0.0, 20480, 12),
    ([20480 * 2 + 333], torch.bfloat16, 9, 64, 0.0249, 0.0, 20480, 11),   # 510 entries, 8 * 128 loads
    ([20480 * 2 + 333], torch.bfloat16, 10, 64, 0.022, 0.0, 20480, 12),   # 451 entries, 9 * 113
    ([20480 * 2 + 333], torch.bfloat16, 10, 64, 0.0223, 0.0, 20480, 12),  # 457 entries, 9 * 115
    ([20480 * 2 + 9001, 20479], torch.bfloat16, 16, 64, 0.02, 0.01, 20480, 18),
    ([32768 + 8200], torch.bfloat16, 12, 1024, 0.01, 0.0, 32768, 14),
    ([12288 * 2 + 4096], torch.bfloat16, 15, 128, 0.02, 0.0, 12288, 17),
    ([20480 + 9001], torch.float32, 15, 64, 0.01, 0.01, 20480, 17),
]


@pytest.mark.parametrize("kind", ["normal", "one row", "ties"])
@pytest.mark.parametrize("sizes,dtype,m,q,k_init,wd,DB,steps", LONG_WINDOW_CASES)
def test_longer_windows(oracle, sizes, dtype, m, q, k_init, wd, DB, steps, kind):
    """kind "one row": the first 1200 coordinates of every other block carry the large gradients
    at every step, so that all rows of the window name them (more shared entries than the stage's
    queue holds); "ties": gradients of few magnitudes, zeros among them."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(m)
    cpu = [(torch.randn(n, generator=gen) * 0.02).to(dtype) for n in sizes]
    oparams = [to_np(p) for p in cpu]
    oref = oracle.OracleMicroAdam(oparams, m, 1e-3, q, k_init, 0.0, weight_decay=wd, d_block_size=DB)
    params = [torch.nn.Parameter(p.clone().cuda()) for p in cpu]
    opt = MicroAdam(params, m=m, lr=1e-3, quant_block_size=q, k_init=k_init, weight_decay=wd)
    opt.d_block_size = DB
    for step in range(steps):
        grads = []
        for n in sizes:
            g = torch.randn(n, generator=gen) * 1e-2
            at = torch.arange(n)
            if kind == "one row":
                g[(at % DB < 1200) & (at // DB % 2 == 0)] *= 100
            elif kind == "ties":
                g = torch.round(g * 200) / 200
            grads.append(g.to(dtype))
        for p, g in zip(params, grads):
            p.grad = g.clone().cuda()
        opt.step()
        oref.step([to_np(g) for g in grads])
        for i, p in enumerate(params):
            assert opt._fusable(p, opt.state[p]) == 1
            if step in (0, 1, m - 1, steps - 1):
                assert_state_equal(opt.state[p], oref.state[i], f"step {step + 1} tensor {i}")
            assert np.array_equal(to_np(p.data), oparams[i]), (step, i)


@pytest.mark.parametrize("alpha", [0.0, 0.5, -2])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("q", [8, 64, 128, 1024, 4096])
def test_fused_route_takes_tensors_shorter_than_a_quantisation_block(oracle, q, dtype, alpha):
    """Beside longer ones, in the same launch; from one element to one less than a block."""
    sizes = sorted({1, 2, 7, 9, q // 2 - 1, q // 2, q - 7, q - 1, q} - {0}) + [20480 + q]
    opt = _run(oracle, sizes, dtype, 3, q, 0.01, alpha, 0.01, 20480, 5, True, zero_step=2)
    assert {opt._fusable(p, opt.state[p]) for p in opt.param_groups[0]["params"]} == \
        {{0.0: 1, 0.5: 3, -2: 4}[alpha]}
    assert opt._uniform is not None


@pytest.mark.parametrize("sizes,dtype,m,k_init", [
    ([20480 * 2 + 9001, 768, 300, 4096], torch.bfloat16, 10, 0.03),  # one tensor with cuts, three beside it
    ([20480 + 9001, 768, 300, 4096], torch.float32, 10, 0.03),
    ([20480 * 2 + 9001, 4096], torch.bfloat16, 18, 0.01),            # two launches, short rows: no cuts
    ([20480 + 9001], torch.float32, 18, 0.01),
])
def test_row_cuts_that_no_step_asks_for_are_left_alone(sizes, dtype, m, k_init):
    """Tensors that ma_fused_step takes in two launches although ma_fused_step_row_cuts answers 0 for
    them, because they ride along with a longer one or because their rows are short: a row_cuts pointer
    they come with is neither written nor read, and the step is that without the pointers."""
    import ctypes
    from ista_daslab_optimizers import MicroAdam, _hip
    gen = torch.Generator().manual_seed(m)
    start = [(torch.randn(n, generator=gen) * 0.02).to(dtype) for n in sizes]
    opts, lists = [], []
    for _ in range(2):
        params = [torch.nn.Parameter(p.clone().cuda()) for p in start]
        opts.append(MicroAdam(params, m=m, lr=1e-3, quant_block_size=64, k_init=k_init))
        lists.append(params)
    guards = {}
    for step in range(m + 2):
        grads = [(torch.randn(n, generator=gen) * 1e-2).to(dtype).cuda() for n in sizes]
        for opt, params in zip(opts, lists):
            for p, g in zip(params, grads):
                p.grad = g
            opt.step()
        if step == 0:
            opt, (table,) = opts[0], opts[0]._tables.values()
            for i, e in enumerate(table.entries):
                probe, h = opt._probe(e.p, e.st)
                words = _hip.lib.ma_fused_step_row_cuts(ctypes.byref(probe), ctypes.byref(h))
                assert (words > 0) == (e.cuts is not None) == (m == 10 and i == 0)
                if words == 0:
                    # (longer than the cuts of such a tensor would be: nothing is written past it)
                    blocks = -(-sizes[i] // 20480)
                    guards[i] = torch.full((m * blocks * 42,), 0x5555, dtype=torch.int16,
                                           device="cuda")
                    table.records[i].row_cuts = guards[i].data_ptr()
    assert guards and all(torch.all(g == 0x5555) for g in guards.values())
    (now,) = opts[0]._tables.values()
    assert now is table and all(table.records[i].row_cuts == g.data_ptr() for i, g in guards.items())
    for a, b in zip(*lists):
        assert torch.equal(a.data, b.data)
        for key in ("error", "min_vals", "max_vals"):
            assert torch.equal(opts[0].state[a][key], opts[1].state[b][key]), key


@pytest.mark.parametrize("kind", [float, np.int64, lambda i: torch.tensor(float(i))],
                         ids=["float", "numpy", "tensor"])
def test_ring_positions_of_another_kind_step_as_before(kind):
    """A ring position that something re-typed between two steps: the list goes through the walk, and
    all positions have moved on behind it."""
    from ista_daslab_optimizers import MicroAdam
    lists, opts = [], []
    for _ in range(2):
        gen = torch.Generator().manual_seed(5)
        lists.append([torch.nn.Parameter((torch.randn(n, generator=gen) * 0.02).cuda())
                      for n in (500, 3000, 64)])
        opts.append(MicroAdam(lists[-1], m=3, lr=1e-3, quant_block_size=64))
    for step in range(5):
        grads = [torch.randn(p.numel(), generator=gen).cuda() for p in lists[0]]
        for opt, params in zip(opts, lists):
            for p, g in zip(params, grads):
                p.grad = g
            if opt is opts[0] and step == 2:
                st = opt.state[params[1]]
                st["index"] = kind(st["index"])
            opt.step()
    for a, b in zip(*lists):
        assert torch.equal(a.data, b.data)
        assert opts[0].state[a]["index"] == opts[1].state[b]["index"] == 2


def test_ring_positions_outside_32_bits_are_refused():
    """2^32 + 1 in a list that goes through one table: refused in front of the launch, not taken for
    row 1."""
    from ista_daslab_optimizers import MicroAdam
    p = torch.nn.Parameter(torch.ones(500, device="cuda"))
    opt = MicroAdam([p], m=3, lr=1e-3, quant_block_size=64)
    for _ in range(2):
        p.grad = torch.ones_like(p)
        opt.step()
    opt.state[p]["index"] = 2 ** 32 + 1
    before = p.data.clone()
    with pytest.raises(OverflowError):
        opt.step()
    assert torch.equal(p.data, before) and opt.state[p]["index"] == 2 ** 32 + 1


RIDING_CASES = [
    # a tensor that takes two launches by its sizes, and short ones of a single-launch form beside it
    ([20480 * 2 + 9001, 768, 300], torch.bfloat16, 10, 0.03),
    ([20480 + 9001, 768, 300], torch.float32, 10, 0.03),
    ([20480 * 2 + 9001, 768, 300], torch.bfloat16, 16, 0.03),
    ([20480 + 9001, 768, 300], torch.float32, 16, 0.03),
    # both single-launch forms beside it, one of them in a full block of a smaller class when alone
    ([20480 + 9001, 12288, 12000, 4096, 5001], torch.bfloat16, 15, 0.02),
    # more short tensors than a launch holds: the second launch has short ones alone
    ([20480 + 9001] + [300 + i for i in range(170)], torch.bfloat16, 10, 0.03),
    # more tensors of the longer one-pass stage than ride along: the shortest ride along with them
    ([20480 + 9001] + [8600] * 257 + [300, 301, 4096], torch.bfloat16, 15, 0.02),
]


@pytest.mark.parametrize("sizes,dtype,m,k_init", RIDING_CASES)
def test_short_tensors_beside_dense_windows(oracle, sizes, dtype, m, k_init):
    """They ride along in the two launches of the longer tensor.  Without its gradient in one step
    they take their own form, whose rows are in no particular order, and ride along again over those
    rows afterwards."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(m)
    cpu = [(torch.randn(n, generator=gen) * 0.02).to(dtype) for n in sizes]
    oparams = [to_np(p) for p in cpu]
    oref = oracle.OracleMicroAdam(oparams, m, 1e-3, 64, k_init, 0.0, weight_decay=0.01, d_block_size=20480)
    params = [torch.nn.Parameter(p.clone().cuda()) for p in cpu]
    opt = MicroAdam(params, m=m, lr=1e-3, quant_block_size=64, k_init=k_init, weight_decay=0.01)
    for step in range(m + 4):
        grads = [(torch.randn(n, generator=gen) * 1e-2).to(dtype) for n in sizes]
        for p, g in zip(params, grads):
            p.grad = g.clone().cuda()
        if step in (3, m + 1):
            params[0].grad = grads[0] = None
        opt.step()
        oref.step([None if g is None else to_np(g) for g in grads])
        for i, p in enumerate(params):
            assert opt._entries[p].route == 1
            if step in (0, 3, 4, m + 1, m + 2, m + 3):
                assert_state_equal(opt.state[p], oref.state[i], f"step {step + 1} tensor {i}")
            assert np.array_equal(to_np(p.data), oparams[i]), (step, i)


@pytest.mark.parametrize("why", ["one turn", "odd address"])
@pytest.mark.parametrize("n", [20480 * 2 + 17100, 18001])
def test_longer_windows_that_fall_back_to_ranges(oracle, n, why):
    """Windows of the longer one-pass stage that it gives up.  "one turn": the large gradients lie on
    every 16th coordinate, the same ones at every step, so that all 3000 entries that share a
    coordinate fall into one turn of its queue; "odd address": the window begins on an odd entry."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(n)
    m, dtype = 15, torch.bfloat16
    start = (torch.randn(n, generator=gen) * 0.02).to(dtype)
    oparams = [to_np(start)]
    oref = oracle.OracleMicroAdam(oparams, m, 1e-3, 64, 0.01, 0.0, weight_decay=0.01, d_block_size=20480)
    p = torch.nn.Parameter(start.clone().cuda())
    opt = MicroAdam([p], m=m, lr=1e-3, quant_block_size=64, weight_decay=0.01)
    for step in range(m + 3):
        g = torch.randn(n, generator=gen) * 1e-2
        if why == "one turn":
            at = torch.arange(n)
            g[(at % 20480 % 16 == 0) & (at % 20480 < 16 * 200)] *= 100
        p.grad = g.to(dtype).cuda()
        opt.step()
        oref.step([to_np(g.to(dtype))])
        st = opt.state[p]
        if step == 0 and why == "odd address":
            for key in ("I", "V"):
                flat = torch.empty(st[key].numel() + 1, dtype=st[key].dtype, device="cuda")
                st[key] = flat[1:].view(st[key].shape).copy_(st[key])
                assert st[key].data_ptr() % 4 == 2
            opt._tables.clear()
            opt._uniform = None
        assert opt._entries[p].route == 1
        assert_state_equal(st, oref.state[0], f"step {step + 1}")
        assert np.array_equal(to_np(p.data), oparams[0]), step


def test_window_kernel_over_rows_out_of_order(oracle):
    """Two launches over a window with rows that are not listed by coordinate, as a checkpoint may hold
    them: the window kernel's general form."""
    from ista_daslab_optimizers import MicroAdam
    gen = torch.Generator().manual_seed(18)
    n, m, dtype = 20480 * 2 + 8192, 18, torch.bfloat16
    start = (torch.randn(n, generator=gen) * 0.02).to(dtype)
    oparams = [to_np(start)]
    oref = oracle.OracleMicroAdam(oparams, m, 1e-3, 64, 0.01, 0.0, d_block_size=20480)
    p = torch.nn.Parameter(start.clone().cuda())
    opt = MicroAdam([p], m=m, lr=1e-3, quant_block_size=64)
    for step in range(m + 3):
        g = (torch.randn(n, generator=gen) * 1e-2).to(dtype)
        p.grad = g.cuda()
        opt.step()
        oref.step([to_np(g)])
        st = opt.state[p]
        assert opt._entries[p].route == 1 and opt._entries[p].cuts is None
        assert_state_equal(st, oref.state[0], f"step {step + 1}")
        assert np.array_equal(to_np(p.data), oparams[0]), step
        if step % 5 == 1:  # this step's row of every block, backwards
            many = st["k_block_size_many"]
            for key in ("I", "V"):
                row = st[key][step % m]
                row.copy_(torch.cat([part.flip(0) for part in row.split(many)]))
