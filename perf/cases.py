"""The work that users of this package have it do, as cases that can be timed and compared.

Two kinds of case:

  kind "step"    one `MicroAdam.step()` over a transformer-shaped parameter list, the window full
                 and the gradient new in every pass, as in training;
  kind "window"  Sparse M-FAC's two passes over a window of sparse gradients: the scalar products
                 of all rows with a dense vector (SP), then a linear combination of the rows (LCG).

A step's parameters lie in one flat buffer, every tensor on a 512-byte boundary (where an
allocator would put it too); its gradients are drawn once into a pool, and every pass takes
another stretch of it, m + 2 of them in turn, so that no gradient recurs inside the window.
Routes of the step that leave the gradient buffer alone get those stretches as `p.grad`; routes
that overwrite it (long or odd quantisation blocks) get them copied into fixed gradient
buffers, which is what a backward pass over persistent buckets does.
"""
import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "ista-daslab-optimizers_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

TOPK_BLOCK = 20480  # MicroAdam's top-k block on this hardware: half of 160 KB of floats
ALIGN = 256         # elements; tensors of a list start on multiples of this
SHIFT = 8 * 13109   # elements between the stretches of the gradient pool two passes take


# ---------------------------------------------------------------------------------- the cases
def _step(name, vocab, hidden, mlp, layers, dtype="bf16", pos=0, kv=0, style="gated", tied=False,
          m=10, k=0.01, q=64, alpha=0.0, wd=0.0, grads="normal", std=1e-3):
    case = dict(kind="step", vocab=vocab, hidden=hidden, mlp=mlp, layers=layers, dtype=dtype,
                pos=pos, kv=kv or hidden, style=style, tied=tied, m=m, k=k, q=q, alpha=alpha,
                wd=wd, grads=grads, std=std)
    return dict(case, name=name) if name else case


def listed():
    return [
        # a toy or test model: 30 small, odd-sized fp32 tensors, most shorter than a top-k block;
        # the time is launches and host work
        _step("small-list-f32", 503, 67, 201, 2, "f32", pos=128, style="biased", tied=True,
              std=1e-2),
        # one fp32 tensor of 2^20 elements (the plumbing configuration), 52 top-k blocks: fewer
        # than the chip has compute units
        _step("one-tensor-1m-f32", 1024, 1024, 0, 0, "f32", tied=True, std=1.0),
        # the GPT-2-small-shaped list of 148 tensors in bf16: an ordinary fine-tuning step
        _step("gpt2-small", 50257, 768, 3072, 12, pos=1024, style="biased", tied=True, std=1e-2),
        # the same list trained in fp32 with weight decay
        _step("gpt2-small-f32-decay", 50257, 768, 3072, 12, "f32", pos=1024, style="biased",
              tied=True, wd=0.01, std=1e-2),
        # the Llama-2-7B-shaped list, the headline configuration and the largest case
        _step("llama2-7b", 32000, 4096, 11008, 32),
        # a dense window (20 rows of 5 %) under heavy-tailed gradients with outlier rows: the
        # 1.3 B outlier configuration's shapes, 12 of its 24 layers
        _step("outlier-window-20", 50304, 2048, 8192, 12, style="plain", tied=True, m=20, k=0.05,
              q=32, grads="student"),
        # quant_block_size=100_000, alpha=0: the setting the reference's README shows; 4 layers
        # of the Llama-2-7B shapes
        _step("readme-q100000", 32000, 4096, 11008, 4, q=100000, wd=0.01),
        # quant_block_size=100_000 with half of the error feedback in the update: the
        # Llama-3-8B-shaped configuration, 8 of its 32 layers (grouped key and value heads)
        _step("llama3-alpha-q100000", 128256, 4096, 14336, 8, kv=1024, q=100000, alpha=0.5),
        # alpha > 0 with short quantisation blocks
        _step("alpha-q64", 32000, 4096, 11008, 4, alpha=0.5),
        # alpha = -2: what quantisation loses goes straight into the parameters
        _step("quant-error", 32000, 2048, 5632, 8, alpha=-2.0, wd=0.01),
        # a quantisation block that neither divides the top-k block nor covers it
        _step("gpt2-small-q10000", 50257, 768, 3072, 12, pos=1024, style="biased", tied=True,
              q=10000, std=1e-2),
        # Sparse M-FAC on a ResNet-50-sized vector, 1024 gradients of 1 %
        dict(name="sparse-mfac-1024", kind="window", d=25557032, m=1024, k=0.01, dtype="bf16",
             values="bf16"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: sizes over their logarithm, odd ones in every second."""
    if rng.random() < 0.12:
        return dict(kind="window", d=_log_uniform(rng, 200_000, 25_000_000),
                    m=_log_uniform(rng, 16, 1024), k=rng.choice([0.005, 0.01, 0.02]),
                    dtype=rng.choice(["bf16", "f32"]), values=rng.choice(["bf16", "f32"]))
    option = rng.choice(["usual", "usual", "usual", "dense window", "long blocks", "long blocks",
                         "alpha", "quant error", "odd blocks"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "f32"])
    largest = {"usual": 1.5e9, "dense window": 5e8, "odd blocks": 1.5e8}.get(option, 1e9)
    if dtype == "f32":
        largest /= 2
    # a list of about `size` parameters: width first, then as many layers as that makes
    size = math.exp(rng.uniform(math.log(2e5), math.log(largest)))
    hidden = _log_uniform(rng, 72, min(4096, max(96, math.sqrt(size / 14))))
    hidden = hidden | 1 if rng.random() < 0.5 else (hidden + 7) // 8 * 8
    mlp = int(hidden * rng.choice([2.6875, 3.5, 4]))
    style = rng.choice(["gated", "biased", "plain"])
    layers = int(max(1, min(32, size / 2 / (4 * hidden ** 2 + 3 * hidden * mlp))))
    vocab = int(max(256, min(130_000, size / 2 / hidden)))
    opts = dict(m=10, k=0.01, q=rng.choice([32, 64, 64, 128]), alpha=0.0)
    if option == "usual":
        opts.update(m=rng.choice([4, 10, 10, 15]), k=rng.choice([0.005, 0.01, 0.01]))
    elif option == "dense window":
        opts.update(m=rng.choice([10, 16, 20]), k=rng.choice([0.02, 0.03, 0.05]))
    elif option == "long blocks":
        opts.update(q=rng.choice([50_000, 100_000, 100_000, 65_536]), alpha=rng.choice([0.0, 0.5]))
    elif option == "alpha":
        opts.update(alpha=rng.choice([0.25, 0.5]))
    elif option == "quant error":
        opts.update(alpha=-2.0)
    else:
        opts.update(q=rng.choice([1000, 8192, 10_000, 16_384]))
    return _step(None, vocab, hidden, mlp, layers, dtype, style=style, tied=rng.random() < 0.5,
                 wd=rng.choice([0.0, 0.01]), grads=rng.choice(["normal", "normal", "student"]),
                 std=rng.choice([1e-3, 1e-2]), **opts)


# ------------------------------------------------------------------------------ what they hold
def _shapes(case):
    h, f, kv = case["hidden"], case["mlp"], case["kv"]
    shapes = [(case["vocab"], h)] + ([(case["pos"], h)] if case["pos"] else [])
    for _ in range(case["layers"]):
        if case["style"] == "gated":     # q, o, k, v projections, three MLP weights, two norms
            shapes += [(h, h)] * 2 + [(kv, h)] * 2 + [(f, h)] * 3 + [(h,)] * 2
        elif case["style"] == "biased":  # two norms with bias, fused qkv, projection, MLP, biases
            shapes += [(h,), (h,), (h, 3 * h), (3 * h,), (h, h), (h,), (h,), (h,), (h, f), (f,),
                       (f, h), (h,)]
        else:                            # the weights alone
            shapes += [(h, 3 * h), (h, h), (h, f), (f, h)]
    if case["style"] == "biased":
        shapes += [(h,), (h,)]
    if not case["tied"]:
        shapes += [(case["vocab"], h)]
    return shapes


def _layout(case):
    """(offset, elements, shape) of every tensor in the flat buffer, and the buffer's length."""
    places, at = [], 0
    for shape in _shapes(case):
        n = math.prod(shape)
        places.append((at, n, shape))
        at += (n + ALIGN - 1) // ALIGN * ALIGN
    return places, at


def _refills(case, places):
    """Whether some tensor's step may overwrite the gradient buffer it is given."""
    q = case["q"]
    inside = 8 <= q <= 4096 and q & (q - 1) == 0
    return not inside or min(n for _, n, _ in places) < q


def _window_geometry(d, k_init):
    """(entries per row of a full top-k block, entries per row) of a tensor of d elements"""
    block = min(d, TOPK_BLOCK)
    full = d // block
    many = math.ceil(block * k_init)
    return many, full * many + math.ceil((d - full * block) * k_init)


_TYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def _student_t(out, std, gen):
    """Student-t with 3 degrees of freedom, a stretch at a time"""
    for part in out.split(1 << 26):
        n = part.numel()
        chi = torch.zeros(n, device=out.device)
        for _ in range(3):
            chi += torch.randn(n, device=out.device, generator=gen).square_()
        part.copy_(torch.randn(n, device=out.device, generator=gen).div_(chi.div_(3).sqrt_()).mul_(std))


class _Step:
    """A training program between two steps."""

    def __init__(self, case, seed):
        from ista_daslab_optimizers import MicroAdam

        dev, dtype = torch.device("cuda:0"), _TYPES[case["dtype"]]
        gen = torch.Generator(device=dev).manual_seed(seed)
        places, total = _layout(case)
        self.flat = torch.zeros(total, dtype=dtype, device=dev)
        self.params = []
        for at, n, shape in places:
            p = self.flat[at:at + n]
            self.params.append(torch.nn.Parameter(p.view(shape)))
        self.flat.normal_(0.0, 0.02, generator=gen)

        turns = case["m"] + 2
        pool = torch.empty(total + turns * SHIFT, dtype=dtype, device=dev)
        if case["grads"] == "student":
            _student_t(pool, case["std"], gen)
        else:
            pool.normal_(0.0, case["std"], generator=gen)
        stretches = [pool[i * SHIFT:i * SHIFT + total] for i in range(turns)]
        if case["grads"] == "student":
            # one row in a hundred, always the same ones, carries gradients a hundred times larger
            cpu = torch.Generator().manual_seed(seed)
            scale = torch.ones(total, dtype=dtype, device=dev)
            for at, n, shape in places:
                if len(shape) == 2:
                    rows = torch.randperm(shape[0], generator=cpu)[:max(1, shape[0] // 100)].to(dev)
                    scale[at:at + n].view(shape)[rows] = 100.0
            stretches = [s * scale for s in stretches]
        self.stretches, self.turn = stretches, 0

        self.bucket = None
        if _refills(case, places):
            self.bucket = torch.empty(total, dtype=dtype, device=dev)
            for p, (at, n, shape) in zip(self.params, places):
                p.grad = self.bucket[at:at + n].view(shape)
        else:
            self.grads = [[s[at:at + n].view(shape) for at, n, shape in places] for s in stretches]

        self.opt = MicroAdam(self.params, m=case["m"], lr=1e-4, quant_block_size=case["q"],
                             k_init=case["k"], alpha=case["alpha"], weight_decay=case["wd"])
        for _ in range(case["m"]):  # fill the window
            self.step()
        # What a pass changes: all parameters, and the error feedback with its statistics of the
        # first tensors of the list (of all of them in the shorter lists).  The window's rows are
        # not among it, as the order of a block's entries inside a row is unspecified; every
        # entry is in the parameters of the next passes.
        self.outputs = {"params": self.flat}
        for i, p in enumerate(self.params[:15]):
            st = self.opt.state[p]
            self.outputs["state%02d" % i] = [st[key] for key in
                                             ("error", "min_vals", "max_vals", "quant_err")
                                             if key in st]

    def step(self):
        turn, self.turn = self.turn, (self.turn + 1) % len(self.stretches)
        if self.bucket is not None:
            self.bucket.copy_(self.stretches[turn])
        else:
            for p, g in zip(self.params, self.grads[turn]):
                p.grad = g
        self.opt.step()


class _Window:
    """Sparse M-FAC's window, a gradient and the coefficients of a combination."""

    def __init__(self, case, seed):
        dev, vtype = torch.device("cuda:0"), _TYPES[case["values"]]
        gen = torch.Generator(device=dev).manual_seed(seed)
        d, m = case["d"], case["m"]
        block = min(d, TOPK_BLOCK)
        full = d // block
        many, k = _window_geometry(d, case["k"])
        few = k - full * many
        self.geometry = (d, m, k, block, many)
        self.I = torch.empty(m, k, dtype=torch.int16, device=dev)
        self.V = torch.empty(m, k, dtype=vtype, device=dev)
        # rows as the block-wise top-k of dense vectors makes them: 8 of them selected, the others
        # with the coordinates of one of these moved round inside the blocks and fresh values
        lengths = torch.full((k,), block, dtype=torch.int32, device=dev)
        if few:
            lengths[full * many:] = d - full * block
        made = []
        for _ in range(min(m, 8)):
            x = torch.randn(d, device=dev, generator=gen).abs_()
            idx = [x[:full * block].view(full, block).topk(many, dim=1, sorted=False).indices.view(-1)]
            if few:
                idx.append(x[full * block:].topk(few, sorted=False).indices)
            made.append(torch.cat(idx).to(torch.int32))
        for r in range(m):
            move = torch.randint(0, block, (1,), device=dev, generator=gen, dtype=torch.int32)
            self.I[r] = (made[r % len(made)] + move) % lengths
            v = torch.randn(k, device=dev, generator=gen)
            self.V[r] = v + 2.5 * v.sign()  # the tails of a normal distribution
        self.g = torch.randn(d, device=dev, generator=gen).to(_TYPES[case["dtype"]])
        self.coef = torch.randn(m, device=dev, generator=gen)
        self.dots = torch.zeros(m, device=dev)
        self.out = torch.zeros(d, dtype=_TYPES[case["dtype"]], device=dev)
        self.bf16 = int(case["values"] == "bf16")


def prepare(case, seed):
    return (_Step if case["kind"] == "step" else _Window)(case, seed)


def run(state):
    if isinstance(state, _Step):
        state.step()
        return state.outputs
    import ista_daslab_cuda_sparse_mfac as sparse_mfac

    d, m, k, block, many = state.geometry
    state.dots.zero_()
    sparse_mfac.SP(0, 0, 23, d, m, k, block, many, state.g, state.I, state.V, state.dots, state.bf16)
    state.out.zero_()
    sparse_mfac.LCG(0, 0, 51, d, m, k, block, many, state.coef, state.I, state.V, state.out,
                    state.bf16)
    return {"dots": state.dots, "out": state.out}


# ------------------------------------------------------------------------- what they have to do
def work(case):
    size = 2 if case["dtype"] == "bf16" else 4
    if case["kind"] == "window":
        d, m = case["d"], case["m"]
        _, k = _window_geometry(d, case["k"])
        entry = 2 + (2 if case["values"] == "bf16" else 4)
        # the window is an input of both passes, which the coefficients lie between; the dense
        # vector in, the combination out
        return {"bytes": 2 * m * k * entry + 2 * d * size + 8 * m, "flops": 4 * m * k}
    total = entries = stats = 0
    for _, n, _ in _layout(case)[0]:
        total += n
        entries += _window_geometry(n, case["k"])[1]
        stats += -(-n // case["q"])
    # gradient in; parameters, 4-bit codes and (min, max) pairs in and out; the window's rows in,
    # one of them out
    nbytes = total * (3 * size + 1) + 8 * stats + 4 * entries * (case["m"] + 1)
    if case["alpha"] == -2:
        nbytes += total * size  # the lost part is part of the state
    if _refills(case, _layout(case)[0]):
        nbytes += 2 * total * size  # the gradient's way into its bucket
    return {"bytes": nbytes, "flops": 20 * total + 6 * entries * case["m"]}


def tolerance(case):
    if case["kind"] == "step":
        # codes, statistics and parameters are settled to the last bit by the step's definition:
        # fp32 operations in a stated order, each rounded once, ties to the lowest index
        return "exact"
    # Sums of many terms in fp32, in any order, and the combination rounded to the vector's type
    # once.  Rows added last to first against first to last, m up to 1024: 1.2e-7 (at most 1.1e-6)
    # in fp32; in bf16 1.8e-5, a sum here and there rounding to the other side (2^-7 of it).
    if case["dtype"] == "bf16":
        return {"rel": 8e-5, "max": 1e-2}
    return {"rel": 5e-7, "max": 5e-6}
