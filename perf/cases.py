"""What the package is used for, as a list of timed cases: `matmul_transpose` on its own, Newton-Schulz
orthogonalisation of single matrices and of stacks, and whole steps of the optimizer.

    listed()            the cases
    draw(rng)           one more case of the ranges they stand for
    prepare(case, seed) what a program holds before the call, on the GPU
    run(state)          one pass through the public entry points
    work(case)          the bytes and operations that a pass cannot do without
    tolerance(case)     how far two correct implementations of the same precision may be apart

A case is a dict.  kind "xxt": y = x x^T of an M x K matrix of `dtype`.  kind "ns": five
Newton-Schulz steps on `batch` (0: a plain 2-D input) matrices of rows x cols.  kind "muon": one
Muon.step on a transformer's matrices, `layers` times (`square` of width x width, `up` of
ffn x width, `down` of width x ffn).
"""
import math

import torch

from flash_muon_amd import Muon, fast_newtonschulz, matmul_transpose, matmul_transpose_assign

STEPS = 5
_DTYPE = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _xxt(M, K, dtype="bf16", **more):
    return dict(kind="xxt", M=M, K=K, dtype=dtype, **more)


def _ns(rows, cols, dtype="bf16", batch=0, **more):
    return dict(kind="ns", rows=rows, cols=cols, dtype=dtype, batch=batch, **more)


def _muon(width, ffn, layers, dtype="bf16", square=4, up=1, down=1, **more):
    return dict(kind="muon", width=width, ffn=ffn, layers=layers, dtype=dtype, square=square, up=up, down=down, **more)


def listed():
    return [
        # the square sweep of the benchmark table, its smallest size: one launch, nearly all latency
        _xxt(1024, 1024, name="xxt_1024"),
        # its second size: fewer tiles than compute units
        _xxt(2048, 2048, name="xxt_2048"),
        # its largest size, the headline: into an output that the caller keeps
        _xxt(8192, 8192, into=True, name="xxt_8192_into"),
        # sides that no tile divides, in half precision
        _xxt(3000, 5000, "f16", name="xxt_3000x5000_f16"),
        # single precision: a Gram matrix of statistics that are kept in fp32
        _xxt(2048, 4096, "f32", name="xxt_2048x4096_f32"),
        # one square gradient of a small model: a chain of short launches
        _ns(1024, 1024, name="ns_1024"),
        # an fp32 gradient of an MLP of 1600 x 6400 (tall, and no multiple of 128)
        _ns(6400, 1600, "f32", name="ns_6400x1600_f32"),
        # the benchmark's wide matrix: bound by the matrix units
        _ns(4096, 16384, name="ns_4096x16384"),
        # a stack of expert matrices as one 3-D gradient
        _ns(1024, 2816, batch=8, name="ns_8x1024x2816"),
        # a GPT-2-small-like model (12 layers of 768) trained with fp32 weights and gradients
        _muon(768, 3072, 12, "f32", name="muon_768_f32"),
        # a model of about 1.3 G parameters with gated MLPs, in bf16
        _muon(2048, 5504, 24, up=2, name="muon_2048"),
        # 8 of the 32 layers of Llama-7B, as one of four pipeline stages holds them, in bf16
        _muon(4096, 11008, 8, up=2, name="muon_llama7b_8_layers"),
    ]


def _size(rng, lo, hi):
    """A size between lo and hi, spread over its logarithm: half of them multiples of 128, a quarter
    multiples of 8, a quarter any number."""
    x = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    unit = rng.choice((128, 128, 8, 1))
    return max(lo, min(hi, int(x / unit + 0.5) * unit))


def draw(rng):
    kind = rng.choice(("xxt", "xxt", "ns", "ns", "muon"))
    if kind == "xxt":
        dtype = rng.choice(("bf16", "bf16", "bf16", "f16", "f32"))
        most = 4096 if dtype == "f32" else 8192
        return _xxt(_size(rng, 512, most), _size(rng, 512, most), dtype, into=rng.random() < 0.3)
    if kind == "ns":
        dtype = rng.choice(("bf16", "bf16", "f32"))
        short, ratio = _size(rng, 256, 4096), rng.choice((1, 1, 4, 2.75, rng.uniform(1, 4)))
        long = short if ratio == 1 else max(short, int(short * ratio))
        if ratio not in (1, 4, 2.75):
            long = max(short, long // 8 * 8)
        rows, cols = (short, long) if rng.random() < 0.5 else (long, short)
        batch = rng.choice((0, 0, 2, 6, 16)) if short <= 2048 else 0
        return _ns(rows, cols, dtype, batch)
    width = max(256, int(math.exp(rng.uniform(math.log(256), math.log(2560)))) // 64 * 64)
    if rng.random() < 0.2:
        width += rng.choice((8, 24, 40))   # no multiple of 64
    gated = rng.random() < 0.5
    ffn = int(width * 2.6875) // 8 * 8 if gated else 4 * width
    return _muon(width, ffn, rng.randint(2, 16), rng.choice(("bf16", "f32")), up=2 if gated else 1)


# ---- inputs -------------------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _gradient_like(shape, dtype, gen):
    """Noise of 1e-3 and a low-rank part with singular values over two decades, as gradients have."""
    rows, cols = shape[-2:]
    rank = min(64, rows, cols)
    lead = shape[:-2]
    g = 1e-3 * torch.randn(*shape, generator=gen, device="cuda")
    u = torch.randn(*lead, rows, rank, generator=gen, device="cuda") / rows ** 0.5
    v = torch.randn(*lead, rank, cols, generator=gen, device="cuda") / cols ** 0.5
    s = torch.exp(torch.rand(*lead, 1, rank, generator=gen, device="cuda") * math.log(1e-2))
    return (g + (u * s) @ v).to(dtype).contiguous()


def _muon_shapes(case):
    w, f = case["width"], case["ffn"]
    return ([(w, w)] * case["square"] + [(f, w)] * case["up"] + [(w, f)] * case["down"]) * case["layers"]


def prepare(case, seed):
    gen = _generator(seed)
    dtype = _DTYPE[case["dtype"]]
    if case["kind"] == "xxt":
        x = torch.randn(case["M"], case["K"], generator=gen, device="cuda").to(dtype)
        into = torch.empty(case["M"], case["M"], dtype=dtype, device="cuda") if case.get("into") else None
        return {"kind": "xxt", "x": x, "into": into}
    if case["kind"] == "ns":
        shape = (case["rows"], case["cols"])
        if case["batch"]:
            shape = (case["batch"],) + shape
        return {"kind": "ns", "g": _gradient_like(shape, dtype, gen)}
    # Weights, gradients and momenta are views of three flat buffers, each matrix on a boundary of 256
    # elements, as trainers with contiguous parameter and gradient buffers keep them; the momenta are
    # those of a run under way.
    shapes = _muon_shapes(case)
    starts, total = [], 0
    for r, c in shapes:
        starts.append(total)
        total += (r * c + 255) // 256 * 256
    flat = [torch.zeros(total, dtype=dtype, device="cuda") for _ in range(3)]
    params = []
    for (r, c), at in zip(shapes, starts):
        views = [f[at:at + r * c].view(r, c) for f in flat]
        for v, scale in zip(views, (0.02, 1e-3, 4e-4)):
            v.copy_(torch.randn(r, c, generator=gen, device="cuda").mul_(scale))
        p = torch.nn.Parameter(views[0])
        p.grad = views[1]
        params.append((p, views[2]))
    opt = Muon([p for p, _ in params], lr=0.02, weight_decay=0.01, momentum=0.95, rank=0, world_size=1)
    for p, momentum in params:
        opt.state[p]["momentum_buffer"] = momentum
    return {"kind": "muon", "opt": opt, "weights": flat[0], "grads": flat[1], "momenta": flat[2]}


def run(state):
    if state["kind"] == "xxt":
        if state["into"] is None:
            return matmul_transpose(state["x"])
        matmul_transpose_assign(state["x"], state["into"])
        return state["into"]
    if state["kind"] == "ns":
        return fast_newtonschulz(state["g"], STEPS)
    state["opt"].step()
    return {"weights": state["weights"], "grads": state["grads"], "momenta": state["momenta"]}


# ---- what a pass cannot do without --------------------------------------------------------------

def _ns_flops(rows, cols):
    """Per step: the distinct elements of the two symmetric products, and the whole third one."""
    m, k = min(rows, cols), max(rows, cols)
    return STEPS * (k * m * (m + 1) + m * m * (m + 1) + 2 * m * m * k)


def work(case):
    size = 4 if case["dtype"] == "f32" else 2
    if case["kind"] == "xxt":
        M, K = case["M"], case["K"]
        return {"bytes": size * (M * K + M * M), "flops": K * M * (M + 1)}
    if case["kind"] == "ns":
        n = max(case["batch"], 1)
        return {"bytes": n * case["rows"] * case["cols"] * (size + 2), "flops": n * _ns_flops(case["rows"], case["cols"])}
    shapes = _muon_shapes(case)
    # weight, gradient and momentum are each read and written
    return {"bytes": sum(6 * size * r * c for r, c in shapes), "flops": sum(_ns_flops(r, c) for r, c in shapes)}


def tolerance(case):
    """About four times what each path shows against the same computation in fp64 (xxt) or with fp32
    iterates (ns, muon)."""
    if case["kind"] == "xxt":
        # 16-bit outputs: a sum in another order rounds the other way now and then, by one unit of the last place
        return {"bf16": {"rel": 1e-3, "max": 1e-2}, "f16": {"rel": 2e-4, "max": 2e-3}, "f32": {"rel": 4e-6}}[case["dtype"]]
    if case["kind"] == "ns":
        # the iterate is rounded to bf16 in every step
        return {"rel": 3e-2}
    # the update is such an iterate, and the weights it is added to are larger; bf16 weights are rounded
    return {"rel": 2e-3 if case["dtype"] == "f32" else 4e-3}
