"""The work that programs built on this library have it do, as timed cases.

Seven paths, each through the entry points a program calls:

  gemm     ``matmul_lt`` with the selector, the launch state and the output tensor kept between calls
  matmul   ``matmul``: everything but the operands left to the library
  train    ``addmm`` and its gradients: a linear layer's forward and backward pass
  a8w8     ``matmul_a8w8_lt`` on operands that are quantised already
  linear8  a quantised linear layer on bf16 activations: ``quantize_tensor_per_channel``, then ``matmul_a8w8``
  moe      ``grouped_matmul_a8w8`` over the experts' routed rows
  mxfp4    ``hadamard_mxfp4_quant`` of the activations, then ``matmul_fp4``

``ta`` / ``tb`` are the storage orders of ``generate_matmul_inputs``: "T" is stored as it is written, (m, k) or (k, n);
"N" is stored transposed and passed as a transposed view.  A weight kept as (out_features, in_features) has tb = "N".
"""
import math

import torch

import tritonblas_amd as tb
from tritonblas_amd.utils import quantize_tensor_per_channel

_DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32,
           "float8_e4m3fn": torch.float8_e4m3fn, "int8": torch.int8}


def listed():
    return [
        # the smallest configuration of the benchmark: a launch-bound product of two row-major matrices
        dict(name="gemm fp16 1024", path="gemm", dtype="float16", m=1024, n=1024, k=1024, ta="T", tb="T"),
        # a training- or prefill-size product in the layout a stored weight has
        dict(name="gemm bf16 8192", path="gemm", dtype="bfloat16", m=8192, n=8192, k=8192, ta="T", tb="N"),
        # single precision, both matrices row-major, as numerical programs hold them
        dict(name="matmul fp32 2048", path="matmul", dtype="float32", m=2048, n=2048, k=2048, ta="T", tb="T"),
        # sizes that are no multiple of anything: padded-free batches, pruned layers, odd vocabularies
        dict(name="matmul bf16 odd", path="matmul", dtype="bfloat16", m=1187, n=3001, k=1531, ta="T", tb="T"),
        # token generation for a small batch with an unquantised weight: latency, host path and weight traffic
        dict(name="decode bf16 8 rows", path="matmul", dtype="bfloat16", m=8, n=14336, k=4096, ta="T", tb="N"),
        # one layer of a training step: output, input gradient, weight gradient, bias gradient
        dict(name="train bf16 4096", path="train", dtype="bfloat16", m=4096, n=14336, k=4096, tb="T"),
        # the benchmark's FP8 prefill and decode products
        dict(name="a8w8 prefill", path="a8w8", dtype="float8_e4m3fn", m=8192, n=28672, k=8192, streamk=False),
        dict(name="a8w8 decode", path="a8w8", dtype="float8_e4m3fn", m=32, n=8192, k=28672, streamk=True),
        # a serving step of a quantised layer: activations arrive in bf16 and are quantised on the way
        dict(name="linear8 512 tokens", path="linear8", dtype="float8_e4m3fn", m=512, n=4096, k=14336),
        # 4096 tokens routed to two of eight experts each
        dict(name="moe 8192 rows", path="moe", rows=8192, experts=8, n=14336, k=4096),
        # rotated MXFP4, a decode batch of the benchmark's FP4 shape list and the benchmark's own large product
        dict(name="mxfp4 64 rows", path="mxfp4", m=64, n=8192, k=1024),
        dict(name="mxfp4 8192 rows", path="mxfp4", m=8192, n=8192, k=16384),
    ]


def _size(rng, lo, hi, steps=(1,)):
    """A size between lo and hi, spread over its logarithm, a multiple of one of ``steps``."""
    step = rng.choice(steps)
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, max(step, int(v / step + 0.5) * step)))


def _within(rng, most, make):
    """The first of make()'s size triples whose product is at most ``most``."""
    while True:
        m, n, k = make()
        if m * n * k <= most:
            return m, n, k


def draw(rng):
    path = rng.choice(("gemm", "matmul", "matmul", "decode", "train", "a8w8", "linear8", "moe", "mxfp4"))
    wide = (64, 8, 1)      # model sizes are round as a rule; batches, slices and vocabularies are not
    if path == "gemm":
        m, n, k = _within(rng, 8192 ** 3, lambda: (_size(rng, 128, 8192, wide), _size(rng, 256, 8192, (64, 8)), _size(rng, 256, 8192, (64, 8))))
        return dict(path="gemm", dtype=rng.choice(("bfloat16", "float16")), m=m, n=n, k=k, ta=rng.choice("TTTN"), tb=rng.choice("NT"))
    if path == "matmul":
        dtype = rng.choice(("bfloat16", "float16", "float32"))
        m, n, k = _within(rng, 2048 ** 3, lambda: (_size(rng, 100, 4096, wide), _size(rng, 200, 4096, wide), _size(rng, 200, 4096, wide)))
        return dict(path="matmul", dtype=dtype, m=m, n=n, k=k, ta=rng.choice("TTTN"), tb=rng.choice("NT"))
    if path == "decode":
        return dict(path="matmul", dtype=rng.choice(("bfloat16", "float16")), m=_size(rng, 1, 64), n=_size(rng, 1024, 28672, (64, 8)),
                    k=_size(rng, 1024, 16384, (64,)), ta="T", tb="N")
    if path == "train":
        m, n, k = _within(rng, 2048 * 14336 * 4096, lambda: (_size(rng, 256, 8192, wide), _size(rng, 512, 14336, (64, 8)), _size(rng, 512, 8192, (64, 8))))
        return dict(path="train", dtype=rng.choice(("bfloat16", "float16")), m=m, n=n, k=k, tb=rng.choice("TN"))
    if path == "a8w8":
        m, n, k = _within(rng, 8192 * 28672 * 8192, lambda: (_size(rng, 1, 8192), _size(rng, 1024, 28672, (64, 16)), _size(rng, 1024, 28672, (64, 16))))
        return dict(path="a8w8", dtype=rng.choice(("float8_e4m3fn", "float8_e4m3fn", "int8")), m=m, n=n, k=k, streamk=rng.random() < 0.3)
    if path == "linear8":
        m, n, k = _within(rng, 4096 * 14336 * 4096, lambda: (_size(rng, 1, 8192), _size(rng, 1024, 28672, (64, 16)), _size(rng, 1024, 28672, (64, 16))))
        return dict(path="linear8", dtype=rng.choice(("float8_e4m3fn", "float8_e4m3fn", "int8")), m=m, n=n, k=k)
    if path == "moe":
        rows, n, k = _within(rng, 8192 * 14336 * 4096, lambda: (_size(rng, 16, 16384), _size(rng, 1024, 14336, (64, 16)), _size(rng, 1024, 8192, (128,))))
        return dict(path="moe", rows=rows, experts=rng.choice((4, 8, 16)), n=n, k=k)
    m, n, k = _within(rng, 8192 * 8192 * 16384, lambda: (_size(rng, 1, 8192), _size(rng, 1024, 16384, (64, 16)), _size(rng, 1024, 16384, (512, 512, 32))))
    return dict(path="mxfp4", m=m, n=n, k=k)


def _normal(gen, shape, dtype, scale=1.0):
    return torch.randn(shape, device="cuda", dtype=torch.float32 if dtype == torch.float32 else torch.bfloat16, generator=gen).mul_(scale).to(dtype)


def _stored(gen, rows, cols, order, dtype, scale=1.0):
    return _normal(gen, (rows, cols), dtype, scale) if order == "T" else _normal(gen, (cols, rows), dtype, scale).T


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    path = case["path"]
    if path in ("gemm", "matmul"):
        m, n, k, dtype = case["m"], case["n"], case["k"], _DTYPES[case["dtype"]]
        a = _stored(gen, m, k, case["ta"], dtype)
        b = _stored(gen, k, n, case["tb"], dtype, k ** -0.5)
        if path == "matmul":
            return dict(path=path, a=a, b=b)
        selector = tb.OrigamiMatmulSelector(m, n, k, dtype, dtype, dtype, a.device)
        return dict(path=path, a=a, b=b, c=torch.empty(m, n, dtype=dtype, device="cuda"), selector=selector, config=tb.matmul_preamble(selector))
    if path == "train":
        m, n, k, dtype = case["m"], case["n"], case["k"], _DTYPES[case["dtype"]]
        x = _normal(gen, (m, k), dtype).requires_grad_()
        w = (_normal(gen, (k, n), dtype, k ** -0.5) if case["tb"] == "T" else _normal(gen, (n, k), dtype, k ** -0.5)).requires_grad_()
        bias = _normal(gen, (n,), dtype, 0.1).requires_grad_()
        return dict(path=path, x=x, w=w, bias=bias, transposed=case["tb"] == "N", grad=_normal(gen, (m, n), dtype))
    if path in ("a8w8", "linear8"):
        m, n, k, dtype = case["m"], case["n"], case["k"], _DTYPES[case["dtype"]]
        x = _normal(gen, (m, k), torch.bfloat16)
        w, w_scale = quantize_tensor_per_channel(_normal(gen, (n, k), torch.bfloat16, k ** -0.5), dtype, axis=1)
        c = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
        if path == "linear8":
            return dict(path=path, x=x, dtype=dtype, w=w.T, w_scale=w_scale, c=c)
        a, a_scale = quantize_tensor_per_channel(x, dtype, axis=1)
        selector = tb.OrigamiMatmulSelector(m, n, k, dtype, dtype, c.dtype, a.device, streamk=case["streamk"])
        return dict(path=path, a=a, a_scale=a_scale, w=w.T, w_scale=w_scale, c=c, selector=selector, config=tb.matmul_preamble(selector),
                    streamk=case["streamk"])
    if path == "moe":
        rows, experts, n, k = case["rows"], case["experts"], case["n"], case["k"]
        a, a_scale = quantize_tensor_per_channel(_normal(gen, (rows, k), torch.bfloat16), torch.float8_e4m3fn, axis=1)
        w, w_scale = quantize_tensor_per_channel(_normal(gen, (experts, n, k), torch.bfloat16, k ** -0.5), torch.float8_e4m3fn, axis=2)
        routed = torch.randint(0, experts, (rows,), device="cuda", generator=gen)
        offsets = torch.zeros(experts + 1, dtype=torch.int32, device="cuda")
        offsets[1:] = torch.bincount(routed, minlength=experts).cumsum(0)
        return dict(path=path, a=a, a_scale=a_scale, w=w, w_scale=w_scale, offsets=offsets, c=torch.empty(rows, n, dtype=torch.bfloat16, device="cuda"))
    m, n, k = case["m"], case["n"], case["k"]
    x = _normal(gen, (m, k), torch.bfloat16)
    x[torch.rand((m, k), device="cuda", dtype=torch.bfloat16, generator=gen) < 1e-3] *= 20     # activations have outliers: the reason for the rotation
    w, w_scale = tb.hadamard_mxfp4_quant(_normal(gen, (n, k), torch.bfloat16, k ** -0.5))
    return dict(path=path, x=x, w=w, w_scale=w_scale, c=torch.empty(m, n, dtype=torch.bfloat16, device="cuda"))


def run(state):
    path = state["path"]
    if path == "gemm":
        return tb.matmul_lt(state["a"], state["b"], state["c"], state["selector"], state["config"])
    if path == "matmul":
        return tb.matmul(state["a"], state["b"])
    if path == "train":
        x, w, bias = state["x"], state["w"], state["bias"]
        y = tb.addmm(bias, x, w.T if state["transposed"] else w)
        return (y,) + torch.autograd.grad(y, (x, w, bias), state["grad"])
    if path == "a8w8":
        return tb.matmul_a8w8_lt(state["a"], state["w"], state["a_scale"], state["w_scale"], state["c"], state["selector"], state["config"],
                                 enable_streamk=state["streamk"])
    if path == "linear8":
        q, scale = quantize_tensor_per_channel(state["x"], state["dtype"], axis=1)
        return tb.matmul_a8w8(q, state["w"], scale, state["w_scale"], state["c"])
    if path == "moe":
        return tb.grouped_matmul_a8w8(state["a"], state["w"], state["a_scale"], state["w_scale"], state["c"], state["offsets"])
    codes, scales = tb.hadamard_mxfp4_quant(state["x"])
    return tb.matmul_fp4(codes, state["w"], state["c"], scales, state["w_scale"])


def work(case):
    n, k = case["n"], case["k"]
    m = case["rows"] if case["path"] == "moe" else case["m"]
    flops = 2.0 * m * n * k
    if case["path"] in ("gemm", "matmul"):
        size = 4 if case["dtype"] == "float32" else 2
        return {"bytes": size * (m * k + k * n + m * n), "flops": flops}
    if case["path"] == "train":
        # forward: x, w, bias -> y; backward: dy, x, w -> dx, dw, dbias
        return {"bytes": 2 * (3 * m * k + 3 * k * n + 2 * m * n + 2 * n), "flops": 3 * flops}
    if case["path"] == "a8w8":
        return {"bytes": m * k + k * n + 2 * m * n + 4 * (m + n), "flops": flops}
    if case["path"] == "linear8":
        return {"bytes": 2 * m * k + k * n + 2 * m * n + 4 * n, "flops": flops}
    if case["path"] == "moe":
        used = min(m, case["experts"])      # experts that can have rows at all
        return {"bytes": m * k + used * (k * n + 4 * n) + 2 * m * n + 4 * (m + case["experts"] + 1), "flops": flops}
    return {"bytes": 2 * m * k + n * k // 2 + n * k // 32 + 2 * m * n, "flops": flops}


def tolerance(case):
    """About four times the distance from the same product in 64 bits: the rounding of the result to its type (in the 2-norm bf16 1.66e-3,
    fp16 2.1e-4), and in single precision the rounding of the sums, which grows with the root of their length (k = 1024: 5.7e-7,
    2048: 8.1e-7, 4096: 1.15e-6)."""
    if case["path"] in ("gemm", "matmul", "train"):
        return {"rel": {"bfloat16": 6.6e-3, "float16": 8.3e-4, "float32": 7.2e-8 * math.sqrt(case["k"])}[case["dtype"]]}
    return {"rel": 6.6e-3}


_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _from_mxfp4(codes, scales):
    """The values that packed e2m1 codes and their block scales stand for (scale byte 0 is 2**-127)."""
    values = torch.tensor(_E2M1, dtype=torch.float64, device=codes.device)
    c = codes.long()
    v = values[torch.stack([c & 15, c >> 4], -1).reshape(codes.shape[0], -1)]
    return v * torch.ldexp(torch.ones((), dtype=torch.float64, device=codes.device), scales.long() - 127).repeat_interleave(32, 1)


def _rotate_and_quantise(x):
    """Every 32 values of a row times H32 / sqrt(32) in single precision (butterflies of stride 1, 2, 4, 8, 16), their scale the power of two
    two below the largest one's, a mantissa of 1.75 and above rounded up; values to the nearest e2m1, ties away from zero."""
    y = x.float().reshape(-1, 32)
    for h in (1, 2, 4, 8, 16):
        y = y.reshape(-1, 16 // h, 2, h)
        y = torch.stack([y[:, :, 0] + y[:, :, 1], y[:, :, 0] - y[:, :, 1]], 2)
    y = y.reshape(-1, 32) * torch.tensor(0x3E3504F3, dtype=torch.int32, device=x.device).view(torch.float32)
    top = ((y.abs().amax(1).view(torch.int32) + 0x200000) >> 23) - 129
    scale = torch.ldexp(torch.ones((), dtype=torch.float64, device=x.device), top.clamp(-127, 127).unsqueeze(1))
    q = y.double() / scale
    mag, steps = q.abs(), torch.tensor((0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0), dtype=torch.float64, device=x.device)
    v = torch.tensor(_E2M1[:8], dtype=torch.float64, device=x.device)[torch.bucketize(mag, steps, right=True)]
    return (torch.copysign(v, q) * scale).reshape(x.shape)


def exact(case, seed):
    """The outputs of run() from plain torch operations in 64 bits.  Operands that the path rounds to 8 or 4 bits are rounded in the same
    way first: what is measured is the product's own error."""
    s, path = prepare(case, seed), case["path"]
    if path in ("gemm", "matmul"):
        return s["a"].double() @ s["b"].double()
    if path == "train":
        x, w, bias, g = (s[name].detach().double() for name in ("x", "w", "bias", "grad"))
        kn = w.T if s["transposed"] else w
        dw = x.T @ g
        return x @ kn + bias, g @ kn.T, dw.T if s["transposed"] else dw, g.sum(0)
    if path in ("a8w8", "linear8"):
        if path == "a8w8":
            q, scale = s["a"], s["a_scale"]
        else:
            x = s["x"].float()
            top = 127.0 if s["dtype"] == torch.int8 else torch.finfo(s["dtype"]).max
            scale = x.abs().amax(1).clamp(min=1e-8) / top
            q = x * (1.0 / scale).unsqueeze(1)
            q = (q.round().clamp(-top, top) if s["dtype"] == torch.int8 else q).to(s["dtype"])
        return (q.double() @ s["w"].double()) * scale.double().reshape(-1, 1) * s["w_scale"].double().reshape(1, -1)
    if path == "moe":
        at = s["offsets"].tolist()
        parts = [(s["a"][lo:hi].double() @ s["w"][e].double().T) * s["w_scale"][e].double().reshape(1, -1) for e, (lo, hi) in enumerate(zip(at, at[1:]))]
        return torch.cat(parts) * s["a_scale"].double().reshape(-1, 1)
    return _rotate_and_quantise(s["x"]) @ _from_mxfp4(s["w"], s["w_scale"]).T
