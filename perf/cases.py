"""The work that a user of this package has it do, as cases to time: products through the BLAS-level entry
``mul_``, configured launches through ``matmul`` / ``plan`` and contractions through ``contract``, over the sizes,
element types, transposes and options of the package's own tests and benchmark.

``listed()`` names the cases, ``draw`` gives others of the same ranges, ``prepare`` makes what a program has in hand
before the call (inputs on the device, the configuration, a plan where a program would keep one), ``run`` is one pass.
"""
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "gemmkernels.jl_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import gemmkernels as gk  # noqa: E402
from gemmkernels import Epilogue, Float16, Float32, Kernel, Transform, configs  # noqa: E402

# element types of a product: (A and B, C and D)
TYPES = {"f16_f32": (torch.float16, torch.float32), "bf16_f32": (torch.bfloat16, torch.float32),
         "f16_f16": (torch.float16, torch.float16), "f32_f32": (torch.float32, torch.float32),
         "f64_f64": (torch.float64, torch.float64)}


def _mul(name, types, M, N, K, ta, tb, alpha, beta):
    return dict(name=name, kind="mul", types=types, M=M, N=N, K=K, ta=ta, tb=tb, alpha=alpha, beta=beta)


def listed():
    return [
        # mul!(C, A, B) on small Float32 matrices, as a program calls it in a loop: the time is launch and host latency
        _mul("mul_f32_256", "f32_f32", 256, 256, 256, False, False, 1.0, 0.0),
        # single precision at full size: scientific codes that do not give up bits
        _mul("mul_f32_4096", "f32_f32", 4096, 4096, 4096, False, False, 1.0, 0.0),
        # double precision at a size that is no multiple of a tile, transposed, with both factors (BLAS's dgemm)
        _mul("mul_f64_1000_tn", "f64_f64", 1000, 1000, 1000, True, False, 1.5, 0.5),
        # half precision in and out at a middle size: a layer of a network (activations times transposed weights)
        _mul("mul_f16_f16_2048_nt", "f16_f16", 2048, 2048, 2048, False, True, 1.0, 0.0),
        # odd extents and odd leading dimensions throughout: no column starts on a 16-byte boundary
        _mul("mul_bf16_odd_4000_tn", "bf16_f32", 4001, 4003, 4005, True, False, 1.0, 0.0),
        # a tall matrix times a few columns, C updated: decoding a batch of 64 with one weight matrix
        _mul("mul_f16_skinny", "f16_f32", 4096, 64, 4096, False, False, 1.0, 1.0),
        # the largest product of the benchmark's sweep, C read and accumulated
        _mul("mul_f16_16384", "f16_f32", 16384, 16384, 4096, False, False, 1.0, 1.0),
        # the headline: C = A B + C at 4096^3, launched from a plan a program keeps
        dict(name="plan_f16_4096", kind="plan", M=4096, N=4096, K=4096, ta=False, tb=False, c=True, fused=False),
        # a layer with its activation: D = relu((A / 2) B + bias)
        dict(name="fused_4096", kind="plan", M=4096, N=4096, K=2048, ta=False, tb=False, c=False, fused=True),
        # complex numbers, interleaved in memory
        dict(name="complex_2048", kind="complex", M=2048, N=2048, K=2048, ta=False, tb=False, c=False, planar=False),
        # the rows of a matrix scaled: D = diag(a) B
        dict(name="diagonal_4096", kind="diagonal", M=4096, N=4096, c=False),
        # a tensor contraction D[a,b,c,d] = sum_ef A[a,e,b,f] B[d,f,c,e]
        dict(name="contraction_64", kind="contraction", a=64, b=64, c=64, d=64, e=64, f=64),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _extent(rng, lo, hi):
    """An extent between lo and hi: whole tiles, vectors of 8 or any number, odd ones among them."""
    x = _log_uniform(rng, lo, hi)
    step = rng.choice((1, 1, 8, 64))
    return max(lo, min(hi, x // step * step))


def draw(rng):
    kind = rng.choice(("mul", "mul", "mul", "mul", "mul", "skinny", "plan", "plan", "complex", "diagonal", "contraction"))
    ta, tb = rng.random() < 0.5, rng.random() < 0.5
    if kind in ("mul", "skinny"):
        types = rng.choice(sorted(TYPES)) if kind == "mul" else rng.choice(("f16_f32", "bf16_f32", "f16_f16"))
        # the Float32 and Float64 products cost more per flop: the most work a drawn one may be
        most = {"f32_f32": 1.3e11, "f64_f64": 3.4e10}.get(types, 1.0e12)
        while True:
            if kind == "mul":
                M, N, K = (_extent(rng, 16, 8192) for _ in range(3))
            else:
                M, N, K = _extent(rng, 1024, 8192), _extent(rng, 8, 128), _extent(rng, 1024, 8192)
            if 2.0 * M * N * K <= most:
                break
        # (an FP16 C that is accumulated over and over would leave its range)
        alpha, beta = rng.choice(((1.0, 0.0), (1.0, 0.0), (1.5, 0.5)) + (() if types == "f16_f16" else ((1.0, 1.0),)))
        case = _mul("", types, M, N, K, ta, tb, alpha, beta)
    elif kind == "plan":
        M, N, K = (64 * _log_uniform(rng, 4, 96) for _ in range(3))
        case = dict(kind="plan", M=M, N=N, K=K, ta=ta, tb=tb, c=rng.random() < 0.5, fused=rng.random() < 0.4)
    elif kind == "complex":
        M, N, K = (64 * _log_uniform(rng, 2, 40) for _ in range(3))
        case = dict(kind="complex", M=M, N=N, K=K, ta=ta, tb=tb, c=rng.random() < 0.3, planar=rng.random() < 0.5)
    elif kind == "diagonal":
        case = dict(kind="diagonal", M=64 * _log_uniform(rng, 4, 128), N=64 * _log_uniform(rng, 4, 128), c=rng.random() < 0.5)
    else:
        case = dict(kind="contraction", a=rng.choice((32, 64)), b=2 * rng.randint(2, 32), c=2 * rng.randint(2, 32),
                    d=rng.choice((32, 64)), e=rng.choice((32, 64)), f=rng.choice((32, 64)))
    case.pop("name", None)
    return case


def _uniform(gen, shape, dtype, lo=-1.0):
    """A column-major device tensor of the logical shape, values uniform in [lo, 1)."""
    flat = torch.rand(tuple(reversed(shape)), generator=gen, device="cuda", dtype=torch.float64 if dtype is torch.float64 else torch.float32)
    flat = (flat * (1.0 - lo) + lo).to(dtype)
    return flat.permute(*reversed(range(len(shape))))


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind = case["kind"]
    if kind == "contraction":
        e = case
        a = _uniform(gen, (e["a"], e["e"], e["b"], e["f"]), torch.float16)
        b = _uniform(gen, (e["d"], e["f"], e["c"], e["e"]), torch.float16)
        d = gk.colmajor_empty((e["a"], e["b"], e["c"], e["d"]), torch.float32)
        return dict(kind=kind, a=a, b=b, d=d)
    if kind == "diagonal":
        M, N = case["M"], case["N"]
        a = torch.rand(M, generator=gen, device="cuda").mul_(2).sub_(1).to(torch.float16)
        b = _uniform(gen, (M, N), torch.float16)
        c = _uniform(gen, (M, N), torch.float32) if case["c"] else None
        d = gk.colmajor_empty((M, N), torch.float32)
        conf = configs.diagonal_config(M, N, zero_c=c is None)
        return dict(kind="matmul", conf=conf, a=a, b=b, c=c, d=d, kernel=Kernel.matmul_singlestage)
    M, N, K, ta, tb = case["M"], case["N"], case["K"], case["ta"], case["tb"]
    sa, sb = (K, M) if ta else (M, K), (N, K) if tb else (K, N)
    if kind == "complex":
        shape = (lambda s: s + (2,)) if case["planar"] else (lambda s: (2,) + s)
        a, b = _uniform(gen, shape(sa), torch.float16), _uniform(gen, shape(sb), torch.float16)
        c = _uniform(gen, shape((M, N)), torch.float32) if case["c"] else None
        d = gk.colmajor_empty(shape((M, N)), torch.float32)
        make = configs.complex_planar_config if case["planar"] else configs.complex_config
        return dict(kind="matmul", conf=make(M, N, K, ta, tb, zero_c=c is None), a=a, b=b, c=c, d=d, kernel=Kernel.matmul_pipelined)
    if kind == "mul":
        ab, cd = TYPES[case["types"]]
        lo = 0.0 if case["types"] == "f32_f32" else -1.0          # (Float32 as in the benchmark's small product)
        a, b, c = _uniform(gen, sa, ab, lo), _uniform(gen, sb, ab, lo), _uniform(gen, (M, N), cd)
        return dict(kind=kind, a=gk.Transpose(a) if ta else a, b=gk.Transpose(b) if tb else b, c=c, alpha=case["alpha"], beta=case["beta"])
    # a configured real product on aligned layouts, kept as a plan
    a, b = _uniform(gen, sa, torch.float16), _uniform(gen, sb, torch.float16)
    c = _uniform(gen, (M, N), torch.float32) if case["c"] else None
    d = gk.colmajor_empty((M, N), torch.float32)
    conf = configs.mfma_config(M, N, K, ta, tb, zero_c=c is None)
    options = {}
    if case["fused"]:
        bias = torch.randn(N, generator=gen, device="cuda")
        options = dict(transform_global_to_shared_a=Transform.Elementwise(lambda x: x * 0.5),
                       transform_shared_to_global_d=Transform.Elementwise(Transform.relu), epilogue=Epilogue.Bias(bias))
    return dict(kind=kind, plan=gk.plan(conf, a, b, c, d, kernel=Kernel.matmul_pipelined, **options))


def run(state):
    kind = state["kind"]
    if kind == "mul":
        return gk.mul_(state["c"], state["a"], state["b"], state["alpha"], state["beta"])
    if kind == "plan":
        return state["plan"]()
    if kind == "contraction":
        return gk.contract("abcd-aebf-dfce", state["a"], state["b"], state["d"])
    return gk.matmul(state["conf"], state["a"], state["b"], state["c"], state["d"], kernel=state["kernel"])


def work(case):
    kind = case["kind"]
    if kind == "contraction":
        M, N, K = case["a"] * case["b"], case["c"] * case["d"], case["e"] * case["f"]
        return {"bytes": 2 * (M * K + K * N) + 4 * M * N, "flops": 2 * M * N * K}
    if kind == "diagonal":
        M, N = case["M"], case["N"]
        return {"bytes": 2 * M + 2 * M * N + 4 * M * N * (2 if case["c"] else 1), "flops": M * N * (2 if case["c"] else 1)}
    M, N, K = case["M"], case["N"], case["K"]
    if kind == "complex":
        return {"bytes": 4 * (M * K + K * N) + 8 * M * N * (2 if case["c"] else 1), "flops": 8 * M * N * K}
    if kind == "mul":
        ab, cd = (torch.empty(0, dtype=t).element_size() for t in TYPES[case["types"]])
        return {"bytes": ab * (M * K + K * N) + cd * M * N * (1 if case["beta"] == 0.0 else 2), "flops": 2 * M * N * K}
    bias = 4 * N if case["fused"] else 0
    return {"bytes": 2 * (M * K + K * N) + 4 * M * N * (2 if case["c"] else 1) + bias, "flops": 2 * M * N * K}


def tolerance(case):
    kind = case["kind"]
    if kind == "diagonal":
        return "exact"                      # one product of two FP16 numbers, exact in FP32, and at most one rounded addition
    # four times what the path differs by from the same products summed in 64 bits
    types = case.get("types", "f16_f32")
    if types == "f64_f64":
        return {"rel": 1e-14, "max": 1e-13}
    if types == "f16_f16":
        return {"rel": 1e-3, "max": 5e-3}   # sums in FP32, one rounding to FP16 at the store
    if types == "f32_f32":
        return {"rel": 5e-6, "max": 5e-5}   # one FP32 fma chain per output
    if case.get("alpha", 1.0) == 1.5:       # A times alpha is rounded to A's 16-bit type
        return {"rel": 1e-3, "max": 5e-3} if types == "f16_f32" else {"rel": 8e-3, "max": 4e-2}
    return {"rel": 3e-6, "max": 3e-5}       # sums in FP32 of exact products
