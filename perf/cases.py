"""Performance cases of the GEMM suite: the calls a user's program makes through
``vibekernel_amd.gemm`` and ``vibekernel_amd.matmul``.

Two kinds of call:

* ``"gemm"``: ``gemm(A, B, out_dtype=...)``, which allocates C and picks the
  kernel version for the shape on every call.
* ``"matmul"``: a serving loop.  The program picks the version once for its
  shape, keeps the output buffer, and calls ``matmul`` for every token.

A holds activations (standard normal), B holds weights (normal with variance
1 / k), so outputs are of order one, as in a network's linear layers.
"""
from __future__ import annotations

import torch

import vibekernel_amd as vk

DTYPES = {"f16": torch.float16, "f32": torch.float32}

# The costliest listed products, which bound the drawn ones.
MAX_MACS = {"f16": 4096 * 50257 * 4096, "f32": 4096 * 4096 * 4096}
MAX_WEIGHTS = {"f16": 50257 * 4096, "f32": 8192 * 8192}


def _case(call, m, n, k, dtype="f16", out=None, name=None):
    case = {"call": call, "m": m, "n": n, "k": k, "dtype": dtype, "out": out or dtype}
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # a per-head projection or a small adapter: the call itself is what costs
        _case("gemm", 64, 64, 64, name="f16_tiny_64x64x64"),
        # one token through a 4096-wide square projection of a decoder
        _case("matmul", 1, 4096, 4096, name="f16_decode_1x4096x4096"),
        # a batch of 16 tokens through an 8192-wide projection
        _case("matmul", 16, 8192, 8192, name="f16_decode_16x8192x8192"),
        # the head of a batch of 32 tokens: a vocabulary of 50,257 columns, fp32 logits
        _case("gemm", 32, 50257, 4096, out="f32", name="f16_head_32x50257x4096_f32out"),
        # a short prompt of 300 tokens through an MLP's up projection
        _case("gemm", 300, 11008, 4096, name="f16_prompt_300x11008x4096"),
        # sizes that are multiples of nothing
        _case("gemm", 1000, 1001, 999, name="f16_ragged_1000x1001x999"),
        # the square product that the suite's benchmark is quoted on
        _case("gemm", 4096, 4096, 4096, name="f16_square_4096"),
        # logits of a whole 4096-token sequence over the same vocabulary
        _case("gemm", 4096, 50257, 4096, name="f16_head_4096x50257x4096"),
        # fp32: the harness's default size
        _case("gemm", 512, 512, 512, "f32", name="f32_square_512"),
        # fp32: few rows against a weight matrix
        _case("matmul", 16, 4096, 4096, "f32", name="f32_decode_16x4096x4096"),
        # fp32: sizes that are multiples of nothing
        _case("gemm", 1000, 1001, 999, "f32", name="f32_ragged_1000x1001x999"),
        # fp32: the benchmark's square
        _case("gemm", 4096, 4096, 4096, "f32", name="f32_square_4096"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _dim(rng, lo, hi):
    """A size from lo to hi: half of them multiples of 64, a quarter multiples
    of 8, a quarter anything."""
    x = _log_uniform(rng, lo, hi)
    step = rng.choice((64, 64, 8, 1))
    return max(lo, min(hi, (x + step // 2) // step * step or step))


def draw(rng):
    dtype = rng.choice(("f16", "f16", "f32"))
    out = rng.choice(("f16", "f16", "f32")) if dtype == "f16" else "f32"
    kind = rng.choice(("decode", "prompt", "general"))
    if kind == "decode":
        call = "matmul"
        m, n, k = _log_uniform(rng, 1, 128), _dim(rng, 256, 50257), _dim(rng, 256, 16384)
    elif kind == "prompt":
        call = rng.choice(("gemm", "matmul"))
        m, n, k = _log_uniform(rng, 129, 4096), _dim(rng, 512, 16384), _dim(rng, 512, 16384)
    else:
        call = "gemm"
        m, n, k = _dim(rng, 32, 4096), _dim(rng, 32, 4096), _dim(rng, 32, 4096)
    # no costlier than the largest listed product: fewer columns, then fewer rows
    n = min(n, MAX_WEIGHTS[dtype] // k)
    m = max(1, min(m, MAX_MACS[dtype] // (n * k)))
    return _case(call, m, n, k, dtype, out)


def _operands(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    m, n, k, dt = case["m"], case["n"], case["k"], DTYPES[case["dtype"]]
    A = torch.randn((m, k), generator=gen, device="cuda", dtype=torch.float32).to(dt)
    B = (torch.randn((k, n), generator=gen, device="cuda", dtype=torch.float32) * k ** -0.5).to(dt)
    return A, B


def prepare(case, seed):
    A, B = _operands(case, seed)
    state = {"call": case["call"], "A": A, "B": B, "out_dtype": DTYPES[case["out"]]}
    if case["call"] == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        state["mnk"] = (m, n, k)
        state["C"] = torch.empty((m, n), dtype=DTYPES[case["out"]], device="cuda")
        state["version"] = vk.pick_version(m, n, k, case["dtype"], case["out"])
    return state


def run(state):
    if state["call"] == "gemm":
        return vk.gemm(state["A"], state["B"], out_dtype=state["out_dtype"])
    m, n, k = state["mnk"]
    vk.matmul(m, n, k, state["A"], state["B"], state["C"], state["version"])
    return state["C"]


def work(case):
    m, n, k = case["m"], case["n"], case["k"]
    size = {"f16": 2, "f32": 4}
    return {"bytes": size[case["dtype"]] * (m * k + k * n) + size[case["out"]] * m * n, "flops": 2 * m * n * k}


def tolerance(case):
    # fp16 output: one rounding of the fp32 sum to fp16 (about 2e-4 in the 2-norm,
    # at most a unit in the last place, 2^-10, between two correct roundings).
    if case["out"] == "f16":
        return {"rel": 8e-4, "max": 2e-3}
    # fp32 output: fp32 sums of k products, in any order.
    return {"rel": 1e-5}


def exact(case, seed):
    A, B = _operands(case, seed)
    return A.double() @ B.double()
