"""The tiled GEMMs' K loops at every number of steps: the loop entered or not,
each length of its remainder, every element of the result.

Integer weights (a power of two times -127..127, every row holding a 127: the
scale is that power of two) and small integer activations: every product sum
is exact in fp32 in any order, so single matrices must match the 64-bit result
exactly, and the SwiGLU pair up to its silu and one rounding.
"""

from __future__ import annotations

import pytest
import torch

from pageserve_amd import _native
from pageserve_amd import quantization as Q

pytestmark = pytest.mark.gpu


def _integers(gpu, gen, n, k, scale=1.0):
    w = torch.randint(-127, 128, (n, k), generator=gen, device=gpu).float()
    w[:, 0] = 127.0
    return w * scale


def _check(gpu, plan, pair, m, n, k, f32):
    gen = torch.Generator(device=gpu).manual_seed(m * 131 + n + k)
    x = torch.randint(-4, 5, (m, k), generator=gen, device=gpu).double()
    xb = x.to(torch.bfloat16)
    if pair:
        g, u = (_integers(gpu, gen, n, k, 2.0**-11) for _ in "gu")
        y = Q.swiglu(xb, Q.QuantizedWeight(g), Q.QuantizedWeight(u))
        gd, ud = x @ g.double().T, x @ u.double().T
        ref = torch.nn.functional.silu(gd) * ud
        # one bf16 rounding (2^-9) and the fp32 silu, a few 2^-23
        ok = torch.allclose(y.double(), ref, rtol=2.0**-8, atol=1e-6)
    else:
        w = _integers(gpu, gen, n, k)
        y = Q.linear(xb, Q.QuantizedWeight(w), out_dtype=torch.float32 if f32 else torch.bfloat16)
        ref = x @ w.double().T
        ok = torch.equal(y, ref.to(y.dtype))
    assert plan in _native.last_plan(), _native.last_plan()
    assert ok, (k // 64, int((y.double() - ref).abs().gt(2.0**-8 * ref.abs() + 1e-6).sum()))


CASES = [
    # unrolled by 3: the pair in 128-token tiles, lm_head's 128 x 128, 64 x 128
    ("gemm_dma", "BM = 128, BN = 64, NMAT = 2", True, 250, 200, range(1, 9)),
    ("gemm_dma", "BM = 128, BN = 128, NMAT = 1", False, 256, 131072, range(1, 7)),
    ("gemm_dma", "BM = 64, BN = 128, NMAT = 1", False, 1100, 3700, range(1, 9)),
    # unrolled by 4: the pair in 64-token tiles
    ("gemm_dma", "BM = 64, BN = 64, NMAT = 2", True, 160, 200, range(1, 11)),
    # two K groups: even and odd numbers of steps, 33 .. 36 in a group
    ("gemm_dma", "KG = 2", False, 1800, 2000, range(65, 72)),
    # the pipelined pair, unrolled by 5
    ("gemm_pipe", "BM = 64, BN = 64, NMAT = 2", True, 100, 200, range(1, 12)),
    ("gemm_pipe", "BM = 96, BN = 64, NMAT = 2", True, 90, 8200, range(1, 12)),
    ("gemm_pipe", "BM = 128, BN = 64, NMAT = 2", True, 128, 8200, range(1, 12)),
    # the pipelined 64 x 128 tile, unrolled by 12 (each count in both output
    # types), and its two K groups (17 .. 28 steps in a group)
    ("gemm_pipe", "KG = 1", False, 1024, 1600, [kb for kb in range(1, 26) for _ in "ab"]),
    ("gemm_pipe", "KG = 2", False, 1024, 1600, range(33, 57)),
]


@pytest.mark.parametrize("kernel,plan,pair,m,n,steps", CASES, ids=[f"{c[0]} {c[1]}" for c in CASES])
def test_every_remainder_of_the_k_loop(gpu, kernel, plan, pair, m, n, steps):
    for i, kb in enumerate(steps):
        print(plan, "K steps", kb, flush=True)
        _check(gpu, plan, pair, m, n, 64 * kb, f32=i % 2 == 1)
        assert f"launch_{kernel[5:]}" in _native.last_plan()
