"""Fused SwiGLU (engine/model.py:188-190) against the oracle.

act = silu(x Wg^T) * (x Wu^T) computed in fp32 and rounded once to bf16;
out = act Wd^T.  The oracle keeps everything in fp32/float64.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import activations, bf16_gpu, report, to_np, weights
from oracle import quantization_oracle as O
from pageserve_amd import quantization as Q

pytestmark = pytest.mark.gpu


def _mlp_weights(gpu, seed, inter, hidden):
    ws = {}
    for j, (name, shape) in enumerate((("gate", (inter, hidden)), ("up", (inter, hidden)),
                                       ("down", (hidden, inter)))):
        w = weights(seed + j, *shape)
        ws[name] = (Q.QuantizedWeight(torch.from_numpy(w).to(gpu)), *O.quantize_per_channel(w))
    return ws


@pytest.mark.parametrize("m,inter,hidden", [(1, 11008, 2048), (4, 11008, 2048), (16, 11008, 2048),
                                            (17, 11008, 2048), (128, 11008, 2048), (512, 11008, 2048),
                                            (3, 100, 48), (40, 300, 208), (20, 64, 16),
                                            (50, 130, 48), (24, 256, 4112),
                                            # 128-token x 64-row tiles: split K, ragged M and N
                                            (100, 256, 4096), (300, 1000, 2048), (65, 64, 64),
                                            (33, 1000, 2048),
                                            # 65..128 tokens: 64-token tiles, LDS-DMA activations
                                            (80, 11008, 2048), (96, 1000, 2112),
                                            # above 128 tokens with a last 128-token tile at most
                                            # half full: 64-token tiles
                                            (160, 11008, 2048), (320, 1000, 2112),
                                            # two token blocks: unsplit, and a long K split into partials
                                            (32, 11008, 2048), (24, 1000, 8192), (21, 300, 1040),
                                            # 14..16 tokens, K <= 2048: three row tiles per workgroup
                                            # (ragged N, tile counts not a multiple of three, a K of
                                            # 17 chunks, a single chunk)
                                            (14, 11008, 2048), (15, 1000, 2048), (16, 130, 1088),
                                            (14, 48, 64), (16, 100, 2048)])
def test_swiglu_matches_oracle(gpu, m, inter, hidden):
    ws = _mlp_weights(gpu, 10 + m + inter, inter, hidden)
    x = activations(m, m, hidden)
    act = Q.swiglu(bf16_gpu(x, gpu), ws["gate"][0], ws["up"][0])
    assert act.dtype == torch.bfloat16 and act.shape == (m, inter)
    ref = O.swiglu(x, ws["gate"][1], ws["gate"][2], ws["up"][1], ws["up"][2])
    acc = O.swiglu_acc(x, ws["gate"][1], ws["gate"][2], ws["up"][1], ws["up"][2])
    report(to_np(act), ref, hidden, f"swiglu m={m}", acc=acc)


@pytest.mark.parametrize("m", [1, 512])
def test_mlp_config(gpu, m):
    """The fused SwiGLU MLP workload: x [m, 2048], gate/up [11008, 2048],
    down [2048, 11008]; out = down(silu(gate(x)) * up(x))."""
    ws = _mlp_weights(gpu, 4000, 11008, 2048)
    x = activations(4100 + m, m, 2048)
    out = Q.mlp(bf16_gpu(x, gpu), ws["gate"][0], ws["up"][0], ws["down"][0])
    ref = O.mlp(x, ws["gate"][1], ws["gate"][2], ws["up"][1], ws["up"][2], ws["down"][1], ws["down"][2])
    report(to_np(out), ref, 11008, f"mlp m={m}", acc=O.mlp_acc(x, ws["gate"][1], ws["gate"][2], ws["up"][1],
                                                              ws["up"][2], ws["down"][1], ws["down"][2]))


def test_swiglu_equals_unfused_composition(gpu):
    """Same as gate and up as separate fp32-output linears, combined in fp32."""
    ws = _mlp_weights(gpu, 77, 1024, 512)
    x = bf16_gpu(activations(3, 8, 512), gpu)
    g = ws["gate"][0].linear(x, out_dtype=torch.float32)
    u = ws["up"][0].linear(x, out_dtype=torch.float32)
    expect = (torch.nn.functional.silu(g) * u).to(torch.bfloat16).float()
    got = Q.swiglu(x, ws["gate"][0], ws["up"][0]).float()
    # same fp32 accumulations; silu rounding may differ by one bf16 ulp
    assert ((got - expect).abs() <= expect.abs() * 2 ** -7 + 1e-6).all()


def test_pair_tiles_plan(gpu):
    """14..16 tokens with K % 64 == 0 and at most 32 chunks run the pair as three
    16-row tiles per workgroup (pair_tiles_kernel); 13 tokens and a 33-chunk K keep
    the one-tile skinny plan.  Every case against the oracle."""
    from pageserve_amd import _native

    for m, inter, hidden, want in ((16, 11008, 2048, True), (14, 1000, 2048, True), (15, 35, 128, True),
                                   (13, 11008, 2048, False), (16, 1000, 2112, False)):
        ws = _mlp_weights(gpu, 900 + m + inter, inter, hidden)
        x = activations(950 + m, m, hidden)
        act = Q.swiglu(bf16_gpu(x, gpu), ws["gate"][0], ws["up"][0])
        plan = _native.last_plan()
        assert ("launch_pair_tiles" in plan) == want, plan
        ref = O.swiglu(x, ws["gate"][1], ws["gate"][2], ws["up"][1], ws["up"][2])
        acc = O.swiglu_acc(x, ws["gate"][1], ws["gate"][2], ws["up"][1], ws["up"][2])
        report(to_np(act), ref, hidden, f"pair tiles m={m} n={inter} k={hidden}", acc=acc)


@pytest.mark.parametrize("m,inter,hidden,tiled", [(17, 4112, 2048, True), (32, 8192, 1024, True), (31, 8208, 1088, True),
                                                  (24, 12288, 64, True), (20, 4096, 512, False),
                                                  (18, 12304, 128, False), (25, 5000, 896, True),
                                                  (20, 11008, 2048, False), (21, 11008, 2048, True),
                                                  (24, 12288, 1600, False), (25, 12288, 1600, True)])
def test_pair_tiles_with_two_token_blocks(gpu, m, inter, hidden, tiled):
    """17..32 tokens at the edges of the two- and three-tile plans (257, 512,
    513 and 768 row tiles; 16 and 17 chunks) and just outside them, a last
    workgroup with missing tiles and a last tile with missing rows, and the
    token counts at which many tiles of a longer K begin."""
    from pageserve_amd import _native

    ws = _mlp_weights(gpu, 700 + m + inter, inter, hidden)
    x = activations(750 + m, m, hidden)
    act = Q.swiglu(bf16_gpu(x, gpu), ws["gate"][0], ws["up"][0])
    assert ("launch_pair_tiles" in _native.last_plan()) == tiled
    ref = O.swiglu(x, *ws["gate"][1:], *ws["up"][1:])
    report(to_np(act), ref, hidden, f"pair tiles m={m} inter={inter} K={hidden}",
           acc=O.swiglu_acc(x, *ws["gate"][1:], *ws["up"][1:]))


@pytest.mark.parametrize("m,inter,hidden,bm", [(65, 11008, 2048, 96), (96, 9000, 1024, 96), (97, 11008, 2048, 128),
                                               (128, 16384, 64, 128), (66, 4864, 896, 64), (127, 8192, 128, 64),
                                               (100, 130, 192, 64)])
def test_pipelined_pair(gpu, m, inter, hidden, bm):
    """65..128 tokens in the three pipelined tile heights: full and ragged
    token tiles, a last tile with missing rows, one to 32 K steps."""
    from pageserve_amd import _native

    ws = _mlp_weights(gpu, 8300 + m + inter, inter, hidden)
    x = activations(8350 + m, m, hidden)
    xt = bf16_gpu(x, gpu)
    act = Q.swiglu(xt, ws["gate"][0], ws["up"][0])
    plan = _native.last_plan()
    assert "launch_pipe" in plan and f"BM = {bm}, BN = 64" in plan, plan
    ref = O.swiglu(x, *ws["gate"][1:], *ws["up"][1:])
    report(to_np(act), ref, hidden, f"pipelined pair m={m} inter={inter} K={hidden}",
           acc=O.swiglu_acc(x, *ws["gate"][1:], *ws["up"][1:]))
    for _ in range(3):
        assert torch.equal(act, Q.swiglu(xt, ws["gate"][0], ws["up"][0]))
