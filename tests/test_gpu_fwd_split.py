"""GPU parity of the 16-bit forward with one tile per workgroup (fwd_split_kernel): shapes for which
1, 2 or 4 waves share a tile's keys, with one or two heads per wave and one or more row tiles per
workgroup, ragged lengths, windows and sink keys that leave some of the sharing waves without an
allowed key, against the float32 oracle with the bar of tests/test_gpu_parity.py; and packed batches.
"""
import math

import pytest
import torch

from conftest import load_mod
from oracle import naive
from test_gpu_parity import assert_close, make_inputs

pytestmark = pytest.mark.gpu

BF, FP = torch.bfloat16, torch.float16

# (B, Hq, Hkv, L, D, W, S, dtype)
CASES = [
    # four waves per tile
    pytest.param(1, 8, 1, 1, 64, 1, 0, BF, id="4w-one-row"),
    pytest.param(1, 8, 1, 33, 64, 33, 0, BF, id="4w-two-halves"),
    pytest.param(1, 16, 2, 257, 64, 257, 0, BF, id="4w-D64-G8"),
    pytest.param(2, 6, 2, 500, 64, 500, 0, FP, id="4w-D64-G3"),
    pytest.param(1, 4, 4, 700, 64, 650, 5, BF, id="4w-D64-G1-sinks"),
    pytest.param(1, 16, 2, 600, 64, 190, 70, BF, id="4w-three-sink-halves"),
    pytest.param(1, 4, 1, 300, 64, 0, 40, BF, id="4w-sinks-only"),
    pytest.param(1, 6, 6, 511, 16, 511, 0, FP, id="4w-D16-one-head"),
    pytest.param(1, 8, 4, 333, 16, 100, 3, BF, id="4w-D16-two-heads"),
    pytest.param(1, 8, 8, 450, 32, 450, 0, BF, id="4w-D32-one-head"),
    pytest.param(1, 16, 1, 640, 32, 300, 4, FP, id="4w-D32-two-heads"),
    # two waves per tile
    pytest.param(1, 64, 8, 1055, 64, 1055, 0, BF, id="2w-D64-G8"),
    pytest.param(1, 16, 16, 2050, 64, 2050, 0, BF, id="2w-D64-G1-two-row-tiles"),
    pytest.param(1, 32, 8, 1000, 128, 1000, 0, BF, id="2w-D128-G4"),
    pytest.param(1, 4, 2, 200, 128, 70, 3, FP, id="2w-D128-G2"),
    pytest.param(4, 16, 16, 3001, 16, 3001, 0, FP, id="2w-D16-two-row-tiles"),
    # one wave per tile
    pytest.param(4, 64, 8, 1023, 64, 1023, 0, BF, id="1w-D64-G8"),
    pytest.param(2, 64, 8, 1500, 64, 300, 4, BF, id="1w-D64-G8-window"),
    pytest.param(8, 16, 16, 1100, 64, 256, 20, BF, id="1w-D64-G1-four-row-tiles"),
    pytest.param(4, 32, 8, 1111, 64, 200, 0, FP, id="1w-D64-G4-two-row-tiles"),
    pytest.param(8, 32, 4, 700, 128, 190, 16, FP, id="1w-D128-G8"),
    pytest.param(8, 32, 16, 650, 128, 190, 0, BF, id="1w-D128-G2-two-row-tiles"),
    # long windows in two rounds and more: fwd_kernel
    pytest.param(8, 32, 4, 700, 128, 200, 16, FP, id="rounds-D128-G8"),
    pytest.param(8, 32, 16, 650, 128, 650, 0, BF, id="rounds-D128-G2"),
    pytest.param(8, 16, 1, 1500, 32, 1500, 0, FP, id="1w-D32-G16"),
]


@pytest.mark.parametrize("B,Hq,Hkv,L,D,W,S,dtype", CASES)
def test_fwd_split(gpu, B, Hq, Hkv, L, D, W, S, dtype):
    print(f"case fwd split B={B} Hq={Hq} Hkv={Hkv} L={L} D={D} W={W} S={S} {dtype}", flush=True)
    ops = load_mod("_ops")
    q, k, v, do = make_inputs(B, Hq, Hkv, L, D, dtype, 21)
    sinks = torch.linspace(-2.0, 3.0, Hq).cuda()
    for sc, sk in ((1.0 / math.sqrt(D), None), (-0.7 / math.sqrt(D), sinks)):
        o, lse = ops.forward(q, k, v, W, S, sc, sinks=sk)
        o2, lse2 = ops.forward(q, k, v, W, S, sc, sinks=sk)
        torch.cuda.synchronize()
        assert torch.equal(o, o2) and torch.equal(lse, lse2)  # deterministic
        if sk is None:
            ref = naive.attention_fwd_bwd(q, k, v, do, W, S, scale=sc, compute_dtype=torch.float32, row_chunk=512)
        else:
            ref = naive.attention_fwd_bwd_sinks(q, k, v, sk, do, W, S, scale=sc, compute_dtype=torch.float32,
                                                row_chunk=512)
        assert_close("O", o, ref[0])
        assert_close("LSE", lse, ref[1])


@pytest.mark.parametrize("Hq,Hkv,D,W", [(8, 1, 64, 900), (16, 2, 64, 200), (4, 4, 64, 900), (8, 2, 128, 900), (6, 2, 32, 900)])
def test_fwd_split_packed(gpu, Hq, Hkv, D, W):
    """Sequences of very different lengths, empty and one-row ones among them."""
    ops = load_mod("_ops")
    cu = [0, 65, 65, 966, 967, 1300]
    total = 1300
    print(f"case fwd split packed Hq={Hq} Hkv={Hkv} D={D} W={W}", flush=True)
    g = torch.Generator().manual_seed(9)
    mk = lambda H: torch.randn(total, H, D, generator=g).bfloat16().cuda()
    q, k, v, do = mk(Hq), mk(Hkv), mk(Hkv), mk(Hq)
    cu_dev = torch.tensor(cu, dtype=torch.int32, device="cuda")
    sc = 1.0 / math.sqrt(D)
    o, lse = ops.forward_varlen(q, k, v, cu_dev, 901, W, 2, sc)
    torch.cuda.synchronize()
    ref = naive.attention_fwd_bwd_varlen(q, k, v, do, torch.tensor(cu), W, 2, sc, compute_dtype=torch.float32,
                                         row_chunk=512)
    assert_close("O", o, ref[0])
    assert_close("LSE", lse, ref[1])
