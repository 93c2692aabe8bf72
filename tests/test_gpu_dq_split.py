"""GPU parity of dQ with one tile per workgroup (bwd_dq_split_kernel): shapes for which 1, 2 or 4 waves
share a tile's keys, one or more row tiles per workgroup, ragged lengths, windows and sink keys whose
gradients the dK/dV kernel takes, against the float32 oracle with the bar of tests/test_gpu_parity.py.
dK, dV (which read this kernel's row statistics; the sink keys' rows, which chunk workgroups add up, with that
file's wider bar) and the learned sinks' gradient are checked too.
"""
import math

import pytest
import torch

from conftest import load_mod
from oracle import naive
from test_gpu_parity import assert_close, make_inputs, naive_reference, sink_rows
from test_gpu_sinks import check_dsinks

pytestmark = pytest.mark.gpu

BF, FP = torch.bfloat16, torch.float16

# (B, Hq, Hkv, L, D, W, S, dtype)
CASES = [
    pytest.param(1, 8, 1, 1, 64, 1, 0, BF, id="one-row"),
    pytest.param(1, 8, 1, 1500, 64, 1500, 0, BF, id="4w-D64-G8"),
    pytest.param(1, 3, 1, 333, 64, 333, 0, FP, id="D64-G3"),
    pytest.param(1, 64, 8, 290, 64, 290, 0, BF, id="2w-D64-G8"),
    pytest.param(1, 16, 16, 2050, 64, 2050, 0, BF, id="D64-G1-row-tiles"),
    pytest.param(1, 16, 2, 600, 64, 190, 70, BF, id="D64-chunked-sinks"),
    pytest.param(1, 4, 4, 100, 64, 90, 8, FP, id="D64-sinks-in-window"),
    pytest.param(4, 64, 8, 1023, 64, 1023, 0, BF, id="1w-D64-G8"),
    pytest.param(8, 16, 16, 1100, 64, 256, 0, BF, id="1w-D64-G1-row-tiles"),
    pytest.param(1, 32, 8, 700, 128, 700, 0, BF, id="2w-D128-G4"),
    pytest.param(1, 3, 3, 257, 128, 60, 0, FP, id="2w-D128-G1"),
    pytest.param(8, 32, 4, 700, 128, 200, 0, FP, id="1w-D128-G8"),
    pytest.param(8, 16, 16, 400, 128, 400, 0, BF, id="1w-D128-G1-row-tiles"),
    # few sink keys whose gradients the dK/dV kernel's chunks take at these windows
    pytest.param(1, 8, 2, 385, 128, 256, 16, BF, id="D128-sinks-in-chunks"),
    pytest.param(2, 6, 2, 1153, 128, 300, 3, FP, id="D128-G3-sinks-in-chunks"),
    pytest.param(1, 4, 1, 1090, 64, 1024, 1, BF, id="D64-G4-one-ragged-chunk"),
    pytest.param(1, 16, 2, 2500, 64, 1100, 16, FP, id="D64-G8-sinks-in-chunks"),
    pytest.param(2, 8, 1, 1200, 64, 1024, 5, BF, id="D64-G8-two-chunks"),
    pytest.param(1, 6, 6, 511, 16, 511, 0, FP, id="4w-D16"),
    pytest.param(4, 16, 16, 3001, 16, 3001, 0, FP, id="D16-row-tiles"),
    pytest.param(1, 16, 1, 900, 32, 900, 0, BF, id="4w-D32"),
    pytest.param(8, 16, 1, 1500, 32, 1500, 0, FP, id="1w-D32"),
]


@pytest.mark.parametrize("B,Hq,Hkv,L,D,W,S,dtype", CASES)
def test_dq_split(gpu, B, Hq, Hkv, L, D, W, S, dtype):
    print(f"case dq split B={B} Hq={Hq} Hkv={Hkv} L={L} D={D} W={W} S={S} {dtype}", flush=True)
    ops = load_mod("_ops")
    q, k, v, do = make_inputs(B, Hq, Hkv, L, D, dtype, 31)
    sinks = torch.linspace(-2.0, 2.0, Hq).cuda()
    for sc, sk in ((1.0 / math.sqrt(D), None), (-0.7 / math.sqrt(D), sinks)):
        o, lse = ops.forward(q, k, v, W, S, sc, sinks=sk)
        grads = ops.backward(q, k, v, o, lse, do, W, S, sc, sinks=sk)
        again = ops.backward(q, k, v, o, lse, do, W, S, sc, sinks=sk)
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(grads, again))  # deterministic
        if sk is None:
            ref = naive.attention_fwd_bwd(q, k, v, do, W, S, scale=sc, compute_dtype=torch.float32, row_chunk=512)
        else:
            ref = naive.attention_fwd_bwd_sinks(q, k, v, sk, do, W, S, scale=sc, compute_dtype=torch.float32,
                                                row_chunk=512)
        assert_close("dQ", grads[0], ref[2])
        # the sink keys' rows sum every row's rounded terms, whatever the learned sinks: without those
        nv = naive_reference(q, k, v, do, W, S, sc) if S > 0 and sk is None else (None,) * 4
        keys = slice(0 if sk is None else S, None)
        assert_close("dK", grads[1][:, :, keys], ref[3][:, :, keys], nv[2], sink_rows(L, S))
        assert_close("dV", grads[2][:, :, keys], ref[4][:, :, keys], nv[3], sink_rows(L, S))
        if sk is not None:
            check_dsinks(grads[3], ref[5], ref[1], ref[0], do, sk, range(Hq))
