"""GPU parity of the float32 kernels where their tiling can go wrong: workgroups of four row tiles of
one head (G = 1, 3) to four heads, ragged ends of 32-row tiles and 64-key blocks, sink blocks whose
later rows go to chunk workgroups (one half or both halves of the block, two blocks), the dK/dV
kernel in pieces, and packed batches.  Oracle and tolerance are those of tests/test_gpu_fp32.py
(float64, 1e-4 + 1e-4 |ref|).
"""
import math

import pytest
import torch

from conftest import load_mod
from oracle import naive
from test_gpu_fp32 import close, inputs, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,L,D,W,S", [
    pytest.param(1, 3, 3, 127, 64, 127, 0, id="G1-four-row-tiles"),
    pytest.param(1, 3, 1, 129, 32, 70, 3, id="G3-one-row-past"),
    pytest.param(2, 4, 2, 95, 16, 31, 1, id="G2-D16"),
    pytest.param(1, 8, 1, 64, 128, 64, 0, id="one-key-block-D128"),
    pytest.param(1, 4, 1, 513, 64, 33, 32, id="sinks-fill-half-0"),
    pytest.param(1, 4, 1, 513, 64, 33, 33, id="sinks-in-both-halves"),
    pytest.param(1, 2, 1, 900, 32, 64, 96, id="two-sink-blocks"),
    pytest.param(1, 2, 2, 700, 128, 1, 16, id="W1-sinks-D128"),
    pytest.param(1, 2, 1, 450, 16, 0, 20, id="sinks-only-D16"),
    # chunks of at most 16 sink keys: ragged ends, odd numbers of items, every head dim
    pytest.param(1, 3, 1, 369, 64, 77, 1, id="one-sink-G3"),
    pytest.param(2, 8, 1, 500, 64, 128, 16, id="16-sinks-G8"),
    pytest.param(1, 4, 1, 513, 64, 33, 17, id="17-sinks"),
    pytest.param(1, 2, 1, 600, 128, 90, 31, id="31-sinks-D128"),
    pytest.param(1, 3, 3, 333, 16, 40, 15, id="sinks-D16"),
    pytest.param(1, 4, 2, 129, 32, 64, 9, id="one-chunk-D32"),
])
def test_fp32_tiles(gpu, B, Hq, Hkv, L, D, W, S):
    run(B, Hq, Hkv, L, D, W, S, seed=5)


@pytest.mark.parametrize("B,Hq,Hkv,L,D,W,S", [
    pytest.param(1, 4, 1, 321, 64, 321, 0, id="full"),
    pytest.param(1, 3, 1, 300, 16, 300, 0, id="G3-D16"),
    pytest.param(2, 4, 2, 290, 128, 150, 5, id="D128-sinks"),
    pytest.param(1, 4, 2, 400, 32, 200, 70, id="two-sink-blocks-D32"),
])
def test_fp32_pieces(gpu, B, Hq, Hkv, L, D, W, S):
    """Every number of pieces up to the plan's, against float64; dQ does not depend on it."""
    ops, libm = load_mod("_ops"), load_mod("_lib")
    lib = libm.lib()
    print(f"case fp32 pieces B={B} Hq={Hq} Hkv={Hkv} L={L} D={D} W={W} S={S}", flush=True)
    q, k, v, do = inputs(B, Hq, Hkv, L, D, 7)
    sc = 1.0 / math.sqrt(D)
    o, lse = ops.forward(q, k, v, W, S, sc)
    ref = naive.attention_fwd_bwd(q, k, v, do, W, S, scale=sc, compute_dtype=torch.float64, row_chunk=2048)
    base = int(lib.fa_bwd_workspace_bytes(B, Hq, Hkv, L, D, W, S))
    full = int(lib.fa_bwd_full_workspace_bytes(B, Hq, Hkv, L, D, W, S, libm.FA_DTYPE_F32, -1))
    per_piece = B * Hkv * ((L + 63) // 64) * 2 * 64 * max(D, 32) * 4
    assert full > base
    ns = 1
    while base + (ns * per_piece if ns > 1 else 0) <= full:
        call = ops.BwdCall(q, k, v, o, lse, do, W, S, sc)
        call.ws = torch.full((base + (ns * per_piece if ns > 1 else 0),), 0xFF, dtype=torch.uint8, device="cuda")
        for t in (call.dq, call.dk, call.dv):
            t.fill_(float("nan"))
        call.run()
        torch.cuda.synchronize()
        for name, got, r in zip(("dQ", "dK", "dV"), (call.dq, call.dk, call.dv), ref[2:5]):
            close(f"{name} in {ns}", got, r)
        ns *= 2


@pytest.mark.parametrize("W,S", [(600, 0), (40, 3)])
def test_fp32_packed(gpu, W, S):
    """A packed batch with empty and one-row sequences (key blocks handed out over the sequences)."""
    ops = load_mod("_ops")
    cu = [0, 333, 333, 334, 400, 1000]
    total, Hq, Hkv, D = 1000, 4, 2, 64
    print(f"case fp32 packed W={W} S={S}", flush=True)
    g = torch.Generator().manual_seed(2)
    mk = lambda H: torch.randn(total, H, D, generator=g).cuda()
    q, k, v, do = mk(Hq), mk(Hkv), mk(Hkv), mk(Hq)
    cu_dev = torch.tensor(cu, dtype=torch.int32, device="cuda")
    sc = 1.0 / math.sqrt(D)
    o, lse = ops.forward_varlen(q, k, v, cu_dev, 600, W, S, sc)
    grads = ops.backward_varlen(q, k, v, o, lse, do, cu_dev, 600, W, S, sc)
    torch.cuda.synchronize()
    ref = naive.attention_fwd_bwd_varlen(q, k, v, do, torch.tensor(cu), W, S, sc, compute_dtype=torch.float64,
                                         row_chunk=1024)
    close("O", o, ref[0])
    for name, got, r in zip(("dQ", "dK", "dV"), grads, ref[2:5]):
        close(name, got, r)
