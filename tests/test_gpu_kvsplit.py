"""GPU parity of the dK/dV kernel split into pieces (bwd_dkdv_kernel with SPLIT and
bwd_dkdv_fold_kernel), at every number of pieces that the workspace allows, against the float32
oracle with the bar of tests/test_gpu_parity.py, and against the unsplit kernel.

A split run adds the same fp32 products in another order, then rounds once to 16 bits, as the unsplit
kernel does.  So the two differ by at most one rounding of the result (2^-8 of it in bfloat16, 2^-11
in float16) plus the fp32 sums' reordering, below 2^-16 of the largest term: |split - unsplit| <=
2 u |unsplit| + 2^-12 rms with u the unit roundoff is checked, four times that second part.
"""
import math

import pytest
import torch

from conftest import load_mod
from oracle import naive
from test_gpu_parity import assert_close, make_inputs, naive_reference, sink_rows

pytestmark = pytest.mark.gpu

BF, FP = torch.bfloat16, torch.float16

# (B, Hq, Hkv, L, D, W, S, dtype, pieces the full workspace gives)
CASES = [
    pytest.param(1, 16, 2, 1001, 64, 1001, 0, BF, 16, id="D64-G8-odd"),
    pytest.param(1, 8, 1, 1537, 64, 1537, 0, FP, 16, id="D64-one-group"),
    pytest.param(2, 6, 2, 700, 64, 650, 4, BF, 8, id="D64-G3-window-dq-sinks"),
    pytest.param(1, 8, 2, 1300, 64, 860, 40, BF, 8, id="D64-G4-chunked-sinks"),
    pytest.param(1, 4, 2, 1300, 64, 600, 70, FP, 4, id="D64-two-sink-blocks"),
    pytest.param(1, 8, 2, 577, 128, 577, 0, BF, 8, id="D128-G4"),
    pytest.param(2, 4, 1, 800, 128, 300, 16, FP, 8, id="D128-window-dq-sinks"),
    pytest.param(1, 4, 1, 1100, 32, 1100, 3, BF, 16, id="D32-sinks-in-window"),
    pytest.param(3, 3, 1, 650, 16, 650, 0, FP, 8, id="D16-G3"),
]


def full_bytes(L, *shape, dtype, total=-1):
    code = load_mod("_ops")._DTYPES[dtype]
    return int(L.fa_bwd_full_workspace_bytes(*shape, code, total))


@pytest.mark.parametrize("B,Hq,Hkv,L,D,W,S,dtype,pieces", CASES)
def test_split_dkdv(gpu, B, Hq, Hkv, L, D, W, S, dtype, pieces):
    print(f"case split B={B} Hq={Hq} Hkv={Hkv} L={L} D={D} W={W} S={S} {dtype}", flush=True)
    ops, lib = load_mod("_ops"), load_mod("_lib").lib()
    q, k, v, do = make_inputs(B, Hq, Hkv, L, D, dtype, 11)
    sc = 1.0 / math.sqrt(D)
    o, lse = ops.forward(q, k, v, W, S, sc)
    base = int(lib.fa_bwd_workspace_bytes(B, Hq, Hkv, L, D, W, S))
    full = full_bytes(lib, B, Hq, Hkv, L, D, W, S, dtype=dtype)
    per_piece = B * Hkv * ((L + 63) // 64) * 2 * 64 * max(D, 32) * 4
    assert full - base == pieces * per_piece  # the plan's number of pieces
    ref = naive.attention_fwd_bwd(q, k, v, do, W, S, scale=sc, compute_dtype=torch.float32, row_chunk=2048)
    nv = naive_reference(q, k, v, do, W, S, sc) if S > 0 else (None,) * 4
    call = ops.BwdCall(q, k, v, o, lse, do, W, S, sc)
    call.ws = torch.full((base,), 0xFF, dtype=torch.uint8, device="cuda")  # no room: unsplit
    call.run()
    dq0, dk0, dv0 = call.dq.clone(), call.dk.clone(), call.dv.clone()
    u = 2.0 ** -8 if dtype == BF else 2.0 ** -11
    ns = 2
    while ns <= pieces:
        call.ws = torch.full((base + ns * per_piece,), 0xFF, dtype=torch.uint8, device="cuda")
        runs = []
        for _ in range(2):
            for t in (call.dq, call.dk, call.dv):
                t.fill_(float("nan"))
            call.run()
            runs.append([t.clone() for t in (call.dq, call.dk, call.dv)])
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(*runs))  # deterministic
        dq, dk, dv = runs[0]
        assert torch.equal(dq, dq0)
        assert_close(f"dK in {ns}", dk, ref[3], nv[2], sink_rows(L, S))
        assert_close(f"dV in {ns}", dv, ref[4], nv[3], sink_rows(L, S))
        for name, x, y in (("dK", dk, dk0), ("dV", dv, dv0)):
            x, y = x.double(), y.double()
            bar = 2 * u * y.abs() + 2.0 ** -12 * y.square().mean().sqrt()
            assert bool(((x - y).abs() <= bar).all()), f"{name} in {ns} pieces is off the unsplit kernel's"
        ns *= 2


@pytest.mark.parametrize("D,dtype", [(64, BF), (128, FP)])
def test_split_dkdv_packed(gpu, D, dtype):
    """A packed batch (key blocks handed out over the sequences; empty and one-row sequences, rows
    outside every sequence) split as far as its workspace allows, against the unsplit run."""
    ops, lib = load_mod("_ops"), load_mod("_lib").lib()
    print(f"case split packed D={D} {dtype}", flush=True)
    cu = [0, 700, 700, 701, 1530, 1601]
    total, Hq, Hkv, W, S = 1640, 8, 2, 829, 4
    B, max_len = len(cu) - 1, 829
    g = torch.Generator().manual_seed(3)
    mk = lambda H: torch.randn(total, H, D, generator=g).to(dtype).cuda()
    q, k, v, do = mk(Hq), mk(Hkv), mk(Hkv), mk(Hq)
    cu_dev = torch.tensor(cu, dtype=torch.int32, device="cuda")
    sc = 1.0 / math.sqrt(D)
    o, lse = ops.forward_varlen(q, k, v, cu_dev, max_len, W, S, sc)
    base = int(lib.fa_bwd_workspace_bytes(B, Hq, Hkv, max_len, D, W, S))
    full = full_bytes(lib, B, Hq, Hkv, max_len, D, W, S, dtype=dtype, total=total)
    assert full > base
    split = ops.backward_varlen(q, k, v, o, lse, do, cu_dev, max_len, W, S, sc)
    real, ops.workspace_bytes = ops.workspace_bytes, lambda *a: base
    try:
        whole = ops.backward_varlen(q, k, v, o, lse, do, cu_dev, max_len, W, S, sc)
    finally:
        ops.workspace_bytes = real
    torch.cuda.synchronize()
    assert torch.equal(split[0], whole[0])
    u = 2.0 ** -8 if dtype == BF else 2.0 ** -11
    for x, y in zip(split[1:], whole[1:]):
        x, y = x.double(), y.double()
        assert bool(((x - y).abs() <= 2 * u * y.abs() + 2.0 ** -12 * y.square().mean().sqrt()).all())
        assert bool((x[1601:] == 0).all())
