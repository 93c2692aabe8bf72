"""GPU parity without a window (W = 0, only the sink keys are seen) where the last row tile of a
sequence holds one row: that row's own key is a sink in a 32-key tile that no window reaches.  Fixed and
packed batches, 16-bit and float32, against the float32 oracle with the bar of tests/test_gpu_parity.py.
"""
import math

import pytest
import torch

from conftest import load_mod
from oracle import naive
from test_gpu_parity import assert_close, make_inputs

pytestmark = pytest.mark.gpu

BF, FP, F32 = torch.bfloat16, torch.float16, torch.float32

CASES = [(L, S, D, G, dtype) for L, S in ((1, 1), (33, 33), (65, 65), (65, 64), (129, 200))
         for D, G, dtype in ((64, 8, BF), (64, 1, FP), (128, 4, BF), (16, 2, FP), (64, 2, F32))]


@pytest.mark.parametrize("L,S,D,G,dtype", CASES)
def test_sinks_only(gpu, L, S, D, G, dtype):
    print(f"case sinks only L={L} S={S} D={D} G={G} {dtype}", flush=True)
    ops = load_mod("_ops")
    q, k, v, do = make_inputs(1, 2 * G, 2, L, D, dtype, 7)
    sc = 1.0 / math.sqrt(D)
    o, lse = ops.forward(q, k, v, 0, S, sc)
    grads = ops.backward(q, k, v, o, lse, do, 0, S, sc)
    torch.cuda.synchronize()
    ref = naive.attention_fwd_bwd(q, k, v, do, 0, S, scale=sc, compute_dtype=torch.float32)
    for name, got, want in zip(("O", "LSE", "dQ", "dK", "dV"), (o, lse, *grads), ref):
        assert_close(name, got, want)


@pytest.mark.parametrize("dtype", [BF, F32])
def test_packed_sequences_of_one_row(gpu, dtype):
    """Each sequence of a packed batch equals the same rows run as a batch of their own."""
    ops = load_mod("_ops")
    lens, Hq, D, S = (1, 40, 33, 1, 65), 8, 64, 70
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], dtype=torch.int32)
    g = torch.Generator().manual_seed(3)
    q, k, v, do = (torch.randn(sum(lens), H, D, generator=g).to(dtype).cuda() for H in (Hq, 2, 2, Hq))
    o, lse = ops.forward_varlen(q, k, v, cu.cuda(), max(lens), 0, S, 0.125)
    grads = ops.backward_varlen(q, k, v, o, lse, do, cu.cuda(), max(lens), 0, S, 0.125)
    torch.cuda.synchronize()
    for b, n in enumerate(lens):
        rows = slice(int(cu[b]), int(cu[b]) + n)
        one = [t[rows].transpose(0, 1).unsqueeze(0).contiguous() for t in (q, k, v, do)]
        ref = naive.attention_fwd_bwd(*one, 0, S, scale=0.125, compute_dtype=torch.float32)
        assert_close("LSE", lse[None, :, rows], ref[1])
        for name, got, want in zip(("O", "dQ", "dK", "dV"), (o, *grads), (ref[0], *ref[2:])):
            assert_close(name, got[rows].transpose(0, 1).unsqueeze(0), want)
