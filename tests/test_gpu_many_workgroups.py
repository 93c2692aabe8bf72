"""GPU tests of packed batches whose B x longest-sequence grids exceed the threads of one launch (2^32, i.e. 2^24
workgroups of 256): thousands of short sequences under a large max_seqlen.  Results against the same batch
with its own longest sequence as max_seqlen, whose parity tests/test_gpu_varlen.py checks."""
import math

import pytest
import torch

from conftest import load_mod

pytestmark = pytest.mark.gpu

BF, F32 = torch.bfloat16, torch.float32

# (max_seqlen, Hq, Hkv, D, W, S, dtype); 4096 sequences
CASES = [
    pytest.param(131072, 8, 1, 64, None, 0, BF, id="forward-and-dq-tiles"),
    pytest.param(131072, 4, 2, 16, None, 0, F32, id="float32-tiles"),
    pytest.param(131072, 2, 2, 16, 128, 4, F32, id="float32-sink-chunks"),
    pytest.param(262144, 4, 1, 64, 1024, 1, BF, id="sink-rows-in-chunks"),
]


@pytest.mark.parametrize("longest,Hq,Hkv,D,W,S,dtype", CASES)
def test_grids_past_one_launch(gpu, longest, Hq, Hkv, D, W, S, dtype):
    print(f"case many workgroups max_seqlen={longest} Hq={Hq} Hkv={Hkv} D={D} W={W} S={S} {dtype}", flush=True)
    if torch.cuda.mem_get_info()[0] < 120 << 30:
        pytest.skip("needs 120 GiB of free device memory for the backward's workspace")
    ops = load_mod("_ops")
    B, scale = 4096, 1.0 / math.sqrt(D)
    g = torch.Generator().manual_seed(D + Hq)
    lens = torch.randint(1, 4, (B,), generator=g)
    lens[1000] = 290
    cu = torch.cat((torch.zeros(1, dtype=torch.int64), lens.cumsum(0))).to(torch.int32).cuda()
    q, k, v, do = (torch.randn(int(lens.sum()), H, D, generator=g).to(dtype).cuda() for H in (Hq, Hkv, Hkv, Hq))
    results = []
    for m in (longest, 290):
        w = m if W is None else W
        o, lse = ops.forward_varlen(q, k, v, cu, m, w, S, scale)
        results.append((o, lse, *ops.backward_varlen(q, k, v, o, lse, do, cu, m, w, S, scale)))
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
    tol = 1e-5 if dtype is F32 else 1e-2  # (the plans differ in the order of fp32 sums, then one rounding)
    for name, a, b in zip(("o", "lse", "dq", "dk", "dv"), *results):
        err = float((a.float() - b.float()).norm() / b.float().norm())
        print(f"  {name}: {err:.2e}")
        assert err <= tol, (name, err)


def test_a_grid_that_does_not_fit_is_refused(gpu):
    """The sliding forward has at least one workgroup per sequence, KV head and 8 query heads: 2^21 sequences
    of 8 KV heads are 2^24 of them, one too many for a launch."""
    ops = load_mod("_ops")
    B = 1 << 21
    cu = torch.zeros(B + 1, dtype=torch.int32, device="cuda")
    cu[-10:] = 4
    q, k, v = (torch.randn(4, H, 64, device="cuda").to(BF) for H in (64, 8, 8))
    with pytest.raises(RuntimeError, match="launch failed"):
        ops.forward_varlen(q, k, v, cu, 8, 8, 0, 0.125)
    o, _ = ops.forward_varlen(q, k, v, cu[-100:].contiguous(), 8, 8, 0, 0.125)
    assert bool(torch.isfinite(o).all())
