"""GPU tests of padded batches whose tokens the variable-length kernels read in place (fa_fwd_ranges,
fa_bwd_ranges): bit for bit the result of gathering the tokens into a packed batch (the path that a
mask with gaps takes, whose parity tests/test_gpu_sinks.py checks), whatever the padded positions hold,
and the packed path's C++ autograd function against the Python one."""
import math

import pytest
import torch

from conftest import load_mod, load_pkg

pytestmark = pytest.mark.gpu

BF, FP, F32 = torch.bfloat16, torch.float16, torch.float32

# (lens, left padded?, L, Hq, Hkv, D, window, dtype, learned sinks, [B, L, H, D] memory)
CASES = [
    pytest.param((300, 41, 257), False, 300, 16, 2, 64, None, BF, True, True, id="right-full"),
    pytest.param((17, 300, 1, 0), True, 311, 8, 1, 64, 128, BF, True, True, id="left-sliding-empty-row"),
    pytest.param((640, 33), False, 1000, 8, 2, 128, 100, FP, False, False, id="D128-longer-than-any-row"),
    pytest.param((90, 500, 450), True, 500, 6, 6, 16, None, BF, False, True, id="D16-one-head-per-group"),
    pytest.param((100, 260), False, 260, 4, 2, 32, None, F32, True, True, id="float32"),
    pytest.param((700, 650, 20, 900), False, 900, 64, 8, 64, 128, BF, True, True, id="sliding-kernels"),
]


def mask_of(lens, L, left):
    pos = torch.arange(L)
    return torch.stack([(pos >= L - n) if left else (pos < n) for n in lens]).cuda()


@pytest.mark.parametrize("lens,left,L,Hq,Hkv,D,window,dtype,learned,blhd", CASES)
def test_in_place_equals_gathered(gpu, lens, left, L, Hq, Hkv, D, window, dtype, learned, blhd):
    print(f"case padded lens={lens} left={left} L={L} Hq={Hq} Hkv={Hkv} D={D} W={window} {dtype}", flush=True)
    gpt_oss = load_mod("gpt_oss")
    mask = mask_of(lens, L, left)
    B = len(lens)
    g = torch.Generator().manual_seed(L)

    def make(H):
        t = torch.randn(B, L, H, D, generator=g).to(dtype).cuda()
        t[~mask] = float("nan")  # padded positions are not read
        return t.transpose(1, 2) if blhd else t.transpose(1, 2).contiguous()

    q, k, v = make(Hq), make(Hkv), make(Hkv)
    do = make(Hq).transpose(1, 2)
    sinks = torch.randn(Hq, generator=g).cuda() if learned else None
    facts = gpt_oss._padding_facts(mask)
    assert facts[1] is not None and facts[3] == max(lens) and facts[4] == sum(lens)
    gathered = facts[:1] + (None, None) + facts[3:5] + (gpt_oss._mask_facts(mask),)
    results = []
    for f in (facts, gathered):
        leaves = [t.clone().requires_grad_() for t in (q, k, v)] + ([sinks.clone().requires_grad_()] if learned else [])
        o = gpt_oss.padded_attention(*leaves[:3], mask, window_size=window, sinks=leaves[3] if learned else None, _facts=f)
        d = torch.where(mask[:, :, None, None], do, torch.zeros_like(do)) if f is gathered else do
        results.append([o, *torch.autograd.grad(o, leaves, d)])
    torch.cuda.synchronize()
    for name, a, b in zip(("o", "dq", "dk", "dv", "dsinks"), *results):
        assert a.shape == b.shape and torch.equal(a, b), name
    o, dq, dk, dv = results[0][:4]
    pad = ~mask
    for t in (o, dq.transpose(1, 2), dk.transpose(1, 2), dv.transpose(1, 2)):
        assert bool((t[pad] == 0).all()) and bool(torch.isfinite(t).all())


def test_facts_of_masks(gpu):
    gpt_oss = load_mod("gpt_oss")
    f = gpt_oss._padding_facts(mask_of((5, 0, 3), 6, True).to(torch.int64))
    assert f[0] is False and f[1].tolist()[0] == 1 and f[1].tolist()[2] == 15 and f[2].tolist() == [5, 0, 3]
    assert f[3:5] == (5, 8) and f[5] is None
    gaps = torch.tensor([[1, 0, 1, 1], [1, 1, 1, 1]]).cuda()
    f = gpt_oss._padding_facts(gaps)
    assert f[0] is False and f[1] is None and f[5][2].tolist() == [0, 3, 7]
    assert gpt_oss._padding_facts(torch.ones(2, 3, device="cuda"))[0] is True
    assert gpt_oss._padding_facts(torch.ones(2, 0, device="cuda"))[0] is True


def test_bad_ranges_stay_inside_the_tensors(gpu):
    """Starts and lengths that reach outside the rows are cut off there, as bad cu_seqlens are."""
    ops = load_mod("_ops")
    b = ops.autograd_binding(torch.empty(1, device="cuda"))
    q, k, v = (torch.randn(100, H, 64, device="cuda").bfloat16() for H in (8, 1, 1))
    starts = torch.tensor([-5, 60, 400], dtype=torch.int32, device="cuda")
    lens = torch.tensor([20, 1 << 30, 7], dtype=torch.int32, device="cuda")
    o = b.swda_varlen(q, k, v, starts, lens, 40, 100, 40, 0, 0.125)
    torch.cuda.synchronize()
    ref = b.swda_varlen(q, k, v, torch.tensor([0, 60], dtype=torch.int32, device="cuda"),
                        torch.tensor([20, 40], dtype=torch.int32, device="cuda"), 40, 60, 40, 0, 0.125)
    assert torch.equal(o, ref) and bool((o[20:60] == 0).all())


def test_rows_far_apart(gpu):
    """q, k and v as slices of one wide buffer whose rows span more than the kernels' 32-bit offsets reach:
    copied closer together, as gathering does."""
    gpt_oss = load_mod("gpt_oss")
    B, L, Hq, Hkv, D, lens = 2, 16500, 4, 1, 64, (16500, 16391)
    wide = torch.empty(B, L, 1 << 16, dtype=BF, device="cuda")
    cut = lambda H, c: wide[..., c:c + H * D].normal_().view(B, L, H, D).transpose(1, 2)
    q, k, v = cut(Hq, 0), cut(Hkv, Hq * D), cut(Hkv, (Hq + 1) * D)
    assert (max(lens) - 1) * q.stride(2) * 2 >= 1 << 31
    do = wide[..., 512:512 + Hq * D].normal_().view(B, L, Hq, D)
    mask = mask_of(lens, L, False)
    results = []
    for x in ((q, k, v), [t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v)]):
        leaves = [t.detach().requires_grad_() for t in x]
        o = gpt_oss.padded_attention(*leaves, mask, window_size=100)
        results.append([o, *torch.autograd.grad(o, leaves, do)])
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.parametrize("Hq,Hkv,D,dtype", [(64, 8, 64, BF), (6, 3, 128, FP), (5, 1, 16, BF), (7, 7, 32, F32)])
def test_rows_of_no_sequence(gpu, Hq, Hkv, D, dtype):
    """A packed buffer with long unused stretches before, between and after its sequences: o, dq, dk and dv are
    0 and lse is -inf on every row outside them, and only there."""
    ops = load_mod("_ops")
    total, starts, lens = 9000, (2500, 2533, 6000), (33, 0, 700)
    rows = torch.zeros(total, dtype=torch.bool)
    for s, n in zip(starts, lens):
        rows[s:s + n] = True
    q, k, v, do = (torch.randn(total, H, D, device="cuda").to(dtype) for H in (Hq, Hkv, Hkv, Hq))
    b = ops.autograd_binding(q)
    leaves = [t.requires_grad_() for t in (q, k, v)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    forms = [(lambda: b.swda_varlen(*leaves, i32(starts), i32(lens), 700, sum(lens), 128, 0, 0.125), rows)]
    cu = i32((2500, 2533, 3000))  # (the first and last rows of the buffer are unused)
    covered = torch.zeros(total, dtype=torch.bool)
    covered[2500:3000] = True
    forms.append((lambda: b.swda_varlen(*leaves, cu, None, 467, 0, 128, 0, 0.125), covered))
    for f, on in forms:
        junk = [torch.full_like(t, 7.0) for t in (q, q, k, v)]
        del junk  # (what unwritten outputs would hold)
        o = f()
        grads = torch.autograd.grad(o, leaves, do)
        for t in (o, *grads):
            assert bool((t[~on] == 0).all()) and bool(torch.isfinite(t).all())
        for t in (o, grads[2]):  # (a first row's dq is 0: it sees one key)
            assert bool((t[on] != 0).any(-1).all())
    _, lse = ops.forward_varlen(q, k, v, cu, 467, 128, 0, 0.125)
    assert torch.equal(torch.isinf(lse), (~covered).cuda().expand_as(lse)) and bool((lse[:, ~covered] < 0).all())


@pytest.mark.parametrize("D,window,sinks", [(64, 128, True), (64, None, False), (128, 200, True)])
def test_packed_function_equals_the_python_one(gpu, D, window, sinks):
    fa = load_pkg()
    cu = torch.tensor([0, 300, 301, 850], dtype=torch.int32, device="cuda")
    leaves = [torch.randn(860, H, D, device="cuda").bfloat16().requires_grad_() for H in (8, 1, 1)]
    sk = torch.randn(8, device="cuda").bfloat16().requires_grad_() if sinks else None
    do = torch.randn(860, 8, D, device="cuda").bfloat16()
    W = 549 if window is None else window
    out = []
    for f in (lambda: fa.flash_swda_with_sink_varlen(*leaves, cu, 549, window, 0, None, sk),
              lambda: fa.FlashSWDAWithSinkVarlen.apply(*leaves, cu, 549, W, 0, None, sk)):
        o = f()
        out.append([o, *torch.autograd.grad(o, leaves + ([sk] if sinks else []), do)])
    for a, b in zip(*out):
        assert torch.equal(a, b) and a.dtype == b.dtype
    with pytest.raises(AssertionError, match="Key and Value"):
        fa.flash_swda_with_sink_varlen(leaves[0], leaves[1][:, :, :32], leaves[2], cu, 549, window)
    with pytest.raises(ValueError, match="max_seqlen is required"):
        fa.flash_swda_with_sink_varlen(*leaves, cu, None, window)


@pytest.mark.parametrize("L", [700, 20000])
def test_mask_facts_are_complete_when_the_host_has_them(gpu, L):
    """Layers on other streams use a mask's facts at once, so nothing may be left to run for them; masks that
    the host works out and, larger, the device."""
    facts = load_mod("gpt_oss")._padding_facts
    mask = torch.zeros(3, L, dtype=torch.long, device=gpu)
    mask[0], mask[1, 50:60] = 1, 1
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        for _ in range(3):
            full, starts, lens, longest, tokens, packed = facts(mask)
            assert stream.query()
            assert (full, longest, tokens, packed) == (False, L, L + 10, None)
            assert starts.tolist() == [0, L + 50, 2 * L] and lens.tolist() == [L, 10, 0]
            assert starts.dtype == lens.dtype == torch.int32 and starts.is_cuda
            mask[0, 5] = 0
            full, starts, lens, longest, tokens, packed = facts(mask)
            assert stream.query() and not full and starts is lens is None
            assert (longest, tokens, packed[3]) == (L - 1, L + 9, L - 1) and packed[2].tolist() == [0, L - 1, L + 9, L + 9]
            mask[0, 5] = 1
            assert facts(torch.ones_like(mask)) == (True, None, None, L, 3 * L, None)
