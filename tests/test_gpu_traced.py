"""Traced and transformed calls of the attention functions: a torch.jit trace records the Python autograd
function (what the binding's kernels write is invisible to it) and computes for other inputs;
forward-mode AD and functorch are refused."""
import pytest
import torch
import torch.autograd.forward_ad as fwad

from conftest import load_mod, load_pkg

pytestmark = pytest.mark.gpu


def forms():
    fa, gpt_oss = load_pkg(), load_mod("gpt_oss")
    cu = torch.tensor([0, 60, 100], dtype=torch.int32, device="cuda")
    mask = torch.ones(2, 50, dtype=torch.bool, device="cuda")
    mask[1, 30:] = False
    sinks = torch.linspace(-1, 1, 8, device="cuda")
    batch, packed = (2, 8, 50, 64), (100, 8, 64)
    return {
        "batch": (batch, lambda q, k, v: fa.flash_swda_with_sink(q, k, v, 20, 2)),
        "learned": (batch, lambda q, k, v: fa.attention(q, k, v, 20, sinks=sinks)),
        "packed": (packed, lambda q, k, v: fa.flash_swda_with_sink_varlen(q, k, v, cu, 60, 60, 0, None, sinks)),
        "padded": (batch, lambda q, k, v: gpt_oss.padded_attention(q, k, v, mask, 40)),
    }


def inputs(shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    kv = (shape[0], 1, *shape[2:])
    return [torch.randn(s, generator=g, device="cuda").bfloat16() for s in (shape, kv, kv)]


@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning")
@pytest.mark.parametrize("form", ["batch", "learned", "packed", "padded"])
@pytest.mark.parametrize("grads", [False, True])
def test_jit_trace(gpu, form, grads):
    shape, f = forms()[form]
    traced = torch.jit.trace(f, tuple(t.requires_grad_(grads) for t in inputs(shape, 1)), check_trace=False)
    other = inputs(shape, 2)
    want = f(*other)
    stale = torch.full_like(want, 7.0)
    del stale  # (what an uninitialised output would hold)
    assert torch.equal(traced(*other), want)


@pytest.mark.parametrize("form", ["batch", "learned", "packed", "padded"])
def test_refused_transforms(gpu, form):
    shape, f = forms()[form]
    q, k, v = inputs(shape, 3)
    with fwad.dual_level(), pytest.raises(NotImplementedError):
        f(fwad.make_dual(q, torch.ones_like(q)), k, v)
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda t: f(t, k, v).float().sum())(q)
    with pytest.raises(RuntimeError):
        torch.vmap(lambda t: f(t, k, v))(q[None])
