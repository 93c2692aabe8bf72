"""GPU test of quantize_fp8's kernels: the codes and the scale are those of the PyTorch expression
(x.float() / descale).clamp(-448, 448).to(float8_e4m3fn), bit for bit, over every 16-bit pattern,
NaNs, infinities, the tensor sizes around a kernel's 16-element unit, and strided layouts."""
import pytest
import torch

from conftest import load_pkg

pytestmark = pytest.mark.gpu


def reference(x, descale=None):
    xf = x.detach().float()
    if descale is None:
        amax = float(xf.abs().max()) if xf.numel() else 0.0
        descale = amax / 448.0 if amax > 0.0 else 1.0
    return (xf / descale).clamp(-448.0, 448.0).to(torch.float8_e4m3fn), float(descale)


def check(x, descale=None):
    got, gd = load_pkg().quantize_fp8(x, descale)
    ref, rd = reference(x, descale)
    assert gd == rd and isinstance(gd, float)
    assert got.dtype == torch.float8_e4m3fn and got.shape == ref.shape and got.stride() == ref.stride()
    assert not got.requires_grad
    nan = torch.isnan(ref.float())
    assert torch.equal(torch.isnan(got.float()), nan)
    g, r = got.view(torch.uint8), ref.view(torch.uint8)
    assert torch.equal(g[~nan], r[~nan])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("descale", [None, 1.0, 0.0123, 7.0, 3e-5])
def test_every_16_bit_value(gpu, dtype, descale):
    x = torch.arange(65536, dtype=torch.int32, device=gpu).to(torch.int16).view(dtype)
    check(x, descale)  # NaNs and infinities included
    check(x[torch.isfinite(x.float())], descale)


@pytest.mark.parametrize("n", [1, 3, 7, 8, 15, 16, 17, 31, 255, 4096, 4099, 1 << 20, (1 << 20) + 5])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_sizes(gpu, n, dtype):
    g = torch.Generator(device=gpu).manual_seed(n)
    x = (torch.randn(n, generator=g, device=gpu) * 3).to(dtype)
    for d in (None, 0.01):
        check(x, d)
    x[n // 2] = -1000.0  # the maximum is a negative element, wherever it lies
    check(x)
    x[n - 1] = float("nan")
    check(x)


def test_layouts_and_special_tensors(gpu):
    x = torch.randn(2, 100, 8, 64, device=gpu).bfloat16().requires_grad_()
    check(x.transpose(1, 2))  # dense: kept in its layout
    check(x[:, :, :4])  # gaps: the PyTorch expression
    check(torch.randn(1025, device=gpu).bfloat16()[1:])  # not 16-byte aligned
    check(torch.zeros(40, device=gpu, dtype=torch.float16))
    check(torch.zeros(0, 4, device=gpu))
    check(torch.randn(64, device=gpu, dtype=torch.float64))
    check(torch.full((33,), float("inf"), device=gpu))
    check(torch.full((33,), 1e-44, device=gpu))
    check(torch.tensor([0.0, -0.0, 1e-30, -3e38], device=gpu))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_nan_codes(gpu, dtype):
    """A NaN's code is 0x7f or 0xff by its sign, as PyTorch's; also NaNs that the scaling makes."""
    bits = torch.int16 if dtype != torch.float32 else torch.int32
    x = torch.randn(8 * 37 + 3, device=gpu).to(dtype)
    quiet = torch.full((), float("nan"), dtype=dtype).view(bits).item() & torch.iinfo(bits).max
    x.view(bits)[5::7] = quiet
    x.view(bits)[3::11] = quiet | torch.iinfo(bits).min
    x[40] = float("inf")
    x[41] = -float("inf")
    for descale in (None, 0.5, float("inf"), float("nan")):
        got, ref = load_pkg().quantize_fp8(x, descale)[0], reference(x, descale)[0]
        assert torch.equal(got.view(torch.uint8), ref.view(torch.uint8)), descale


class _Sub(torch.Tensor):
    pass


def test_traced_and_transformed_calls(gpu):
    """Calls that are recorded or transformed run the PyTorch expression: traces compute, on other
    inputs too, and vmap, functorch, fake tensors, subclasses and compilation work as with it."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.proxy_tensor import make_fx

    fa = load_pkg()
    f = lambda t: fa.quantize_fp8(t, 0.5)[0]
    x, y = torch.randn(4, 64, device=gpu), torch.randn(4, 64, device=gpu)
    same = lambda a, t: torch.equal(a.view(torch.uint8), reference(t, 0.5)[0].view(torch.uint8))
    for traced in (torch.jit.trace(f, (x,), check_trace=False), make_fx(f)(x),
                   torch.compile(f, backend="eager", fullgraph=True)):
        stale = torch.full((4, 64), 7, dtype=torch.uint8, device=gpu)
        del stale  # (what uninitialised outputs would hold)
        assert same(traced(y), y)
    assert same(torch.vmap(f)(x), x)
    assert same(torch.func.functionalize(f)(x), x)
    assert not torch.func.grad(lambda t: f(t).float().sum())(x).any()
    mode = FakeTensorMode()
    fake = mode.from_tensor(x)
    with mode:
        assert f(fake).shape == (4, 64)
    assert f(fake).dtype == torch.float8_e4m3fn
    assert type(f(x.as_subclass(_Sub))) is _Sub and same(f(x.as_subclass(_Sub)).as_subclass(torch.Tensor), x)


def test_graph_capture(gpu):
    """Under capture a given scale quantises in the graph; without one, which the host would have to read
    back, the call is refused before it enqueues anything."""
    fa = load_pkg()
    x = torch.randn(3, 1000, device=gpu).bfloat16()
    check(x, 0.02)
    count = torch.zeros(1, device=gpu)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        count.add_(1)
        codes = fa.quantize_fp8(x, 0.02)[0]
        with pytest.raises(RuntimeError, match="capture"):
            fa.quantize_fp8(x)
    for i in range(3):
        x.normal_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(codes.view(torch.uint8), reference(x, 0.02)[0].view(torch.uint8)) and int(count) == i + 1
    check(x)
