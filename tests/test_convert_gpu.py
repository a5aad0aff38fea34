"""GPU tests of the weight conversion kernels (quantiser, packers) against the
sequence of tensor operations that defines them, evaluated on the same GPU: the
integers, the packed words and every half are the same bits."""
import os
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "awesome-cute_amd"))


@pytest.fixture(scope="module")
def env():
    import torch
    import marlin
    assert torch.cuda.is_available()
    return torch, marlin


def _weights(torch, k, n, by_column, seed):
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(seed)
    shape = (n, k) if by_column else (k, n)
    w = torch.randn(shape, dtype=torch.half, device="cuda:0", generator=gen)
    w *= 2.0 ** torch.randint(-20, 12, shape, device="cuda:0", generator=gen)  # subnormals to thousands
    w = w.t() if by_column else w
    w[: k // 2, 0] = 0.0   # a column whose first groups are all zero
    w[:, 1] = 7.5          # ties: w / s = 7.5 and halves of it
    w[1::2, 1] = 1.25
    w[0, 2] = float("inf")
    w[k - 1, 3] = float("nan")
    return w


def _quantise(torch, w, gs):
    k, n = w.shape
    wg = w.contiguous().reshape(k // gs, gs, n)
    s = wg.abs().amax(dim=1, keepdim=True) * (2 / 15)
    q = torch.clamp(torch.round(wg / s).int() + 8, 0, 15)
    return ((q - 8).to(w.dtype) * s).reshape(k, n), q.reshape(k, n), s.reshape(k // gs, n)


def _same(torch, got, want):
    assert got.shape == want.shape and got.dtype == want.dtype
    if want.dtype == torch.half:  # NaN of any payload
        assert torch.equal(got.isnan(), want.isnan())
        got, want = (torch.nan_to_num(x.contiguous(), 0.0, posinf=float("inf"), neginf=float("-inf"))
                     .view(torch.int16) for x in (got, want))
    assert torch.equal(got.contiguous(), want.contiguous())


@pytest.mark.parametrize("by_column", [False, True])
@pytest.mark.parametrize("k,n,gs", [(4, 4, 4), (12, 260, 12), (128, 64, 128), (256, 520, 128), (384, 1096, 128), (120, 512, 40),
                                    (136, 72, -1), (4096, 64, -1), (2304, 136, 1152), (512, 256, 256)])
def test_quantise_is_the_tensor_sequence(env, k, n, gs, by_column):
    torch, marlin = env
    w = _weights(torch, k, n, by_column, seed=k + n)
    got = marlin.quantize(w, gs)
    for g, want in zip(got, _quantise(torch, w, k if gs == -1 else gs)):
        _same(torch, g, want)
    assert got[0].stride() == w.stride() and got[1].stride() == w.stride()


@pytest.mark.parametrize("by_column", [False, True])
@pytest.mark.parametrize("k,n,gs", [(128, 256, 128), (256, 512, 128), (384, 768, 128), (128, 256, -1), (1152, 1280, -1)])
def test_pack_is_the_tensor_sequence(env, k, n, gs, by_column):
    torch, marlin = env
    fake, q, s = marlin.quantize(_weights(torch, k, n, by_column, seed=k * n), gs)
    linear = torch.nn.Linear(k, n, bias=False, device="cuda:0", dtype=torch.half)
    linear.weight.data = fake.t()
    groups = s.shape[0]
    for scales in (s.t(), s.t().contiguous()):
        layer = marlin.Layer(k, n, gs).to("cuda:0")
        layer.pack(linear, scales)
        again = torch.clamp(torch.round(fake / s.repeat_interleave(k // groups, 0)).int() + 8, 0, 15)
        assert torch.equal(layer.B.cpu(), marlin.pack_weights(again.cpu()))
        _same(torch, layer.s, marlin.pack_scales(s, groups > 1))


@pytest.mark.parametrize("k,n,gs", [(2048, 64, -1), (1920, 1028, -1), (4352, 260, 2176), (1921, 132, -1)])
def test_long_groups_in_chunks(env, k, n, gs):
    """Groups of many chunks of 128 rows, whole and ragged, one and two per column."""
    torch, marlin = env
    w = _weights(torch, k, n, False, seed=k + n)
    w[k - 1, 5] = 3.0e4  # the largest of its group, in the last chunk
    for g, want in zip(marlin.quantize(w, gs), _quantise(torch, w, k if gs == -1 else gs)):
        _same(torch, g, want)


@pytest.mark.parametrize("by_column", [False, True])
def test_pack_takes_any_half(env, by_column):
    """Every bit pattern as a weight, under scales of any bits: zeros, infinities, NaN, negative
    and subnormal ones, quotients beyond a half and beyond an integer."""
    torch, marlin = env
    gen = torch.Generator(device="cuda:0")
    k = n = 256
    linear = torch.nn.Linear(k, n, bias=False, device="cuda:0", dtype=torch.half)
    layer = marlin.Layer(k, n, 128).to("cuda:0")
    for seed in range(8):
        gen.manual_seed(seed)
        w = torch.randperm(65536, device="cuda:0", generator=gen).to(torch.int16).view(torch.half).reshape(n, k)
        s = torch.randint(-32768, 32768, (n, 2), device="cuda:0", generator=gen).to(torch.int16).view(torch.half)
        s[:6, 0] = torch.tensor([0.0, -0.0, float("inf"), float("nan"), 2.0 ** -24, 65504.0])
        s[6:n // 2] = torch.rand((n // 2 - 6, 2), device="cuda:0", generator=gen).half() * 0.02
        linear.weight.data = w if by_column else w.t().contiguous().t()
        layer.pack(linear, s)
        q = torch.clamp(torch.round(w.t() / s.t().repeat_interleave(128, 0)).int() + 8, 0, 15)
        assert torch.equal(layer.B.cpu(), marlin.pack_weights(q.cpu()))


@pytest.mark.parametrize("k,n", [(16, 64), (48, 576), (256, 1088)])
def test_packed_integers(env, k, n):
    torch, marlin = env
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(n)
    q = torch.randint(0, 16, (k, n), dtype=torch.int32, device="cuda:0", generator=gen)
    want = marlin.pack_weights(q.cpu())
    assert torch.equal(marlin.pack_weights(q).cpu(), want)
    assert torch.equal(marlin.pack_weights(q.t().contiguous().t()).cpu(), want)  # other layouts and types
    assert torch.equal(marlin.pack_weights(q.to(torch.int64)).cpu(), want)


def test_what_looks_on_sees_the_tensor_operations(env):
    torch, marlin = env
    import torch.autograd.forward_ad as forward_ad
    from torch.fx.experimental.proxy_tensor import make_fx
    w = torch.randn((3, 256, 64), device="cuda:0").half()
    want = [torch.stack(x) for x in zip(*(_quantise(torch, x, 128) for x in w))]
    for got, expected in zip(torch.vmap(lambda x: marlin.quantize(x, 128))(w), want):
        _same(torch, got, expected)
    graph = make_fx(lambda x: marlin.quantize(x, 128))(w[0])  # traced on one weight, run on another
    for got, expected in zip(graph(w[1]), want):
        _same(torch, got, expected[1])
    with forward_ad.dual_level():
        fake, _, s = marlin.quantize(forward_ad.make_dual(w[0], torch.ones_like(w[0])), 128)
        assert forward_ad.unpack_dual(fake).tangent is not None
        assert forward_ad.unpack_dual(s).tangent is not None


def test_layers_whose_buffers_were_changed(env):
    torch, marlin = env
    k, n = 256, 512
    fake, _, s = marlin.quantize(torch.randn((k, n), device="cuda:0").half() * 0.02, 128)
    linear = torch.nn.Linear(k, n, bias=False, device="cuda:0", dtype=torch.half)
    linear.weight.data = fake.t()
    layer = marlin.Layer(k, n, 128).to("cuda:0")
    versions = layer.B._version, layer.s._version
    layer.pack(linear, s.t())
    assert layer.B._version > versions[0] and layer.s._version > versions[1]
    wide = marlin.Layer(k, n, 128).to("cuda:0").float()  # scales held in 32 bits
    wide.pack(linear, s.t())
    assert torch.equal(wide.s, layer.s.float()) and torch.equal(wide.B, layer.B)
    x = torch.randn((3, k), device="cuda:0").half()
    y = layer(x)
    layer.B = torch.nn.Parameter(layer.B, requires_grad=False)  # a parameter in the buffer's place
    assert torch.equal(layer(x), y)


@pytest.mark.parametrize("by_column", [False, True])
@pytest.mark.parametrize("gs", [128, -1])
def test_pack_reads_everything_before_it_writes(env, gs, by_column):
    """Scales in the layer's own buffer, and a weight whose memory the packed words go to."""
    torch, marlin = env
    k, n = 512, 768
    w = torch.randn((k, n), device="cuda:0").half() * 0.02
    fake, _, s = marlin.quantize(w, gs)

    def linear():
        lin = torch.nn.Linear(k, n, bias=False, device="cuda:0", dtype=torch.half)
        lin.weight.data = fake.t().contiguous() if by_column else fake.clone().t()
        return lin

    want = marlin.Layer(k, n, gs).to("cuda:0")
    want.pack(linear(), s.t())
    layer = marlin.Layer(k, n, gs).to("cuda:0")
    layer.s.copy_(s)
    layer.pack(linear(), layer.s.t())
    assert torch.equal(layer.B, want.B) and torch.equal(layer.s, want.s)
    layer, lin = marlin.Layer(k, n, gs).to("cuda:0"), linear()
    memory = lin.weight.data if by_column else lin.weight.data.t()
    layer.B = memory.view(torch.int32).view(-1)[:layer.B.numel()].view(layer.B.shape)
    layer.pack(lin, s.t())
    assert torch.equal(layer.B, want.B) and torch.equal(layer.s, want.s)


def test_more_than_a_grid_holds(env):
    """Sizes beyond the kernels' grids take the tensor operations: the same as in parts."""
    torch, marlin = env
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(2)
    k, n = 16 * 65536, 64
    q = torch.randint(0, 16, (k, n), dtype=torch.int32, device="cuda:0", generator=gen)
    assert torch.equal(marlin.pack_weights(q),
                       torch.cat([marlin.pack_weights(half) for half in q.split(k // 2)]))
    k, n = 128 * 8192, 256
    w = torch.randint(-8, 8, (k, n), device="cuda:0", generator=gen).half()
    s = torch.ones((k // 128, n), device="cuda:0").half()
    linear = torch.nn.Linear(k, n, bias=False, device="meta", dtype=torch.half)
    linear.weight = torch.nn.Parameter(w.t())
    layer = marlin.Layer(k, n, 128).to("cuda:0")
    layer.pack(linear, s.t())
    assert torch.equal(layer.B, torch.cat([marlin.pack_weights((half + 8).int()) for half in w.split(k // 2)]))
    del q, w, linear, layer
    wide = torch.randn((65536, 8192), dtype=torch.half, device="cuda:0", generator=gen)  # columns
    got = marlin.quantize(wide.t(), 4)
    for part, rows in zip(got, (8192, 8192, 2048)):
        assert part.shape == (rows, 65536)
    half = marlin.quantize(wide[:32768].t(), 4)
    assert all(torch.equal(a[:, :32768], b) for a, b in zip(got, half))


def test_layers_made_in_inference_mode(env):
    """Packing writes to the buffers: refused outside inference mode as any write to them is."""
    torch, marlin = env
    k, n = 128, 256
    fake, _, s = marlin.quantize(torch.randn((k, n), device="cuda:0").half(), 128)
    linear = torch.nn.Linear(k, n, bias=False, device="cuda:0", dtype=torch.half)
    linear.weight.data = fake.t()
    with torch.inference_mode():
        layer = marlin.Layer(k, n, 128).to("cuda:0")
        layer.pack(linear, s.t())
        before = layer.B.clone()
    with pytest.raises(RuntimeError, match="[Ii]nference"):
        layer.pack(linear, s.t())
    other = marlin.Layer(k, n, 128).to("cuda:0")
    with torch.inference_mode():
        other.pack(linear, s.t())
    assert torch.equal(other.B, before)


def test_function_modes_see_the_tensor_operations(env):
    torch, marlin = env
    from torch.overrides import TorchFunctionMode
    seen = []

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(getattr(func, "__name__", ""))
            return func(*args, **(kwargs or {}))

    w = torch.randn((256, 128), device="cuda:0").half()
    want = marlin.quantize(w, 128)
    with Mode():
        got = marlin.quantize(w, 128)
    assert "round" in seen and "clamp" in seen
    for g, x in zip(got, want):
        _same(torch, g, x)
    seen.clear()
    with torch.device("cuda:0"):  # says where new tensors go, no more
        for g, x in zip(marlin.quantize(w, 128), want):
            _same(torch, g, x)
