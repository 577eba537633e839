"""The native host path of the linears: the calls it takes return the Python
path's bits, every other form is left to that path, which still answers or
refuses it as before."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from inputs import normal_bias, normal_weight, outlier_activations

pytestmark = pytest.mark.gpu


def setup(backend, M, N, K, dt, R=0):
    G = backend.pick_groupsize(K)
    x = outlier_activations(M, K, seed=M + 4).to(dt).cuda()
    qw, s = backend.quantize_convrot_w4a4_weight(normal_weight(N, K, seed=N).cuda(), convrot_groupsize=G)
    g = torch.Generator(device="cuda").manual_seed(7)
    lora = tuple((torch.randn(sh, generator=g, device="cuda") * 0.02).to(torch.bfloat16)
                 for sh in ((R, K), (N, R))) if R else None
    return x, qw, s, normal_bias(N, seed=5).cuda(), G, lora, backend.prepare_convrot_w4a4_weight_bf6(qw)


def python_path(native, x, qw, s, b, G, lora, w6, eager):
    epi = {torch.bfloat16: native.EPI_BF16_EAGER if eager else native.EPI_BF16, torch.float16: native.EPI_F16,
           torch.float32: native.EPI_F32}[x.dtype]
    D, U = lora or (None, None)
    x2 = x.reshape(-1, x.shape[-1])
    y = native.convrot_w4a4_linear_packed(x2, qw, s, b, D, U, 1.0, epi, G) if w6 is None else \
        native.convrot_w4a4_linear_bf6(x2, w6, s, b, D, U, 1.0, epi, G, qw.shape[0])
    return y.reshape(*x.shape[:-1], -1)


@pytest.mark.parametrize("M,N,K", [(1, 300, 256), (48, 1000, 1152), (130, 700, 320), (600, 5000, 384)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("R", [0, 32])
def test_same_bits(backend, native, gpu, M, N, K, dt, R):
    if R and dt == torch.float32:
        R = 0
    x, qw, s, b, G, lora, w6 = setup(backend, M, N, K, dt, R)
    host = native.host_module()
    for bias in (b, b.float(), b.bfloat16(), None):
        for eager in (False, True):
            y = host.w4a4(x, qw, s, bias, G, eager, lora, w6)
            assert y.dtype == dt and torch.equal(y, python_path(native, x, qw, s, bias, G, lora, w6, eager))
    x3 = x[:M // 2 * 2].reshape(2, M // 2, K) if M > 1 else x[None]
    y3 = backend.convrot_w4a4_linear(x3, qw, s, bias=b, convrot_groupsize=G, lora=lora, qweight_bf6=w6)
    assert y3.shape == (*x3.shape[:-1], N)
    assert torch.equal(y3, python_path(native, x3, qw, s, b, G, lora, w6, False))
    p = torch.nn.Parameter(b, requires_grad=True)        # a layer's bias; the linear has no gradient
    assert not host.w4a4(x, qw, s, p, G, False, lora, w6).requires_grad


@pytest.mark.parametrize("M,N,K", [(1, 300, 256), (130, 700, 320), (600, 5000, 384)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
def test_w8a8_same_bits(backend, native, gpu, M, N, K, dt):
    x = outlier_activations(M, K, seed=M + 4).to(dt).cuda()
    q = torch.randint(-127, 128, (N, K), generator=torch.Generator().manual_seed(N)).to(torch.int8).cuda()
    s, t = torch.rand(N, generator=torch.Generator().manual_seed(1)).cuda(), native.int8_to_i8t(q)
    epi = {torch.bfloat16: native.EPI_BF16, torch.float16: native.EPI_F16, torch.float32: native.EPI_F32}[dt]
    for b in (normal_bias(N, seed=5).cuda(), None):
        y = native.host_module().w8a8(x, q, s, b, 64, t)
        assert y.dtype == dt and torch.equal(y, native.convrot_w8a8_linear_i8t(x, t, s, b, epi, 64, N))


def test_without_the_host_module(backend, native, gpu, monkeypatch, tmp_path):
    """The linears answer, bit for bit, where the host module is missing."""
    x, qw, s, b, G, lora, w6 = setup(backend, 130, 700, 256, torch.bfloat16, 32)
    q = torch.randint(-127, 128, (700, 256), generator=torch.Generator().manual_seed(2)).to(torch.int8).cuda()
    t = native.int8_to_i8t(q)

    def both():
        return (backend.convrot_w4a4_linear(x, qw, s, bias=b, convrot_groupsize=G, lora=lora, qweight_bf6=w6),
                backend.convrot_w8a8_linear(x, q, s, bias=b, qweight_i8t=t))
    want = both()
    monkeypatch.setattr(native._build, "host_path", lambda: str(tmp_path / "_host.so"))
    monkeypatch.setattr(native, "_host", None)
    monkeypatch.setattr(native, "_host_error", None)
    assert all(torch.equal(y, w) for y, w in zip(both(), want))


def test_other_forms_go_to_python(backend, native, gpu):
    M, N, K = 48, 384, 256
    x, qw, s, b, G, lora, w6 = setup(backend, M, N, K, torch.bfloat16, 32)
    host = native.host_module()
    want = backend.convrot_w4a4_linear(x, qw, s, bias=b, convrot_groupsize=G, qweight_bf6=w6)
    wide = torch.zeros((M, K + 8), dtype=x.dtype, device="cuda")
    wide[:, 1:1 + K] = x
    flat = torch.zeros(M * K + 8, dtype=x.dtype, device="cuda")
    off = flat[1:1 + M * K].reshape(M, K)                # contiguous, 2-byte aligned
    off.copy_(x)
    taken = [(wide[:, 1:1 + K], qw, s, b, w6), (off, qw, s, b, w6), (x, qw, s.double(), b, w6), (x, qw, s, b.double(), w6),
             (x, qw, s, b, None), (x, qw, torch.stack([s, s], 1)[:, 0], b, w6),
             (x, qw, s, torch.stack([b, b], 1)[:, 0], w6)]
    for xx, q, ss, bb, w in taken:
        assert host.w4a4(xx, q, ss, bb, G, False, None, w) is None
        y = backend.convrot_w4a4_linear(xx, q, ss, bias=bb, convrot_groupsize=G, qweight_bf6=w)
        assert torch.equal(y, want)
    assert backend.convrot_w4a4_linear(x[:0], qw, s, bias=b, qweight_bf6=w6).shape == (0, N)
    f64 = backend.convrot_w4a4_linear(x.double(), qw, s, bias=b, qweight_bf6=w6)
    assert f64.dtype == torch.float64

    class Seen(TorchDispatchMode):
        n = 0

        def __torch_dispatch__(self, f, types, args=(), kwargs=None):
            Seen.n += 1
            return f(*args, **(kwargs or {}))
    with Seen():
        assert host.w4a4(x, qw, s, b, G, False, None, w6) is None
        assert torch.equal(backend.convrot_w4a4_linear(x, qw, s, bias=b, qweight_bf6=w6), want)
    assert Seen.n > 0
    D, U = lora
    for bad in [dict(convrot_groupsize=128), dict(quant_group_size=32), dict(linear_dtype="fp8"), dict(bias=b[:-1]),
                dict(wscales=s[:-1]), dict(qweight=qw[:, :-64]), dict(qweight_bf6=w6[:-256]),
                dict(lora=(D.half(), U)), dict(lora=(D, U[:-1]))]:
        kw = dict(x=x, qweight=qw, wscales=s, bias=b, qweight_bf6=w6)
        kw.update(bad)
        with pytest.raises(ValueError):
            backend.convrot_w4a4_linear(**kw)
    with pytest.raises(RuntimeError):
        backend.convrot_w4a4_linear(x, qw, s, bias=b.cpu(), qweight_bf6=w6)


def test_w8a8_bad_operands_are_refused(backend, native, gpu):
    """Lengths and shapes the host module leaves to Python raise there, before any launch."""
    M, N, K = 48, 384, 256
    x = outlier_activations(M, K, seed=3).cuda()
    q = torch.randint(-127, 128, (N, K), generator=torch.Generator().manual_seed(1)).to(torch.int8).cuda()
    s, b, t = torch.ones(N, device="cuda"), normal_bias(N, seed=5).cuda(), native.int8_to_i8t(q)
    good = dict(x=x, qweight=q, wscales=s, bias=b, qweight_i8t=t)
    want = backend.convrot_w8a8_linear(**good)
    for bad in [dict(wscales=s[:-1]), dict(wscales=s[:1]), dict(bias=b[:-1]), dict(qweight_i8t=t[:-256]),
                dict(qweight=q[:, :-64]), dict(convrot_groupsize=128)]:
        with pytest.raises(ValueError):
            backend.convrot_w8a8_linear(**{**good, **bad})
    with pytest.raises(RuntimeError):
        backend.convrot_w8a8_linear(**{**good, "bias": b.cpu()})
    assert torch.equal(backend.convrot_w8a8_linear(**{**good, "wscales": s[:, None], "bias": b[None]}), want)


def test_streams_and_threads(backend, native, gpu):
    """Calls on several streams from several threads: their intermediates never meet."""
    import threading
    sets = [setup(backend, m, 1000, 1152, torch.bfloat16) for m in (1, 48, 200, 600)]
    want = [backend.convrot_w4a4_linear(x, qw, s, bias=b, convrot_groupsize=G, qweight_bf6=w6)
            for x, qw, s, b, G, _, w6 in sets]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        x, qw, s, b, G, _, w6 = sets[i]
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            ys = [backend.convrot_w4a4_linear(x, qw, s, bias=b, convrot_groupsize=G, qweight_bf6=w6) for _ in range(40)]
        st.synchronize()
        bad.extend(i for y in ys if not torch.equal(y, want[i]))
    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad


@pytest.mark.parametrize("K,mode,R", [(512, "int4", 0), (512, "int4", 32), (1600, "int4", 0), (1600, "int4", 32), (512, "int8", 0)])
def test_layers_take_the_host_path(backend, native, gpu, monkeypatch, K, mode, R):
    """A loaded layer's forward (its codes a meta-device shape where a tile layout
    is the operand) is answered by the host module in every activation type."""
    import types
    from test_gpu_footprint import _ops
    host, taken = native.host_module(), []

    def seen(name):
        def call(*a):
            y = getattr(host, name)(*a)
            taken.append((name, y is not None))
            return y
        return call
    monkeypatch.setattr(native, "_host", types.SimpleNamespace(w4a4=seen("w4a4"), w8a8=seen("w8a8")))
    Ops, parent, N = _ops(), torch.nn.Module(), 384
    parent.lin = Ops.Linear(K, N, bias=True)
    Ops.int8_exact = {"lin"} if mode == "int8" else set()
    try:
        parent.load_state_dict({"lin.weight": normal_weight(N, K, seed=1).float(), "lin.bias": normal_bias(N, seed=2).float()},
                               strict=False)
    finally:
        Ops.int8_exact = set()
    lin = parent.lin
    assert lin._qmode == mode
    if R:
        g = torch.Generator(device="cuda").manual_seed(1)
        lin._dyn_fused = tuple((torch.randn(sh, generator=g, device="cuda") * 0.02).to(torch.bfloat16)
                               for sh in ((R, K), (N, R)))
        lin._dyn_lora, lin._dyn_rest = [], []
    types_ = (torch.bfloat16, torch.float16) if R else (torch.bfloat16, torch.float16, torch.float32)
    for dt in types_:
        y = lin(outlier_activations(48, K, seed=3).to(dt).cuda()[None])
        assert y.shape == (1, 48, N) and y.dtype == dt
    assert taken == [("w8a8" if mode == "int8" else "w4a4", True)] * len(types_)
