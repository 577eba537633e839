"""Calls that share a stream's workspace from several threads: a call's launches
are queued without another call's in between."""
import threading
import time

import pytest
import torch

from inputs import normal_bias, normal_weight, outlier_activations


class CountingLibrary:
    """Stands in for the kernel library: every call that is handed a workspace
    stays inside for a moment, and two at once on one workspace are noted."""

    def __init__(self):
        self.inside, self.calls, self.met = {}, 0, []
        self.lock = threading.Lock()

    def __getattr__(self, name):
        if name.endswith("_workspace"):
            return lambda *a: 4096
        if name.endswith("choose_nsplit"):
            return lambda *a: 2

        def call(*a):
            ws = a[-3]
            with self.lock:
                self.calls += 1
                n = self.inside[ws] = self.inside.get(ws, 0) + 1
                if n > 1:
                    self.met.append(name)
            time.sleep(0.02)
            with self.lock:
                self.inside[ws] -= 1
            return 0
        return call


def calls(native):
    x = torch.zeros((4, 128), dtype=torch.bfloat16)
    s, out = torch.ones(8), []
    out.append(lambda: native.convrot_w8a8_linear_i8t(x, torch.zeros((256, 128), dtype=torch.int8), s, None,
                                                      native.EPI_BF16, 64, 8))
    out.append(lambda: native.convrot_w4a4_linear_packed(x, torch.zeros((8, 64), dtype=torch.int8), s, None, None, None,
                                                         1.0, native.EPI_BF16, 64))
    for epi in (native.EPI_BF16, native.EPI_F16):
        out.append(lambda epi=epi: native.convrot_w4a4_linear_bf6(x, torch.zeros((256, 96), dtype=torch.uint8), s, None,
                                                                  None, None, 1.0, epi, 64, 8))
    out.append(lambda: native.lora_down(x, torch.zeros((32, 128), dtype=torch.bfloat16)))
    b6 = torch.zeros((256, 96), dtype=torch.uint8)
    out.append(lambda: native.int4_convrot_gemm_bf6(b6, b6, torch.ones(4), s, None, native.EPI_BF16))
    return out


def test_one_call_at_a_time_on_a_workspace(native, monkeypatch):
    """Threads on one stream: no library call starts on the workspace while
    another has launches to queue on it."""
    lib = CountingLibrary()
    monkeypatch.setattr(native, "load_library", lambda: lib)
    monkeypatch.setattr(native, "_check_cuda", lambda *t: None)
    monkeypatch.setattr(native, "_stream", lambda device: 7)
    monkeypatch.setattr(native, "_workspaces", type(native._workspaces)())
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    errors, todo = [], calls(native)
    start = threading.Barrier(len(todo))

    def work(i):
        try:
            start.wait(timeout=60)
            for k in range(4):
                todo[(i + k) % len(todo)]()
        except BaseException as e:          # noqa: BLE001 - reported below
            errors.append(e)
    ts = [threading.Thread(target=work, args=(i,)) for i in range(len(todo))]
    [t.start() for t in ts]
    [t.join(timeout=120) for t in ts]
    assert not errors, errors
    assert lib.calls == 4 * len(todo) and not lib.met


@pytest.mark.gpu
def test_threads_on_one_stream(backend, native, gpu):
    """Two threads on the default stream with different inputs: W8A8 and W4A4
    products that split k, a packed width in a strided form, a LoRA."""
    work = []
    for i, (M, N, K) in enumerate([(512, 3072, 12288), (300, 3072, 6144)]):
        x = outlier_activations(M, K, seed=20 + i).cuda()
        b = normal_bias(N, seed=30 + i).cuda()
        q = torch.randint(-127, 128, (N, K), generator=torch.Generator().manual_seed(i)).to(torch.int8).cuda()
        s, t = torch.full((N,), 1e-3 * (i + 1), device="cuda"), native.int8_to_i8t(q)
        assert native.load_library().cr_convrot_w8a8_linear_i8t_split(M, N, K)
        qw, s4 = backend.quantize_convrot_w4a4_weight(normal_weight(N, K, seed=40 + i).cuda())
        w6 = backend.prepare_convrot_w4a4_weight_bf6(qw)
        assert native.load_library().cr_convrot_w4a4_linear_bf6_split(M, N, K)
        g = torch.Generator(device="cuda").manual_seed(i)
        lora = tuple((torch.randn(sh, generator=g, device="cuda") * 0.02).to(torch.bfloat16) for sh in ((32, K), (N, 32)))
        xp = torch.zeros((M, 328), dtype=torch.bfloat16, device="cuda")
        xp[:, :320] = outlier_activations(M, 320, seed=50 + i).cuda()
        qp, sp = backend.quantize_convrot_w4a4_weight(normal_weight(N, 320, seed=60 + i).cuda(), convrot_groupsize=64)
        work.append([
            lambda x=x, q=q, s=s, b=b, t=t: backend.convrot_w8a8_linear(x, q, s, bias=b, qweight_i8t=t),
            lambda x=x, qw=qw, s4=s4, b=b, w6=w6, lora=lora: backend.convrot_w4a4_linear(x, qw, s4, bias=b, lora=lora,
                                                                                         qweight_bf6=w6),
            lambda xp=xp, qp=qp, sp=sp, b=b: backend.convrot_w4a4_linear(xp[:, :320], qp, sp, bias=b, convrot_groupsize=64),
            lambda x=x, qw=qw, s4=s4, w6=w6: backend.convrot_w4a4_linear(x, qw, s4, qweight_bf6=w6)])
    want = [[f() for f in fs] for fs in work]
    torch.cuda.synchronize()
    bad, start = [], threading.Barrier(2)

    def run(i):
        try:
            start.wait(timeout=60)
            ys = [(k, work[i][k]()) for _ in range(25) for k in range(len(work[i]))]
            torch.cuda.synchronize()
            bad.extend((i, k) for k, y in ys if not torch.equal(y, want[i][k]))
        except BaseException as e:          # noqa: BLE001 - reported below
            bad.append(e)
    ts = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    [t.start() for t in ts]
    [t.join(timeout=90) for t in ts]
    assert not bad, bad
