"""The native form of kquant's calls (csrc/host/torch_calls.cpp): it takes plain calls and gives what the Python form gives, and leaves
everything else to the Python form, which accepts or refuses it as it did."""
import ctypes
import importlib.util
import subprocess
import sys
import threading

import numpy as np
import pytest
import torch

from test_gpu_fused import gpu  # noqa: F401  (fixture)

Q4_K, Q6_K = 12, 14


class _General:
    """Stands in for the native module: every call goes to the Python form."""

    def __init__(self, native):
        self.stream = native.stream

    def __getattr__(self, name):
        return lambda *a: NotImplemented


@pytest.fixture
def both(monkeypatch):
    """Runs a call in its native form and in Python's; says whether the native one took it."""
    from backpack_amd import kquant
    native = kquant._native()

    class Watched(_General):
        took = None

        def __getattr__(self, name):
            def f(*a):
                r = getattr(native, name)(*a)
                Watched.took = r is not NotImplemented
                return r
            return f

    def run(f, *a, **k):
        out = []
        for form in (Watched(native), _General(native)):
            monkeypatch.setattr(kquant, "_native", lambda form=form: form)
            try:
                out.append(("value", f(*a, **k)))
            except Exception as e:  # noqa: BLE001  (both forms have to raise the same)
                out.append(("raised", type(e), str(e)))
        return out[0], out[1], Watched.took
    return run


def _same(a, b):
    assert a[0] == b[0], (a, b)
    if a[0] == "raised":
        assert a[1:] == b[1:]
        return
    xs, ys = (v[1] if isinstance(v[1], tuple) else (v[1],) for v in (a, b))
    assert len(xs) == len(ys)
    for x, y in zip(xs, ys):
        assert x.dtype == y.dtype and x.shape == y.shape and x.device == y.device and torch.equal(x, y)


def test_calls_on_host_tensors_are_refused_as_before(both):
    from backpack_amd import kquant
    w = kquant.KQuantPacked(torch.zeros(144 * 4 + 16, dtype=torch.uint8), Q4_K, 4, 256, 36, 1)
    for f, a in ((kquant.matmul, (torch.zeros(1, 256), w)), (kquant.matmul_fused, (torch.zeros(1, 256), w)), (kquant.matmul_argmax, (torch.zeros(1, 256), w)),
                 (kquant.prefill_rows_bf16, (torch.zeros(1, 256), 256)), (kquant.dequant_rows, (w, torch.zeros(3, dtype=torch.int32)))):
        n, g, took = both(f, *a)
        assert not took and n[0] == g[0] == "raised" and n[1] is g[1] is AssertionError


def test_native_calls_are_there_for_every_thread_at_every_moment():
    """Between any two instructions of a thread's first call another thread's call gets the native module."""
    from backpack_amd import kquant as loaded
    spec = importlib.util.spec_from_file_location("backpack_amd.kquant_once_more", loaded.__file__)
    kquant = importlib.util.module_from_spec(spec)       # as it is ahead of its first call
    sys.modules[spec.name] = kquant                      # (its dataclass looks its module up)
    spec.loader.exec_module(kquant)
    state, asked = vars(kquant), []

    def another_thread():
        got, before = [], dict(state)
        t = threading.Thread(target=lambda: got.append(kquant._native()))
        t.start()
        t.join()
        state.update(before)      # (the traced call goes on as if alone)
        asked.append(got[0])

    def trace(frame, event, arg):
        if frame.f_code is not kquant._native.__code__:
            return None
        frame.f_trace_opcodes = True
        if event == "opcode":
            another_thread()
        return trace
    sys.settrace(trace)
    try:
        mine = kquant._native()
    finally:
        sys.settrace(None)
        del sys.modules[spec.name]
    assert mine is not None and len(asked) > 20 and all(a is mine for a in asked)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 3, 20])
def test_native_calls_give_what_the_general_form_gives(gpu, both, M):  # noqa: F811
    from backpack_amd import capi, kquant
    K, N, E = 512, 272, 4
    rng = np.random.default_rng(M)
    f32 = lambda *s: gpu.dev(rng.standard_normal(s).astype(np.float32))  # noqa: E731
    _, _, w = gpu.make_weight(Q4_K, N, K, seed=1)
    _, _, gate = gpu.make_weight(Q4_K, E * 256, K, seed=2)
    _, _, up = gpu.make_weight(Q4_K, E * 256, K, seed=3)
    _, _, down = gpu.make_weight(Q6_K, E * K, 256, seed=4)
    x, bias, res, nw = f32(M, K), f32(N), f32(M, N), f32(K)
    ws = torch.empty(capi.lib().bpk_kq_matmul_fused_workspace_bytes(M, N, K), dtype=torch.uint8, device="cuda")
    idx = gpu.dev(np.stack([rng.permutation(E)[:2] for _ in range(M)]).astype(np.int32))
    rows = gpu.dev(rng.integers(0, N, M).astype(np.int32))
    calls = [(kquant.matmul, (x, w), {}), (kquant.matmul, (x.view(M, 1, K), w), {"bias": bias}), (kquant.matmul, (x.bfloat16(), w), {"bias": bias}),
             (kquant.matmul, (x, w), {"out": torch.zeros(M, N, device="cuda")}), (kquant.matmul, (x.requires_grad_(), w), {}),
             (kquant.matmul_fused, (x, w, capi.PRO_RMS_NORM), {"norm_w": nw, "eps": 1e-5, "residual": res, "bias": bias, "workspace": ws}),
             (kquant.matmul_fused, (x, w), {"epilogue": capi.EPI_SILU_MUL}), (kquant.matmul_fused, (f32(M, 2 * K), w, capi.PRO_SILU_MUL), {}),
             (kquant.matmul_argmax, (x, w), {"bias": bias}), (kquant.prefill_rows_bf16, (x, K, capi.PRO_RMS_NORM, nw, 1e-5), {}),
             (kquant.prefill_rows_bf16, (f32(M, 2 * K), K, capi.PRO_GELU_MUL), {}), (kquant.dequant_rows, (w, rows), {}),
             (kquant.moe_route, (x, f32(E, K), 2), {}), (kquant.moe_route, (x, f32(E, K), 2, False), {}),
             (kquant.moe_ffn, (x, gate, up, down, idx, f32(M, 2), E), {})]
    for f, a, k in calls:
        n, g, took = both(f, *a, **k)
        assert took and n[0] == "value", (f, n)
        _same(n, g)
    # on a stream that is not the default one
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    want = kquant.matmul(x, w)
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        assert kquant._stream() == s.cuda_stream
        got = kquant.matmul(x, w)
    s.synchronize()
    assert torch.equal(got, want)


@pytest.mark.gpu
def test_calls_that_are_not_plain_are_answered_as_before(gpu, both):  # noqa: F811
    from backpack_amd import kquant
    K, N = 512, 64
    _, packed, w = gpu.make_weight(Q4_K, N, K, seed=5)
    x = torch.randn(4, K, device="cuda")

    class Sub(torch.Tensor):
        pass

    class Owned:   # a weight whose memory is no tensor's
        def data_ptr(self):
            return w.data.data_ptr()
    owned = kquant.KQuantPacked(Owned(), w.type, N, K, w.row_stride_words, w.n_blocks)
    for f, a, k, fine in [(kquant.matmul, (x.as_subclass(Sub), w), {}, True), (kquant.matmul, (x, owned), {}, True),
                          (kquant.matmul, (x, w), {"out": torch.zeros(4, N, device="cuda"), "y_offset": 0}, True), (kquant.matmul_fused, (x, w), {"eps": 0}, True),
                          (kquant.matmul, (x[:, ::2], w), {}, False), (kquant.matmul, (x.half(), w), {}, False), (kquant.matmul, (x, w), {"y_offset": 4}, False),
                          (kquant.matmul, (x.t(), w), {}, False), (kquant.matmul, (x, w), {"out": torch.zeros(N, 4, device="cuda").t()}, False),
                          (kquant.matmul_fused, (x, w), {"prologue": 7}, False), (kquant.moe_route, (x, torch.randn(4, K, device="cuda"), 0), {}, False),
                          (kquant.matmul, (x, kquant.KQuantPacked(w.data, 99, N, K, w.row_stride_words, w.n_blocks)), {}, False),
                          (kquant.matmul, (x, kquant.KQuantPacked(w.data, w.type, N, K, 1, w.n_blocks)), {}, False)]:
        n, g, _ = both(f, *a, **k)
        assert (n[0] == "value") == fine, (f, n)
        _same(n, g)


_ALLOCATOR = r"""
#include <hip/hip_runtime_api.h>
extern "C" int PyGILState_Check(void);
extern "C" { int taken, locked; }
extern "C" void* take(ssize_t n, int, hipStream_t) {
    void* p = nullptr;
    ++taken;
    locked += PyGILState_Check();
    return hipMalloc(&p, n) == hipSuccess ? p : nullptr;
}
extern "C" void give(void* p, ssize_t, int, hipStream_t) { (void)hipFree(p); }
"""
_kept = []     # the allocator outlives what it has given


@pytest.mark.gpu
def test_outputs_are_allocated_without_the_interpreter_lock(gpu, tmp_path):  # noqa: F811
    """A device allocation may wait for the device; a host callback in a stream may wait for the lock.  Asked from an allocator that
    the calls' outputs come from."""
    from backpack_amd import capi, kquant
    src, so = tmp_path / "a.cpp", tmp_path / "a.so"
    src.write_text(_ALLOCATOR)
    subprocess.run(["g++", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", str(src), "-o", str(so), "-L/opt/rocm/lib",
                    "-lamdhip64"], check=True, timeout=60)
    M, K, N, E = 2, 256, 64, 4
    x, idx, wt = torch.randn(M, K, device="cuda"), torch.zeros(M, 2, dtype=torch.int32, device="cuda"), torch.rand(M, 2, device="cuda")
    _, _, w = gpu.make_weight(Q4_K, N, K, seed=1)
    _, _, experts = gpu.make_weight(Q4_K, E * 256, K, seed=2)
    router, rows = torch.randn(E, K, device="cuda"), torch.zeros(3, dtype=torch.int32, device="cuda")
    calls = [lambda: kquant.matmul(x, w), lambda: kquant.matmul_fused(x, w, capi.PRO_RMS_NORM, norm_w=x[0], eps=1e-5), lambda: kquant.matmul_argmax(x, w),
             lambda: kquant.prefill_rows_bf16(x, K), lambda: kquant.dequant_rows(w, rows), lambda: kquant.moe_route(x, router, 2),
             lambda: kquant.moe_ffn(x, experts, experts, experts, idx, wt, E)]
    native = kquant._native()
    for c in calls:
        c()                    # (what the library allocates once is there)
    torch.cuda.synchronize()
    _kept.append(torch.cuda.memory.CUDAPluggableAllocator(str(so), "take", "give"))
    seen = ctypes.CDLL(str(so))
    taken, locked = (ctypes.c_int.in_dll(seen, n) for n in ("taken", "locked"))
    assert native is kquant._native()
    for i, c in enumerate(calls):
        pool = torch.cuda.MemPool(_kept[-1].allocator())
        before = taken.value
        with torch.cuda.use_mem_pool(pool):
            y = c()
        torch.cuda.synchronize()
        assert taken.value > before and locked.value == 0, (i, taken.value - before, locked.value)
        del y, pool
