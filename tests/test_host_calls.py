"""The operators' host side in C++ against the one in Python: the same entry points on the same tensors, so the same bits; what it does not
take goes on in Python, with its results and its errors."""
import pytest
import torch


@pytest.mark.parametrize("content", [None, "not a shared object"])
def test_calls_go_on_without_the_module(tmp_path, monkeypatch, content):
    from lego_amd import ops, runtime
    monkeypatch.setattr(runtime, "_calls", None)
    monkeypatch.setattr(runtime, "CALLS_PATH", tmp_path / "host_calls.so")
    monkeypatch.setattr(ops, "_calls", None)
    if content:
        runtime.CALLS_PATH.write_text(content)
    with pytest.warns(RuntimeWarning, match="in Python"), pytest.raises(ValueError, match="GPU"):
        ops.softmax(torch.ones(4, 8))
    with pytest.raises(ValueError, match="GPU"):       # said once
        ops.transpose(torch.ones(4, 8))


def test_refused_calls_keep_their_errors():
    from lego_amd import ops
    x = torch.ones(4, 8)
    for call in (lambda: ops.transpose(x), lambda: ops.softmax(x), lambda: ops.matmul(x.half(), x.half().t()), lambda: ops.stencil_f3d(torch.ones(8, 8, 8), torch.ones(8, 8, 8)),
                 lambda: ops.lego_group_gemm_fn([x.half()], [x.half().t()])):
        with pytest.raises(ValueError, match="GPU"):
            call()
    with pytest.raises(NotImplementedError):
        ops.matmul(x, x, activation="relu")
    with pytest.raises(ValueError, match="same length"):
        ops.lego_group_gemm_fn([x], [])


def test_a_function_in_the_place_of_the_call_sees_the_calls(monkeypatch):
    from lego_amd import ops, runtime
    monkeypatch.setattr(ops, "_calls", in_cpp := object())
    assert ops._host() is in_cpp
    monkeypatch.setattr(runtime, "call", lambda entry, *args: None)
    assert ops._host() is ops._InPython
    monkeypatch.undo()
    assert ops._host() is not ops._InPython


def _both(monkeypatch, call, taken=True):
    """What the call gives through C++ and in Python; whether C++ took it."""
    from lego_amd import ops, runtime
    module, took = runtime.host_calls(), []

    class Watched:
        def __getattr__(self, name):
            def run(*args):
                out = getattr(module, name)(*args)
                took.append(out is not None)
                return out
            return run
    monkeypatch.setattr(ops, "_calls", Watched())
    got = call()
    assert took[0] == taken
    monkeypatch.setattr(ops, "_calls", ops._InPython)
    want = call()
    for u, v in zip(got if isinstance(got, list) else [got], want if isinstance(want, list) else [want]):
        assert type(u) is type(v) and u.shape == v.shape and u.dtype == v.dtype and u.device == v.device and u.stride() == v.stride()
        assert u.requires_grad == v.requires_grad and torch.equal(u, v)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_gpu_rows_and_transposes(monkeypatch, dtype):
    from lego_amd import ops
    print(f"host calls {dtype}", flush=True)
    for shape in ((1, 1), (3, 65), (64, 128), (257, 40)):
        x = torch.randn(shape, device="cuda").to(dtype)
        for v in (x, x.flatten()[:-1].view(1, -1) if x.numel() > 1 else x, x.clone().requires_grad_(dtype == torch.float32)):
            _both(monkeypatch, lambda: ops.softmax(v))
            _both(monkeypatch, lambda: ops.transpose(v))
    _both(monkeypatch, lambda: ops.transpose(torch.arange(12, device="cuda", dtype=torch.int32).view(3, 4)))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,out", [(torch.float16, torch.float16), (torch.bfloat16, torch.float16), (torch.bfloat16, torch.bfloat16),
                                       (torch.float8_e5m2, torch.float16), (torch.float8_e4m3fn, torch.float16)])
def test_gpu_products(monkeypatch, dtype, out):
    from lego_amd import ops
    eight = torch.finfo(dtype).bits == 8
    for M, N, K in ((16, 64, 32), (1, 16, 16), (64, 48, 1), (1, 1, 64), (130, 136, 96), (16, 64, 4096), (33, 17, 65), (33, 17, 4097), (64, 1024, 512)):
        for ta in (0, 1):
            for tb in (0, 1):
                a = torch.randint(-2, 3, (K, M) if ta else (M, K), device="cuda").to(dtype)
                b = torch.randint(-2, 3, (N, K) if tb else (K, N), device="cuda").to(dtype)
                a, b = a.t() if ta else a, b.t() if tb else b
                # of one row or column either layout is the other, and the first one is what is seen
                la = int(not a.is_contiguous())
                taken = eight or not (la and M % 8)
                print(f"host calls {dtype} {M}x{N}x{K} {ta}{tb}", flush=True)
                _both(monkeypatch, lambda: ops.matmul(a, b, activation="leaky_relu" if M == 16 else "", out_dtype=out), taken)


@pytest.mark.gpu
@pytest.mark.parametrize("in_cpp", [True, False])
@pytest.mark.parametrize("dtype,M,N,K,ta,tb,uses", [
    (torch.float8_e5m2, 16, 64, 4096, 0, 0, "parts"), (torch.float8_e5m2, 24, 64, 4096, 0, 1, "parts"), (torch.float8_e4m3fn, 32, 64, 4104, 1, 0, "parts"),
    (torch.float8_e5m2, 24, 64, 4096, 1, 0, "copies"), (torch.float8_e4m3fn, 32, 64, 4104, 0, 0, "copies"), (torch.float8_e5m2, 32, 64, 4104, 1, 1, "copies"),
    (torch.float8_e5m2, 33, 17, 65, 0, 0, "nothing"), (torch.float8_e4m3fn, 64, 64, 64, 0, 1, "nothing"), (torch.float16, 16, 64, 4104, 0, 0, "parts"),
    (torch.float16, 33, 17, 65, 0, 1, "nothing"), (torch.bfloat16, 496, 135, 3878, 0, 0, "copies"), (torch.float16, 16, 4096, 4096, 0, 1, "nothing")])
def test_gpu_products_bring_a_workspace_only_where_it_is_used(monkeypatch, in_cpp, dtype, M, N, K, ta, tb, uses):
    """What a call allocates besides its result, on either route: room for sums of whole tiles, for copies of operands with ragged rows, or nothing."""
    import ctypes
    from lego_amd import ops, runtime
    print(f"workspace {dtype} {M}x{N}x{K} {ta}{tb} {'C++' if in_cpp else 'Python'}", flush=True)
    need, size = ctypes.c_ulonglong(0), torch.finfo(dtype).bits // 8
    runtime.call("lego_hip_gemm_layout_workspace_bytes", M, N, K, ta, tb, size, ctypes.byref(need))
    need = need.value
    assert {"parts": need > 0 and need % 65536 == 0, "copies": need >= size * (M * K + K * N) + 2 * M * N, "nothing": need == 0}[uses]
    # some two hundred products of -4 .. 4 a sum: below 2048, exact in fp16
    a = (torch.randint(-2, 3, (K, M) if ta else (M, K), device="cuda") * (torch.rand((K, M) if ta else (M, K), device="cuda") < 200.0 / K)).to(dtype)
    b = torch.randint(-2, 3, (N, K) if tb else (K, N), device="cuda").to(dtype)
    a, b = a.t() if ta else a, b.t() if tb else b
    monkeypatch.setattr(ops, "_calls", runtime.host_calls() if in_cpp else ops._InPython)

    def allocated():
        stats = torch.cuda.memory_stats()
        return stats["allocation.all.allocated"], stats["requested_bytes.all.allocated"]
    before = allocated()
    c = ops.matmul(a, b)
    assert tuple(after - first for after, first in zip(allocated(), before)) == (1 + (need > 0), 2 * M * N + need)
    assert c.shape == (M, N) and torch.equal(c.double(), a.double() @ b.double())


@pytest.mark.gpu
def test_gpu_groups_and_stencils(monkeypatch):
    from lego_amd import ops
    print("host calls, groups and stencils", flush=True)
    made = lambda sizes: ([torch.randint(-2, 3, (m, k), device="cuda").half() for m, _, k in sizes], [torch.randint(-2, 3, (k, n), device="cuda").half() for _, n, k in sizes])
    for sizes, taken in (([(64, 64, 64)], True), ([(33, 16, 72), (128, 128, 64)], True), ([(33, 17, 65), (128, 128, 64)], True), ([(33, 17, 65)], False),
                         ([(8, 8, 8)] * 65, False), ([(8, 8, 2001), (8, 8, 8)], True), ([(64, 64, 2577)] + [(1024, 1024, 1024)] * 16, False)):
        a, b = made(sizes)
        _both(monkeypatch, lambda: ops.lego_group_gemm_fn(a, b), taken)
    x, c = torch.rand(16, 16, 16, device="cuda"), torch.rand(8, 8, 8, device="cuda")
    for radius in (1, 2, 3):
        for bricks in (False, True):
            _both(monkeypatch, lambda: ops.stencil_f3d(x, c, radius, bricks))
            _both(monkeypatch, lambda: ops.stencil_laplacian(x, c[0, 0].contiguous(), radius, bricks))
    _both(monkeypatch, lambda: ops.stencil_f3d(x, c, 1, 0), False)


@pytest.mark.gpu
def test_gpu_calls_that_are_not_taken(monkeypatch):
    from lego_amd import ops, runtime
    print("host calls: subclasses, modes, forward mode, streams", flush=True)
    calls = runtime.host_calls()
    x = torch.randn(16, 64, device="cuda")
    sub = x.as_subclass(type("Sub", (torch.Tensor,), {}))
    assert calls.softmax(sub) is None and calls.transpose(sub) is None and calls.matmul(sub, sub, "", torch.float16) is None
    assert calls.softmax(x.t()) is None and calls.softmax(x.double()) is None and calls.softmax(x[:0]) is None and calls.softmax(x.cpu()) is None and calls.softmax(3) is None
    h = x.half()
    assert calls.matmul(h, h, "", torch.float16) is None and calls.matmul(h, h.t(), "relu", torch.float16) is None and calls.matmul(h, h.t(), "", torch.float32) is None
    assert calls.matmul(h[:, ::2], h.t()[::2], "", torch.float16) is None and calls.group([h], (h.t().contiguous(),)) is None and calls.transpose() is None
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    for mode in (Dispatch, Function):
        with mode():
            assert calls.softmax(x) is None and calls.matmul(h, h.t(), "", torch.float16) is None
    with torch.autograd.forward_ad.dual_level():
        assert calls.softmax(torch.autograd.forward_ad.make_dual(x, x)) is None
    seen = []
    torch.vmap(lambda t: seen.append(calls.softmax(t)) or t)(x[None])
    assert seen == [None]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        y = calls.softmax(x)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(y, calls.softmax(x))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = ops.matmul(h, h.t())
    for _ in range(3):
        h.copy_(torch.randn_like(x))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ops.matmul(h, h.t()))
