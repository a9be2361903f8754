"""LayerNorm's autograd node in C++ against the one in Python: the same kernels on the same tensors, so the same bits; what it
does not take goes through the node in Python, with its results and its errors."""
import pytest
import torch


def test_refused_calls_keep_their_errors():
    from lego_amd import ops
    w = torch.ones(8)
    with pytest.raises(ValueError, match="GPU"):
        ops.lego_layer_norm(torch.ones(4, 8), (8,), w, w, 1e-5)
    with pytest.raises(ValueError, match="normalized_shape"):
        ops.lego_layer_norm(torch.ones(4, 8), (4,), w, w, 1e-5)


@pytest.mark.parametrize("content", [None, "not a shared object"])
def test_calls_go_on_without_the_node_in_cpp(tmp_path, monkeypatch, content):
    """Not built, or an object that does not load (another torch's): one warning, and the node in Python takes the calls."""
    from lego_amd import ops, runtime
    monkeypatch.setattr(runtime, "_node", None)
    monkeypatch.setattr(runtime, "NODE_PATH", tmp_path / "layernorm_node.so")
    monkeypatch.setattr(ops, "_node_apply", None)
    if content:
        runtime.NODE_PATH.write_text(content)
    w = torch.ones(8)
    with pytest.warns(RuntimeWarning, match="in Python"), pytest.raises(ValueError, match="GPU"):
        ops.lego_layer_norm(torch.ones(4, 8), (8,), w, w, 1e-5)


def test_the_node_is_built_again_for_another_torch(tmp_path, monkeypatch):
    import subprocess
    from lego_amd import build
    built = []

    def run(cmd, **kwargs):
        built.append(cmd)
        build.NODE_PATH.write_text("")
        return subprocess.CompletedProcess(cmd, 0, "", "")
    monkeypatch.setattr(build, "NODE_PATH", tmp_path / "layernorm_node.so")
    monkeypatch.setattr(build.subprocess, "run", run)
    for _ in range(3):
        build.build_node(incremental=True)
    assert len(built) == 1
    monkeypatch.setattr(torch, "__version__", "0.0")
    build.build_node(incremental=True)
    build.build_node(incremental=True)
    assert len(built) == 2


def _inputs(shape, dtype, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    n = shape[-1]
    make = lambda *s: torch.randn(*s, device="cuda", generator=g).to(dtype)
    return make(*shape).requires_grad_(), (1 + 0.1 * make(n)).requires_grad_(), (0.1 * make(n)).requires_grad_(), make(*shape)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(1, 64), (19, 192), (3, 5, 247), (512, 768), (640,)])
def test_gpu_same_bits_as_the_node_in_python(shape, dtype):
    from lego_amd import ops, runtime
    print(f"layernorm node {shape} {dtype}", flush=True)
    x, w, b, dy = _inputs(shape, dtype)
    y = runtime.layernorm_node().apply(x, (shape[-1],), w, b, 1e-5)
    assert y is not None                     # the node in C++ took it
    got = (y.detach(),) + torch.autograd.grad(y, (x, w, b), dy)
    want_y = ops.LEGOLayerNorm.apply(x, (shape[-1],), w, b, 1e-5)
    want = (want_y.detach(),) + torch.autograd.grad(want_y, (x, w, b), dy)
    for u, v in zip(got, want):
        assert u.shape == v.shape and u.dtype == v.dtype and torch.equal(u, v)
    # a gradient in another layout: a sum's is one element, expanded
    gx, = torch.autograd.grad(ops.lego_layer_norm(x, (shape[-1],), w, b, 1e-5).sum(), (x,))
    hx, = torch.autograd.grad(ops.LEGOLayerNorm.apply(x, (shape[-1],), w, b, 1e-5).sum(), (x,))
    assert torch.equal(gx, hx)


@pytest.mark.gpu
def test_gpu_hooks_streams_versions_and_modes():
    from lego_amd import ops, runtime
    print("layernorm node: hooks, streams, versions, modes", flush=True)
    x, w, b, dy = _inputs((64, 256), torch.float16)
    want = torch.autograd.grad(ops.LEGOLayerNorm.apply(x, (256,), w, b, 1e-5), (x, w, b), dy)
    packed = []

    def pack(t):
        packed.append(tuple(t.shape))
        return t.cpu()
    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
        y = ops.lego_layer_norm(x, (256,), w, b, 1e-5)
    assert packed == [(64, 256), (256,), (256,), (64,), (64,)]
    assert all(torch.equal(u, v) for u, v in zip(torch.autograd.grad(y, (x, w, b), dy), want))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        y = ops.lego_layer_norm(x, (256,), w, b, 1e-5)
        got = torch.autograd.grad(y, (x, w, b), dy)
    torch.cuda.current_stream().wait_stream(side)
    assert all(torch.equal(u, v) for u, v in zip(got, want))
    y = ops.lego_layer_norm(x, (256,), w, b, 1e-5)
    with torch.no_grad():
        w.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward(dy)
    with torch.no_grad():
        assert not ops.lego_layer_norm(x, (256,), w, b, 1e-5).requires_grad
    # not for the node in C++: an eps that is no float, a transposed matrix, a subclass, forward mode, a dispatch mode, vmap
    node = runtime.layernorm_node().apply
    assert node(x, (256,), w, b, 1) is None and node(x, [256], w, b, 1e-5) is None
    assert node(torch.randn(256, 64, device="cuda").half().t(), (256,), w, b, 1e-5) is None
    assert node(x.detach().as_subclass(type("Sub", (torch.Tensor,), {})), (256,), w, b, 1e-5) is None
    assert torch.equal(ops.lego_layer_norm(x, [256], w, b, 1e-5), ops.LEGOLayerNorm.apply(x, (256,), w, b, 1e-5))
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x.detach(), dy)
        assert node(dual, (256,), w, b, 1e-5) is None
    from torch.utils._python_dispatch import TorchDispatchMode

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    with Mode():
        assert node(x, (256,), w, b, 1e-5) is None
    for call in (ops.lego_layer_norm, ops.LEGOLayerNorm.apply):
        with pytest.raises(Exception):
            torch.vmap(lambda t: call(t, (256,), w.detach(), b.detach(), 1e-5))(x.detach()[None])


@pytest.mark.gpu
@pytest.mark.parametrize("eps", [-1.0, -1e-3, float("nan")])
def test_gpu_refused_eps_keeps_its_error(eps):
    """An eps that the entry point refuses, before anything is launched, is the error of the call in Python: its entry and code."""
    from lego_amd import ops, runtime
    print(f"layernorm node, eps {eps}", flush=True)
    x, w, b, _ = _inputs((4, 64), torch.float32)
    assert runtime.layernorm_node().apply(x, (64,), w, b, eps) is None
    with pytest.raises(runtime.LegoHipError) as refused:
        ops.lego_layer_norm(x, (64,), w, b, eps)
    assert refused.value.entry == "lego_hip_layernorm_fwd_f32" and refused.value.code == 1
    assert runtime.layernorm_node().apply(x, (64,), w, b, 0.0) is not None
