"""Grouped products whose deep problems are in parts along K: which calls are, the room they ask for, and their results.  Operands are
whole numbers whose sums are exact in fp32 and in the result."""
import ctypes

import pytest
import torch


def _room(problems):
    from lego_amd import runtime
    size, limit = ctypes.c_ulonglong(), ctypes.c_int()
    runtime.call("lego_hip_grouped_gemm_f16_room", (ctypes.c_int * (3 * len(problems)))(*sum(problems, ())), len(problems), ctypes.byref(size), ctypes.byref(limit))
    return size.value, limit.value


def _copies(problems):
    from lego_amd import runtime
    size = ctypes.c_ulonglong()
    runtime.call("lego_hip_grouped_gemm_f16_workspace_bytes", (ctypes.c_int * (3 * len(problems)))(*sum(problems, ())), len(problems), ctypes.byref(size))
    return size.value


def test_parts_where_a_chain_is_what_a_launch_waits_for():
    for problems in ([(64, 64, 4096), (512, 512, 256)], [(152, 512, 3280), (64, 64, 1920)], [(64, 72, 2577), (33, 9, 100)], [(128, 128, 2048)]):
        size, limit = _room(problems)
        tiles = 0
        for m, n, k in problems:
            depth = -(-(-(-k // 8) * 8) // 64)
            parts = -(-depth // limit)
            parts = -(-depth // -(-depth // parts))
            tiles += parts * -(-m // 128) * -(-n // 128) if parts > 1 else 0
        assert 0 < tiles <= 1024 and size == _copies(problems) + 65536 * tiles, problems
    for problems in ([(4096, 4096, 4096)], [(512, 512, 192)] * 8, [(64, 64, 2577)] + [(1024, 1024, 1024)] * 16, [(64, 64, 4096)] * 65, [(64, 64, 64)]):
        assert _room(problems) == (_copies(problems), 0), problems
    from lego_amd import runtime
    with pytest.raises(runtime.LegoHipError):
        _room([(0, 64, 64)])


_CALLS = [[(128, 128, 64 * 17)], [(1, 8, 64 * 33 + 8), (130, 136, 64 * 20), (64, 64, 8)],
          [(300, 264, 64 * 24), (129, 128, 64 * 5 + 16), (64, 520, 64 * 31)], [(64, 72, 2577), (33, 9, 100), (200, 160, 1984)],
          [(8, 65, 4111), (64, 64, 4096), (5, 127, 2049), (128, 8, 512)], [(16 + i, 64, 64 * (i % 40 + 1)) for i in range(64)]]


@pytest.mark.gpu
@pytest.mark.parametrize("problems", _CALLS)
def test_gpu_parts(problems):
    """Parts of equal and of unequal length beside whole problems, ragged rows and k-tiles, as many problems as a launch carries; with room for
    the copies alone the same results from whole chains, and nothing written past the room."""
    from lego_amd import ops, runtime
    print(f"grouped in parts, {len(problems)} problems", flush=True)
    size, limit = _room(problems)
    assert limit > 0
    g = torch.Generator().manual_seed(len(problems))
    a = [(torch.randint(-2, 3, (m, k), generator=g) * (torch.rand(m, k, generator=g) < 200.0 / k)).half() for m, _, k in problems]
    b = [torch.randint(-2, 3, (k, n), generator=g).half() for _, n, k in problems]
    want = [(x.float() @ y.float()).half() for x, y in zip(a, b)]
    ad, bd = [x.cuda() for x in a], [y.cuda() for y in b]
    for c, w in zip(ops.lego_group_gemm_fn(ad, bd), want):
        assert torch.equal(c.cpu(), w)
    pointers = lambda ts: (ctypes.c_void_p * len(ts))(*[t.data_ptr() for t in ts])
    for room in (size, _copies(problems)):
        ws = torch.full((room + 64,), 0x5a, dtype=torch.uint8, device="cuda")
        cd = [torch.full_like(w, 9, device="cuda") for w in want]
        runtime.call("lego_hip_grouped_gemm_f16_ws", pointers(ad), pointers(bd), pointers(cd), (ctypes.c_int * (3 * len(problems)))(*sum(problems, ())),
                     len(problems), ws.data_ptr(), room, None)
        assert all(torch.equal(c.cpu(), w) for c, w in zip(cd, want)) and (ws[room:] == 0x5a).all()
