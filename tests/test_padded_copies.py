"""Products whose operand rows are not whole 16-byte chunks, on zero-padded copies: 8-bit ones, and grouped calls with such problems
among others.  Small whole numbers: every sum is exact, whatever the workspace held."""
import ctypes

import pytest
import torch


def _size(entry, *args):
    from lego_amd import runtime
    need = ctypes.c_ulonglong(0)
    runtime.call(entry, *args, ctypes.byref(need))
    return need.value


def test_padded_sizes_hold_the_copies():
    for M, N, K, ta, tb in ((17, 65, 4000, 0, 0), (320, 1984, 7959, 0, 1), (33, 64, 512, 1, 0), (5000, 3001, 100, 0, 0)):
        r = lambda v: (v + 15) // 16 * 16
        need = _size("lego_hip_gemm_fp8_padded_bytes", M, N, K, ta, tb)
        assert need >= r(M) * r(K) + r(K) * r(N) + 2 * r(M) * r(N) and need % 16 == 0
    for M, N, K, ta, tb in ((33, 64, 512, 0, 0), (64, 64, 512, 1, 1), (32, 64, 4104, 1, 0), (100, 100, 100, 0, 0)):     # whole chunks, or too little work
        assert _size("lego_hip_gemm_fp8_padded_bytes", M, N, K, ta, tb) == 0
    sizes = (ctypes.c_int * 9)(64, 64, 64, 5, 9, 17, 100, 64, 63)
    assert _size("lego_hip_grouped_gemm_f16_workspace_bytes", sizes, 3) == 2 * (8 * 24 + 24 * 16 + 8 * 16 + 104 * 64 + 64 * 64 + 104 * 64)
    assert _size("lego_hip_grouped_gemm_f16_workspace_bytes", sizes, 1) == 0


def test_copies_of_a_grouped_call_take_bounded_room():
    """Sixteen ragged products of 4095 a side: copies of five of them at a time, not of all sixteen (1.6 GB)."""
    one = 3 * 2 * 4096 * 4096
    for count, need in ((1, one), (5, 5 * one), (16, 5 * one)):
        sizes = (ctypes.c_int * (3 * count))(*[4095] * (3 * count))
        assert _size("lego_hip_grouped_gemm_f16_workspace_bytes", sizes, count) == need
    sizes = (ctypes.c_int * 9)(20000, 20001, 64, 2000, 9999, 16, 64, 64, 64)       # one beyond the bound keeps its own room
    assert _size("lego_hip_grouped_gemm_f16_workspace_bytes", sizes, 3) == 2 * (20000 * 64 + 64 * 20008 + 20000 * 20008)


def _apart(*problems):
    from lego_amd import runtime
    flags = (ctypes.c_int * len(problems))()
    runtime.call("lego_hip_grouped_gemm_f16_apart", (ctypes.c_int * (3 * len(problems)))(*sum(problems, ())), len(problems), flags)
    return [i for i, f in enumerate(flags) if f]


def test_deep_problems_leave_a_grouped_call_by_the_work_beside_them():
    """A ragged problem's chain of k-tiles runs beside the others' work, however many they are, or in parts on its own."""
    for few in (2, 3, 5):
        assert _apart(*[(64, 64, 64)] * few, (64, 64, 4095)) == [few]              # next to nothing beside it
        assert _apart((512, 512, 8191), *[(512, 512, 512)] * few) == [0]
    assert _apart(*[(64, 64, 64)] * 15, (64, 64, 4095)) == [15]                     # many, and still nothing
    assert _apart(*[(1024, 1024, 1024)] * 16, (64, 64, 2577)) == []                 # a chain beside rounds of tiles
    assert _apart(*[(64, 64, 4095)] * 4) == []                                      # chains beside each other
    assert _apart(*[(3001, 2999, 3003)] * 8) == []                                  # rounds of the whole chip
    assert _apart(*[(64, 64, 4096)] * 4) == [] and _apart((64, 65, 1984), (64, 64, 64)) == []      # whole chunks, or not split
    assert _apart(*[(64, 64, 64)] * 100, (64, 64, 16383)) == [100]                  # more than a launch carries


@pytest.mark.gpu
@pytest.mark.parametrize("fp8", [torch.float8_e5m2, torch.float8_e4m3fn])
@pytest.mark.parametrize("M,N,K", [(1, 65, 257), (17, 64, 4097), (33, 100, 264), (128, 129, 256), (1000, 1001, 271), (2500, 3001, 72)])
def test_gpu_8bit_products_of_any_shape(fp8, M, N, K):
    from lego_amd import ops, runtime
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randint(-1, 2, (M, K), generator=g).float() * (torch.randint(0, 4, (M, K), generator=g) == 0)
    b = torch.randint(-1, 2, (K, N), generator=g).float()
    want = a @ b
    assert want.abs().max() < 2048
    for ta in (0, 1):
        for tb in (0, 1):
            print(f"8-bit on copies {fp8} {M}x{N}x{K} ta={ta} tb={tb}", flush=True)
            a8 = a.to(fp8).t().contiguous().cuda() if ta else a.to(fp8).cuda()
            b8 = b.to(fp8).t().contiguous().cuda() if tb else b.to(fp8).cuda()
            assert torch.equal(ops.matmul(a8.t() if ta else a8, b8.t() if tb else b8).cpu().float(), want)
            need = _size("lego_hip_gemm_fp8_padded_bytes", M, N, K, ta, tb)
            if not need:
                continue
            # a workspace full of NaN, operands and result at any element, nothing written around the result
            ws = torch.full((need,), 0x7f, dtype=torch.uint8, device="cuda")
            ad, bd = (torch.cat([t.view(torch.uint8).new_zeros(3), t.view(torch.uint8).reshape(-1)])[3:] for t in (a8, b8))
            c = torch.full((M * N + 64,), 7.0, dtype=torch.float16, device="cuda")
            runtime.call("lego_hip_gemm_fp8_padded", ad.data_ptr(), bd.data_ptr(), c.data_ptr() + 2 * 29, M, N, K, ta, tb, 0,
                         0 if fp8 == torch.float8_e4m3fn else 1, ws.data_ptr(), need, None)
            assert torch.equal(c[29:29 + M * N].view(M, N).cpu().float(), want)
            assert (c[:29] == 7).all() and (c[29 + M * N:] == 7).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,transposed_first", [(5, 520, 1023, False), (5, 521, 1024, False), (5, 520, 1024, True), (67, 520, 1023, True), (5, 520, 376, False), (5, 1030, 1601, True),
                                                      (5, 1030, 1201, False), (5, 1030, 2101, False), (5, 520, 1601, False)])
def test_gpu_column_major_rows_of_no_whole_chunks(M, N, K, transposed_first, monkeypatch):
    """A small column-major A is stored row-major first where the product would run by elements, not where copies take it."""
    from lego_amd import ops
    print(f"tn {M}x{N}x{K}", flush=True)
    calls, transpose = [], ops.transpose
    monkeypatch.setattr(ops, "transpose", lambda t: calls.append(t.shape) or transpose(t))
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randint(-1, 2, (M, K), generator=g).half()
    b = torch.randint(-1, 2, (K, N), generator=g).half()
    got = ops.matmul(a.t().contiguous().cuda().t(), b.t().contiguous().cuda().t() if N > 1024 else b.cuda())
    assert torch.equal(got.cpu().float(), a.float() @ b.float()) and bool(calls) == transposed_first


@pytest.mark.gpu
def test_gpu_grouped_in_runs_of_bounded_copies():
    """Copies of 680 MB in all, in two runs through the same room, with whole-chunk problems among them; nothing beyond the room is written."""
    from lego_amd import ops, runtime
    print("grouped, copies in runs", flush=True)
    problems = [(90000, 1001, 9), (64, 64, 64), (90000, 1001, 17), (90000, 1999, 33), (8, 16, 8), (33, 72, 63)]
    g = torch.Generator(device="cuda").manual_seed(5)
    a = [torch.randint(-2, 3, (m, k), device="cuda", generator=g).half() for m, _, k in problems]
    b = [torch.randint(-2, 3, (k, n), device="cuda", generator=g).half() for _, n, k in problems]
    want = [(x.float() @ y.float()).half() for x, y in zip(a, b)]
    for c, w in zip(ops.lego_group_gemm_fn(a, b), want):
        assert torch.equal(c, w)
    sizes = (ctypes.c_int * 18)(*sum(problems, ()))
    need = _size("lego_hip_grouped_gemm_f16_workspace_bytes", sizes, 6)
    assert need <= 512 << 20 < sum(2 * 8 * -(-m // 8) * 8 * -(-n // 8) for m, n, _ in problems if n % 8)
    ws = torch.full((need + 64,), 0x5a, dtype=torch.uint8, device="cuda")
    c = [torch.zeros_like(w) for w in want]
    pointers = lambda ts: (ctypes.c_void_p * 6)(*[t.data_ptr() for t in ts])
    runtime.call("lego_hip_grouped_gemm_f16_ws", pointers(a), pointers(b), pointers(c), sizes, 6, ws.data_ptr(), need, None)
    assert all(torch.equal(x, w) for x, w in zip(c, want)) and (ws[need:] == 0x5a).all()


@pytest.mark.gpu
@pytest.mark.parametrize("problems", [[(1, 65, 64), (64, 64, 64), (33, 72, 63)], [(5, 9, 2111), (64, 64, 64), (130, 1, 1)],
                                      [(9, 31, 2050), (64, 64, 64), (33, 72, 63), (3, 8, 8)],
                                      [(64, 64, 64), (9, 31, 8190), (33, 72, 63), (3, 8, 8), (17, 8, 4100)], [(65, 63, 100)],
                                      [(16 + i, 63 + i, 65 + i) for i in range(70)]])
def test_gpu_grouped_with_ragged_problems(problems):
    """Problems of whole chunks and others, deep ones, and more than the launches of the copies and of the products carry."""
    from lego_amd import ops
    print(f"grouped, {len(problems)} problems", flush=True)
    g = torch.Generator().manual_seed(len(problems))
    a = [torch.randint(-2, 3, (m, k), generator=g).half() * (torch.rand(m, k, generator=g) < 200.0 / k).half() for m, _, k in problems]
    b = [torch.randint(-2, 3, (k, n), generator=g).half() for _, n, k in problems]
    for x, y, c in zip(a, b, ops.lego_group_gemm_fn([x.cuda() for x in a], [y.cuda() for y in b])):
        assert torch.equal(c.cpu().double(), x.double() @ y.double())
