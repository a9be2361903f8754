"""The kernel for products of any shape and alignment, at the edges of what it reads in vectors: small whole numbers, so that every sum
is exact, between NaNs that any element from outside an operand would bring into the result."""
import ctypes

import pytest
import torch

F16, BF16, E5M2, E4M3 = torch.float16, torch.bfloat16, torch.float8_e5m2, torch.float8_e4m3fn


def _room(M, N, K, ta, tb, size):
    from lego_amd import runtime
    need = ctypes.c_ulonglong(0)
    runtime.call("lego_hip_gemm_layout_workspace_bytes", M, N, K, ta, tb, size, ctypes.byref(need))
    return need.value


def test_small_ragged_products_need_no_copies_and_deep_ones_do():
    for size in (1, 2):
        for M, N, K, ta, tb in ((64, 852, 65, 1, 0), (55, 511, 93, 1, 1), (9, 781, 577, 0, 1), (1, 1, 1, 0, 0)):
            assert _room(M, N, K, ta, tb, size) == 0
        for M, N, K, ta, tb in ((496, 135, 3878, 0, 0), (1618, 2024, 485, 0, 1), (3001, 2999, 3003, 1, 1)):
            assert _room(M, N, K, ta, tb, size) >= size * (M * K + K * N) + 2 * M * N
    assert _room(64, 64, 64, 0, 0, 2) == 0 and _room(16, 16, 8192, 0, 0, 2) > 0       # whole chunks: parts as before


def _entry(dtype, a, b, c, M, N, K, ta, tb, activation=0, stream=0):
    from lego_amd import runtime
    stream = torch.cuda.current_stream().cuda_stream if stream == 0 else stream
    if dtype in (E5M2, E4M3):
        runtime.call("lego_hip_gemm_fp8_ex", a, b, c, M, N, K, ta, tb, activation, int(dtype == E5M2), stream)
    else:
        runtime.call("lego_hip_gemm_f16_ex" if dtype == F16 else "lego_hip_gemm_bf16_f16_ex", a, b, c, M, N, K, ta, tb, activation, stream)


_TALL = [(F16, 4194305, 63, 63, 0), (BF16, 4194241, 9, 130, 0), (E4M3, 4194310, 60, 33, 1), (E5M2, 4200000, 63, 41, 0)]


@pytest.mark.parametrize("dtype,M,N,K,ta", _TALL)
def test_more_rows_of_tiles_than_a_grid_dimension_has_are_taken(dtype, M, N, K, ta):
    """Without a GPU a call that is taken gets as far as the launch, which finds no device; one that is refused does not."""
    from lego_amd import runtime
    if torch.cuda.is_available():
        pytest.skip("the operands are addresses of nothing")
    assert _room(M, N, K, ta, 0, torch.finfo(dtype).bits // 8) == 0 < _room(5000000, 100, 60, 0, 0, 2)      # A of 600 MB in two columns of tiles
    with pytest.raises(runtime.LegoHipError) as refused:
        _entry(dtype, 1 << 20, 1 << 21, 1 << 22, M, N, K, ta, 0, stream=None)
    assert refused.value.code == 100      # hipErrorNoDevice


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,M,N,K,ta", _TALL)
def test_gpu_more_rows_of_tiles_than_a_grid_dimension_has(dtype, M, N, K, ta):
    """Whole numbers, exact in every type: every row of a product of 65537 rows of tiles and more, the last one ragged."""
    from lego_amd import ops
    print(f"tall {dtype} {M}x{N}x{K} {ta}", flush=True)
    a = torch.randint(-2, 3, (K, M) if ta else (M, K), device="cuda", dtype=torch.int8).to(dtype)
    b = torch.randint(-2, 3, (K, N), device="cuda").to(dtype)
    a = a.t() if ta else a
    got = ops.matmul(a, b)
    for first in range(0, M, 1 << 20):
        rows = slice(first, first + (1 << 20))
        assert torch.equal(got[rows].float(), a[rows].float() @ b.float()), first


def _between(t, dtype, before, after=16):
    """``t`` row-major inside a buffer of NaNs, ``before`` elements in."""
    flat = torch.full((before + t.numel() + after,), float("nan")).to(dtype)
    flat[before:before + t.numel()] = t.contiguous().view(-1).to(dtype)
    return flat.cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F16, BF16, E5M2, E4M3])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (1, 2, 129), (3, 1, 193), (2, 3, 64), (5, 7, 65), (4, 68, 128), (63, 65, 127), (65, 62, 192),
                                   (66, 130, 321), (17, 9, 576), (130, 67, 640), (1, 64, 67)])
def test_any_shape_reads_nothing_outside_its_operands(dtype, M, N, K):
    """One row or column, K about whole k-tiles of 64 and turns of four of them, sides about whole fours and tiles of 64."""
    g = torch.Generator().manual_seed(M + N + K)
    a, b = torch.randint(-3, 4, (M, K), generator=g).float(), torch.randint(-3, 4, (K, N), generator=g).float()
    a[:, 4:] *= torch.rand(max(K - 4, 0), generator=g) < 100.0 / K      # sums below 2048: exact in fp16
    want = (a.double() @ b.double()).half()
    assert want.abs().max() < 2048
    size = 1 if dtype in (E5M2, E4M3) else 2
    for ta in (0, 1):
        for tb in (0, 1):
            for before in (1, 16):
                ad, bd = _between(a.t() if ta else a, dtype, before), _between(b.t() if tb else b, dtype, before + 2)
                c = torch.full((M * N + 22,), 7.0, dtype=F16, device="cuda")
                print(f"{dtype} {M}x{N}x{K} {ta}{tb} {before}", flush=True)
                _entry(dtype, ad.data_ptr() + size * before, bd.data_ptr() + size * (before + 2), c.data_ptr() + 2 * 3, M, N, K, ta, tb)
                got = c.cpu()
                assert torch.equal(got[3:3 + M * N].view(M, N), want), (ta, tb, before)
                assert (got[:3] == 7).all() and (got[3 + M * N:] == 7).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [E5M2, E4M3])
def test_any_shape_widens_every_byte(dtype):
    """All 256 values of a type, infinities and NaNs among them, by elements (K = 1) and in vectors along k and along rows."""
    values = torch.arange(256, dtype=torch.uint8).view(dtype)
    want = values.float().half()
    for K in (1, 129):
        a = torch.zeros(256, K).to(dtype)
        a.view(torch.uint8)[torch.arange(256), torch.arange(256) % K] = torch.arange(256, dtype=torch.uint8)
        b = torch.ones(K, 3).to(dtype).cuda()
        for ta in (0, 1):
            c = torch.empty(256, 3, dtype=F16, device="cuda")
            ad = (a.view(torch.uint8).t().contiguous() if ta else a.view(torch.uint8)).cuda()
            _entry(dtype, ad.data_ptr(), b.data_ptr(), c.data_ptr(), 256, 3, K, ta, 0)
            got = c.cpu()
            for col in range(3):
                assert torch.equal(got[:, col].isnan(), want.isnan()) and torch.equal(got[:, col].nan_to_num(9.0), want.nan_to_num(9.0)), (K, ta)
