"""Products of few tiles whose K is past the reach of a buffer descriptor (128 rows of 2 GiB and more): in parts along K as shorter ones, on two operand buffers.
A quarter or less of A is not zero, so that sums of whole numbers are exact in fp32 and in the result."""
import ctypes

import pytest
import torch

F16, E5M2 = torch.float16, torch.float8_e5m2


def _room(M, N, K, ta, tb, size):
    from lego_amd import runtime
    out = ctypes.c_ulonglong(0)
    runtime.call("lego_hip_gemm_layout_workspace_bytes", M, N, K, ta, tb, size, ctypes.byref(out))
    return out.value


@pytest.mark.parametrize("M,N,K,size,parts", [(64, 64, 1 << 23, 2, 64), (16, 128, (1 << 24) + 16, 1, 64), (1, 2048, 1 << 23, 2, 32), (16384, 16, 1 << 23, 2, 4),
                                              (128, 128 * 128, 1 << 23, 2, 4), (128, 129 * 128, 1 << 23, 2, 0)])
def test_far_products_have_room_for_parts(M, N, K, size, parts):
    tiles = -(-M // 128) * -(-N // 128)
    assert _room(M, N, K, 0, 0, size) == parts * tiles * 65536


def test_far_products_on_copies_have_room_for_parts():
    M, N, K = 16, 63, (1 << 23) + 1
    assert _room(M, N, K, 0, 0, 2) == 2 * (M * (K + 7) + (K + 7) * 64 + M * 64) + 64 * 65536


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,M,N,K,ta,tb", [(F16, 16, 64, (1 << 23) + 8, 0, 0), (F16, 40, 24, 1 << 23, 0, 1), (F16, 16, 63, (1 << 23) + 1, 0, 0),
                                               (E5M2, 32, 16, (1 << 24) + 16, 0, 0), (E5M2, 16, 48, 1 << 24, 1, 1)])
def test_gpu_far_products(dtype, M, N, K, ta, tb):
    from lego_amd import ops
    print(f"far {dtype} {M}x{N}x{K} {ta}{tb}", flush=True)
    shape = (K, M) if ta else (M, K)
    # some 200 products of -2 .. 2 a sum: below 2048 by 100 standard deviations
    a = (torch.randint(-1, 2, shape, device="cuda", dtype=torch.int8) * (torch.rand(shape, device="cuda") < 300.0 / K)).to(dtype)
    b = torch.randint(-2, 3, (N, K) if tb else (K, N), device="cuda", dtype=torch.int8).to(dtype)
    a[0, 0] = a[-1, -1] = 1      # both ends of K
    a, b = a.t() if ta else a, b.t() if tb else b
    want = sum(a[:, k:k + (1 << 20)].float() @ b[k:k + (1 << 20)].float() for k in range(0, K, 1 << 20))
    assert torch.equal(ops.matmul(a, b).float(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,M,N,K,ta,tb", [(F16, 24, 8192, 8192, 0, 1), (F16, 64, 8192, 8160, 1, 1), (F16, 8192, 40, 8192, 0, 0), (E5M2, 24, 8192, 16384, 0, 1),
                                               (F16, 24, 8191, 8185, 0, 1)])
def test_gpu_three_quarters_of_the_parts(dtype, M, N, K, ta, tb):
    """Parts of a multiple of 32 k-tiles along k-major operands: the launch takes fewer of them than there is room for."""
    from lego_amd import ops
    print(f"parts {dtype} {M}x{N}x{K} {ta}{tb}", flush=True)
    shape = (K, M) if ta else (M, K)
    a = (torch.randint(-1, 2, shape, device="cuda", dtype=torch.int8) * (torch.rand(shape, device="cuda") < 300.0 / K)).to(dtype)
    b = torch.randint(-2, 3, (N, K) if tb else (K, N), device="cuda", dtype=torch.int8).to(dtype)
    a, b = a.t() if ta else a, b.t() if tb else b
    assert torch.equal(ops.matmul(a, b).float(), a.float() @ b.float())
