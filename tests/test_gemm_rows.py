"""Products of up to sixteen rows against a transposed B, which a kernel of their own takes: every element type, ragged columns, a last
line of k that is not whole, fewer lines than wavefronts.  Small whole numbers: sums are exact in any order."""
import pytest
import torch


def _columns(M, N, K, bytes, ta=0, tb=1):
    import ctypes
    from lego_amd import runtime
    columns = ctypes.c_int(-1)
    runtime.call("lego_hip_gemm_rows_plan", M, N, K, ta, tb, bytes, ctypes.byref(columns))
    return columns.value


def test_columns_of_a_workgroup_and_where_tiles_stay():
    assert _columns(16, 4096, 4096, 2) == 16 and _columns(16, 8192, 8192, 2) == 32 and _columns(16, 16384, 8192, 2) == 64
    for N in range(8256, 8192 + 1024, 64):        # one round of 32 columns and a little: no second round nearly empty
        assert _columns(1, N, 4096, 2) == 16 and _columns(16, N, 4096, 2) != 32
    for M in (1, 16):
        assert _columns(M, 4096, 128, 2) == _columns(M, 4096, 256, 1) == 0 and _columns(M, 4096, 512, 1) == 16       # next to nothing to read
        assert _columns(M, 1024, 8192, 2) == 0                                   # K long beside N
        assert _columns(M, 65536, 4096, 2) == 0                                  # tiles fill the chip
        assert _columns(M, 4096, 4096, 2, ta=1) == _columns(M, 4096, 4096, 2, tb=0) == _columns(17, 4096, 4096, 2) == 0
    assert _columns(8, 40960, 4096, 2) and not _columns(9, 40960, 4096, 2)
    assert _columns(8, 2048, 6144, 2) and not _columns(9, 2048, 6144, 2)         # more rows: A is read too often
    assert _columns(8, 8448, 10240, 2) and not _columns(9, 8448, 10240, 2)
    assert _columns(8, 5120, 5120, 2) and not _columns(9, 5120, 5120, 2) and _columns(9, 5120, 4096, 2) and _columns(9, 5120, 8192, 1)
    assert _columns(1, 4 << 20, 16 << 20, 1) == 0                                # rows beyond a descriptor


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,out", [(torch.float16, torch.float16), (torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float16),
                                       (torch.float8_e4m3fn, torch.float16), (torch.float8_e5m2, torch.float16)])
@pytest.mark.parametrize("M,N,K", [(1, 1024, 16), (16, 1024, 64), (3, 1040, 528), (16, 1032, 4096), (7, 4096, 1040), (15, 6160, 272), (16, 6176, 2064),
                                   (3, 8264, 512), (16, 16392, 592), (9, 24584, 528)])
def test_gpu_few_rows_against_a_transposed_matrix(dtype, out, M, N, K):
    from lego_amd import ops
    print(f"gemm rows {dtype} {M}x{N}x{K}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randint(-1, 2, (M, K), generator=g).float() * (torch.rand(M, K, generator=g) < 100.0 / K)
    b = torch.randint(-1, 2, (K, N), generator=g).float()
    want = a @ b
    assert want.abs().max() <= 256
    bd = b.t().contiguous().to(dtype).cuda().t()
    got = ops.matmul(a.to(dtype).cuda(), bd, out_dtype=out)
    assert got.dtype == out and torch.equal(got.cpu().float(), want)
    leaky = torch.where(want >= 0, want, 0.01 * want)
    got = ops.matmul(a.to(dtype).cuda(), bd, activation="leaky_relu", out_dtype=out).cpu().float()
    assert (got - leaky).abs().max() <= 256 * 0.01 * 2.0 ** (-8 if out == torch.bfloat16 else -11)


@pytest.mark.gpu
def test_gpu_row_past_the_matrix_reaches_nothing():
    """Infinities around the operands (the same storage, before and after) stay out of every sum; nothing is written past C."""
    import ctypes
    from lego_amd import runtime
    print("gemm rows, infinities around the operands", flush=True)
    M, N, K = 5, 1032, 72
    def inside(t):
        buf = torch.full((t.numel() + 256,), float("inf"), dtype=torch.float16, device="cuda")
        buf[128:128 + t.numel()] = t.reshape(-1).cuda()
        return buf, buf.data_ptr() + 256
    a, b = torch.ones(M, K).half(), torch.ones(N, K).half()
    (ab, ap), (bb, bp) = inside(a), inside(b)
    c = torch.full((M * N + 256,), 7.0, dtype=torch.float16, device="cuda")
    runtime.call("lego_hip_gemm_f16_ex", ap, bp, c.data_ptr() + 256, M, N, K, 0, 1, 0, None)
    assert (c[128:128 + M * N] == K).all() and (c[:128] == 7).all() and (c[128 + M * N:] == 7).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e5m2])
def test_gpu_few_rows_allocate_the_result_alone(dtype):
    """No room for partial sums that the kernel for few rows does not form; the same product against a row-major B still has it."""
    from lego_amd import ops
    print(f"gemm rows, memory, {dtype}", flush=True)
    a, b = torch.zeros(16, 4096, device="cuda").to(dtype), torch.zeros(4096, 4096, device="cuda").to(dtype)

    def peak(b):
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        c = ops.matmul(a, b)
        del c
        return torch.cuda.max_memory_allocated() - before
    assert peak(b.t()) == 2 * 16 * 4096 < peak(b)
