"""Products on 128 x 128 tiles with four operand buffers in LDS: as many k-tiles as the buffers and one more or fewer, edges of
tiles and k-tiles, sums along K in parts.  Operands are whole numbers whose sums are exact in fp32 and in the result."""
import ctypes

import pytest
import torch

_BYTES = {torch.float16: 2, torch.bfloat16: 2, torch.float8_e5m2: 1, torch.float8_e4m3fn: 1}


def _plan(M, N, K, element_bytes=2):
    from lego_amd import runtime
    out = (ctypes.c_int * 2)()
    runtime.call("lego_hip_gemm_parts_plan", M, N, K, element_bytes, out)
    return tuple(out)


def test_parts_and_buffers_follow_the_measured_crossovers():
    assert _plan(512, 512, 512) == (1, 4) and _plan(1024, 1024, 1024) == (1, 4) and _plan(512, 512, 1024)[0] > 2
    assert _plan(2048, 2048, 2048) == (1, 4) and _plan(2049, 2048, 2048) == (1, 2)            # a tile per CU, and more
    assert _plan(1024, 2048, 3584) == (2, 4) and _plan(1000, 2048, 2048, 1) == (1, 4)
    assert _plan(64, 64, 1 << 20)[0] == 64 and _plan(64, 64, 1 << 23) == (1, 2)               # past a descriptor's reach
    for M, N, K, size in ((1, 64, 64, 2), (1, 64, 4096, 2), (1408, 1408, 8192, 2), (256, 2048, 4096, 1), (16, 8192, 8192, 2)):
        parts, depth = _plan(M, N, K, size)[0], -(-K * size // 128)
        assert parts == 1 or (parts * -(-M // 128) * -(-N // 128) <= 256 and 2 * parts <= depth)
    from lego_amd import runtime
    with pytest.raises(runtime.LegoHipError):
        _plan(1, 1, 1, 4)


def _operands(M, N, K, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    # a quarter of A's values is not zero: sums of up to 4500 products stay below 2048 by 40 standard deviations; in {0, +-1}, so that a
    # bfloat16 result of up to 256 is exact too where its sum is
    a = torch.randint(-1, 2, (M, K), generator=g).float() * (torch.randint(0, 4, (M, K), generator=g) == 0)
    b = torch.randint(-1, 2, (K, N), generator=g).float()
    return a, b, (a @ b).to(torch.bfloat16 if dtype == torch.bfloat16 else torch.float16)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", list(_BYTES))
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_gpu_every_depth_around_the_buffers(dtype, layout):
    from lego_amd import ops
    chunk, bk = 16 // _BYTES[dtype], 128 // _BYTES[dtype]
    for tiles, rest in ((1, 0), (1, chunk), (2, 0), (3, 0), (3, chunk), (4, 0), (4, chunk), (5, 0), (6, chunk), (9, 0)):
        for M, N in ((128, 128), (chunk, chunk), (128 + chunk, 256 - chunk)):
            K = tiles * bk + rest
            assert _plan(M, N, K, _BYTES[dtype]) == (1, 4)
            a, b, want = _operands(M, N, K, dtype, K)
            print(f"gemm four buffers {dtype} {layout} {M}x{N}x{K}", flush=True)
            ad = (a.t().contiguous().to(dtype).cuda().t() if layout[0] == "t" else a.to(dtype).cuda())
            bd = (b.t().contiguous().to(dtype).cuda().t() if layout[1] == "t" else b.to(dtype).cuda())
            got = ops.matmul(ad, bd, out_dtype=want.dtype)
            assert torch.equal(got.cpu(), want), (M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float8_e5m2])
@pytest.mark.parametrize("M,N,K128", [(1, 16, 16), (128, 144, 17), (256, 256, 21), (48, 2048, 33), (320, 64, 36)])
def test_gpu_sums_in_parts(dtype, M, N, K128):
    """Depths (of 128 bytes a row) from where parts begin, whole and with a ragged last k-tile, parts of unequal lengths."""
    from lego_amd import ops
    for K in (K128 * 128 // _BYTES[dtype], K128 * 128 // _BYTES[dtype] + 16 // _BYTES[dtype]):
        assert _plan(M, N, K, _BYTES[dtype])[0] > 1
        a, b, want = _operands(M, N, K, dtype, K)
        for ta, tb in ((0, 0), (1, 1) if M % 16 == 0 else (0, 0)):
            print(f"gemm in parts {dtype} {M}x{N}x{K} {ta}{tb}", flush=True)
            ad = a.t().contiguous().to(dtype).cuda().t() if ta else a.to(dtype).cuda()
            bd = b.t().contiguous().to(dtype).cuda().t() if tb else b.to(dtype).cuda()
            assert torch.equal(ops.matmul(ad, bd, out_dtype=want.dtype).cpu(), want)
            leaky = torch.where(want.float() >= 0, want.float(), 0.01 * want.float())
            got = ops.matmul(ad, bd, activation="leaky_relu", out_dtype=want.dtype).cpu().float()
            assert (got - leaky).abs().max() <= 2048 * 0.01 * 2.0 ** (-8 if want.dtype == torch.bfloat16 else -11)


@pytest.mark.gpu
def test_gpu_grouped_problems_of_many_depths():
    """Ragged tiles and k-tiles, one to seven k-tiles deep, in one launch with a workgroup per CU."""
    from lego_amd import ops
    sizes = [(1, 8, 8), (128, 128, 64), (130, 136, 200), (256, 8, 192), (5, 264, 256), (300, 304, 320), (64, 64, 448)]
    made = [_operands(*s, torch.float16, i) for i, s in enumerate(sizes)]
    print("grouped four buffers", flush=True)
    got = ops.lego_group_gemm_fn([a.half().cuda() for a, _, _ in made], [b.half().cuda() for _, b, _ in made])
    assert all(torch.equal(c.cpu(), want) for c, (_, _, want) in zip(got, made))
