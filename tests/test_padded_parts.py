"""Products on zero-padded copies that are split along K: the sums stay inside the workspace that is asked for."""
import ctypes

import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(130, 130, 8200), (130, 136, 8201), (129, 200, 4097), (7, 65, 4000), (257, 250, 3001)])
def test_sums_stay_in_the_workspace(M, N, K):
    """M that is no multiple of 8, where M rounded up has another number of parts: 130 x 136 x 8200 43, 136 x 136 x 8200 33."""
    from lego_amd import runtime
    print(f"sums on padded copies {M}x{N}x{K}", flush=True)
    need = ctypes.c_ulonglong(0)
    for room in ("lego_hip_gemm_workspace_bytes", "lego_hip_gemm_layout_workspace_bytes"):
        runtime.call(room, M, N, K, *((0, 1, 2) if "layout" in room else ()), ctypes.byref(need))
        assert need.value > 0
        a, b = torch.randint(-2, 3, (M, K)).half(), torch.randint(-2, 3, (N, K)).half()
        a = a * (torch.rand(M, K) < 200.0 / K)
        guard = 64 << 20      # more than all parts that any estimate gives
        ws = torch.full((need.value + guard,), 85, dtype=torch.uint8, device="cuda")
        ad, bd, c = a.cuda(), b.cuda(), torch.empty(M, N, dtype=torch.half, device="cuda")
        runtime.call("lego_hip_gemm_ex_ws", 0, ad.data_ptr(), bd.data_ptr(), c.data_ptr(), M, N, K, 0, 1, 0, ws.data_ptr(), need.value,
                     torch.cuda.current_stream().cuda_stream)
        assert torch.equal(c.cpu().double(), a.double() @ b.double().t())
        assert (ws[need.value:] == 85).all()


def test_a_large_operand_in_whole_chunks_is_no_copy():
    """Ragged columns against a large A that is read where it is: on copies of the rest, not by the kernel for any shape; a ragged K keeps that one."""
    from lego_amd import runtime
    need = ctypes.c_ulonglong(0)
    for M, N, K, copies in ((6174, 68, 5808, True), (7452, 277, 5680, True), (6831, 315, 3176, True), (7778, 110, 2114, False), (1073, 427, 2368, False)):
        runtime.call("lego_hip_gemm_layout_workspace_bytes", M, N, K, 0, 1, 2, ctypes.byref(need))
        assert (need.value > 0) == copies, (M, N, K)
