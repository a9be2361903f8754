"""Needleman-Wunsch: the oracle is pinned on the CPU, the kernel against the oracle on the GPU."""
from pathlib import Path

import numpy as np
import pytest
import sympy as sp
import torch

from lego_amd.kernels import nw
from oracle import kernels as ok


def _loops(ref, penalty):
    n1 = ref.shape[0]
    m = [[0] * n1 for _ in range(n1)]
    for i in range(n1):
        m[i][0] = -i * penalty
        m[0][i] = -i * penalty
    for i in range(1, n1):
        for j in range(1, n1):
            m[i][j] = max(m[i - 1][j - 1] + int(ref[i, j]), m[i][j - 1] - penalty, m[i - 1][j] - penalty)
    return np.array(m, dtype=np.int32)


def test_oracle_matches_the_plain_double_loop():
    rng = np.random.default_rng(0)
    for n, penalty in ((7, 10), (16, 3), (33, 1)):
        ref = rng.integers(-4, 12, size=(n + 1, n + 1)).astype(np.int32)
        assert np.array_equal(ok.needleman_wunsch(ref, penalty), _loops(ref, penalty))


def test_oracle_closed_form_without_substitution_scores():
    """With zero scores a diagonal step is free and a gap costs ``penalty``: m[i][j] = -|i-j|*penalty."""
    n = 40
    got = ok.needleman_wunsch(np.zeros((n + 1, n + 1), dtype=np.int32), 7)
    i, j = np.meshgrid(np.arange(n + 1), np.arange(n + 1), indexing="ij")
    assert np.array_equal(got, -np.abs(i - j) * 7)


def test_rotation_through_lds_is_free_of_bank_conflicts():
    """Slot k of lane tx is row (k - tx) mod 64 of column tx: in the kernel's LDS tile the 64 lanes
    of every such access, and of every row access, fall into 64 different banks."""
    b = nw.B
    i, j = sp.symbols("i j", integer=True, nonnegative=True)
    f = sp.lambdify([i, j], nw.rotation_layout()[i, j], "math")
    words = set()
    for k in range(b):
        slots = [int(f((k - tx) % b, tx)) for tx in range(b)]
        assert len({w % 64 for w in slots}) == 64
        words.update(slots)
        assert len({int(f(k, tx)) % 64 for tx in range(b)}) == 64
    assert words == set(range(b * b))


def test_tile_layout_is_the_anti_diagonal_enumeration():
    """The reference's layout of the tile (nw_sympy.py:9-11): a bijection of the 64 x 64 tile in
    which the cells of one anti-diagonal are consecutive and ordered by row."""
    b = nw.B
    i, j = sp.symbols("i j", integer=True, nonnegative=True)
    f = sp.lambdify([i, j], nw.tile_layout()[i, j], "math")
    table = np.array([[int(f(a, c)) for c in range(b)] for a in range(b)])
    assert sorted(table.ravel().tolist()) == list(range(b * b))
    pos = 0
    for d in range(2 * b - 1):
        for a in range(max(0, d - b + 1), min(d, b - 1) + 1):
            assert table[a, d - a] == pos
            pos += 1


@pytest.mark.gpu
@pytest.mark.parametrize("n,penalty", [(64, 10), (256, 10), (1024, 3), (2048, 10)])
def test_gpu_matches_oracle(n, penalty):
    from lego_amd import ops
    print(f"needleman-wunsch n={n} penalty={penalty}", flush=True)
    g = torch.Generator().manual_seed(20 + n)
    ref = torch.randint(-4, 12, (n + 1, n + 1), generator=g, dtype=torch.int32)
    want = torch.from_numpy(ok.needleman_wunsch(ref.numpy(), penalty))
    m = torch.zeros((n + 1, n + 1), dtype=torch.int32)
    m[:, 0] = -torch.arange(n + 1, dtype=torch.int32) * penalty
    m[0, :] = -torch.arange(n + 1, dtype=torch.int32) * penalty
    got = ops.needleman_wunsch(ref.cuda(), m.cuda(), penalty).cpu()
    assert torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [64, 128, 192, 256, 320, 384, 448, 576, 1088, 4160])
def test_gpu_single_launch_agrees_with_a_launch_per_anti_diagonal(n):
    """Strips of 128 columns, two per workgroup, the last one half empty or missing; any borders and scores, down to half
    the type's lowest value.  Up to n = 256 (one workgroup, which both entry points take) the oracle's borders are used."""
    from lego_amd import ops, runtime
    print(f"needleman-wunsch n={n}, one launch", flush=True)
    g = torch.Generator().manual_seed(n)
    ref = torch.randint(-40, 60, (n + 1, n + 1), generator=g, dtype=torch.int32)
    ref[torch.rand(n + 1, n + 1, generator=g) < 0.01] = -(1 << 30)
    m = torch.randint(-1000, 1000, (n + 1, n + 1), generator=g, dtype=torch.int32)
    m[5, 0] = m[0, 7] = -(1 << 30)
    if n <= 256:
        m[:, 0] = m[0, :] = -3 * torch.arange(n + 1, dtype=torch.int32)
        want = torch.from_numpy(ok.needleman_wunsch(ref.numpy(), 3))
    else:
        mat, r = m.cuda(), ref.cuda()
        runtime.call("lego_hip_nw_i32", r.data_ptr(), mat.data_ptr(), n, 3, None)
        want = mat.cpu()
    for _ in range(2):      # the second call finds the first one's workspace in the allocator
        got = ops.needleman_wunsch(ref.cuda(), m.cuda(), 3).cpu()
        assert torch.equal(got, want)


_ONE_LANE = """
#include <algorithm>
#include <climits>
using std::max;
#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_mov_dpp(v, ...) (v)
#define __builtin_amdgcn_update_dpp(edge, v, ...) (edge)      // lane 0: the column to its left
typedef int int2v __attribute__((vector_size(8)));
constexpr int kP = %(P)d;
inline int slot_at(int slot, int) { return 2 * slot; }
%(code)s
int main()
{
  const int ends[] = {INT_MIN, INT_MIN + 1, -1, 0, 1, INT_MAX - 1, INT_MAX};
  for (int penalty : ends) for (int score : ends) for (int edge : ends) {
    int2v scores[kP];
    for (auto& s : scores) s = int2v{plus(score, penalty), plus(minus(0, score), penalty)};
    alignas(8) int out[2 * kP];
    int ga = minus(edge, penalty), gb = ga, gnw = ga;
    run_phase<false>(4, 0, penalty, scores, minus(edge, penalty), out, ga, gb, gnw);
    // the recurrence as it is written down, modulo 2^32
    int up_a = edge, up_b = edge, corner = edge;
    for (int i = 0; i < kP; ++i) {
      const int a = max(max(plus(corner, score), minus(up_a, penalty)), minus(edge, penalty));
      const int b = max(max(plus(up_a, minus(0, score)), minus(up_b, penalty)), minus(a, penalty));
      if (a != plus(out[2 * i], penalty) || b != plus(out[2 * i + 1], penalty)) return 1;
      corner = edge, up_a = a, up_b = b;
    }
  }
}
"""


def test_sums_wrap_as_the_language_promises(tmp_path):
    """The recurrence of one lane, as the generator prints it, over the ends of the type: with a trap on signed overflow, which
    the compiler may otherwise take as never happening, it runs through and gives the cells modulo 2^32."""
    import re
    import subprocess
    from lego_amd.kernels import nw as gen
    text = (Path(__file__).resolve().parents[1] / "lego_amd" / "csrc" / "generated" / "nw_i32.hip").read_text()
    code = "\n".join(re.findall(r"^__device__ __forceinline__ int (?:plus|minus)\(.*$", text, re.M))
    code += "\n" + re.search(r"template <bool kStart>\n.*?\n}\n", text, re.S).group(0)
    src = tmp_path / "lane.cpp"
    src.write_text(_ONE_LANE % {"P": gen.P, "code": code})
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-fsanitize=signed-integer-overflow", "-fsanitize-undefined-trap-on-error",
                    str(src), "-o", str(tmp_path / "lane")], check=True)
    assert subprocess.run([str(tmp_path / "lane")]).returncode == 0
    assert not re.search(r"[-+] penalty|nw \+ ", re.sub(r"//.*", "", text))      # nor anywhere else in the kernels


@pytest.mark.gpu
@pytest.mark.parametrize("n,penalty", [(320, 2 ** 31 - 1), (384, -(2 ** 31)), (576, -7)])
def test_gpu_single_launch_wraps_as_the_tiles_do(n, penalty):
    """Scores, borders and penalties over the whole range of the type: sums are modulo 2^32 in both forms of the recurrence,
    and what is compared has the same bits."""
    from lego_amd import ops, runtime
    print(f"needleman-wunsch n={n}, whole range", flush=True)
    g = torch.Generator().manual_seed(n + 1)
    lo, hi = -(2 ** 31), 2 ** 31 - 1
    ref = torch.randint(lo, hi, (n + 1, n + 1), generator=g, dtype=torch.int32).cuda()
    m = torch.randint(lo, hi, (n + 1, n + 1), generator=g, dtype=torch.int32).cuda()
    want = m.clone()
    runtime.call("lego_hip_nw_i32", ref.data_ptr(), want.data_ptr(), n, penalty, None)
    assert torch.equal(ops.needleman_wunsch(ref, m, penalty), want)


@pytest.mark.gpu
def test_gpu_rejects_bad_sizes():
    from lego_amd import ops
    from lego_amd.runtime import LegoHipError
    with pytest.raises(LegoHipError):
        ops.needleman_wunsch(torch.zeros(101, 101, dtype=torch.int32, device="cuda"),
                             torch.zeros(101, 101, dtype=torch.int32, device="cuda"), 10)


@pytest.mark.gpu
def test_gpu_maximum_size_closed_form():
    """The largest size the entry point takes, n = 32768: with zero scores a diagonal step is free and a
    gap costs the penalty, so m[i][j] = -|i - j| * penalty."""
    from lego_amd import ops
    print("needleman-wunsch n=32768, zero scores", flush=True)
    n, penalty = 32768, 3
    ref = torch.zeros((n + 1, n + 1), dtype=torch.int32, device="cuda")
    m = torch.zeros((n + 1, n + 1), dtype=torch.int32, device="cuda")
    border = -torch.arange(n + 1, dtype=torch.int32, device="cuda") * penalty
    m[0, :] = border
    m[:, 0] = border
    ops.needleman_wunsch(ref, m, penalty)
    idx = torch.arange(n + 1, device="cuda", dtype=torch.int32)
    for rows in (slice(0, 130), slice(16000, 16130), slice(n - 129, n + 1)):
        want = -(idx[rows, None] - idx[None, :]).abs() * penalty
        assert torch.equal(m[rows], want)


def _wrapped(ref, m, penalty):
    """The recurrence modulo 2^32 over any borders, one anti-diagonal at a time."""
    ref, m = ref.numpy(), m.numpy().copy()
    p = np.array([penalty], dtype=np.int32)
    for d in range(2, 2 * len(m) - 1):
        i = np.arange(max(1, d - len(m) + 1), min(d - 1, len(m) - 1) + 1)
        j = d - i
        m[i, j] = np.maximum(np.maximum(m[i - 1, j - 1] + ref[i, j], m[i, j - 1] - p), m[i - 1, j] - p)
    return torch.from_numpy(m)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [128, 192, 256, 320, 576])
@pytest.mark.parametrize("where", ["near", "score", "score last", "top", "left", "penalty", "negative"])
def test_gpu_values_beyond_the_near_form(n, where):
    """The kernel leaves its shorter form of the recurrence where a value is too far from zero for it: at the bounds themselves, and where
    the first one beyond is a score in any strip, a border's cell, or the penalty."""
    from lego_amd import ops
    print(f"needleman-wunsch n={n}, {where}", flush=True)
    g = torch.Generator().manual_seed(7 * n)
    limit, penalty = (1 << 28) // (n + 256), 9
    ref = torch.randint(-4, 12, (n + 1, n + 1), generator=g, dtype=torch.int32)
    m = torch.randint(-99, 99, (n + 1, n + 1), generator=g, dtype=torch.int32)
    if where == "near":              # scores and penalty as large as the shorter form takes them
        ref = torch.where(ref > 4, limit, -limit).to(torch.int32)
        penalty = (1 << 27) // (n + 256)
        m[n // 3, 0] = -(1 << 27)
    elif where == "score":
        ref[n // 2, n // 3], ref[n // 2 + 1, n - 5] = limit + 1, 2 ** 31 - 1
    elif where == "score last":
        ref[n, n], ref[n - 20, 1] = -(2 ** 31), -limit - 1
    elif where == "top":
        m[0, n - 3], m[0, 1] = 2 ** 31 - 1, (1 << 28) + 1000
    elif where == "left":
        m[n // 2, 0], m[n // 2 + 40, 0] = 2 ** 31 - 5, -(2 ** 31)
    elif where == "penalty":
        penalty = (1 << 27) // (n + 256) + 1
    else:
        penalty = -3
    want = _wrapped(ref, m, penalty)
    got = ops.needleman_wunsch(ref.cuda(), m.cuda(), penalty)
    assert torch.equal(got.cpu(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [192, 320, 1088])
@pytest.mark.parametrize("where", ["highest", "above", "lowest", "below", "growing", "border", "left", "penalty", "penalty above"])
def test_gpu_bounds_of_the_near_form(n, where):
    """Either side of each bound up to which the kernel keeps its shorter form, and values that pass the bound, or the type's end, in the course of it."""
    from lego_amd import ops
    print(f"needleman-wunsch n={n}, bound: {where}", flush=True)
    g = torch.Generator().manual_seed(11 * n)
    penalty = 10
    ref = torch.randint(-4, 12, (n + 1, n + 1), generator=g, dtype=torch.int32)
    m = torch.randint(-99, 99, (n + 1, n + 1), generator=g, dtype=torch.int32)
    some = torch.rand(n + 1, n + 1, generator=g) < 0.3
    if where in ("highest", "above"):
        ref = torch.where(some, (1 << 23) + (where == "above"), ref)
    elif where in ("lowest", "below"):
        ref = torch.where(some, -(1 << 30) - (where == "below"), ref)
        m[n // 2:, 0] -= 1 << 29      # a sum with the lowest score that is still inside the type
    elif where == "growing":          # a whole diagonal of matches from 2^28 on: past 2^29 after 128 rows, past the type's end after 896
        ref, m = torch.full_like(ref, 1 << 21), m + (1 << 28)
    elif where == "border":
        m[0, n // 2], m[0, n - 1] = (1 << 29) - penalty * n, (1 << 29) + 1
    elif where == "left":
        m[n // 3, 0], m[n - 40, 0], m[n - 20, 0] = -(1 << 29), (1 << 29) - penalty * n, (1 << 29) + 1
    else:
        penalty = (1 << 27) // (n + 256) + (where == "penalty above")
        m[:, 0] = m[0, :] = -penalty * torch.arange(n + 1, dtype=torch.int32)
    want = _wrapped(ref, m, penalty)
    got = ops.needleman_wunsch(ref.cuda(), m.cuda(), penalty)
    assert torch.equal(got.cpu(), want)
