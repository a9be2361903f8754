"""LU decomposition without pivoting: oracle pins on the CPU, parity on the GPU."""
import numpy as np
import pytest
import scipy.linalg
import torch

from lego_amd.kernels import lud as lud_gen
from oracle import kernels as ok


def _dominant(n, seed):
    """Strictly column-diagonally-dominant: partial pivoting never swaps, so a library LU with
    pivoting is the decomposition without pivoting."""
    rng = np.random.default_rng(seed)
    a = rng.uniform(-1, 1, (n, n))
    a[np.arange(n), np.arange(n)] = np.abs(a).sum(axis=0) + 1.0
    return a


def test_oracle_matches_scipy_on_dominant_matrices():
    for n in (5, 64, 130):
        a = _dominant(n, n)
        p, l, u = scipy.linalg.lu(a)
        assert np.array_equal(p, np.eye(n))
        got = ok.lud(a)
        assert np.allclose(np.tril(got, -1) + np.eye(n), l, atol=1e-12)
        assert np.allclose(np.triu(got), u, atol=1e-10)


def test_oracle_reconstructs_the_matrix():
    a = _dominant(96, 7)
    got = ok.lud(a)
    l, u = np.tril(got, -1) + np.eye(96), np.triu(got)
    assert np.allclose(l @ u, a, atol=1e-10)


def test_coarsening_places_every_block_element_once():
    """The reference's ``inv``: virtual thread (ii, jj, tid) -> (i, j, tid/T, tid%T); with
    r = i*T + ty, c = j*T + tx the R*R*T*T virtual threads cover the block exactly once."""
    import sympy as sp
    ii, jj, tid = sp.symbols("ii jj tid", integer=True, nonnegative=True)
    f = sp.lambdify([ii, jj, tid], lud_gen.coarsening(ii, jj, tid), "math")
    T, R = lud_gen.T, lud_gen.R
    seen = set()
    for a in range(R):
        for b in range(R):
            for t in range(T * T):
                i, j, ty, tx = (int(v) for v in f(a, b, t))
                assert (i, j, ty, tx) == (a, b, t // T, t % T)
                seen.add((i * T + ty, j * T + tx))
    assert len(seen) == (R * T) ** 2


def _plan(n):
    """The launches of lego_hip_lud_f32 for an n x n matrix: (kind, workgroups, s, steps, side, run) each."""
    import ctypes
    from lego_amd import runtime
    count = ctypes.c_int(0)
    runtime.call("lego_hip_lud_f32_plan", n, None, 0, ctypes.byref(count))
    buf = (ctypes.c_int * (6 * count.value))()
    runtime.call("lego_hip_lud_f32_plan", n, buf, count.value, ctypes.byref(count))
    return [tuple(buf[6 * i:6 * i + 6]) for i in range(count.value)]


@pytest.mark.parametrize("nb", list(range(1, 14)) + [63, 64, 76, 77, 78, 79, 100, 129, 256, 511, 512])
def test_launches_take_every_block_through_every_step_once(nb):
    """What each launch reads is final when it starts, and every block has every step before its own once.  Panels of `steps` steps apply
    the earlier of them to the later by substitution; the diagonal block that a launch factors is the next launch's."""
    plan = _plan(64 * nb)
    kind, workgroups, _, _, side, _ = plan[0]
    assert (kind, workgroups) == (0, 1) and 1 <= side <= min(2, nb)
    done, factored = 0, side               # steps applied to all blocks behind them; side of the factored diagonal block at `done`
    for panels, trailing in zip(plan[1::2], plan[2::2]):
        kind, workgroups, s, steps, _, _ = panels
        q = nb - s - steps
        assert kind == 1 and (s, steps) == (done, factored) and q > 0
        assert workgroups * 2 * 16 == 64 * q                 # two wavefronts of sixteen columns, and two of sixteen rows
        kind, workgroups, s2, steps2, side, run = trailing
        assert kind == 2 and (s2, steps2) == (s, steps) and 1 <= side <= min(2, q) and 1 <= run <= lud_gen.GROUP
        done, factored = done + steps, side
        if q > side:
            assert (workgroups - 1) % lud_gen.XCDS == 0 and workgroups - 1 >= -(-q // run) * -(-q // 2)
    assert len(plan) % 2 == 1 and done + factored == nb
    assert factored == min(2, nb)          # a single block at the end would wait for panels of two steps


_WALK = """
#include <cstdio>
#include <cstdlib>
#include <vector>
#define __host__
#define __device__
#define __forceinline__ inline
%(code)s
// every block of the square by one workgroup: the first has the diagonal block of `side` blocks, and beside a single one its neighbour
bool covered_once(unsigned q, unsigned run, unsigned side, unsigned workgroups)
{
  std::vector<int> seen(q * q, 0);
  for (unsigned r = 0; r < side; ++r) for (unsigned c = 0; c < 2 && c < q; ++c) ++seen[r * q + c];
  for (unsigned wg = 0; wg + 1 < workgroups; ++wg) {
    unsigned from = 0, to = 0, pair = 0;
    if (!part_of(wg, workgroups - 1, q, run, side, from, to, pair)) continue;
    if (to > q || to - from > run || 2 * pair >= q) return false;
    for (unsigned r = from; r < to; ++r) for (unsigned c = 2 * pair; c < 2 * pair + 2 && c < q; ++c) ++seen[r * q + c];
  }
  for (int s : seen) if (s != 1) return false;
  return true;
}
int main()
{
  for (unsigned q = 1; q <= 510; q = q < 40 ? q + 1 : q * 9 / 8) {
    const unsigned chosen = trailing_rows(q);
    if (chosen < 1 || chosen > %(group)d) return 1;
    for (unsigned run = 1; run <= %(group)d; ++run)
      for (unsigned side = 1; side <= 2 && side <= q; ++side)
        if (!covered_once(q, run, side, trailing_grid(q, run))) { std::printf("q %%u run %%u side %%u\\n", q, run, side); return 2; }
  }
  return 0;
}
"""


def test_trailing_launch_covers_the_square_once(tmp_path):
    """The decomposition of the trailing update as the generator prints it, compiled for the host: for squares of 1 to 510 blocks and every
    length of run, each block is one workgroup's, the first one's part left out of the others'."""
    import re
    import subprocess
    from pathlib import Path
    text = (Path(__file__).resolve().parents[1] / "lego_amd" / "csrc" / "generated" / "lud_f32.hip").read_text()
    code = "\n".join(re.search(p + r".*?\n}\n", text, re.S).group(0) for p in (
        r"__host__ __device__ __forceinline__ bool part_of\(", r"inline unsigned trailing_rows\(", r"inline unsigned trailing_grid\("))
    src = tmp_path / "walk.cpp"
    src.write_text(_WALK % {"code": code, "group": lud_gen.GROUP})
    subprocess.run(["g++", "-std=c++17", "-O1", str(src), "-o", str(tmp_path / "walk")], check=True)
    res = subprocess.run([str(tmp_path / "walk")], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout


def test_trailing_walk_gives_each_xcd_a_contiguous_piece():
    """The layouts that print the kernel's index expressions: positions of the walk in group-major order, pairs of block columns inside a
    group, and for every XCD (every XCDS-th workgroup id) consecutive ones."""
    import sympy as sp
    ng, q2, per, pid, wg = sp.symbols("ng q2 per pid wg", integer=True, nonnegative=True)
    order = sp.lambdify([ng, q2, pid], lud_gen.block_order(ng, q2, 1, pid), "math")
    remap = sp.lambdify([per, wg], lud_gen.xcd_remap(per, wg), "math")
    X = lud_gen.XCDS
    for groups, pairs in ((1, 1), (3, 2), (8, 31), (16, 62)):
        assert [tuple(int(v) for v in order(groups, pairs, p)) for p in range(groups * pairs)] == [(g, c, 0) for g in range(groups) for c in range(pairs)]
    for pieces in (1, 2, 31):
        for x in range(X):
            assert [int(remap(pieces, w)) for w in range(x, X * pieces, X)] == list(range(x * pieces, (x + 1) * pieces))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [64, 128, 512, 1024])
def test_gpu_matches_oracle(n):
    from lego_amd import ops
    print(f"lud n={n}", flush=True)
    a = _dominant(n, 100 + n).astype(np.float32)
    want = ok.lud(a)
    got = ops.lud(torch.from_numpy(a.copy()).cuda()).cpu().numpy().astype(np.float64)
    scale = np.abs(want).max()
    assert np.abs(got - want).max() <= 2e-5 * scale
    l, u = np.tril(got, -1) + np.eye(n), np.triu(got)
    assert np.abs(l @ u - a).max() <= 1e-4 * scale


@pytest.mark.gpu
@pytest.mark.parametrize("n", [192, 320, 576, 1088, 1152])
def test_gpu_odd_block_counts(n):
    """A last block that is no pair, a second column of blocks past the matrix: the factors against the oracle's, each rounded some n
    times at the size of the pivots."""
    from lego_amd import ops
    print(f"lud n={n}", flush=True)
    a = _dominant(n, 300 + n).astype(np.float32)
    want = ok.lud(a)
    got = ops.lud(torch.from_numpy(a.copy()).cuda()).cpu().numpy().astype(np.float64)
    assert np.linalg.norm(got - want) <= n * 2.0 ** -24 * np.linalg.norm(want)
    assert np.abs(got - want).max() <= 2e-5 * np.abs(want).max()


def _lud_by_blocks(a, b=128):
    """The oracle's elimination on diagonal blocks, triangular solves and products in 64 bits around them."""
    m = np.array(a, dtype=np.float64)
    for k in range(0, len(m), b):
        e = min(k + b, len(m))
        m[k:e, k:e] = ok.lud(m[k:e, k:e])
        m[k:e, e:] = scipy.linalg.solve_triangular(m[k:e, k:e], m[k:e, e:], lower=True, unit_diagonal=True)
        m[e:, k:e] = scipy.linalg.solve_triangular(m[k:e, k:e], m[e:, k:e].T, trans=1).T
        m[e:, e:] -= m[e:, k:e] @ m[k:e, e:]
    return m


def test_oracle_by_blocks_is_the_oracle():
    a = _dominant(300, 4)
    assert np.allclose(_lud_by_blocks(a, 64), ok.lud(a), rtol=1e-12, atol=1e-11)


@pytest.mark.gpu
@pytest.mark.parametrize("n,runs", [(1600, {1, 2}), (2624, {1, 2, 3, 4}), (4160, {1, 2, 3, 4, 5, 6, 7, 8})])
def test_gpu_run_lengths(n, runs):
    """Trailing squares whose workgroups take runs of several block rows, the last ones short: bounds as for the odd block counts."""
    from lego_amd import ops
    print(f"lud n={n}", flush=True)
    assert {record[5] for record in _plan(n) if record[0] == 2} == runs
    a = _dominant(n, 500 + n).astype(np.float32)
    want = _lud_by_blocks(a)
    got = ops.lud(torch.from_numpy(a.copy()).cuda()).cpu().numpy().astype(np.float64)
    assert np.linalg.norm(got - want) <= n * 2.0 ** -24 * np.linalg.norm(want)
    assert np.abs(got - want).max() <= 2e-5 * np.abs(want).max()


@pytest.mark.gpu
def test_gpu_rejects_bad_sizes():
    from lego_amd import ops
    from lego_amd.runtime import LegoHipError
    with pytest.raises(LegoHipError):
        ops.lud(torch.eye(100, device="cuda"))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [4928, 8256, 16384, 32768])
def test_gpu_large_matrix_reproduces_its_factors(n):
    """77 and 129 blocks, odd counts, n = 16384, the largest size the reference publishes, and n = 32768, the
    largest the entry point takes (a 4 GiB matrix: offsets beyond 32 bits): L*U gives the
    matrix back (fp32, diagonally dominant)."""
    from lego_amd import ops
    print(f"lud n={n}", flush=True)
    a = torch.rand(n, n, device="cuda", generator=torch.Generator(device="cuda").manual_seed(61))
    a.diagonal().add_(float(n))
    w = a.clone()
    ops.lud(w)
    lower = torch.tril(w, -1)
    lower.diagonal().fill_(1.0)
    back = lower @ torch.triu(w)
    assert ((back - a).norm() / a.norm()).item() <= 1e-5


@pytest.mark.gpu
def test_gpu_call_replays_from_a_hip_graph():
    """Captured into a graph, on a stream that an eager call has used before and on a new one, every replay
    gives the bits of the eager result, with eager work and synchronisation between the replays."""
    from lego_amd import ops
    print("lud n=8256 captured into a graph", flush=True)
    n = 8256
    a = torch.rand(n, n, device="cuda", generator=torch.Generator(device="cuda").manual_seed(62))
    a.diagonal().add_(float(n))
    w = a.clone()
    ops.lud(w)
    torch.cuda.synchronize()
    want = w.clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        w.copy_(a)
        ops.lud(w)                       # warm-up on a side stream, outside the capture
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    for capture_stream in (side, torch.cuda.Stream()):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=capture_stream):
            ops.lud(w)
        for trial in range(3):
            w.copy_(a)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(w, want), trial
            other = a[:512, :512] @ a[:512, :512]   # eager work between the replays
            torch.cuda.synchronize()
            del other
        del graph


def _factored(a):
    from lego_amd import ops
    return ops.lud(torch.from_numpy(a.astype(np.float32)).cuda()).cpu().numpy().astype(np.float64)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [64, 128, 192])
@pytest.mark.parametrize("scale", [1.0, 1e-30, 1e30, 2.0 ** -130, 2.0 ** -136])
def test_gpu_pivots_of_any_magnitude(n, scale):
    """Pivots near the ends of the exponent range take true divisions; the last scale makes them subnormal, below 2^-128,
    where a reciprocal overflows.  The rounding of the elements themselves, n of them summed, bounds L - L' and
    (U - U') / scale."""
    print(f"lud n={n} scale={scale}", flush=True)
    a = (_dominant(n, n + 1) * scale).astype(np.float32)
    assert scale > 2.0 ** -136 or np.abs(np.diagonal(a)).max() < 2.0 ** -128
    got = _factored(a)
    want = ok.lud(a.astype(np.float64))
    spacing = max(2.0 ** -24, 2.0 ** -149 / (scale * n))      # of the pivots, which are about n * scale
    assert np.abs(np.tril(got - want, -1)).max() <= 4 * n * spacing
    assert np.abs(np.triu(got - want)).max() / scale <= 4 * n * n * spacing


@pytest.mark.gpu
@pytest.mark.parametrize("n", [128, 192])
def test_gpu_upper_triangle_is_its_own_decomposition(n):
    """Ones above a small diagonal: L = I and U the matrix itself, exactly, though the inverse of a 16 x 16 tile of it is beyond
    the range of floats."""
    a = np.triu(np.ones((n, n)), 1) + np.float64(np.float32(0.003)) * np.eye(n)
    assert np.array_equal(_factored(a), a)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["normal", "uniform"])
@pytest.mark.parametrize("n", [128, 256])
def test_gpu_residual_is_that_of_elimination(n, kind):
    """Matrices that no diagonal dominates, whose blocks and tiles may be ill-conditioned: A - L U against |L| |U| stays within
    twice that of the elimination done in float32, element by element, on the host."""
    print(f"lud n={n} {kind}", flush=True)

    def residual(a, w):
        low, up = np.tril(w, -1) + np.eye(n), np.triu(w)
        return np.linalg.norm(a - low @ up) / np.linalg.norm(np.abs(low) @ np.abs(up))

    for seed in range(6):
        rng = np.random.default_rng(seed)
        a = (rng.standard_normal((n, n)) if kind == "normal" else rng.uniform(0, 1, (n, n))).astype(np.float32)
        host = a.copy()
        for k in range(n - 1):
            host[k + 1:, k] /= host[k, k]
            host[k + 1:, k + 1:] -= np.outer(host[k + 1:, k], host[k, k + 1:])
        a = a.astype(np.float64)
        assert residual(a, _factored(a)) <= 2 * residual(a, host.astype(np.float64)), seed


@pytest.mark.gpu
@pytest.mark.parametrize("at,value", [((10, 100), np.inf), ((100, 10), np.inf), ((10, 100), np.nan), ((100, 40), np.nan),
                                      ((63, 64), -np.inf), ((64, 63), np.inf), ((0, 190), np.inf), ((150, 160), np.nan), ((40, None), 0.0)])
def test_gpu_non_finite_elements_stay_where_elimination_takes_them(at, value):
    """An infinity or NaN in a panel of the first step, in a later block, or a zero pivot (a row of zeros): what elimination
    leaves finite is finite and the same, but for diagonal blocks that have other elements: rows that are done take
    the multiplier 0 there, and 0 times an infinity is none."""
    print(f"lud {value} at {at}", flush=True)
    a = _dominant(192, 3).astype(np.float32)
    a[at[0], slice(None) if at[1] is None else at[1]] = value
    with np.errstate(all="ignore"):
        want = ok.lud(a.astype(np.float64))
    got = _factored(a)
    finite = np.isfinite(want)
    assert not np.isfinite(got[~finite]).any()
    for k in range(0, 192, 64):
        block = finite[k:k + 64, k:k + 64]
        block &= block.all()
    assert want.size // 4 < np.count_nonzero(finite) < want.size
    assert np.isfinite(got[finite]).all()
    assert np.abs(got[finite] - want[finite]).max() <= 2e-5 * np.abs(want[finite]).max()
