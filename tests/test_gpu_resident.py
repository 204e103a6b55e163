"""Resident launches (a system held on the chip for a batch of iterations)
against the separate launches of each Krylov phase: the same rows, threads and
order of additions, so iterates, iteration counts and residuals are equal bit
for bit.  Per-launch profiling keeps a solve to the separate launches, which
gives the reference."""
import numpy as np
import pytest

import ogs5_amd as ox
from ogs5_amd import mesh as M
from ogs5_amd import workloads as W
from ogs5_amd.workloads import Scenario, Step
from devbuf import DevArray

pytestmark = pytest.mark.gpu

MESH = {"line": M.line_mesh, "quad": M.quad_mesh, "hex": M.hex_mesh, "tet": M.tet_mesh}


def _scenario(kind, shape, seed=3, permute=False):
    """A flow problem with a random conductivity per element; permute: nodes
    renumbered at random (no symmetric diagonal copy: rows read from CRS)."""
    m = MESH[kind](*shape)
    rng = np.random.default_rng(seed)
    if permute:
        to = rng.permutation(m.n_nodes)
        back = np.argsort(to)
        m.x, m.y, m.z = m.x[back], m.y[back], m.z[back]
        m.conn = to[m.conn]
    left, right = m.nodes_where(0, 0.0), m.nodes_where(0, float(m.x.max()))
    idx = np.concatenate([left, right]).astype(np.int64)
    val = np.concatenate([np.full(left.size, 10.0), np.zeros(right.size)])
    return Scenario(kind, m, ox.LIQUID_FLOW, np.full(m.n_elem, 1e-4),
                    1e-4 * np.exp(rng.standard_normal(m.n_elem)), 1, idx, val,
                    np.zeros(0, np.int64), np.zeros(0), rng.uniform(0, 1, m.n_nodes),
                    [Step(100.0, 1.0)], max_iter=40)


def _solve(sc, system, separate, **kw):
    system[1].profile(separate)
    r = W.run_gpu(sc, system=system, **kw)
    return r["x"], r["info"][-1]


def _same(a, b):
    assert {k: a[1][k] for k in ("iterations", "error", "converged", "bnorm", "outer")} == {
        k: b[1][k] for k in ("iterations", "error", "converged", "bnorm", "outer")}
    assert np.array_equal(a[0], b[0])


# sizes: one row; a chunk and one row more; the partial sums' q = 1, 2 and 4
# neighbours per thread; the largest resident system of each row length and
# the next one up
# (FP64 also: one workgroup, of 256, 1024 and 2048 rows, and one row more)
CG = [("line", (1,)), ("line", (255,)), ("line", (256,)), ("line", (1023,)), ("line", (1024,)),
      ("line", (2047,)), ("line", (2048,)), ("line", (4096,)),
      ("quad", (1, 1)), ("quad", (33, 21)), ("quad", (63, 31)), ("quad", (64, 63)),
      ("tet", (3, 7, 7)), ("hex", (3, 7, 7)),
      ("tet", (11, 12, 11)), ("tet", (12, 12, 12)), ("hex", (9, 9, 9)), ("hex", (10, 9, 9)), ("quad", (255, 255)), ("quad", (256, 255)),
      ("quad", (361, 362)), ("quad", (511, 511)), ("quad", (512, 511)),
      ("tet", (1, 1, 1)), ("tet", (9, 7, 5)), ("tet", (50, 50, 49)), ("tet", (50, 50, 50)),
      ("hex", (1, 1, 1)), ("hex", (9, 7, 5)), ("hex", (50, 50, 49)), ("hex", (50, 50, 50))]


@pytest.mark.parametrize("prec", [ox.FP64, ox.FP32_IR])
@pytest.mark.parametrize("kind,shape", CG)
def test_cg_equals_separate_launches(kind, shape, prec):
    sc = _scenario(kind, shape)
    system = W.make_system(sc, prec)
    for max_iter in (1, 40):  # stops at the limit; ends by itself where it converges
        sc.max_iter = max_iter
        _same(_solve(sc, system, False), _solve(sc, system, True))
    system[1].close()


@pytest.mark.parametrize("prec", [ox.FP64, ox.FP32_IR])
@pytest.mark.parametrize("kind,shape", [("quad", (40, 31)), ("tet", (7, 8, 6)), ("hex", (8, 9, 7))])
def test_cg_rows_read_from_crs(kind, shape, prec):
    """Random node numbers (no banded pattern), and the banded pattern with
    the row-only elimination (not symmetric: no diagonal copy)."""
    for sc, bc in ((_scenario(kind, shape, permute=True), ox.DIRICHLET_SYMMETRIC),
                   (_scenario(kind, shape), ox.DIRICHLET_ROW)):
        sc.max_iter = 25
        system = W.make_system(sc, prec)
        _same(_solve(sc, system, False, dirichlet=bc), _solve(sc, system, True, dirichlet=bc))
        system[1].close()


@pytest.mark.parametrize("permute", [False, True])
@pytest.mark.parametrize("kind,shape", [("line", (300,)), ("quad", (61, 50)), ("quad", (300, 240)),
                                        ("tet", (9, 8, 10)), ("hex", (14, 11, 13))])
def test_refinement_steps_in_the_launch(kind, shape, permute):
    """FP32-IR solves to the tolerance (several reliable updates, taken inside
    the launch) and to a limit between two of them; FP64 rows from the diagonal
    copy and from CRS; a second solve on the same system."""
    sc = _scenario(kind, shape, permute=permute)
    sc.steps = sc.steps * 2
    system = W.make_system(sc, ox.FP32_IR)
    for max_iter in (5000, 37):
        sc.max_iter = max_iter
        got = _solve(sc, system, False)
        _same(got, _solve(sc, system, True))
        assert got[1]["converged"] == (max_iter == 5000)
        assert max_iter != 5000 or got[1]["outer"] >= 2  # updates, the last one final
    system[1].close()


# sizes as above; the largest resident system of 256-thread workgroups
# (65,536 rows) and of 512-thread ones (131,072) and the next one up
BI = [("line", (1,)), ("line", (255,)), ("line", (1023,)), ("line", (1024,)), ("line", (2047,)),
      ("line", (2048,)), ("quad", (1, 1)), ("quad", (33, 21)), ("tet", (9, 9, 9)),
      ("tet", (10, 9, 9)), ("hex", (9, 9, 9)), ("hex", (10, 9, 9)),
      ("quad", (361, 361)), ("quad", (361, 362)), ("tet", (1, 1, 1)), ("tet", (9, 7, 5)),
      ("tet", (39, 39, 39)), ("tet", (40, 40, 40)), ("tet", (50, 50, 50)),
      ("hex", (1, 1, 1)), ("hex", (9, 7, 5)), ("hex", (39, 39, 39)), ("hex", (40, 40, 40)),
      # past a thread per row: 1, 2 and 4 rows per thread
      ("quad", (600, 440)), ("tet", (64, 64, 64)), ("quad", (1000, 600))]


@pytest.mark.parametrize("prec", [ox.FP64, ox.FP32_IR])
@pytest.mark.parametrize("kind,shape", BI)
def test_bicgstab_equals_separate_launches(kind, shape, prec):
    """Row-only elimination (rows read from CRS) and the symmetric one (from
    the diagonal copy); stops at a limit and at the tolerance."""
    sc = _scenario(kind, shape)
    system = W.make_system(sc, prec)
    for bc in (ox.DIRICHLET_ROW, ox.DIRICHLET_SYMMETRIC):
        for max_iter in (1, 30):
            sc.max_iter = max_iter
            kw = dict(method=ox.BICGSTAB, dirichlet=bc)
            _same(_solve(sc, system, False, **kw), _solve(sc, system, True, **kw))
    system[1].close()


@pytest.mark.parametrize("prec", [ox.FP64, ox.FP32_IR])
def test_group_of_several_resident_launches(prec):
    """A group with more workgroups than the chip holds, rows of 9 and 27
    entries, and one member past the resident size: each member's result is
    that of its own separate launches."""
    scs = [_scenario("quad", (200 + k, 199), seed=k) for k in range(8)]
    scs += [_scenario("hex", (12, 11, 10)), _scenario("quad", (530, 520))]
    for sc in scs:
        sc.max_iter = 150
    got = W.run_group(scs, precision=prec)
    for sc, x, info in zip(scs, got["x"], got["info"]):
        system = W.make_system(sc, prec)
        _same((x, info[0]), _solve(sc, system, True))
        system[1].close()


@pytest.mark.parametrize("prec", [ox.FP64, ox.FP32_IR])
@pytest.mark.parametrize("method,bc", [(ox.CG, ox.DIRICHLET_SYMMETRIC), (ox.BICGSTAB, ox.DIRICHLET_ROW)])
def test_group_members_prepared_together(prec, method, bc):
    """Members on and off a banded pattern, of several sizes, over two steps
    (the matrix copies of the first are stale in the second): each member's
    result is that of its own solves."""
    scs = [_scenario("line", (1,)), _scenario("quad", (16, 15)), _scenario("quad", (40, 33), permute=True),
           _scenario("hex", (9, 8, 7)), _scenario("tet", (7, 6, 5), permute=True)]
    for sc in scs:
        sc.steps, sc.max_iter = [Step(100.0, 1.0), Step(30.0, 1.0)], 60
    got = W.run_group(scs, precision=prec, method=method, dirichlet=bc)
    for sc, x, info in zip(scs, got["x"], got["info"]):
        system = W.make_system(sc, prec)
        _same((x, info[-1]), _solve(sc, system, False, method=method, dirichlet=bc))
        system[1].close()


@pytest.mark.parametrize("n,width", [(1, 1), (300, 3), (2048, 9), (2049, 9), (5000, 27), (5000, 29), (262144, 3),
                                     (262145, 3)])
@pytest.mark.parametrize("method", [ox.CG, ox.BICGSTAB])
def test_noalloc_rows_and_sizes(n, width, method):
    """Caller-held CRS rows of up to 27 entries run resident, longer ones and
    larger systems do not; twice in a row from the same start, the same bits,
    and the residual they report."""
    rng = np.random.default_rng(n)
    k = np.arange(-(width // 2), width - width // 2)
    cols = np.arange(n)[:, None] + k
    have = (cols >= 0) & (cols < n)
    sym = np.where(k == 0, width + 1.0, -1.0 / (1.0 + np.abs(k)))
    val = np.broadcast_to(sym, cols.shape)[have]
    ptr = np.concatenate([[0], np.cumsum(have.sum(1))]).astype(np.int32)
    col = cols[have].astype(np.int32)
    b = rng.standard_normal(n)
    dev = [DevArray(a) for a in (ptr, col, np.ascontiguousarray(val), b)]
    xs = []
    for _ in range(2):
        x = DevArray(np.zeros(n))
        info, _ = ox.solve_crs_noalloc(n, *(d.ptr for d in dev), x.ptr, tol=1e-12, max_iter=500,
                                       method=method)
        assert info["converged"] == 1
        xs.append(x.get())
    assert np.array_equal(*xs)
    row = np.repeat(np.arange(n), np.diff(ptr))
    r = b - np.bincount(row, val * xs[0][col], n)
    # the recurrence's residual and the true one differ by rounding
    assert np.linalg.norm(r) <= 1e-11 * np.linalg.norm(b)


@pytest.mark.parametrize("prec", [ox.FP64, ox.FP32_IR])
@pytest.mark.parametrize("shape", [(9, 7), (70, 60)])
@pytest.mark.parametrize("bc", [ox.DIRICHLET_ROW, ox.DIRICHLET_SYMMETRIC])
def test_formats_are_tuned_when_asked_for(shape, prec, bc):
    """A solve in resident launches times no SpMV format; asking for the
    formats does, and changes no later solve."""
    sc = _scenario("quad", shape)
    system = W.make_system(sc, prec)
    s = system[1]
    kw = dict(method=ox.BICGSTAB, dirichlet=bc)
    first = _solve(sc, system, False, **kw)
    stands = bc == ox.DIRICHLET_SYMMETRIC  # the diagonal copy, format 25
    timed = [f for f, _ in s.spmv_tuning()]
    half = len(timed) // 2 if prec == ox.FP32_IR else len(timed)
    for part, fmt in ((timed[:half], s.spmv_format()), (timed[half:], s.spmv_format(fp32=True))):
        if part:
            assert len(set(part)) == len(part) > 1 and (fmt == 25 if stands else fmt in part)
    _same(_solve(sc, system, False, **kw), first)
    _same(_solve(sc, system, True, **kw), first)
    s.set_spmv_variant(0)
    _same(_solve(sc, system, False, **kw), first)
    s.close()
