"""Systems solved by teams of every size against the same systems solved by one
workgroup each: the same bits, iterations and residuals, with other systems
taken alone beside them, and with more teams' systems than teams."""
import numpy as np
import pytest

from unap_amd import hip, meshgen

pytestmark = pytest.mark.gpu

FIELDS = ("nIterations", "converged", "singular", "initial", "final", "previous")


def _box(dims, kind, seed):
    p0, shift = (5.0, 1e-3) if kind == meshgen.CONVDIFF else (-3.0, 1e-6)
    return meshgen.box_system(*dims, kind, p0, 0.0, shift, seed)


P, C = meshgen.POISSON_LOGUNIF, meshgen.CONVDIFF
# levels of about 1000 .. 2500 rows, not multiples of a wavefront's; and small ones, down to one cell
LARGE = [((33, 31, 29), P), ((30, 27, 35), C), ((29, 23, 31), P), ((37, 33, 35), C)]
SMALL = [((1, 1, 1), P), ((1, 1, 2), C), ((5, 4, 3), C), ((16, 17, 15), P), ((19, 18, 17), C), ((9, 8, 40), P)]


@pytest.mark.parametrize("max_iter,rel_tol", [(1000, 1e-8), (3, 1e-8), (1, 0.0)])
def test_same_bits_as_one_workgroup(max_iter, rel_tol):
    systems = [_box(d, k, i) for i, (d, k) in enumerate(LARGE + SMALL + LARGE)]
    B = hip.Batch(systems, ["PCG" if s.symmetric else "PBiCGStab" for s in systems])
    b = np.concatenate([s.b for s in systems])
    x0 = np.random.default_rng(3).uniform(-1, 1, b.size)
    for rows in (64, 128, 256):
        B.set_config(1024, 1, rows)
        B.set_team(1)
        x, p = B.solve(b, x=x0, max_iter=max_iter, rel_tol=rel_tol)
        assert B.team() == (1, 0)
        for size in (2, 3, 4, 8, 0):
            B.set_team(size)
            y, q = B.solve(b, x=x0, max_iter=max_iter, rel_tol=rel_tol)
            got, wide = B.team()
            assert got == size if size else got in (4, 8)
            assert wide >= len(LARGE)
            assert np.array_equal(x, y), size
            for i in range(len(systems)):
                assert [p[i][f] for f in FIELDS] == [q[i][f] for f in FIELDS], (size, i)


def test_more_systems_than_teams():
    systems = [_box((26 + i % 5, 29 - i % 3, 30), C if i % 2 else P, i) for i in range(80)]
    B = hip.Batch(systems, ["PCG" if s.symmetric else "PBiCGStab" for s in systems])
    b = np.concatenate([s.b for s in systems])
    B.set_config(1024, 1, 128)
    out = []
    for size in (1, 8, 0):
        B.set_team(size)
        out.append(B.solve(b, max_iter=40, rel_tol=1e-8)[0])
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])


def test_refused_sizes():
    s = _box((5, 4, 3), P, 1)
    B = hip.Batch([s], ["PCG"])
    for size in (-1, 9):
        with pytest.raises(hip.UnapHipError):
            B.set_team(size)


def test_tuner_times_a_launch_of_teams_once():
    systems = [_box(d, k, i) for i, (d, k) in enumerate(LARGE[:2])]
    B = hip.Batch(systems, ["PCG" if s.symmetric else "PBiCGStab" for s in systems])
    x, _ = B.solve(np.concatenate([s.b for s in systems]), max_iter=20)
    bs, wg, _ = B.config()
    assert bs in (256, 512, 1024) and (bs < 1024 or wg == 1)
    B.set_config(1024, 2, 256)  # accepted, and the same as (1024, 1)
    y, _ = B.solve(np.concatenate([s.b for s in systems]), max_iter=20)
    assert B.config() == (1024, 2, 256) and B.team()[0] > 1
    B.set_config(1024, 1, 256)
    assert np.array_equal(y, B.solve(np.concatenate([s.b for s in systems]), max_iter=20)[0])
