"""GPU parity of the cooperative-signalling projections where the guarded
decisions, the kept rays and the combines' cases meet: bit-equal to the oracle
(rows, the crowding sum over n, the signalling maximum)."""
import numpy as np
import pytest

from oracle import cs_oracle as co

pytestmark = pytest.mark.gpu
PI = np.pi


def _run(R, fov, focal, objs, mets, max_proj, norm):
    import torch
    from abm_amd.cs import CSProjection
    dev = torch.device("cuda")
    T = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev)
    off = np.concatenate([[0], np.cumsum([len(o) for o in objs])]).astype(np.int64)
    cat = np.concatenate([np.asarray(o, dtype=np.float64).reshape(-1, 2) for o in objs])
    met = T(np.concatenate(mets))
    args = (T(np.asarray(focal, dtype=np.float64)), T(off), T(cat))
    proj, sig = CSProjection(R, fov, max_proj), CSProjection(R, fov, None)
    return (proj.sum(*args, T(np.full(len(focal), float(norm)))).cpu().numpy(),
            sig.max(*args, met).cpu().numpy(), sig.rows(*args, met).cpu().numpy(), off)


# object counts around a wavefront and the 64 quotients of the sum; rays of less
# than a word to thousands; the mask keeping all, a part and next to nothing
@pytest.mark.parametrize("R, fov", [(8, 1.0), (31, 0.5), (64, 0.25), (333, 0.45), (1200, 1.0), (1200, 0.02),
                                    (5000, 0.45)])
def test_counts_and_maxima_match_oracle(gpu, R, fov):
    rng = np.random.RandomState(R)
    fv = (-fov * PI, fov * PI)
    counts = [0, 1, 2, 63, 64, 65, 130]
    focal, objs, mets = [], [], []
    for k, n in enumerate(counts * 2):
        # the second half on a lattice, headings in eighths of a turn: objects on
        # bin ties, on the ends of the field of view, coincident, overlapping
        lattice = k >= len(counts)
        th = PI / 4 * rng.randint(0, 8) if lattice else rng.uniform(0, 2 * PI)
        focal.append((100.0, 100.0, 5.0, th))
        o = 100.0 + (2.0 * rng.randint(-20, 21, (n, 2)) if lattice else rng.uniform(-90, 90, (n, 2)))
        objs.append(o)
        mets.append(np.where(rng.rand(n) < 0.2, 0.0, rng.uniform(0, 1, n)))
    max_proj = 0.1 * R
    s, m, rows, off = _run(R, fv, focal, objs, mets, max_proj, 7)
    for k, (x, y, r, th) in enumerate(focal):
        pos = [np.array(p) for p in objs[k]]
        want = co.projection_field(fv, R, np.array([x, y]), r, th, pos, list(mets[k]), None)
        assert np.array_equal(rows[off[k]:off[k + 1]], want), (k, "rows")
        assert np.array_equal(m[k], want.max(axis=0) if len(pos) else np.zeros(R)), (k, "max")
        got = co.crowd_density_proj(fv, R, np.array([x, y]), r, th, pos, 7, max_proj) if pos else np.zeros(R)
        assert np.array_equal(s[k], got), (k, "sum")


def test_size_limit_at_equality(gpu):
    # a projection exactly as large as the limit is drawn (cs_supcalc.py:298-307)
    R, r, d = 1000, 6.0, 80.0
    size = 2 * np.arctan(r / d) / (2 * PI) * R
    focal, objs = [(50.0, 50.0, r, 0.3)] * 3, [[(50.0 + d, 50.0)]] * 3
    for limit in (size, np.nextafter(size, 0), np.nextafter(size, 1e9)):
        s, _, _, _ = _run(R, (-PI, PI), focal, objs, [np.ones(1)] * 3, float(limit), 1)
        want = co.crowd_density_proj((-PI, PI), R, np.array([50.0, 50.0]), r, 0.3, [np.array(objs[0][0])], 1,
                                     float(limit))
        assert np.array_equal(s[0], want), limit
