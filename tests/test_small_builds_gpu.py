"""Neighbour lists of one small periodic structure (prepared by one workgroup)
against the same structure as the first of a batch of two (prepared launch by
launch): every array bit for bit, on the first build and on a repeated one.
The sizes lie around the tiles of 64 atoms, the 1,024 threads and the limit of
3,072 atoms; the cells are cubic, skewed, left-handed, flat, shorter than the
cutoff and, where a limit is passed, such that the general way takes over."""
import numpy as np
import pytest

from mtpx import capi
from mtpx import synth as S

pytestmark = pytest.mark.gpu

CUTOFF = 5.0


def _structure(n, shape, seed, density=0.06):
    rng = S.rng_for(920, seed)
    a = (n / density) ** (1 / 3)
    cell = np.diag([a, a, a])
    if shape == "skewed":
        cell = cell @ np.array([[1.0, 0.35, -0.2], [0.1, 0.9, 0.4], [-0.3, 0.2, 1.1]])
    elif shape == "left-handed":
        cell = cell[[1, 0, 2]]
    elif shape == "flat":
        cell = np.diag([a * 2.2, a * 2.0, a / 4.4])
    elif shape == "vacuum":
        cell = np.diag([a, a, 5 * a])
    f = rng.random((n, 3))
    if n > 4:  # on the boundary, outside the cell, on one another's faces
        f[0], f[1], f[2], f[3] = (0, 0, 0), (0.5, 0, 1.0), (3.25, -2.5, 0.1), (-1e-17, 0.2, 0.7)
    if shape == "vacuum":
        f[:, 2] = 0.4 + 0.2 * f[:, 2]
    return S.Structure(cell, f @ cell, (S.uniform(rng, n) * 2).astype(np.int32), np.ones(3, np.int32))


def _lists(ctx):
    d = ctx.get_neighbors()
    return {k: d[k] for k in ("offsets", "idx", "types", "vec", "dist", "center_types")}


@pytest.mark.parametrize("shape", ["cubic", "skewed", "left-handed", "flat", "vacuum"])
@pytest.mark.parametrize("n", [1, 2, 33, 63, 64, 65, 108, 1023, 1024, 1025, 2049, 3071, 3072, 3073])
def test_small_build_equals_the_batch_build(ctx, n, shape):
    st = _structure(n, shape, n)
    other = _structure(7, "cubic", 3)
    text = S.random_model("shapeev-10.mtp", 2, 8, 1.0, CUTOFF, -0.05, 0.05, S.rng_for(921))
    ctx.load_model_text(text)
    ctx.set_structures([st, other], CUTOFF)
    want = _lists(ctx)
    P = want["offsets"][n]
    wantF = ctx.compute_batch()[1][:n]
    for _ in range(2):
        ctx.build_neighbors(st.cell, st.pbc, st.pos, st.types, CUTOFF)
        got = _lists(ctx)
        assert np.array_equal(got["offsets"], want["offsets"][:n + 1])
        for k in ("idx", "types", "vec", "dist"):
            assert np.array_equal(got[k], want[k][:P]), k
        assert np.array_equal(got["center_types"], want["center_types"][:n])
        # the mirrors: the same derivatives at the same slots; the launch
        # splits the atoms over other waves, which no sum of an atom crosses
        F = ctx.efs()[1]
        assert np.array_equal(F, wantF)


def _check(ctx, st, cutoff=CUTOFF):
    """The lists of st alone on ctx against those of a batch in a context of
    its own, which neither sizes nor fills ctx's bins."""
    c = capi.Context(0)
    try:
        c.set_structures([st, _structure(7, "cubic", 3)], cutoff)
        want = _lists(c)
    finally:
        c.close()
    ctx.build_neighbors(st.cell, st.pbc, st.pos, st.types, cutoff)
    got = _lists(ctx)
    P = want["offsets"][st.n]
    assert np.array_equal(got["offsets"], want["offsets"][:st.n + 1])
    for k in ("idx", "types", "vec", "dist"):
        assert np.array_equal(got[k], want[k][:P]), k
    return int(np.diff(got["offsets"]).max())


def _mean_list(st):
    return st.n / abs(np.linalg.det(st.cell)) * 4 / 3 * np.pi * CUTOFF ** 3


def test_bins_that_overflow_fall_back():
    """A cluster in a large cell.  On a fresh context its lists outgrow the
    bins sized by the mean density (one and a half times the mean list and 32)
    and it is counted; the next builds use bins of the longest list and a
    quarter, which a denser cluster outgrows again."""
    rng = S.rng_for(922)
    cluster = lambda n: S.Structure(np.eye(3) * 20.0, 4.0 * rng.random((n, 3)) + 8.0,
                                    np.zeros(n, np.int32), np.ones(3, np.int32))
    dense, denser, sparse = cluster(300), cluster(500), _structure(500, "cubic", 5)
    c = capi.Context(0)
    try:
        longest = _check(c, dense)
        assert longest > 1.5 * _mean_list(dense) + 32
        _check(c, sparse)
        assert _check(c, denser) > longest + longest // 4 + 8
        for st in (dense, denser, sparse):
            _check(c, st)
    finally:
        c.close()


def test_more_points_than_the_preparation_holds():
    """Atoms crowded around the corner of the cell: each has seven images
    within the cutoff of the bounding box, 20,800 points where the mean density
    promises 5,000, so the one-workgroup preparation gives the build up."""
    rng = S.rng_for(923)
    n, a, rc = 2600, 16.0, 2.0
    st = S.Structure(np.eye(3) * a, rng.uniform(-0.95 * rc, 0.95 * rc, (n, 3)),
                     (S.uniform(rng, n) * 2).astype(np.int32), np.ones(3, np.int32))
    assert n * (1 + 2 * rc / a) ** 3 < 18432 < 8 * n
    c = capi.Context(0)
    try:
        for _ in range(2):
            _check(c, st, rc)
        _check(c, _structure(997, "cubic", 6))
    finally:
        c.close()
