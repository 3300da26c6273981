"""Neighbour lists of one small periodic structure (prepared by one workgroup)
against the same structure as the first of a batch of two (prepared launch by
launch): every array bit for bit, on the first build and on a repeated one.
The sizes lie around the tiles of 64 atoms, the 1,024 threads and the limit of
3,072 atoms; the cells are cubic, skewed, left-handed, flat, shorter than the
cutoff and, where a limit is passed, such that the general way takes over."""
import numpy as np
import pytest

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


def test_bins_that_overflow_fall_back(ctx):
    """A cluster in a large cell: its lists outgrow bins sized by the mean
    density, and the next, sparser build uses the larger bins."""
    rng = S.rng_for(922)
    pos = 4.0 * rng.random((300, 3)) + 8.0
    dense = S.Structure(np.eye(3) * 20.0, pos, np.zeros(300, np.int32), np.ones(3, np.int32))
    for st in (dense, _structure(500, "cubic", 5), dense):
        ctx.set_structures([st, _structure(7, "cubic", 3)], CUTOFF)
        want = _lists(ctx)
        P = want["offsets"][len(st.types)]
        ctx.build_neighbors(st.cell, st.pbc, st.pos, st.types, CUTOFF)
        got = _lists(ctx)
        assert len(got["idx"]) == P
        for k in ("idx", "types", "vec", "dist"):
            assert np.array_equal(got[k], want[k][:P]), k
