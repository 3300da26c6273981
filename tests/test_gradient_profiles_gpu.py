"""Loss and gradient of every gradient-kernel profile against the oracle.

The kernel's five variants are levels 10, 16 and 20, the small run-time profile
(other structures and general radial bases of up to four radial functions) and
the generic one.  Species counts pass the groups of four that the radial
gradient takes at a time; list lengths pass the places where the neighbour
passes change course (sixteen neighbours a product, 32 or 64 a part, batches of
64).  Bar: 1e-9 of the largest value, the bar of the training parity tests."""
import numpy as np
import pytest

from helpers import assert_loss_grad_close, loss_case
from mtpx import synth as S

pytestmark = pytest.mark.gpu

PROFILES = {
    "level10": ("shapeev-10.mtp", 8, {}), "level16": ("shapeev-16.mtp", 8, {}),
    "level20": ("shapeev-20.mtp", 10, {}), "small": ("shapeev-06.mtp", 6, {}),
    "odd-R": ("shapeev-16.mtp", 7, {}), "M8": ("ps1-7b-517.mtp", 8, {}),
    "M8-nu": ("pot4b.mtp", 8, {}), "R16": ("shapeev-10.mtp", 16, {}),
    "poly5": ("shapeev-16.mtp", 8, {"basis": "RBChebyshevPoly5"}),
    "level20-poly5": ("shapeev-20.mtp", 10, {"basis": "RBChebyshevPoly5"}),
}
COUNTS = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 80, 95, 96, 97, 127, 128, 129]


def _model(name, Z, seed=940):
    template, R, kw = PROFILES[name]
    return S.random_model(template, Z, R, 1.0, 5.0, -0.05, 0.05, S.rng_for(seed, Z), **kw)


def _crystal(Z, k):
    rng = S.rng_for(941, 10 * Z + k)
    s = S.displace(S.strain(S.lattice("bcc", (2, 3, 3 + k), 2.87), rng, 0.03), rng, 0.15)
    s.types = (S.uniform(rng, s.n) * Z).astype(np.int32)
    return s


def _cluster(n, Z):
    """n atoms in a ball of radius 2.4 (all pairs within 4.8 A)."""
    rng = S.rng_for(942, n)
    pos = np.zeros((0, 3))
    while len(pos) < n:
        p = S.uniform(rng, 3, -2.4, 2.4)
        if p @ p < 2.4 ** 2 and (not len(pos) or np.min(np.sum((pos - p) ** 2, 1)) > 0.25 ** 2):
            pos = np.vstack([pos, p])
    types = (S.uniform(rng, n) * Z).astype(np.int32)
    return S.Structure(np.eye(3) * 50.0, pos + 25.0, types, np.zeros(3, np.int32))


@pytest.mark.parametrize("name,Z", [("level10", 2), ("level10", 9), ("level16", 5), ("level20", 5),
                                    ("small", 6), ("odd-R", 3), ("M8", 2), ("M8", 5), ("M8-nu", 2),
                                    ("R16", 3), ("poly5", 5), ("level20-poly5", 2)])
def test_loss_grad_matches_oracle(ctx, name, Z):
    text = _model(name, Z)
    ctx.load_model_text(text)
    assert_loss_grad_close(ctx, loss_case(text, [_crystal(Z, k) for k in range(3)], 943), 1e-9)


@pytest.mark.parametrize("name", ["level10", "level16", "level20", "small", "M8", "poly5"])
def test_every_list_length(ctx, name):
    text = _model(name, 2)
    ctx.load_model_text(text)
    for n in COUNTS:
        case = loss_case(text, [_cluster(n + 1, 2)], 944)
        assert np.all(np.diff(case["nbs"][0].offsets) == n)
        assert_loss_grad_close(ctx, case, 1e-9)
