"""E/F/S and energies at the neighbour counts where the neighbour passes
change course: the moment products take sixteen neighbours at a time and
batches of 64, the force pass one batch at a time.  A cluster of n + 1 atoms
within the cutoff of each other gives every atom a list of n entries.  Each
kernel profile runs: levels 10, 16 and 20 (the last with a second group of
radial functions), the run-time profiles (eight radial functions), a general
radial basis and an MTP-M head.  Bar: 1e-10 of the largest value, the bar of
the E/F/S parity tests."""
import numpy as np
import pytest

from helpers import assert_efs_close, oracle_case, rel_err, upload_oracle_lists
from mtpx import synth as S

pytestmark = pytest.mark.gpu

COUNTS = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 80, 127, 128, 129]


def _model(name):
    rng = S.rng_for(910)
    mk = lambda t, Z, R, **kw: S.random_model(t, Z, R, 1.0, 5.0, -0.05, 0.05, rng, **kw)
    if name == "level16-head":
        return S.mtpm_model(mk("shapeev-16.mtp", 2, 8), "mtp_m_q2", rng)
    return {"level10": lambda: mk("shapeev-10.mtp", 1, 8), "level16": lambda: mk("shapeev-16.mtp", 3, 8),
            "level20": lambda: mk("shapeev-20.mtp", 4, 10), "small": lambda: mk("shapeev-06.mtp", 2, 6),
            "odd-R": lambda: mk("shapeev-16.mtp", 2, 7), "M8": lambda: mk("ps1-7b-517.mtp", 2, 8),
            "M8-nu": lambda: mk("pot4b.mtp", 2, 8),
            "poly5": lambda: mk("shapeev-16.mtp", 2, 8, basis="RBChebyshevPoly5")}[name]()


def _cluster(n, Z):
    """n atoms in a ball of radius 2.4 (all pairs within 4.8 A)."""
    rng = S.rng_for(911, n)
    pos = np.zeros((0, 3))
    while len(pos) < n:
        p = S.uniform(rng, 3, -2.4, 2.4)
        if p @ p < 2.4 ** 2 and (not len(pos) or np.min(np.sum((pos - p) ** 2, 1)) > 0.25 ** 2):
            pos = np.vstack([pos, p])
    types = (S.uniform(rng, n) * Z).astype(np.int32)
    return S.Structure(np.eye(3) * 50.0, pos + 25.0, types, np.zeros(3, np.int32))


@pytest.mark.parametrize("name", ["level10", "level16", "level20", "small", "odd-R", "M8", "M8-nu",
                                  "poly5", "level16-head"])
def test_every_list_length(ctx, name):
    text = _model(name)
    ctx.load_model_text(text)
    for n in COUNTS:
        ref = oracle_case(text, _cluster(n + 1, ctx.info["Z"]))
        assert np.all(np.diff(ref["nb"].offsets) == n)
        upload_oracle_lists(ctx, ref["nb"])
        assert_efs_close(ctx.efs(), ref, 1e-10)
        assert_efs_close(ctx.efs(deterministic=True), ref, 1e-10)
        E, se = ctx.energy()
        assert rel_err(se, ref["se"]) < 1e-10 and rel_err(E[0], ref["E"]) < 1e-10
