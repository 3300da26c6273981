"""Byte-repeatable results where split rule tasks meet: these structures have
pieces of one task that end in the same step of the product rules on different
lanes, whose LDS adds then share an instruction.  Ordered E/F/S and the loss
gradient give the same bytes on every call, with other work between the calls
and in another context."""
import numpy as np
import pytest

from helpers import loss_case, oracle_case, upload_oracle_lists
from mtpx import capi
from mtpx import synth as S

pytestmark = pytest.mark.gpu


def _structure(n):
    rng = S.rng_for(950, n)
    s = S.displace(S.strain(S.lattice("fcc", (n, n, n), 3.56), rng, 0.03), rng, 0.1)
    s.types = (S.uniform(rng, s.n) * 2).astype(np.int32)
    return s


@pytest.mark.parametrize("template,R", [("shapeev-10.mtp", 8), ("shapeev-16.mtp", 8),
                                        ("shapeev-20.mtp", 10), ("potential.mtp", 8),
                                        ("ps1-7b-517.mtp", 8)])
def test_results_repeat_byte_for_byte(template, R):
    text = S.random_model(template, 2, R, 1.5, 5.0, -0.05, 0.05, S.rng_for(951))
    s, other = _structure(5), _structure(3)
    ref = oracle_case(text, s)
    labels = loss_case(text, [other], 952)["labels"]
    seen = set()
    for _ in range(2):
        c = capi.Context(0)
        try:
            c.load_model_text(text)
            for _ in range(6):
                upload_oracle_lists(c, ref["nb"])  # handed over: gathered by the reverse index
                efs = [np.asarray(v).tobytes() for v in c.efs(deterministic=True)]
                c.build_neighbors(s.cell, s.pbc, ref["pos"], s.types, 5.0)
                built = [np.asarray(v).tobytes() for v in c.efs()]
                off = c.set_structures([s, other], 5.0)
                tf = np.concatenate([np.zeros((s.n, 3)), labels[0].forces])
                act, wE, wF, wS = capi.loss_weights(capi.LossSettings.make(), off,
                                                    np.ones((2, 3), np.int32), tf)
                c.set_labels(act, np.array([0.0, labels[0].energy]), wE, tf, wF,
                             np.array([np.zeros((3, 3)), labels[0].stress]), wS)
                f, g, _ = c.loss_grad()
                seen.add((*efs, *built, np.asarray(f).tobytes(), g.tobytes()))
        finally:
            c.close()
    assert len(seen) == 1
