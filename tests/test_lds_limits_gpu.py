"""Models whose work space just fits a CU's 160 KB of LDS.

What a single wave needs beside its own work space is the radial coefficients
(Z^2 M R), the moment coefficients and map, the force polynomials' table and,
for E/F/S, the adjoint seeds; the moment and step tables stay in global memory
where they do not fit.  These species counts leave at most three kilobytes of
the LDS, less than those tables take.  Bars: 1e-10 for E/F/S, 1e-9 for loss and
gradient, as in the other parity tests."""
import numpy as np
import pytest

from helpers import assert_efs_close, assert_loss_grad_close, loss_case, oracle_case, upload_oracle_lists
from mtpx import synth as S

pytestmark = pytest.mark.gpu


def _structure(Z, seed):
    rng = S.rng_for(930, seed)
    s = S.displace(S.lattice("fcc", (3, 3, 3), 3.56), rng, 0.1)
    s.types = (S.uniform(rng, s.n) * Z).astype(np.int32)
    return s


def _model(template, Z, R):
    return S.random_model(template, Z, R, 1.5, 5.0, -0.05, 0.05, S.rng_for(931, Z))


@pytest.mark.parametrize("template,Z,R", [("shapeev-02.mtp", 44, 10), ("shapeev-06.mtp", 44, 5),
                                          ("shapeev-16.mtp", 34, 4), ("shapeev-16.mtp", 17, 16),
                                          ("potential.mtp", 24, 8), ("ps1-7b-517.mtp", 23, 4),
                                          ("pot4b.mtp", 12, 13)])
def test_efs_of_many_species(ctx, template, Z, R):
    text = _model(template, Z, R)
    ref = oracle_case(text, _structure(Z, 1))
    ctx.load_model_text(text)
    upload_oracle_lists(ctx, ref["nb"])
    assert_efs_close(ctx.efs(), ref, 1e-10)


@pytest.mark.parametrize("template,Z,R", [("shapeev-10.mtp", 17, 11), ("shapeev-20.mtp", 16, 6),
                                          ("shapeev-20-t.mtp", 16, 6), ("pot4b.mtp", 13, 5)])
def test_gradient_of_many_species(ctx, template, Z, R):
    text = _model(template, Z, R)
    ctx.load_model_text(text)
    assert_loss_grad_close(ctx, loss_case(text, [_structure(Z, 2), _structure(Z, 3)], 932), 1e-9)


@pytest.mark.parametrize("M", [3, 5])
def test_force_table_longer_than_the_moments(ctx, M):
    """M radial functions of degree 0 and no products: the force polynomials'
    table (an even count per function) is longer than the moments, so the
    staged adjoints lie behind the wave's blocks instead of over them."""
    topo = dict(K=M, M=M, basic=[[mu, 0, 0, 0] for mu in range(M)], times=[], map=list(range(M)))
    n = 4 * M * 8 + 2 + M
    text = S.write_mtp(topo, 2, 8, 1.5, 5.0, 0.01, S.uniform(S.rng_for(933, M), n, -0.05, 0.05))
    s = _structure(2, 4)
    ref = oracle_case(text, s)
    ctx.load_model_text(text)
    upload_oracle_lists(ctx, ref["nb"])
    assert_efs_close(ctx.efs(), ref, 1e-10)
    assert_efs_close(ctx.efs(deterministic=True), ref, 1e-10)
    assert_loss_grad_close(ctx, loss_case(text, [s, _structure(2, 5)], 934), 1e-9)
