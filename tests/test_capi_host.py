"""Host-side C-ABI checks that need no GPU: the library loads and exports
every entry point include/mtpx.h declares; the host-only functions (wrap,
the .mtp parser, the loss weights) agree with the oracle; context creation
fails cleanly without a device."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from helpers import rel_err
from mtpx import capi
from mtpx import synth as S


def test_library_exports_every_declared_symbol():
    L = capi.lib()
    names = capi.declared_symbols()
    assert len(names) >= 28
    for name in names:
        assert hasattr(L, name), name


def test_create_without_device_fails_cleanly():
    import torch
    if torch.cuda.is_available():
        pytest.skip("a device is present")
    h = C.c_void_p()
    rc = capi.lib().mtpx_create(0, C.byref(h))
    assert rc == -5 and not h.value


def test_wrap_is_bit_exact_against_oracle():
    rng = S.rng_for(900)
    for k in range(20):
        s = S.lattice("fcc" if k % 2 else "bcc", (2, 3, 2), 3.6)
        s = S.displace(S.strain(s, rng, 0.2), rng, 2.0)
        cell = s.cell.copy()
        cell[1] += 0.3 * cell[0]
        cell[2] -= 0.2 * cell[1]
        pos = s.pos * (1.0 + 3 * rng.random())
        pbc = np.array([1, 1, 1], np.int32) if k % 3 else np.array([1, 0, 1], np.int32)
        a = capi.wrap(cell, pbc, pos)
        b = O.wrap(cell, pbc, pos)
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64))


def _lattice_offsets(delta, basis):
    """Least-squares coefficients of delta over the rows of basis."""
    k, *_ = np.linalg.lstsq(basis.T, delta.T, rcond=None)
    return k.T


def test_singular_cell_wrap_known_answers():
    """wrap_singular_cell (base/structures.cpp:97-130): a line (rank 1) wraps
    x into [0, L); the non-periodic coordinates are untouched."""
    cell = np.array([[3.0, 0, 0], [0, 0, 0], [0, 0, 0]])
    pos = np.array([[7.5, 1.0, -2.0], [-0.5, 4.0, 9.0], [0.0, 0.0, 0.0], [3.0, 1.0, 1.0]])
    out = capi.wrap(cell, [1, 0, 0], pos)
    assert np.array_equal(out[:, 1:], pos[:, 1:])
    assert np.array_equal(out[:, 0], [1.5, 2.5, 0.0, 0.0])
    # nothing periodic: unchanged
    assert np.array_equal(capi.wrap(cell, [0, 0, 0], pos), pos)


@pytest.mark.parametrize("seed", range(4))
def test_singular_cell_wrap_slab(seed):
    """A slab: two periodic rows and a zero (or dependent) third row.  Every
    position moves by an integer combination of the periodic rows and lands
    with dual coordinates in [0, 1)."""
    rng = np.random.default_rng(seed)
    a1 = rng.standard_normal(3) * 3
    a2 = rng.standard_normal(3) * 3
    third = np.zeros(3) if seed % 2 == 0 else a1 + a2  # singular either way
    cell = np.array([a1, a2, third])
    pos = rng.standard_normal((50, 3)) * 10
    out = capi.wrap(cell, [1, 1, 0], pos)
    basis = np.array([a1, a2])
    k = _lattice_offsets(pos - out, basis)
    assert np.abs(k - np.round(k)).max() < 1e-9
    # the component normal to the plane is kept
    nrm = np.cross(a1, a2)
    assert np.abs((out - pos) @ nrm).max() < 1e-9 * np.abs(pos @ nrm).max()
    dual = np.linalg.solve(basis @ basis.T, basis)
    c = out @ dual.T
    assert c.min() > -1e-12 and c.max() < 1 + 1e-12
    # a second pass moves nothing by more than rounding
    assert np.abs(capi.wrap(cell, [1, 1, 0], out) - out).max() < 1e-12


def test_singular_cell_wrap_refusals():
    """Dependent periodic rows and non-finite rows raise, as the reference
    throws."""
    a = np.array([2.0, 0.5, 0.0])
    pos = np.zeros((1, 3))
    with pytest.raises(capi.MtpxError):
        capi.wrap(np.array([a, 2 * a, [0, 0, 0]]), [1, 1, 0], pos)
    with pytest.raises(capi.MtpxError):
        capi.wrap(np.array([a, [np.inf, 0, 0], [0, 0, 0]]), [1, 1, 0], pos)
    with pytest.raises(capi.MtpxError):  # all three periodic and singular
        capi.wrap(np.array([a, [0, 1.0, 0], a]), [1, 1, 1], pos)


@pytest.mark.parametrize("name", ["shapeev-10.mtp", "shapeev-16.mtp", "shapeev-20.mtp",
                                  "shapeev-20-t.mtp", "shapeev-06.mtp"])
def test_parser_matches_oracle(name):
    text = S.random_model(name, 3, 8, 2.0, 5.0, -0.1, 0.1, S.rng_for(3))
    info, coef = capi.parse_model_text(text)
    m = O.Model(text)
    assert (info["Z"], info["M"], info["R"], info["K"], info["B"], info["T"], info["S"]) == \
        (m.Z, m.M, m.R, m.K, m.B, m.T, m.S)
    assert np.array_equal(coef, m.coeffs)


def test_parser_defaults_match_oracle():
    """No scaling line (default 0.01) and no coefficient lines (defaults)."""
    text = S.read_template("shapeev-06.mtp")
    info, coef = capi.parse_model_text(text)
    m = O.Model(text)
    assert np.array_equal(coef, m.coeffs)


@pytest.mark.parametrize("bad", ["", "MTP\nversion = 1.1.0\nspecies_count = x\n",
                                 "not an mtp file"])
def test_parser_rejects_malformed_text(bad):
    with pytest.raises(capi.MtpxError):
        capi.parse_model_text(bad)


SETTINGS = [O.LossSettings.make(),
            O.LossSettings.make(eng_pow=2.0, force_pow=1.0, stress_pow=0.0),
            O.LossSettings.make(force_norm_f=1.0, force_norm_p=1.5, force_norm_d=0.1)]


@pytest.mark.parametrize("k", range(len(SETTINGS)))
def test_loss_weights_reproduce_oracle_loss(k):
    """mtpx_loss_weights applied to the oracle's own residuals gives the loss
    the oracle's AddLossGard computes, structure by structure."""
    st = SETTINGS[k]
    text = S.random_model("shapeev-10.mtp", 2, 8, 2.0, 5.0, -0.1, 0.1, S.rng_for(31))
    m = O.Model(text)
    rng = S.rng_for(32)
    structs, labels, nbs = [], [], []
    for j in range(5):
        s = S.displace(S.lattice("fcc", (2, 2, 1 + j % 2), 3.6), rng, 0.15)
        s.types = (S.uniform(rng, s.n) * 2).astype(np.int32)
        s.pos = O.wrap(s.cell, s.pbc, s.pos)
        nb = O.Neighbors.build(s.cell, s.pbc, s.pos, s.types, m.cutoff)
        E, F, St, _ = O.efs(m, nb)
        lb = O.Labels(s.n, energy=E + 0.1 * (rng.random() - 0.5),
                      forces=F + 0.05 * (rng.random((s.n, 3)) - 0.5),
                      stress=St + 0.2 * (rng.random((3, 3)) - 0.5), fitness=0.5 + rng.random())
        if j == 1:
            lb.forces = None
        if j == 2:
            lb.stress = None
        if j == 3:
            lb.atomic_fitness = rng.random(s.n)
        structs.append((s, E, F, St))
        labels.append(lb)
        nbs.append(nb)
    off = np.cumsum([0] + [lb.n for lb in labels]).astype(np.int32)
    has = np.array([[lb.energy is not None, lb.forces is not None, lb.stress is not None]
                    for lb in labels], np.int32)
    tf = np.concatenate([lb.forces if lb.forces is not None else np.zeros((lb.n, 3))
                         for lb in labels])
    af = np.concatenate([lb.atomic_fitness if lb.atomic_fitness is not None else np.ones(lb.n)
                         for lb in labels])
    fit = np.array([lb.fitness for lb in labels])
    cs = capi.LossSettings.make(*[getattr(st, f[0]) for f in st._fields_])
    active, wE, wF, wS = capi.loss_weights(cs, off, has, tf, fit, af)
    for c, ((s, E, F, St), lb, nb) in enumerate(zip(structs, labels, nbs)):
        loss_o, _, _ = O.add_loss_grad(m, nb, st, lb)
        loss = 0.0
        if active[c, 1]:
            loss += np.sum(wF[off[c]:off[c + 1]] * np.sum((F - lb.forces) ** 2, axis=1))
        if active[c, 2]:
            loss += wS[c] * np.sum((St - lb.stress) ** 2)
        if active[c, 0]:
            loss += wE[c] * (E - lb.energy) ** 2
        assert rel_err(loss, loss_o) < 1e-12


def test_loss_weights_flags():
    cs = capi.LossSettings.make(weight_stress=0.0)
    active, wE, wF, wS = capi.loss_weights(cs, [0, 3, 3, 5], [[1, 1, 1], [1, 1, 1], [0, 1, 0]])
    assert active.tolist() == [[1, 1, 0], [0, 0, 0], [0, 1, 0]]
    assert wS.tolist() == [0.0, 0.0, 0.0] and wE[1] == 0.0 and wE[2] == 0.0


def test_compiled_linear_walk_is_current(tmp_path):
    """The level-16 walk compiled into the linear-fit kernel
    (csrc/lin_plan_level16.inc) equals what the library's plan code computes
    for the level-16 template today (regenerated with gen_lin_plan.cpp)."""
    import os
    import shutil
    import subprocess
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc is not available")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    pkg = os.path.join(root, "imr-mlp_amd")
    exe = str(tmp_path / "gen_lin_plan")
    subprocess.run([hipcc, "-O1", "-std=c++17", "-w", "-I", os.path.join(root, "include"),
                    "-I", os.path.join(pkg, "csrc"), os.path.join(pkg, "gen_lin_plan.cpp"),
                    os.path.join(pkg, "csrc", "model.cpp"), os.path.join(pkg, "csrc", "metadata.cpp"),
                    "-o", exe], check=True)
    rel = "tests/golden/templates/shapeev-16.mtp"
    out = subprocess.run([exe, rel, "LinPlanLevel16"], cwd=root, check=True,
                         capture_output=True, text=True).stdout
    with open(os.path.join(pkg, "csrc", "lin_plan_level16.inc")) as f:
        assert f.read() == out
    # another structure gives another plan (the kernel keeps the run-time walk)
    other = subprocess.run([exe, "tests/golden/templates/shapeev-20.mtp", "LinPlanLevel16"],
                           cwd=root, check=True, capture_output=True, text=True).stdout
    assert other.split("struct", 1)[1] != out.split("struct", 1)[1]
    for text in (out, other):
        _check_lin_chunks(text)


def _check_lin_chunks(text):
    """The chunks of a generated plan partition the scalars into groups of at
    most 6 scalars and 128 (slot, scalar) entries, and share slots: they form
    fewer slots per site than chunks of consecutive scalars would."""
    import re
    S = int(re.search(r"nslots = (\d+), nchunks = (\d+), S = (\d+)", text).group(3))
    nch = int(re.search(r"nchunks = (\d+)", text).group(1))
    s0 = [int(v) for v in re.search(r"chunk_s0\[\d+\] = \{([^}]*)\}", text).group(1).split(",")]
    scal = [int(v) for v in re.search(r"scalar\[\d+\] = \{([^}]*)\}", text).group(1).split(",")]
    body = re.search(r"mask\[\d+\]\[\d+\] = \{(.*?)\};", text, re.S).group(1)
    masks = [[int(v) for v in row.split(",")] for row in re.findall(r"\{([^{}]*)\}", body)]
    assert sorted(scal) == list(range(S)) and len(s0) == nch + 1 and s0[-1] == S
    slots_of = {}
    for c in range(nch):
        w = s0[c + 1] - s0[c]
        assert 1 <= w <= 6
        ent = sum(bin(v).count("1") for v in masks[c])
        assert ent <= 128 or w == 1
        assert all(v >> w == 0 for v in masks[c])
        for k in range(w):
            slots_of[scal[s0[c] + k]] = {sl for sl, v in enumerate(masks[c]) if v >> k & 1}
    formed = sum(len(set().union(*(slots_of[scal[q]] for q in range(s0[c], s0[c + 1]))))
                 for c in range(nch))
    consecutive = sum(len(set().union(*(slots_of[q] for q in range(a, min(a + 6, S)))))
                      for a in range(0, S, 6))
    assert formed < consecutive


@pytest.mark.parametrize("first,step,last", [(20000, 40, 24000), (5000, 100000, 2000000),
                                             (160000, 32, 170000)])
def test_pinned_buffers_grow_in_strides(tmp_path, first, step, last):
    """Requests that grow a little from call to call pin memory a few times,
    not on every call, and never hold more than half again what was asked for
    (tests/pinned_growth.cpp; the smallest buffer has 4096 bytes)."""
    import math
    import os
    import shutil
    import subprocess
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc is not available")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    exe = str(tmp_path / "pinned_growth")
    subprocess.run([hipcc, "-O1", "-std=c++17", "-w", "-I", os.path.join(root, "include"),
                    "-I", os.path.join(root, "imr-mlp_amd", "csrc"),
                    os.path.join(root, "tests", "pinned_growth.cpp"), "-o", exe], check=True)
    def run(limit):
        out = subprocess.run([exe, str(first), str(step), str(last), str(limit)], check=True,
                             capture_output=True, text=True).stdout
        return [int(t) for t in out.split()]

    allocations, held = run(10 * last)
    assert allocations <= 2 + math.ceil(math.log(last / first) / math.log(1.5))
    assert held <= max(4096, 1.5 * last)
    # with room for no more than the last request every request is still met
    assert last - step < run(last)[1] <= last


@pytest.fixture(scope="module")
def rule_dump(tmp_path_factory):
    """tests/rule_tables_dump.cpp built against the library's plan code."""
    import os
    import shutil
    import subprocess
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc is not available")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    pkg = os.path.join(root, "imr-mlp_amd")
    exe = str(tmp_path_factory.mktemp("rules") / "rule_tables_dump")
    subprocess.run([hipcc, "-O1", "-std=c++17", "-w", "-I", os.path.join(root, "include"),
                    "-I", os.path.join(pkg, "csrc"),
                    os.path.join(root, "tests", "rule_tables_dump.cpp"),
                    os.path.join(pkg, "csrc", "model.cpp"), os.path.join(pkg, "csrc", "metadata.cpp"),
                    "-o", exe], check=True)
    return root, exe


NAMES = ["shapeev-02.mtp", "shapeev-10.mtp", "shapeev-16.mtp", "shapeev-20.mtp", "pot4b.mtp",
         "ps1-7b-517.mtp", "dup-scalar.mtp"]


class _Dump:
    """The dump of one template, read in order."""

    def __init__(self, rule_dump, name):
        import os
        import subprocess
        root, exe = rule_dump
        out = subprocess.run([exe, os.path.join("tests", "golden", "templates", name)], cwd=root,
                             check=True, capture_output=True, text=True).stdout
        self.v = np.array(out.split(), dtype=np.int64)
        self.pos = 0
        self.K, self.B, self.T, self.K4, self.dummy, self.red0, self.pad, self.M = self.take(8)
        self.basic = self.take(4 * self.B).reshape(-1, 4)
        self.times = self.take(4 * self.T).reshape(-1, 4)
        self.fwd, self.bwd = self.table(), self.table()
        (self.lin_dummy, self.one, self.L0, self.nL, self.lin_priv, nslots, nchunks,
         S) = self.take(8)
        self.lin = nchunks >= 0
        if self.lin:
            self.slot_basic, self.map = self.take(nslots), self.take(S)
            self.chunk_s0, self.chunk_scalar = self.take(nchunks + 1), self.take(S)
            self.slot_mask = self.take(nchunks * nslots).reshape(nchunks, nslots)
            self.slot_L = self.take(nchunks * nslots * 6).reshape(nchunks, nslots, 6)
            self.lin_fwd, self.lin_tab = self.table(), self.table()
        self.moments = []
        for _ in range(self.take(1)[0]):
            nu, n, groups = self.take(3)
            self.moments.append((nu, groups, self.take(64 * n).reshape(n, 64),
                                 self.take(192 * n).reshape(n, 3, 64)))
        assert self.pos == len(self.v)

    def take(self, n):
        self.pos += n
        return self.v[self.pos - n:self.pos]

    def table(self):
        nlev, nsteps = self.take(2)
        ls = self.take(nlev + 1)
        return ls, self.take(128 * nsteps).reshape(nsteps, 64, 2)


def _fields(x, y):
    """l, r, w, c, last of a step entry."""
    c = (y >> 17) & 0x3FFF
    return x & 0xFFFF, (x >> 16) & 0xFFFF, y & 0xFFFF, c - (c >> 13 << 14), y < 0


def _check_shape(tab, dummy, pad):
    """A level is as long as its longest lane; the padding after the last
    level reads the zero slot and writes nothing."""
    ls, steps = tab
    assert len(steps) == ls[-1] + pad
    l, r, _, c, last = _fields(steps[..., 0], steps[..., 1])
    blank = (l == dummy) & (r == dummy) & (c == 0) & ~last
    assert blank[ls[-1]:].all()
    for a, b in zip(ls[:-1], ls[1:]):
        assert b == a or not blank[b - 1].all()


def _replay(ws, tab):
    """A step table applied level by level as run_rules applies it: a level's
    operands are read as they stood when the level began, and a lane's sum is
    added to the target of the entry that ends a task or a piece of one."""
    ls, steps = tab
    for a, b in zip(ls[:-1], ls[1:]):
        snap = ws.copy()
        acc = np.zeros(64)
        for st in range(a, b):
            l, r, w, c, last = _fields(steps[st, :, 0], steps[st, :, 1])
            acc += c * snap[l] * snap[r]
            np.add.at(ws, w[last], acc[last])
            acc[last] = 0.0
        assert not acc.any()  # every sum found its target


@pytest.mark.parametrize("name", NAMES)
def test_rule_tables_apply_the_product_rules(rule_dump, name):
    """The step tables the kernels read, replayed on random basic moments and
    seeds, give the moments of the product rules in file order
    (potential_mtp.cpp:2918-2924) and the adjoints of backpropagate_moments
    (:3292-3305, reverse file order); the zero slot stays zero."""
    d = _Dump(rule_dump, name)
    for tab in (d.fwd, d.bwd):
        _check_shape(tab, d.dummy, d.pad)
    rng = np.random.default_rng(11)
    ws = np.zeros(d.red0)
    ws[:d.B] = rng.uniform(0.5, 1.5, d.B)
    m = ws[:d.K].copy()
    for l, r, c, o in d.times:
        m[o] += c * m[l] * m[r]
    _replay(ws, d.fwd)
    assert np.allclose(ws[:d.K], m, rtol=1e-12, atol=1e-12 * np.abs(m).max())
    assert not ws[d.dummy:].any()

    seed = rng.uniform(-1.0, 1.0, d.K)
    ws[d.K4:d.K4 + d.K] = seed
    A = seed.copy()
    for l, r, c, o in d.times[::-1]:
        A[r] += c * A[o] * m[l]
        A[l] += c * A[o] * m[r]
    _replay(ws, d.bwd)
    assert np.allclose(ws[d.K4:d.K4 + d.K], A, rtol=1e-11, atol=1e-12 * np.abs(A).max())
    assert not ws[d.dummy:].any()


@pytest.mark.parametrize("name", ["shapeev-10.mtp", "shapeev-16.mtp", "ps1-7b-517.mtp",
                                  "dup-scalar.mtp"])
def test_linear_tables_give_the_scalar_jacobian(rule_dump, name):
    """The linear fit's step tables: the forward rules again, then
    L[s][b] = dm_s/dm_b at the work-space index that slot_L names for every
    scalar of a chunk and every slot of its mask, and 0 outside the masks."""
    d = _Dump(rule_dump, name)
    assert d.lin
    for tab in (d.lin_fwd, d.lin_tab):
        _check_shape(tab, d.lin_dummy, d.pad)
    canon = np.arange(d.B)
    for b in range(d.B):
        canon[b] = next(k for k in range(b + 1) if np.array_equal(d.basic[k], d.basic[b]))
    rng = np.random.default_rng(12)
    ws = np.zeros(d.lin_priv)
    ws[:d.B] = rng.uniform(0.5, 1.5, d.B)[canon]
    m, J = ws[:d.K].copy(), np.zeros((d.K, d.B))
    J[np.arange(d.B), canon] = 1.0
    for l, r, c, o in d.times:
        m[o] += c * m[l] * m[r]
        J[o] += c * (m[r] * J[l] + m[l] * J[r])
    _replay(ws, d.lin_fwd)
    assert np.allclose(ws[:d.K], m, rtol=1e-12, atol=1e-12 * np.abs(m).max())
    ws[d.one:d.L0 + d.nL] = 0.0
    ws[d.one] = 1.0
    _replay(ws, d.lin_tab)
    assert not ws[d.lin_dummy] and ws[d.one] == 1.0
    scale = 1e-12 * np.abs(J).max()
    for ch in range(len(d.chunk_s0) - 1):
        for k, s in enumerate(d.chunk_scalar[d.chunk_s0[ch]:d.chunk_s0[ch + 1]]):
            got = np.zeros(d.B)
            for sl, b in enumerate(d.slot_basic):
                if d.slot_mask[ch, sl] >> k & 1:
                    got[b] = ws[d.slot_L[ch, sl, k]]
            assert np.allclose(got, J[d.map[s]], rtol=1e-12, atol=scale)


@pytest.mark.parametrize("name", NAMES)
def test_moment_tables_place_every_moment_and_tangent(rule_dump, name):
    """moment_table for every profile degree that holds the model: the sums of
    f Y, h Y and t Y over the table's (function, monomial) entries, with its
    shifts and factors, are the basic moments f_mu u^a and their tangents
    h_mu u^a + t_mu . grad u^a, each moment that occurs once or first in the
    file.  (Values for one neighbour; the sums over neighbours are linear.)"""
    d = _Dump(rule_dump, name)
    rng = np.random.default_rng(13)
    u = rng.uniform(0.4, 0.9, 3)
    f, h, t = rng.uniform(0.5, 1.5, d.M), rng.uniform(0.5, 1.5, d.M), rng.uniform(0.5, 1.5, (d.M, 3))
    Y = lambda p: np.prod([u[k] ** p[k] for k in range(3)]) if min(p) >= 0 else 0.0
    want, wantq, seen = np.zeros(d.B), np.zeros(d.B), set()
    for b, (mu, *p) in enumerate(d.basic.tolist()):
        if (mu, *p) in seen:
            continue
        seen.add((mu, *p))
        want[b] = f[mu] * Y(p)
        wantq[b] = h[mu] * Y(p) + sum(
            t[mu, k] * p[k] * Y([p[j] - (j == k) for j in range(3)]) for k in range(3))
    assert d.moments
    for nu, groups, tab, shift in d.moments:
        mono = [(a, b, c) for c in range(nu + 1) for b in range(nu - c + 1)
                for a in range(nu - c - b + 1)]
        got, gotq, entry = np.zeros(d.B), np.zeros(d.B), 0
        for ch in range((len(mono) + 15) // 16):
            for g in range(2):
                if not groups >> (2 * ch + g) & 1:
                    continue
                for lane in range(64):
                    mu, e = 4 * g + lane // 16, 16 * ch + lane % 16
                    to = [tab[entry, lane], *(shift[entry, :, lane] & 0xFFFF)]
                    if mu >= d.M or e >= len(mono):
                        assert all(w == 0xFFFF for w in to)
                        continue
                    y = Y(mono[e])
                    if to[0] != 0xFFFF:
                        got[to[0]] += f[mu] * y
                        gotq[to[0]] += h[mu] * y
                    for k in range(3):
                        if to[1 + k] != 0xFFFF:
                            gotq[to[1 + k]] += (shift[entry, k, lane] >> 16) * t[mu, k] * y
                entry += 1
            assert groups >> (2 * ch) & 1  # the compile-time profiles count on group 0
        assert entry == len(tab)
        assert np.allclose(got, want, rtol=1e-13) and np.allclose(gotq, wantq, rtol=1e-13)
