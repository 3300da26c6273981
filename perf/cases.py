"""Performance cases: the calls a program makes on this library, over the sizes it meets.

A case is a plain dict.  `op` names the call:

  md        one molecular-dynamics step: lists from host positions, then E/F/S
  efs       E/F/S on resident lists
  mc        one Monte-Carlo trial: lists from host positions, then energies
  screen    a batch of structures: lists of all of them, then batch E/F/S
  sites     one time step of a LAMMPS pair style: CSR with ghost atoms, kept topology
  train     one loss + gradient evaluation of a training batch
  linear    the normal equations of a linear fit

`template` is the moment structure (level 10, 16, 20), `species` Z, `basis`
the radial basis kind, `head` an MTP-M head or "".  `atoms` counts all atoms,
spread over `structures` structures of different sizes; `liquid` chooses
disordered structures instead of strained, displaced crystals with vacancies.
All floating-point work is in 64 bits.
"""
import math
import os
import re
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("imr-mlp_amd"))

from mtpx import capi, synth  # noqa: E402

#: Per template: radial basis size, min_dist, max_dist (angstrom).
MODELS = {"shapeev-10.mtp": (8, 2.0, 5.0), "shapeev-16.mtp": (8, 1.9, 5.0), "shapeev-20.mtp": (10, 1.5, 5.5)}
SCALING = 0.01
POLY5_B = -1.0 / 3.0  # write_mtp's rb_b of a Poly5 basis
LINEAR_VALUES = 1000  # d(scalar moment) / d(basic moment) that are not always zero, level 16
HEAD_Q, HEAD_H1 = 3, 16  # an mtp_m_n1 head: descriptors, hidden units
FCC_A, LIQUID_DENSITY = 3.56, 0.06


def case(name, op, template, atoms, species=2, structures=1, liquid=False, basis="RBChebyshev", head=""):
    c = dict(op=op, template=template, atoms=atoms, species=species, structures=structures, liquid=liquid, basis=basis, head=head)
    return dict(c, name=name) if name else c


def listed():
    return [
        # a small cell relaxed or run step by step: the shortest call, where launches and copies count
        case("md_l10_108", "md", "shapeev-10.mtp", 108, species=1),
        # an ordinary MD cell of an odd size
        case("md_l16_997", "md", "shapeev-16.mtp", 997),
        # a large MD cell (the benchmark's cell) with the lists rebuilt from the host's positions
        case("md_l16_32000", "md", "shapeev-16.mtp", 32000),
        # the benchmark's E/F/S on resident lists
        case("efs_l16_32000", "efs", "shapeev-16.mtp", 32000),
        # the largest: a level-20 four-species cell
        case("efs_l20_256000", "efs", "shapeev-20.mtp", 256000, species=4),
        # a radial basis the compiled profiles do not cover
        case("efs_poly5_l16_4001", "efs", "shapeev-16.mtp", 4001, basis="RBChebyshevPoly5"),
        # a potential with a neural site-energy head
        case("efs_n1_l16_4000", "efs", "shapeev-16.mtp", 4000, head="mtp_m_n1"),
        # high-throughput screening: many small structures of different sizes at once
        case("screen_l16_200", "screen", "shapeev-16.mtp", 16800, structures=200),
        # one LAMMPS time step of a mid-sized subdomain with its ghost atoms
        case("sites_l16_5324", "sites", "shapeev-16.mtp", 5324),
        # a small training set: one L-BFGS evaluation
        case("train_l16_40", "train", "shapeev-16.mtp", 4400, structures=40),
        # a large training set of disordered structures, level 20
        case("train_l20_1000", "train", "shapeev-20.mtp", 160000, species=3, structures=1000, liquid=True),
        # the assembly of a linear fit
        case("linear_l16_1000", "linear", "shapeev-16.mtp", 160000, structures=1000),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    op = rng.choice(["md", "md", "efs", "efs", "mc", "screen", "sites", "train", "linear"])
    level = rng.choice([10, 16, 16, 20]) if op != "linear" else 16
    species = rng.randint(1, 4) if op != "linear" else 2
    liquid = rng.random() < 0.3
    most = {"md": 60000, "efs": 200000, "mc": 20000, "sites": 20000, "screen": 40000, "train": 120000, "linear": 120000}[op]
    if level == 20 and op in ("md", "sites"):
        most //= 2
    structures = 1
    if op in ("screen", "train", "linear"):
        structures = _log_int(rng, 2, 700)
        atoms = min(most, structures * rng.randint(20, 170) + rng.randint(0, 9))
    else:
        atoms = _log_int(rng, 33, most)
    basis = "RBChebyshevPoly5" if op in ("md", "efs", "mc", "train") and rng.random() < 0.15 else "RBChebyshev"
    if basis != "RBChebyshev" or (liquid and op != "train"):
        atoms = min(atoms, 60000)
    head = "mtp_m_n1" if op in ("md", "efs", "mc", "screen", "sites") and rng.random() < 0.15 else ""
    return case("", op, "shapeev-%d.mtp" % level, atoms, species, structures, liquid, basis, head)


# ---- inputs ------------------------------------------------------------------


class Cell:
    def __init__(self, cell, pos, types):
        self.cell, self.pos, self.types, self.pbc = cell, pos, types, np.ones(3, np.int32)
        self.n = len(types)


def _boxes(n):
    """Near-cubic (a, b, c) with a b c >= n, as tight as such a box gets."""
    a = max(1, int(round(n ** (1 / 3))))
    best = None
    for p in range(max(1, a - 2), a + 3):
        for q in range(max(1, a - 2), a + 3):
            r = -(-n // (p * q))
            if max(p, q, r) <= 2 * min(p, q, r) + 1 and (best is None or p * q * r < best[0]):
                best = (p * q * r, (p, q, r))
    return best[1]


def _structure(rng, n, species, liquid):
    """n atoms: a jittered grid at liquid density, or an FCC crystal with
    vacancies, strained and thermally displaced; random species, periodic."""
    if liquid:
        reps = np.array(_boxes(n))
        a, basis = LIQUID_DENSITY ** (-1 / 3), np.zeros((1, 3))
    else:
        reps = np.array(_boxes(-(-n // 4)))
        a, basis = FCC_A, synth.FCC_BASIS
    grid = np.stack(np.meshgrid(*[np.arange(r) for r in reps], indexing="ij"), -1).reshape(-1, 1, 3)
    frac = ((grid + basis) / reps).reshape(-1, 3)
    if len(frac) > n:
        frac = frac[np.sort(rng.permutation(len(frac))[:n])]
    cell = np.diag(reps * a).astype(np.float64)
    pos = frac @ cell
    if liquid:
        pos = pos + rng.uniform(-0.45, 0.45, pos.shape)
    else:
        e = rng.uniform(-0.02, 0.02, 6)
        strain = np.eye(3) + np.array([[e[0], e[3], e[4]], [e[3], e[1], e[5]], [e[4], e[5], e[2]]])
        cell, pos = cell @ strain, pos @ strain + 0.1 * rng.standard_normal(pos.shape)
    return Cell(cell, capi.wrap(cell, np.ones(3, np.int32), pos), rng.integers(0, species, n).astype(np.int32))


def _structures(c, seed):
    rng = np.random.default_rng([seed, 1])
    k = c["structures"]
    if k == 1:
        sizes = [c["atoms"]]
    else:  # sizes from half to one and a half times the mean
        w = rng.uniform(0.5, 1.5, k)
        sizes = np.maximum(1, np.floor(w / w.sum() * c["atoms"]).astype(int))
        sizes[-1] += max(0, c["atoms"] - sizes.sum())
    return [_structure(rng, int(n), c["species"], c["liquid"]) for n in sizes]


_TOPO = {}


def _topology(template):
    """The moment structure of a template: basic [B][4], times [T][4], map [S], M."""
    if template not in _TOPO:
        text = synth.read_template(template)

        def ints(key):
            m = re.search(r"^%s\s*=\s*\{(.*?)\}\s*$" % key, text, re.M | re.S)
            return np.array([int(v) for v in re.findall(r"-?\d+", m.group(1))])

        K = int(re.search(r"alpha_moments_count\s*=\s*(\d+)", text).group(1))
        M = int(re.search(r"radial_funcs_count\s*=\s*(\d+)", text).group(1))
        _TOPO[template] = dict(K=K, M=M, basic=ints("alpha_index_basic").reshape(-1, 4),
                               times=ints("alpha_index_times").reshape(-1, 4), map=ints("alpha_moment_mapping"))
    return _TOPO[template]


def _coefficients(c, seed):
    """Flat [radial | species | moment] and, with a head, its own coefficients."""
    t, Z = _topology(c["template"]), c["species"]
    R = MODELS[c["template"]][0]
    rng = np.random.default_rng([seed, 2])
    x = rng.uniform(-0.05, 0.05, Z * Z * t["M"] * R + Z + len(t["map"]))
    if not c["head"]:
        return x, None
    q, S = HEAD_Q, len(t["map"])
    return x, dict(species=rng.uniform(-0.1, 0.1, Z), dspecies=rng.uniform(-0.1, 0.1, (q, Z)),
                   moment=rng.uniform(-0.1, 0.1, (q, S)), w1=rng.uniform(-0.5, 0.5, (HEAD_H1, q)),
                   out=rng.uniform(-0.5, 0.5, HEAD_H1), b1=rng.uniform(-0.5, 0.5, HEAD_H1))


def _model_text(c, seed):
    R, rmin, rmax = MODELS[c["template"]]
    x, head = _coefficients(c, seed)
    topo = _topology(c["template"])
    text = synth.write_mtp(topo, c["species"], R, rmin, rmax, SCALING, x, basis=c["basis"])
    if head is None:
        return text

    def line(key, v):
        return "%s = {%s}" % (key, ", ".join("%.17e" % u for u in np.concatenate([np.ravel(a) for a in v])))

    body = [ln for ln in text.rstrip("\n").split("\n") if not ln.startswith(("species_coeffs", "moment_coeffs"))]
    body += [line("species_coeffs", [head["species"], head["dspecies"]]), line("moment_coeffs", [head["moment"]]),
             line("model_coeffs", [head["w1"], head["out"], head["b1"]]),
             "# mtp_model = mtp_m_n1", "# mtp_descriptor_count = %d" % HEAD_Q,
             "# mtp_model_coeffs_count = %d" % (HEAD_H1 * (HEAD_Q + 2)), "# mtp_activation = TANH",
             "# mtp_hidden1 = %d" % HEAD_H1, "# mtp_hidden2 = 0"]
    return "\n".join(body) + "\n"


def _labels(c, seed, sizes):
    """Targets of the size of early training residuals: E [nconf], F [N][3], S [nconf][3][3]."""
    rng = np.random.default_rng([seed, 3])
    k, n = len(sizes), int(np.sum(sizes))
    s = rng.standard_normal((k, 3, 3))
    return (0.2 * np.sqrt(sizes) * rng.standard_normal(k), 0.3 * rng.standard_normal((n, 3)),
            (s + s.transpose(0, 2, 1)) * np.sqrt(np.asarray(sizes, float))[:, None, None])


class State:
    pass


def prepare(c, seed):
    s = State()
    s.op = c["op"]
    s.rmax = MODELS[c["template"]][2]
    s.ctx = capi.Context(0)
    s.ctx.load_model_text(_model_text(c, seed))
    s.ctx.set_timings(False)
    cells = _structures(c, seed)
    if s.op in ("md", "mc"):
        s.cell = cells[0]
    elif s.op == "screen":
        s.cells = cells
    elif s.op == "efs":
        st = cells[0]
        s.ctx.build_neighbors(st.cell, st.pbc, st.pos, st.types, s.rmax)
    elif s.op == "sites":
        s.request = _ghost_request(s.ctx, cells[0], s.rmax)
        s.ctx.compute_sites(**s.request)  # the step at which the pair style rebuilds its lists
        s.request["reuse"] = True
    else:
        off = s.ctx.set_structures(cells, s.rmax)
        E, F, S = _labels(c, seed, np.diff(off))
        act, wE, wF, wS = capi.loss_weights(capi.LossSettings.make(), off, np.ones((len(cells), 3), np.int32), F)
        s.ctx.set_labels(act, E, wE, F, wF, S, wS)
    return s


def _ghost_request(ctx, st, rmax):
    """The periodic cell as a pair style sees it: owned atoms first, then its
    ghosts: every periodic image within the cutoff of an owned atom, and as
    many of the skin's further images as fill the shell the styles exchange."""
    ctx.build_neighbors(st.cell, st.pbc, st.pos, st.types, rmax)
    nb = ctx.get_neighbors()
    ctr = np.repeat(np.arange(st.n), np.diff(nb["offsets"]))
    far = st.pos[ctr] + nb["vec"]
    shift = np.rint((far - st.pos[nb["idx"]]) @ np.linalg.inv(st.cell)).astype(np.int64)
    key = ((nb["idx"].astype(np.int64) * 64 + shift[:, 0] + 32) * 64 + shift[:, 1] + 32) * 64 + shift[:, 2] + 32
    outside = np.any(shift != 0, axis=1)
    images, first, which = np.unique(key[outside], return_index=True, return_inverse=True)
    neighbors = nb["idx"].copy()
    neighbors[outside] = st.n + which
    gidx, gshift = nb["idx"][outside][first], shift[outside][first]
    side = (st.n / (4 / FCC_A ** 3)) ** (1 / 3)
    rest = 200 + int(1.2 * st.n * ((1 + 2 * rmax / side) ** 3 - 1)) - len(images)
    assert rest >= 0
    gidx = np.concatenate([gidx, np.arange(rest) % st.n])
    gshift = np.concatenate([gshift, np.full((rest, 3), 9)])
    x = np.concatenate([st.pos, st.pos[gidx] + gshift @ st.cell])
    return dict(offsets=nb["offsets"], neighbors=neighbors.astype(np.int32), nlocal=st.n, x=x,
                types=np.concatenate([st.types, st.types[gidx]]), site_virial=False, accumulate=False)


def run(s):
    if s.op == "efs":
        return s.ctx.efs()
    if s.op in ("md", "mc"):
        st = s.cell
        s.ctx.build_neighbors(st.cell, st.pbc, st.pos, st.types, s.rmax)
        return s.ctx.efs() if s.op == "md" else s.ctx.energy()
    if s.op == "screen":
        s.ctx.set_structures(s.cells, s.rmax)
        return s.ctx.compute_batch()
    if s.op == "sites":
        r = s.ctx.compute_sites(**s.request)
        return r["energy"], r["virial6"], r["force"], r["site_energy"]
    if s.op == "train":
        return s.ctx.loss_grad()
    return s.ctx.linear_system()


def work(c):
    """Flops of the mathematics (monomials, radial functions and moments once
    per neighbour; a value and three derivatives per moment backwards; the
    products forwards and backwards), bytes of the inputs and outputs."""
    t, n = _topology(c["template"]), float(c["atoms"])
    R, _, rmax = MODELS[c["template"]]
    M, B, T, S, Z = t["M"], len(t["basic"]), len(t["times"]), len(t["map"]), c["species"]
    nu = int(t["basic"][:, 1:].sum(1).max())
    mono = math.comb(nu + 3, 3)
    density = LIQUID_DENSITY if c["liquid"] else 4 / FCC_A ** 3
    per_entry_list = 40.0
    P = n * density * 4 / 3 * math.pi * rmax ** 3
    ncoef = Z * Z * M * R + Z + S
    radial = 8.0 * R + 2 * M * R
    forward, force = radial + mono + 2.0 * B, radial + 2 * M * R + 7.0 * B + 20
    flops = P * forward + n * (3.0 * T + 2 * S)
    io = n * 28 + 8.0 * ncoef
    if c["op"] != "mc":
        flops += P * force + n * 6.0 * T
        io += n * 32
    if c["op"] == "efs":
        io += P * per_entry_list
    if c["op"] == "sites":
        io += P * 4 + n * 28
    if c["op"] == "train":  # tangents forwards, second adjoints backwards, radial coefficients
        flops += P * (2 * forward + 9.0 * B + 4 * M * R) + n * 18.0 * T
        io += P * per_entry_list + n * 56
    if c["op"] == "linear":  # sparse site Jacobian walks; A^T A over the force rows
        p = Z + S
        flops = P * (forward + 6.0 * B + 6.0 * LINEAR_VALUES) + n * 6.0 * T + 3 * n * p * (p + 3)
        io += P * per_entry_list + 8.0 * p * (p + 1)
    return {"bytes": io, "flops": flops}


def tolerance(c):
    # all in 64 bits; forces are sums of some 10^4 terms that cancel (up to 1e-13 against exact())
    return {"rel": 4e-13, "max": 4e-11}


# ---- the same in plain torch -------------------------------------------------------


def _neighbors(st, rc, dev):
    """Padded lists by direct search: idx, vec [n][m][.], mask [n][m]."""
    n = st.n
    pos = torch.tensor(st.pos, device=dev)
    cell = torch.tensor(st.cell, device=dev)
    inv = torch.linalg.inv(cell)
    height = 1.0 / torch.linalg.norm(inv, dim=0)
    reach = [int(math.ceil(rc / float(h))) for h in height]
    frac = pos @ inv
    rows, idx, vec = [], [], []
    wide = all(float(h) > 2 * rc for h in height)  # at most one image of a pair within the cutoff
    shifts = None if wide else torch.tensor([[a, b, d] for a in range(-reach[0], reach[0] + 1)
                                             for b in range(-reach[1], reach[1] + 1)
                                             for d in range(-reach[2], reach[2] + 1)], dtype=torch.float64, device=dev)
    step = max(1, int(4e7 // (n * (1 if wide else len(shifts)))))
    for i0 in range(0, n, step):
        i1 = min(n, i0 + step)
        if wide:
            df = frac[None, :, :] - frac[i0:i1, None, :]
            sh = -torch.round(df)
            d2 = ((df + sh) @ cell).square().sum(-1)
            i, j = torch.nonzero(d2 <= rc * rc, as_tuple=True)
            v = pos[j] - pos[i + i0] + sh[i, j] @ cell
        else:
            d0 = pos[None, :, :] - pos[i0:i1, None, :]
            d2 = (d0[:, :, None, :] + shifts @ cell).square().sum(-1)
            i, j, k = torch.nonzero(d2 <= rc * rc, as_tuple=True)
            v = d0[i, j] + shifts[k] @ cell
        keep = v.square().sum(-1) > 1e-12
        rows.append(i[keep] + i0), idx.append(j[keep]), vec.append(v[keep])
    return torch.cat(rows), torch.cat(idx), torch.cat(vec)


def _basis(c, d):
    R, lo, hi = MODELS[c["template"]]
    ksi = (2 * d - (hi + lo)) / (hi - lo)
    if c["basis"] == "RBChebyshev":
        env = (d - hi) ** 2
    else:
        x = (d - lo) / (hi - lo)
        env = torch.where(d < lo, torch.zeros_like(d), (1 - x) ** 4 * (1 + (4 + POLY5_B) * x))
    Q = [SCALING * env, SCALING * ksi * env]
    for _ in range(2, R):
        Q.append(2 * ksi * Q[-1] - Q[-2])
    return torch.stack(Q[:R], -1)


def _site_moments(c, radial, ti, tj, vec, mask):
    """Every moment of every site: a list of K tensors [n]."""
    t = _topology(c["template"])
    d = torch.where(mask, vec.square().sum(-1), torch.ones_like(mask, dtype=vec.dtype)).sqrt()
    f = torch.einsum("nmr,nmkr->nmk", _basis(c, d), radial[ti[:, None], tj]) * mask[..., None]
    u = vec / d[..., None]
    powers = [[torch.ones_like(d)] for _ in range(3)]
    for a in range(3):
        for _ in range(int(t["basic"][:, 1:].max())):
            powers[a].append(powers[a][-1] * u[..., a])
    mono, m = {}, [None] * t["K"]
    for b, (mu, p, q, r) in enumerate(t["basic"].tolist()):
        if (p, q, r) not in mono:
            mono[p, q, r] = powers[0][p] * powers[1][q] * powers[2][r]
        m[b] = (f[..., mu] * mono[p, q, r]).sum(1)
    for left, right, k, out in t["times"].tolist():
        v = k * m[left] * m[right]
        m[out] = v if m[out] is None else m[out] + v
    return m


def _site_energy(c, m, ti, species, moment, head, dev):
    t = _topology(c["template"])
    if head is None:
        return species[ti] + torch.stack([m[k] for k in t["map"]], -1) @ moment
    h = {k: torch.tensor(v, device=dev) for k, v in head.items()}
    Q = h["dspecies"][:, ti].T + torch.stack([m[k] for k in t["map"]], -1) @ h["moment"].T
    return h["species"][ti] + torch.tanh(Q @ h["w1"].T + h["b1"]) @ h["out"]


def _padded(st, rc, dev):
    """All lists of a set of structures, as chunks of sites: (first site, types, idx, vec, mask)."""
    base, chunks = 0, []
    group, sites = [], 0
    for k, one in enumerate(st):
        r, j, v = _neighbors(one, rc, dev)
        group.append((r + sites, j + base, v, torch.tensor(one.types, device=dev, dtype=torch.long), k))
        base, sites = base + one.n, sites + one.n
        if sites >= 12000 or k == len(st) - 1:
            rows, idx, vec = (torch.cat([g[q] for g in group]) for q in range(3))
            types = torch.cat([g[3] for g in group])
            chunks.append((base - sites, sites, types, rows, idx, vec))
            group, sites = [], 0
    for first, n, types, rows, idx, vec in chunks:
        order = torch.argsort(rows, stable=True)
        rows, idx, vec = rows[order], idx[order], vec[order]
        count = torch.bincount(rows, minlength=n)
        start = torch.cumsum(count, 0) - count
        at = torch.arange(len(rows), device=dev) - start[rows]
        for i0 in range(0, n, 16000):
            i1 = min(n, i0 + 16000)
            pick = (rows >= i0) & (rows < i1)
            m = max(1, int(count[i0:i1].max()))
            J = torch.zeros((i1 - i0, m), dtype=torch.long, device=dev)
            V = torch.zeros((i1 - i0, m, 3), dtype=torch.float64, device=dev)
            ok = torch.zeros((i1 - i0, m), dtype=torch.bool, device=dev)
            r, a = rows[pick] - i0, at[pick]
            J[r, a], V[r, a], ok[r, a] = idx[pick], vec[pick], True
            V[~ok] = torch.tensor([1.0, 0.0, 0.0], dtype=torch.float64, device=dev)
            yield first + i0, types[i0:i1], J, V, ok


def exact(c, seed):
    entries = c["atoms"] * (95 if "20" in c["template"] else 60)
    if c["op"] in ("train", "linear") and entries > 12e6 or entries > 30e6:
        return None
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    st = _structures(c, seed)
    t, Z = _topology(c["template"]), c["species"]
    R, _, rc = MODELS[c["template"]]
    x, head = _coefficients(c, seed)
    nrad = Z * Z * t["M"] * R
    x = torch.tensor(x, device=dev)
    radial0, species, moment = x[:nrad].reshape(Z, Z, t["M"], R), x[nrad:nrad + Z], x[nrad + Z:]
    sizes = np.array([s.n for s in st])
    N, nc = int(sizes.sum()), len(st)
    conf = torch.repeat_interleave(torch.arange(nc, device=dev), torch.tensor(sizes, device=dev))
    types = torch.cat([torch.tensor(s.types, device=dev, dtype=torch.long) for s in st])
    fitting = c["op"] in ("train", "linear")
    if fitting:
        tE, tF, tS = (torch.tensor(v, device=dev) for v in _labels(c, seed, sizes))
        wE = 1.0 / torch.tensor(sizes, dtype=torch.float64, device=dev)
        wF, wS = 0.01, 1e-4 * wE
    E = torch.zeros(nc, dtype=torch.float64, device=dev)
    F = torch.zeros(N, 3, dtype=torch.float64, device=dev)
    S = torch.zeros(nc, 3, 3, dtype=torch.float64, device=dev)
    site = torch.zeros(N, dtype=torch.float64, device=dev)
    p = Z + len(t["map"])
    if c["op"] == "linear":
        eC = torch.zeros(nc, p, dtype=torch.float64, device=dev)
        fC = torch.zeros(N, 3, p, dtype=torch.float64, device=dev)
        sC = torch.zeros(nc, 3, 3, p, dtype=torch.float64, device=dev)
    gradient, loss, metrics = torch.zeros_like(x), 0.0, torch.zeros(7, dtype=torch.float64, device=dev)
    train = c["op"] == "train"
    for first, ti, J, V, ok in _padded(st, rc, dev):
        n = len(ti)
        tj = types[J]
        cf = conf[first:first + n]
        V = V.requires_grad_(True)
        xr = x.clone().requires_grad_(train)
        radial = xr[:nrad].reshape(Z, Z, t["M"], R)
        m = _site_moments(c, radial, ti, tj, V, ok)
        if c["op"] == "linear":
            eC.index_add_(0, cf, torch.nn.functional.one_hot(ti, p).double())
            for s, k in enumerate(t["map"].tolist()):
                D, = torch.autograd.grad(m[k].sum(), V, retain_graph=True)
                eC[:, Z + s].index_add_(0, cf, m[k].detach())
                fC[first:first + n, :, Z + s] += D.sum(1)
                fC[:, :, Z + s].index_add_(0, J.reshape(-1), -D.reshape(-1, 3))
                sC[:, :, :, Z + s].index_add_(0, cf, -torch.einsum("nma,nmb->nab", D, V.detach()))
            continue
        e = _site_energy(c, m, ti, xr[nrad:nrad + Z], xr[nrad + Z:], head, dev)
        if c["op"] == "mc":
            site[first:first + n] = e.detach()
            E.index_add_(0, cf, e.detach())
            continue
        D, = torch.autograd.grad(e.sum(), V, create_graph=train)
        Fl = torch.zeros_like(F).index_add(0, J.reshape(-1), -D.reshape(-1, 3))
        Fl = Fl.index_add(0, torch.arange(first, first + n, device=dev), D.sum(1))
        Sl = torch.zeros_like(S).index_add(0, cf, -torch.einsum("nma,nmb->nab", D, V))
        El = torch.zeros_like(E).index_add(0, cf, e)
        if train:  # a chunk holds whole structures
            k = torch.unique(cf)
            a = slice(first, first + n)
            dE, dF, dS = El[k] - tE[k], Fl[a] - tF[a], Sl[k] - tS[k]
            le, lf = (wE[k] * dE ** 2).sum(), wF * dF.square().sum()
            ls = (wS[k] * dS.square().sum((1, 2))).sum()
            g, = torch.autograd.grad(le + lf + ls, xr)
            gradient += g / nc
            loss += float(le + lf + ls) / nc
            q = torch.tensor(sizes, device=dev)[k]
            metrics += torch.stack([le + lf + ls, le, lf, ls, ((dE / q) ** 2).sum(), dF.square().sum(),
                                    dS.square().sum()]).detach()
        else:
            E, F, S = E + El.detach(), F + Fl.detach(), S + Sl.detach()
            site[first:first + n] = e.detach()
    host = lambda v: v.cpu().numpy()  # noqa: E731
    if train:
        return loss, host(gradient), host(metrics)
    if c["op"] == "linear":
        rows = [eC * wE.sqrt()[:, None], fC.reshape(-1, p) * math.sqrt(wF),
                sC.reshape(-1, p) * wS.sqrt().repeat_interleave(9)[:, None]]
        rhs = [tE * wE.sqrt(), tF.reshape(-1) * math.sqrt(wF), tS.reshape(-1) * wS.sqrt().repeat_interleave(9)]
        A, y = torch.cat(rows), torch.cat(rhs)
        return host(A.T @ A), host(A.T @ y)
    if c["op"] == "mc":
        return host(E), host(site)
    if c["op"] == "screen":
        return host(E), host(F), host(S), host(site)
    if c["op"] == "sites":  # forces stay on the ghosts there: only energy and virial compare
        v = host(S[0])
        return float(E[0]), np.array([v[0, 0], v[1, 1], v[2, 2], (v[0, 1] + v[1, 0]) / 2, (v[0, 2] + v[2, 0]) / 2,
                                      (v[1, 2] + v[2, 1]) / 2]), None, host(site)
    return float(E[0]), host(F), host(S[0]), host(site)
