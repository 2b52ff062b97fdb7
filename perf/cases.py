"""The work that a user of this framework has it do, as measurable cases.

The framework solves block-tridiagonal Green's function problems for batches
of energy points: the selected solve (G^R, G^<, G^>) and the selected
inversion, the open boundary conditions before them, the system-matrix
assembly, and the same solve on block-sparse stacks.  Everything is complex128;
FP64 is the precision of every path that is used in earnest (the complex64
products are an opt-in whose errors do not allow serving).

Inputs are those of the synthetic tight-binding device of
``quatrex_amd.workloads`` (Hermitian H with ``CN(0, 1) / sqrt(b)`` blocks,
couplings scaled by 0.3, contacts ``-0.5 i``), drawn on the GPU, with
self-energies that differ per energy and have off-diagonal blocks, as a
self-consistent loop hands them over.
"""

import math

import numpy as np
import torch

from quatrex_amd import solve as S
from quatrex_amd.boundary_conditions import OBCSystem, SanchoRubio, Spectral, compute_contact_obc
from quatrex_amd.dsdb import DSDBCOO
from quatrex_amd.greens_function_solver import RGF
from quatrex_amd.layout import Geometry
from quatrex_amd.nevp import Beyn

ETA = 1e-3
BOUNDARY = -0.5j
C128 = torch.complex128


def listed():
    return [
        # one energy point of the smallest device: a call's latency and nothing else
        dict(name="solve_8x32_1", kind="solve", n_blocks=8, block=32, ragged=False, energies=1,
             retarded=True, current=False),
        # a sweep over small blocks, where a thousand energy points fit one call
        dict(name="solve_32x32_1024", kind="solve", n_blocks=32, block=32, ragged=False, energies=1024,
             retarded=True, current=False),
        # blocks of odd and unequal sizes with contacts as boundary blocks and the
        # layer currents: the last iteration of a self-consistent loop
        dict(name="current_12x77_48", kind="solve", n_blocks=12, block=77, ragged=True, energies=48,
             retarded=True, current=True),
        # the screened Coulomb interaction: lesser and greater only
        dict(name="coulomb_16x128_64", kind="solve", n_blocks=16, block=128, ragged=False, energies=64,
             retarded=False, current=False),
        # few energies of a device with wide blocks
        dict(name="solve_12x512_16", kind="solve", n_blocks=12, block=512, ragged=False, energies=16,
             retarded=True, current=False),
        # the headline device, as many energies as leave room for the rest of a program
        dict(name="solve_32x256_64", kind="solve", n_blocks=32, block=256, ragged=False, energies=64,
             retarded=True, current=False),
        # a serving slot: a captured sweep of a few requests, replayed
        dict(name="graph_20x256_8", kind="graph", n_blocks=20, block=256, ragged=False, energies=8,
             retarded=True, current=False),
        # retarded only: density of states, transmission
        dict(name="inverse_24x192_32", kind="inverse", n_blocks=24, block=192, ragged=False, energies=32),
        # both steps of a contact: Sancho-Rubio surface function and self-energies
        dict(name="contact_208_64", kind="contact", block=208, energies=64),
        # the default contact solver: Beyn's contour integral and mode selection
        dict(name="spectral_128_32", kind="spectral", block=128, chains=4, energies=32),
        # the drop-in on block-sparse stacks (half of each tridiagonal block stored)
        dict(name="sparse_20x96_64", kind="sparse", n_blocks=20, block=96, energies=64, fill=0.5),
        # the electron solver's system matrix before each solve
        dict(name="assemble_32x256_32", kind="assemble", n_blocks=32, block=256, ragged=False, energies=32,
             overlap=True),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "solve", "graph", "inverse", "contact", "spectral", "sparse",
                       "assemble"])
    if kind == "contact":
        return dict(kind=kind, block=_log_uniform(rng, 24, 320), energies=_log_uniform(rng, 2, 96))
    if kind == "spectral":
        chains = rng.randint(1, 6)
        return dict(kind=kind, block=chains * _log_uniform(rng, 8, 192 // chains), chains=chains,
                    energies=_log_uniform(rng, 2, 48))
    if kind == "sparse":
        return dict(kind=kind, n_blocks=_log_uniform(rng, 3, 24), block=_log_uniform(rng, 8, 128),
                    energies=_log_uniform(rng, 2, 64), fill=round(rng.uniform(0.2, 0.9), 2))
    if kind == "graph":
        return dict(kind=kind, n_blocks=_log_uniform(rng, 4, 40), block=_log_uniform(rng, 24, 512), ragged=False,
                    energies=rng.randint(1, 8), retarded=True, current=False)
    n, b = _log_uniform(rng, 2, 48), _log_uniform(rng, 8, 512)
    ragged = rng.random() < 0.35
    # no more work than the largest listed case, and no more memory
    cap = min(1024, 9.0e12 / (8.0 * b ** 3 * 34 * n), 2.4e10 / (144.0 * n * b * b))
    if kind == "assemble":
        cap = min(256, 1.2e10 / (192.0 * n * b * b))
    energies = _log_uniform(rng, 1, max(2.0, cap))
    if kind == "assemble":
        return dict(kind=kind, n_blocks=n, block=b, ragged=ragged, energies=energies, overlap=rng.random() < 0.5)
    if kind == "inverse":
        return dict(kind=kind, n_blocks=n, block=b, ragged=ragged, energies=energies)
    current = rng.random() < 0.4
    return dict(kind=kind, n_blocks=n, block=b, ragged=ragged, energies=energies,
                retarded=current or rng.random() < 0.7, current=current)


# --- inputs -------------------------------------------------------------------


def _sizes(case):
    """Block sizes: all equal, or spread by up to a quarter around ``block``."""
    n, b = case["n_blocks"], case["block"]
    if not case.get("ragged"):
        return (b,) * n
    top = 512
    return tuple(min(top, max(1, b + (7 * i * i + 3 * i) % (b // 2 + 1) - b // 4)) for i in range(n))


class _Draw:
    def __init__(self, seed):
        self.dev = torch.device("cuda", torch.cuda.current_device())
        self.gen = torch.Generator(device=self.dev)
        self.gen.manual_seed(seed)

    def cn(self, *shape):
        """CN(0, 1) entries."""
        return torch.randn(shape, dtype=C128, device=self.dev, generator=self.gen)

    def uniform(self, n, lo, hi):
        return lo + (hi - lo) * torch.rand(n, dtype=torch.float64, device=self.dev, generator=self.gen)


def _herm(x):
    return x.mH.resolve_conj()


def _hamiltonian(d, sizes):
    """Packed (diag, upper, lower) of one Hermitian H, and lists of its blocks."""
    dd, uu, ll = [], [], []
    for i, b in enumerate(sizes):
        x = d.cn(b, b) / math.sqrt(b)
        dd.append(0.5 * (x + _herm(x)))
        if i + 1 < len(sizes):
            u = 0.3 * d.cn(b, sizes[i + 1]) / math.sqrt(b)
            uu.append(u)
            ll.append(_herm(u))
    return dd, uu, ll


def _flat(blocks, dev):
    return torch.cat([b.reshape(-1) for b in blocks]) if blocks else torch.empty(0, dtype=C128, device=dev)


def _system(d, sizes, energies, fold):
    """A = (E + i eta) - H - Sigma_B per energy, packed; the contacts folded in or left out."""
    g = Geometry(sizes)
    dd, uu, ll = _hamiltonian(d, sizes)
    z = d.uniform(energies, -1.0, 1.0) + 1j * ETA
    diag = (-_flat(dd, d.dev)).expand(energies, -1).clone()
    for i, b in enumerate(sizes):
        idx = int(g.diag_offsets[i]) + torch.arange(b, device=d.dev) * (b + 1)
        shift = z - BOUNDARY if fold and i in (0, len(sizes) - 1) else z
        diag[:, idx] += shift[:, None]
    off = [(-_flat(x, d.dev)).expand(energies, -1).clone() for x in (uu, ll)]
    return g, (diag, off[0], off[1])


def _self_energies(d, g, energies):
    """Sigma^<_ii = i f Y Y^H / b, Sigma^>_ii = -i (1 - f) Y Y^H / b with an occupation
    f per energy, and small off-diagonal blocks (upper parts; the matrices are
    skew-Hermitian)."""
    base = []
    for b in g.block_sizes:
        y = d.cn(b, b)
        base.append(y @ _herm(y) / b)
    base = _flat(base, d.dev)
    off = 0.05 * d.cn(g.offdiag_size) / math.sqrt(g.max_block)
    f = d.uniform(energies, 0.05, 0.95)[:, None]
    lesser = (1j * f * base, 1j * f * off)
    greater = (-1j * (1 - f) * base, -1j * (1 - f) * off)
    return lesser, greater


def _contacts(d, g, energies):
    """Retarded, lesser and greater boundary blocks of both contacts."""
    lists = [[None] * g.n_blocks for _ in range(3)]
    for i, mu in ((0, 0.7), (g.n_blocks - 1, 0.2)):
        b = g.block_sizes[i]
        x = d.cn(energies, b, b) / math.sqrt(b)
        gamma = torch.eye(b, dtype=C128, device=d.dev) + 0.05 * (x + _herm(x))  # positive
        re = 0.05 * d.cn(energies, b, b) / math.sqrt(b)
        new = (0.5 * (re + _herm(re)) - 0.5j * gamma, 1j * mu * gamma, 1j * (mu - 1) * gamma)
        for k in range(3):
            lists[k][i] = new[k] if lists[k][i] is None else lists[k][i] + new[k]
    return lists


def _solve_inputs(case, seed):
    d = _Draw(seed)
    E = case["energies"]
    g, a = _system(d, _sizes(case), E, fold=not case["current"])
    sl, sg = _self_energies(d, g, E)
    obc = _contacts(d, g, E) if case["current"] else None
    return d, g, a, sl, sg, obc


def _lead(case, seed):
    """A lead's (a_10, a_00, a_01) per energy: the first cell of a random device."""
    d = _Draw(seed)
    E, b = case["energies"], case["block"]
    dd, uu, _ = _hamiltonian(d, (b, b))
    z = d.uniform(E, -1.0, 1.0) + 1j * ETA
    eye = torch.eye(b, dtype=C128, device=d.dev)
    a_00 = z[:, None, None] * eye - dd[0]
    a_01 = (-uu[0]).expand(E, b, b).clone()
    return a_00, a_01, _herm(a_01).contiguous(), d.uniform(E, 0.05, 0.95)


def _chains(case, seed):
    """A lead of a few one-dimensional chains per cell in a random orbital basis:
    two modes per chain, on the unit circle up to eta."""
    d = _Draw(seed)
    E, b, c = case["energies"], case["block"], case["chains"]
    n = b // c
    site = torch.diag(torch.ones(n - 1, dtype=C128, device=d.dev), 1)
    h = torch.zeros((b, b), dtype=C128, device=d.dev)
    t = torch.zeros((b, b), dtype=C128, device=d.dev)
    eps = d.uniform(c, -0.3, 0.3).tolist()
    for k in range(c):
        s = slice(k * n, (k + 1) * n)
        h[s, s] = site + site.T + eps[k] * torch.eye(n, dtype=C128, device=d.dev)
        t[(k + 1) * n - 1, k * n] = 1.0
    u = torch.linalg.qr(d.cn(b, b).cpu())[0].to(d.dev)
    h, t = u @ h @ _herm(u), u @ t @ _herm(u)
    z = d.uniform(E, -1.2, 1.2) + 1j * ETA
    eye = torch.eye(b, dtype=C128, device=d.dev)
    a_ii = z[:, None, None] * eye - h
    return a_ii, (-t).expand(E, b, b).clone(), (-_herm(t)).expand(E, b, b).clone()


def _pattern(case):
    """Stored entries of a block-sparse stack in block-sorted order: (rows, cols, part,
    offset inside the packed part); structurally symmetric, diagonal always stored.
    The pattern is the device's: other inputs have the same one."""
    g = Geometry.uniform(case["n_blocks"], case["block"])
    rng = np.random.default_rng(case["n_blocks"] * 1000 + case["block"])
    b, bo = case["block"], g.block_offsets
    rows, cols, part, off = [], [], [], []
    upper = [rng.random((b, b)) < case["fill"] for _ in range(g.n_blocks - 1)]
    for i in range(g.n_blocks):
        m = rng.random((b, b)) < case["fill"]
        for j, mask, p in ((i - 1, upper[i - 1].T if i else None, 2), (i, m | m.T | np.eye(b, dtype=bool), 0),
                           (i + 1, upper[i] if i + 1 < g.n_blocks else None, 1)):
            if mask is None:
                continue
            r, c = np.nonzero(mask)
            base = (g.diag_offsets[i], g.offdiag_offsets[min(i, g.n_blocks - 2)], g.offdiag_offsets[max(i - 1, 0)])[p]
            rows.append(bo[i] + r)
            cols.append(bo[j] + c)
            part.append(np.full(r.size, p))
            off.append(int(base) + r * b + c)
    return g, np.concatenate(rows), np.concatenate(cols), np.concatenate(part), np.concatenate(off)


def _sparse_inputs(case, seed):
    """Packed A, Sigma^<, Sigma^> restricted to the pattern, and each stack's stored entries."""
    d = _Draw(seed)
    E = case["energies"]
    g, rows, cols, part, off = _pattern(case)
    _, a = _system(d, g.block_sizes, E, fold=True)
    sl, sg = _self_energies(d, g, E)
    skew = [(x[0], x[1], _lower_of(g, x[1], -1.0)) for x in (sl, sg)]
    at = [torch.as_tensor(off[part == p], device=d.dev) for p in range(3)]
    where = [torch.as_tensor(np.nonzero(part == p)[0], device=d.dev) for p in range(3)]
    packed, data = [], []
    for m in (a, *skew):
        v = torch.empty((E, rows.size), dtype=C128, device=d.dev)
        kept = []
        for p in range(3):
            v[:, where[p]] = m[p][:, at[p]]
            k = torch.zeros_like(m[p])
            k[:, at[p]] = m[p][:, at[p]]
            kept.append(k)
        packed.append(tuple(kept))
        data.append(v)
    return g, rows, cols, (at, where), packed, data


def _lower_of(g, upper, sign):
    """The packed lower part sign * upper^H."""
    out = torch.empty_like(upper)
    for i in range(g.n_blocks - 1):
        g.lower(out, i)[...] = sign * g.upper(upper, i).mH
    return out


def _assembly_inputs(case, seed):
    d = _Draw(seed)
    E = case["energies"]
    g = Geometry(_sizes(case))
    h = tuple(_flat(x, d.dev) for x in _hamiltonian(d, g.block_sizes))
    overlap = None
    if case["overlap"]:
        dd, uu, ll = _hamiltonian(d, g.block_sizes)
        dd = [torch.eye(x.shape[0], dtype=C128, device=d.dev) + 0.1 * x for x in dd]
        overlap = (_flat(dd, d.dev), 0.1 * _flat(uu, d.dev), 0.1 * _flat(ll, d.dev))
    z = d.uniform(E, -1.0, 1.0) + 1j * ETA
    v = d.uniform(g.n, -0.2, 0.2)
    sl, sg = _self_energies(d, g, E)
    sig = [(x[0], x[1], _lower_of(g, x[1], -1.0)) for x in (sl, sg)]
    w = 0.1 * d.uniform(E, 0.5, 1.5)[:, None]
    sr = tuple(w * x for x in h)
    return g, z, h, overlap, v, sr, sig[0], sig[1]


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("solve", "graph"):
        d, g, a, sl, sg, obc = _solve_inputs(case, seed)
        E = case["energies"]
        gr = S.packed_empty(g, E, d.dev) if case["retarded"] else None
        gl, gg = (S.packed_empty(g, E, d.dev) for _ in range(2))
        cur = torch.empty((E, g.n_blocks + 1), dtype=C128, device=d.dev) if case["current"] else None
        args = (g, a, sl, sg)
        kw = dict(g_lesser=gl, g_greater=gg, g_retarded=gr, obc=obc, current=cur)
        graph = S.SolveGraph(*args, **kw) if kind == "graph" else None
        return dict(kind=kind, args=args, kw=kw, graph=graph, out=dict(r=gr, l=gl, g=gg, j=cur))
    if kind == "inverse":
        d = _Draw(seed)
        g, a = _system(d, _sizes(case), case["energies"], fold=True)
        return dict(kind=kind, g=g, a=a, x=S.packed_empty(g, case["energies"], d.dev))
    if kind == "contact":
        a_00, a_01, a_10, occ = _lead(case, seed)
        return dict(kind=kind, a=(a_10, a_00, a_01), occ=occ,
                    obc=OBCSystem(SanchoRubio(max_iterations=100, convergence_tol=1e-6), memoization_mode="off"))
    if kind == "spectral":
        beyn = Beyn(r_o=2.0, r_i=0.5, m_0=4 * case["chains"], num_quad_points=32)
        return dict(kind=kind, a=_chains(case, seed), obc=Spectral(beyn, max_decay=1.5 * math.log(2.0)))
    if kind == "sparse":
        g, rows, cols, _, _, data = _sparse_inputs(case, seed)
        stacks = [DSDBCOO(v, rows, cols, g.block_sizes, (case["energies"],)) for v in data]
        # one structure: the stacks of a program share their index maps
        a = stacks[0]
        sl, sg = (a._structure_view(s.data) for s in stacks[1:])
        out = tuple(DSDBCOO.zeros_like(a) for _ in range(3))
        return dict(kind=kind, rgf=RGF(), a=a, sl=sl, sg=sg, out=out)
    g, z, h, overlap, v, sr, sl, sg = _assembly_inputs(case, seed)
    return dict(kind=kind, args=(g, z, h), kw=dict(overlap=overlap, potential=v, sigma_retarded_herm=sr,
                                                   sigma_lesser=sl, sigma_greater=sg),
                a=S.packed_empty(g, case["energies"], z.device))


def run(state):
    kind = state["kind"]
    if kind == "solve":
        S.selected_solve(*state["args"], **state["kw"])
        return state["out"]
    if kind == "graph":
        state["graph"].launch()
        return state["out"]
    if kind == "inverse":
        S.selected_inv(state["g"], state["a"], x=state["x"])
        return state["x"]
    if kind == "contact":
        return compute_contact_obc(*state["a"], state["occ"], 0.0, state["obc"], contact="left")
    if kind == "spectral":
        return state["obc"](*state["a"], contact="left"), state["obc"].n_reflected
    if kind == "sparse":
        state["rgf"].selected_solve(state["a"], state["sl"], state["sg"], out=state["out"], return_retarded=True)
        return [x.data for x in state["out"]]
    S.assemble_system(*state["args"], a=state["a"], **state["kw"])
    return state["a"]


# --- what a pass cannot do without ------------------------------------------------


def work(case):
    kind, E = case["kind"], case["energies"]
    if kind in ("contact", "spectral"):
        b = case["block"]
        if kind == "contact":
            # 11 decimation steps of 6 products and an inverse, the last inverse, one
            # fixed-point step and the self-energies
            return dict(bytes=16.0 * 6 * b * b * E, flops=8.0 * b ** 3 * (7 * 11 + 1 + 3 + 2) * E)
        # an inverse and two thin products per quadrature node, then the pseudo-inverse
        # product, an inverse and two fixed-point steps
        m = 4 * case["chains"]
        return dict(bytes=16.0 * 4 * b * b * E, flops=8.0 * (64 * (b ** 3 + b * b * m) + 8 * b ** 3) * E)
    g = Geometry(_sizes(case))
    bs, d, u = g.block_sizes, g.diag_size, g.offdiag_size
    mid = [bs[i] * bs[i + 1] * (bs[i] + bs[i + 1]) / 2 for i in range(g.n_blocks - 1)]
    if kind == "assemble":
        one = d + 2 * u
        return dict(bytes=16.0 * (4 * E + (2 if case["overlap"] else 1)) * one, flops=12.0 * E * one)
    if kind == "inverse":
        return dict(bytes=16.0 * 2 * (d + 2 * u) * E, flops=8.0 * (sum(8 * x for x in mid) + bs[0] ** 3) * E)
    flops = 8.0 * (sum(34 * x for x in mid) + 5 * bs[0] ** 3) * E
    if kind == "sparse":
        nnz = case["fill"] * (d + 2 * u)
        return dict(bytes=16.0 * 6 * nnz * E, flops=flops)
    full = d + 2 * u
    nbytes = full + 2 * (d + u) + 2 * full + (full if case["retarded"] else 0)
    if case["current"]:
        nbytes += 3 * (bs[0] ** 2 + bs[-1] ** 2)
    return dict(bytes=16.0 * nbytes * E, flops=flops)


# --- the same results by plain torch in 64 bits -------------------------------------


def _inv(x):
    # on the host: torch's batched device inverse is wrong for some odd sizes
    # (residual 0.6 for 48 matrices of 65 x 65)
    return torch.linalg.inv(x.cpu()).to(x.device)


def _plain_retarded(g, a, obr=None):
    """Left-connected g_i, then the tridiagonal blocks of the inverse."""
    N = g.n_blocks
    A = lambda i: g.diag(a[0], i) - (obr[i] if obr is not None and obr[i] is not None else 0)  # noqa: E731
    left = [_inv(A(0))]
    for j in range(1, N):
        left.append(_inv(A(j) - g.lower(a[2], j - 1) @ left[-1] @ g.upper(a[1], j - 1)))
    x = tuple(torch.zeros_like(t) for t in a)
    full = left[-1]
    g.diag(x[0], N - 1)[...] = full
    for i in range(N - 2, -1, -1):
        u, l = left[i] @ g.upper(a[1], i), g.lower(a[2], i) @ left[i]
        g.upper(x[1], i)[...] = -u @ full
        g.lower(x[2], i)[...] = -full @ l
        full = left[i] + u @ full @ l
        g.diag(x[0], i)[...] = full
    return left, x


def _plain_solve(g, a, sl, sg, obc):
    """G^R and G^<> = G^R Sigma^<> G^R^H on the tridiagonal blocks, and the layer currents.

    Sigma^<> are skew-Hermitian; only their diagonal and upper blocks are given."""
    N, E = g.n_blocks, a[0].shape[0]
    left, gr = _plain_retarded(g, a, obc[0] if obc else None)
    outs, folded, carried = [], [], []
    for k, s in ((1, sl), (2, sg)):
        def sig(i):
            v = g.diag(s[0], i)
            return v + obc[k][i] if obc and obc[k][i] is not None else v
        w = [sig(0)]
        fold = [None]
        small = [left[0] @ w[0] @ left[0].mH]
        for j in range(1, N):
            aji, up = g.lower(a[2], j - 1), g.upper(s[1], j - 1)
            q = aji @ left[j - 1] @ up
            fold.append(aji @ small[-1] @ aji.mH + q.mH - q)
            small.append(left[j] @ (fold[j] + sig(j)) @ left[j].mH)
        x = tuple(torch.zeros_like(t) for t in a)
        full = small[-1]
        whole = [None] * N
        whole[-1] = full
        for i in range(N - 2, -1, -1):
            aij, aji, up = g.upper(a[1], i), g.lower(a[2], i), g.upper(s[1], i)
            gj = g.diag(gr[0], i + 1)
            u, r = left[i] @ aij, gj @ aji
            bb = left[i] @ up @ gj.mH
            off = -small[i] @ r.mH + bb - u @ full
            g.upper(x[1], i)[...] = off
            g.lower(x[2], i)[...] = -off.mH
            t = u @ r @ small[i] - bb @ u.mH
            full = small[i] + u @ full @ u.mH + t - t.mH
            whole[i] = full
        for i in range(N):
            g.diag(x[0], i)[...] = 0.5 * (whole[i] - whole[i].mH)
        outs.append(x)
        folded.append(fold)
        carried.append(whole)
    cur = None
    if obc:
        cur = torch.empty((E, N + 1), dtype=C128, device=a[0].device)
        tr = lambda p, q: (p * q.transpose(-1, -2)).sum((-1, -2))  # noqa: E731
        for j in range(1, N):
            cur[:, j] = tr(folded[1][j], carried[0][j]) - tr(carried[1][j], folded[0][j])
        for slot, i, sign in ((0, 0, 1.0), (N, N - 1, -1.0)):
            cur[:, slot] = sign * (tr(obc[2][i], carried[0][i]) - tr(carried[1][i], obc[1][i]))
    return gr, outs[0], outs[1], cur


def _plain_surface(a_00, a_01, a_10, tol):
    """Surface Green's function by decimation."""
    eps, surf, al, be = a_00, a_00, a_10, a_01
    for _ in range(100):
        g = _inv(eps)
        ag, bg = al @ g, be @ g
        surf = surf - ag @ be
        eps = eps - ag @ be - bg @ al
        al, be = ag @ al, bg @ be
        if float(torch.linalg.norm((al.abs() + be.abs()).reshape(al.shape[0], -1), dim=1).max()) / 2 < tol:
            break
    x = _inv(surf)
    return _inv(a_00 - a_10 @ x @ a_01)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("solve", "graph"):
        d, g, a, sl, sg, obc = _solve_inputs(case, seed)
        gr, gl, gg, cur = _plain_solve(g, a, sl, sg, obc)
        return dict(r=gr if case["retarded"] else None, l=gl, g=gg, j=cur)
    if kind == "inverse":
        d = _Draw(seed)
        g, a = _system(d, _sizes(case), case["energies"], fold=True)
        return _plain_retarded(g, a)[1]
    if kind == "contact":
        a_00, a_01, a_10, occ = _lead(case, seed)
        sigma = a_10 @ _plain_surface(a_00, a_01, a_10, 1e-6) @ a_01
        gamma, f = 1j * (sigma - sigma.mH), occ[:, None, None]
        return sigma, 1j * f * gamma, 1j * (f - 1) * gamma
    if kind == "spectral":
        return _plain_surface(*_chains(case, seed), 1e-13), None
    if kind == "sparse":
        g, rows, cols, (at, where), packed, data = _sparse_inputs(case, seed)
        gr, gl, gg, _ = _plain_solve(g, packed[0], packed[1][:2], packed[2][:2], None)
        outs = []
        for x in (gl, gg, gr):
            v = torch.empty_like(data[0])
            for p in range(3):
                v[:, where[p]] = x[p][:, at[p]]
            outs.append(v)
        return outs
    g, z, h, overlap, v, sr, sl, sg = _assembly_inputs(case, seed)
    bo, out = g.block_offsets, []
    for p, view in enumerate((g.diag, g.upper, g.lower)):
        x = -(sr[p] + (sg[p] - sl[p]) / 2 + h[p])
        for i in range(g.n_blocks - (p > 0)):
            r, c = (i, i) if p == 0 else (i, i + 1) if p == 1 else (i + 1, i)
            vr, vc = v[int(bo[r]):int(bo[r + 1]), None], v[None, int(bo[c]):int(bo[c + 1])]
            if overlap is not None:
                s = view(overlap[p], i)
                view(x, i)[...] += z[:, None, None] * s - s * (vr + vc) / 2
            elif p == 0:
                view(x, i).diagonal(dim1=-2, dim2=-1)[...] += z[:, None] - vr[:, 0]
        out.append(x)
    return tuple(out)
