"""Performance cases: the work a user of this library has it do.

Molecular dynamics (``md``): chunks of 100 steps of the active Kob-Andersen
system, each chunk ending with the frame x_u and the statistics line, as a run
loop has them; from a single small box over ensembles of replicas in launch
groups to one box of 10^6 particles, with FP64 and with FP32 pair forces.
Trajectory analysis (``ana``): MSD, overlap, S4 and Fs of a trajectory whose
frames are on the device (a parsed text file, a stored run), from the creation
of the handle to its slot results.  S4 on |q| shells (``shells``) and g_uu(r)
(``guu``) of a frame store.  Frame text written from a run (``text_write``) and
read back (``text_read``).

Inputs come from the seed alone, through numpy and torch.  ``exact`` restates
each computation in 64-bit torch.
"""
import ctypes
import math

import numpy as np
import torch

import activechi4_amd as ac4

RHO = 1.2
DT = 0.005
STEPS = 100   # MD steps of one pass: frames are sampled every 100 steps
FACTOR = 1.4  # lag ladder of the analyses
OVERLAP_A = 0.3


def listed():
    return [
        # The smallest run: N=1000 in FP64, stepped eagerly as the `run`
        # executable does; bound by launches and latency.
        dict(name="md_n1000_fp64", kind="md", n=1000, replicas=1, fp32=False, graph=False, groups=1, tpp=0, skin=0.35,
             T=0.6, f0=1.5, tau=200),
        # One mid-size production box with FP32 pair forces, graph-replayed.
        dict(name="md_n10000_fp32", kind="md", n=10000, replicas=1, fp32=True, graph=True, groups=1, tpp=0, skin=0.35,
             T=0.5, f0=1.0, tau=200),
        # The reference's compile-time system (N=50000) in FP64, eager.
        dict(name="md_n50000_fp64", kind="md", n=50000, replicas=1, fp32=False, graph=False, groups=1, tpp=0,
             skin=0.35, T=0.5, f0=1.0, tau=200),
        # The batched ensemble: 64 replicas of uneven N (log-uniform up to
        # 5000) in three launch groups at the autotuner's kernel shape, with
        # the in-situ overlap sampled every chunk.
        dict(name="md_ensemble64_fp32", kind="md", n=5000, replicas=64, fp32=True, graph=True, groups=3, tpp=2,
             skin=0.45, T=0.5, f0=1.0, tau=200),
        # The large single box.
        dict(name="md_box1m_fp32", kind="md", n=1000000, replicas=1, fp32=True, graph=True, groups=1, tpp=0,
             skin=0.35, T=0.5, f0=1.0, tau=200),
        # All four observables of a short trajectory of the CPU-runnable size:
        # bound by the per-frame path.
        dict(name="ana_n1000_all", kind="ana", n=1000, origins=60, gap=50, obs=15, flag=0),
        # The reference Analysis' own observables and N on a trajectory of its
        # frame schedule.
        dict(name="ana_n50000_s4", kind="ana", n=50000, origins=60, gap=50, obs=7, flag=0),
        # The self-intermediate scattering function of the A particles.
        dict(name="ana_n20011_fs", kind="ana", n=20011, origins=20, gap=100, obs=8, flag=1),
        # S4 on |q| shells at one lag over the origins of a large box.
        dict(name="shells_n300000", kind="shells", n=300000, pairs=8, nshell=108, ndir=64),
        # g_uu(r) of the active tenth of N=50000 over 20 origins.
        dict(name="guu_n50000", kind="guu", n=50000, origins=20, gap=100),
        # One frame of N=50000 as text, as the run loop writes it.
        dict(name="text_write_n50000", kind="text_write", n=50000),
        # A chunk of trajectory text read back: 20 frames of N=50000.
        dict(name="text_read_n50000", kind="text_read", n=50000, frames=20),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box_n(n):
    """n rounded down to whole tiles (the start of a large box is a periodic
    arrangement of one relaxed tile)."""
    t3 = _tiles(n) ** 3
    return n // t3 * t3


def draw(rng):
    kind = rng.choice(["md", "md", "md", "ens", "ana", "ana", "shells", "guu", "text_write", "text_read"])
    T, f0, tau = round(rng.uniform(0.45, 0.8), 3), round(rng.uniform(0.0, 2.0), 3), _logint(rng, 20, 2000)
    if kind == "md":
        fp32 = rng.random() < 0.5
        n = _box_n(_logint(rng, 700, 500000 if fp32 else 60000))
        return dict(kind="md", n=n, replicas=1, fp32=fp32, graph=rng.random() < 0.5, groups=1, tpp=0,
                    skin=rng.choice([0.3, 0.35, 0.45]), T=T, f0=f0, tau=tau)
    if kind == "ens":
        reps = rng.randint(6, 48)
        return dict(kind="md", n=_logint(rng, 1500, 5000), replicas=reps, fp32=rng.random() < 0.7, graph=True,
                    groups=rng.randint(1, 3), tpp=rng.choice([0, 1, 2, 4]), skin=rng.choice([0.3, 0.35, 0.45]), T=T,
                    f0=f0, tau=tau)
    if kind == "ana":
        obs = rng.choice([3, 7, 7, 15, 8])
        n = _logint(rng, 700, 10000 if obs & 8 else 50000)
        return dict(kind="ana", n=n, origins=rng.randint(8, 40 if not obs & 8 else 20), gap=rng.choice([40, 50, 100]),
                    obs=obs, flag=rng.randint(0, 1))
    if kind == "shells":
        nshell = rng.randint(9, 108)
        return dict(kind="shells", n=_logint(rng, 5000, 250000), pairs=rng.randint(2, 8), nshell=nshell,
                    ndir=rng.randint(5, 256 // ((nshell + 26) // 27)) if nshell > 27 else rng.randint(5, 128))
    if kind == "guu":
        return dict(kind="guu", n=_logint(rng, 3000, 45000), origins=rng.randint(4, 20), gap=rng.choice([50, 100]))
    n = _logint(rng, 1000, 400000 if kind == "text_write" else 50000)
    if kind == "text_write":
        return dict(kind=kind, n=n)
    return dict(kind=kind, n=n, frames=max(1, min(20, _logint(rng, 50000, 900000) // n)))


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, int(seed))


def run(state):
    return state["run"](state)


def exact(case, seed):
    f = _EXACT.get(case["kind"])
    with torch.no_grad():
        return f(case, int(seed)) if f else None


def work(case):
    k, n = case["kind"], case["n"]
    if k == "md":
        n = sum(_sizes(case))
        # per particle-step: positions, unwrapped positions and momenta read
        # and written once; 39 pairs within the cutoff (each once), about 45
        # operations a pair, and the integrator
        return {"bytes": 144.0 * n * STEPS + 24.0 * n, "flops": (39 * 45 + 100.0) * n * STEPS}
    if k == "ana":
        fr, pairs = _walk_of(case)
        np_, no = len(pairs), len({p[0] for p in pairs})
        obs = case["obs"]
        flops = n * np_ * (15.0 * bool(obs & 1) + 15.0 * bool(obs & 2))
        if obs & 4:  # 573 phases per particle and origin, masked sums of their cos and sin over the lags
            flops += n * (573.0 * 8 * no + 573.0 * 2 * np_)
        if obs & 8:  # 573 phases per particle and pair
            flops += n * 573.0 * 8 * np_
        return {"bytes": 28.0 * n * len(fr) + 8.0 * 324 * np_ * (bool(obs & 4) + bool(obs & 8)), "flops": flops}
    if k == "shells":
        # half the particles overlap; per particle, direction and shell one
        # phase advance and two sums
        return {"bytes": 48.0 * n * case["pairs"], "flops": 0.5 * n * case["pairs"] * case["nshell"] * case["ndir"] * 8.0}
    if k == "guu":
        na = n // 10
        return {"bytes": 48.0 * na * case["origins"], "flops": 25.0 * na * (na - 1) / 2 * case["origins"]}
    if k == "text_write":
        return {"bytes": 55.0 * n, "flops": 0.0}
    return {"bytes": 55.0 * n * case["frames"], "flops": 0.0}


# ------------------------------------------------------- the model in torch
SIG = (1.0, 0.8, 0.88)
EPS = (1.0, 1.5, 0.5)
C0, C2 = 0.0162665594880, -0.001949973872640


class _Box:
    """Replicas of the Kob-Andersen mixture, concatenated, as torch tensors:
    pair lists by distance search and forces over padded lists."""

    def __init__(self, sizes, types, dtype, dev, skin):
        self.sizes, self.dtype, self.dev, self.skin = sizes, dtype, dev, skin
        self.L_of = [(n / RHO) ** 0.33333333 for n in sizes]
        self.L = torch.cat([torch.full((n, 1), l, dtype=dtype, device=dev) for n, l in zip(sizes, self.L_of)])
        self.ty = types
        self.sig = torch.tensor(SIG, dtype=dtype, device=dev)
        self.eps = torch.tensor(EPS, dtype=dtype, device=dev)
        self.nb = None

    def build(self, x):
        """Neighbours of every particle within 2.5 + skin, padded with the
        particle itself."""
        rows, cols, off, skin = [], [], 0, self.skin
        rc2 = (2.5 + skin) ** 2
        for n, L in zip(self.sizes, self.L_of):
            xr = x[off:off + n]
            nc = int(L / (2.5 + skin))
            if n <= 12000 or nc < 4:
                step = max(1, 30000000 // n)
                for a in range(0, n, step):
                    d = xr[a:a + step, None, :] - xr[None, :, :]
                    d -= torch.round(d)
                    m = (d * d).sum(-1) * (L * L) < rc2
                    r, c = m.nonzero(as_tuple=True)
                    keep = r + a != c
                    rows.append(r[keep] + (off + a))
                    cols.append(c[keep] + off)
            else:
                cell3 = (xr - torch.floor(xr)).mul(nc).long().clamp_(0, nc - 1)
                cell = (cell3[:, 2] * nc + cell3[:, 1]) * nc + cell3[:, 0]
                order = torch.argsort(cell, stable=True)
                cnt = torch.bincount(cell, minlength=nc ** 3)
                cap = int(cnt.max())
                start = torch.cumsum(cnt, 0) - cnt
                slot = start[:, None] + torch.arange(cap, device=self.dev)[None, :]
                mem = torch.where(torch.arange(cap, device=self.dev)[None, :] < cnt[:, None],
                                  order[slot.clamp(max=n - 1)], torch.full_like(slot, -1))
                sh = torch.tensor([(i, j, k) for k in (-1, 0, 1) for j in (-1, 0, 1) for i in (-1, 0, 1)],
                                  device=self.dev)
                step = max(1, 40000000 // (27 * cap))
                for a in range(0, n, step):
                    c3 = (cell3[a:a + step, None, :] + sh[None]) % nc
                    cand = mem[(c3[..., 2] * nc + c3[..., 1]) * nc + c3[..., 0]].reshape(c3.shape[0], -1)
                    d = xr[a:a + step, None, :] - xr[cand.clamp(min=0)]
                    d -= torch.round(d)
                    own = torch.arange(a, a + c3.shape[0], device=self.dev)[:, None]
                    m = ((d * d).sum(-1) * (L * L) < rc2) & (cand >= 0) & (cand != own)
                    r, c = m.nonzero(as_tuple=True)
                    rows.append(r + (off + a))
                    cols.append(cand[r, c] + off)
            off += n
        r, c = torch.cat(rows), torch.cat(cols)
        del rows, cols
        cnt = torch.bincount(r, minlength=off)
        place = torch.arange(len(r), device=self.dev) - (torch.cumsum(cnt, 0) - cnt)[r]
        self.nb = torch.arange(off, device=self.dev)[:, None].repeat(1, int(cnt.max()))
        self.nb[r, place] = c
        self.ref = x.clone()

    def forces(self, x, energy=False):
        """Pair forces (real units); with energy also the sums of the pair
        energy and virial of every replica."""
        stale = self.nb is None
        if not stale:
            d = x - self.ref
            stale = 2.0 * float(((d - torch.round(d)) * self.L).norm(dim=1).max()) >= self.skin
        if stale:
            self.build(x)
        n, k = self.nb.shape
        F = torch.empty_like(x)
        pe = torch.empty(n, dtype=self.dtype, device=self.dev)
        vir = torch.empty_like(pe)
        step = max(1, 30000000 // k)
        for a in range(0, n, step):
            nb = self.nb[a:a + step]
            d = x[a:a + step, None, :] - x[nb]
            d -= torch.round(d)
            d *= self.L[a:a + step, None, :]
            r2 = (d * d).sum(-1)
            ab = self.ty[a:a + step, None] + self.ty[nb]
            s2i = 1.0 / (self.sig * self.sig)[ab]
            q = r2 * s2i
            inside = (q < 6.25) & (r2 > 0)
            r2 = torch.where(inside, r2, torch.ones_like(r2))
            q = torch.where(inside, q, torch.ones_like(q))
            s6 = 1.0 / (q * q * q)
            eps = torch.where(inside, self.eps[ab], torch.zeros_like(q))
            grad = 8.0 * eps * (6.0 * s6 * (s6 - 0.5) / r2 - C2 * s2i)
            F[a:a + step] = (grad[..., None] * d).sum(1)
            if energy:
                pe[a:a + step] = (4.0 * eps * (s6 * (s6 - 1.0) + C0 + C2 * q)).sum(1)
                vir[a:a + step] = (grad * r2).sum(1)
        if not energy:
            return F
        return F, [0.5 * float(v.sum()) for v in pe.split(self.sizes)], [
            0.5 * float(v.sum()) / 3.0 for v in vir.split(self.sizes)]


def _tiles(n):
    """Tiles per axis of the relaxed start of a box of n particles."""
    return max(1, math.ceil((n / 12000.0) ** (1.0 / 3.0)))


def _liquid(sizes, T, seed):
    """A start near equilibrium for each replica: simple-cubic sites, 80:20
    species, an overlap-removing descent and a short rescaled run in FP32 (large
    boxes: one tile of up to 12000 particles, repeated, each copy displaced a
    little).  Returns per replica a dict of host arrays of the state."""
    rng = np.random.default_rng(seed)
    dev = torch.device("cuda")
    tiles = [_tiles(n) for n in sizes]
    base = [n // t ** 3 for n, t in zip(sizes, tiles)]
    x0, ty = [], []
    for n in base:
        m = math.ceil(n ** (1.0 / 3.0) - 1e-9)
        site = rng.permutation(m ** 3)[:n]
        p = np.stack([site % m, site // m % m, site // (m * m)], 1) + 0.5 + rng.normal(0.0, 0.03, (n, 3))
        x0.append(p / m)
        t = np.zeros(n, dtype=np.int64)
        t[rng.permutation(n)[:n // 5]] = 1
        ty.append(t)
    x = torch.tensor(np.concatenate(x0), dtype=torch.float32, device=dev)
    v = torch.tensor(rng.normal(0.0, math.sqrt(T), (len(x), 3)), dtype=torch.float32, device=dev)
    box = _Box(base, torch.tensor(np.concatenate(ty), device=dev), torch.float32, dev, 0.7)
    for _ in range(40):
        F = box.forces(x)
        x = x + (F * 0.002).clamp(-0.04, 0.04) / box.L
    F = box.forces(x)
    for k in range(120):
        v = v + F * (0.5 * DT)
        x = x + v * DT / box.L
        F = box.forces(x)
        v = v + F * (0.5 * DT)
        v = v * torch.sqrt(T / (v * v).mean())
    x = (x - torch.floor(x)).double().cpu().numpy()
    out, off = [], 0
    for n, m, t in zip(sizes, base, tiles):
        p, L = x[off:off + m], (n / RHO) ** 0.33333333
        s = dict(type=ty[len(out)])
        off += m
        if t > 1:
            shift = np.stack(np.meshgrid(*[np.arange(t)] * 3, indexing="ij"), -1).reshape(-1, 1, 3)
            p = ((p[None] + shift) / t).reshape(-1, 3) + rng.normal(0.0, 0.02 / L, (n, 3))
            s["type"] = np.tile(s["type"], t ** 3)
        p = p - np.floor(p)
        p[p >= 1.0] = 0.0
        mom = rng.normal(0.0, math.sqrt(T), (n, 3))
        mom -= mom.mean(0)
        mom *= math.sqrt(3.0 * (n - 1) * T / (mom * mom).sum())
        na = int(n * 0.1)
        act = np.full(n, -1, dtype=np.int32)
        act[rng.permutation(n)[:na]] = np.arange(na)
        s.update(x=p, p=mom, act=act, k=rng.integers(0, 2, (3, na)) * 2 - 1, key=int(rng.integers(1, 1 << 62)))
        dof = 3.0 * n - 3.0
        Q = np.array([dof * T * 0.04, T * 0.04, T * 0.04])
        s["chain"] = np.concatenate([np.zeros(3), rng.normal(0.0, 1.0, 3) * np.sqrt(T * Q), Q])
        out.append(s)
    return out


def _sizes(case):
    r, n = case["replicas"], case["n"]
    if r == 1:
        return [n]
    # log-uniform over [n/5, n], the same sizes for every seed
    g = np.random.default_rng(20261202)
    return [int(v) for v in np.round(np.exp(g.uniform(math.log(n / 5.0), math.log(n), r)))]


def _groups(case):
    """Launch group of every replica: the largest first, each to the group
    that holds the fewest particles."""
    sizes, load = _sizes(case), [0] * case["groups"]
    of = [0] * len(sizes)
    for r in sorted(range(len(sizes)), key=lambda r: (-sizes[r], r)):
        of[r] = load.index(min(load))
        load[of[r]] += sizes[r]
    return of


# ----------------------------------------------------------------------- MD
def _md_load(md, r, s):
    c = [np.ascontiguousarray(s["x"][:, a]) for a in range(3)]
    p = [np.ascontiguousarray(s["p"][:, a]) for a in range(3)]
    md.set_state(r, *c, *c, *p, s["type"], s["act"], *s["k"])
    md.set_chain(r, s["chain"])


def _md_prepare(case, seed):
    states = _liquid(_sizes(case), case["T"], seed)
    ps = [ac4.ReplicaParams(n, RHO, case["T"], case["f0"], -1, case["tau"], s["key"])
          for n, s in zip(_sizes(case), states)]
    ac4.load()
    plan = _groups(case)
    ac4.set_tuning(case["tpp"], 3)
    ac4.set_skin(case["skin"])
    try:
        mds = []
        for g in range(case["groups"]):
            mine = [r for r in range(len(ps)) if plan[r] == g]
            md = ac4.MD([ps[r] for r in mine], precision=ac4.FP32 if case["fp32"] else ac4.FP64)
            for k, r in enumerate(mine):
                _md_load(md, k, states[r])
            if case["replicas"] > 1:
                md.overlap_enable(STEPS, 10 * STEPS, 10, 100, OVERLAP_A)
            mds.append(md)
    finally:
        ac4.set_tuning()
        ac4.set_skin()
    return dict(run=_md_run, mds=mds, graph=case["graph"], ensemble=case["replicas"] > 1)


def _md_run(s):
    mds = s["mds"]
    if s["ensemble"]:
        ac4.step_multi(mds, STEPS)
        for md in mds:
            md.overlap_sample()
        out = []
        for md in mds:
            out += [np.concatenate(md.export_xu(), 1), np.stack(md.chi4(range(md.R))[:2])]
        return out
    md = mds[0]
    md.step(STEPS, graph=s["graph"])
    return [md.export_xu()[0], np.array(list(md.stats(0).values()))]


def _philox(i, comp, s, key):
    """The words of Philox-4x32-10 at counters (i, comp, s, 0)."""
    m32 = np.uint64(0xFFFFFFFF)
    i = np.asarray(i).astype(np.uint64)
    c = [i, np.full_like(i, comp), np.full_like(i, s), np.zeros_like(i)]
    k0, k1 = key & 0xFFFFFFFF, key >> 32
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & m32, (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1),
             p0 & m32]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return [w.astype(np.float64) for w in c]


def _shuffle(k, s, key):
    """The swap shuffle of each direction component: for i, swap with (int)(n u_i)."""
    for a in range(3):
        n = k.shape[1]
        j = (n * (_philox(np.arange(n), a, s, key)[0] / 4294967296.0)).astype(np.int64).tolist()
        v = k[a].tolist()
        for i in range(n):
            v[i], v[j[i]] = v[j[i]], v[i]
        k[a] = v


def _nhc_u4(t, order, S, T, dof, q, pe):
    for j in order:
        g = S - dof * T if j == 0 else pe[j - 1] ** 2 / q[j - 1] - T
        if j == 2:
            pe[j] += t * g
        else:
            x = t * pe[j + 1] / q[j + 1]
            pe[j] = pe[j] * math.exp(-x) + t * g * (1.0 - math.exp(-x)) / x


def _nhc_half(S, T, dof, c):
    eta, pe, q = c
    _nhc_u4(DT * 0.25, (2, 1, 0), S, T, dof, q, pe)
    s = math.exp(-0.5 * DT * pe[0] / q[0])
    for i in range(3):
        eta[i] += 0.5 * DT * pe[i] / q[i]
    _nhc_u4(DT * 0.25, (0, 1, 2), S * s * s, T, dof, q, pe)
    return s, S * s * s


def _md_exact(case, seed):
    """The Nose-Hoover steps in 64 bits over all replicas together."""
    sizes, T, f0, tau = _sizes(case), case["T"], case["f0"], case["tau"]
    if sum(sizes) > 400000:
        return None
    states = _liquid(sizes, T, seed)
    dev = torch.device("cuda")
    cat = lambda k, d: torch.tensor(np.concatenate([s[k] for s in states]), dtype=d, device=dev)  # noqa: E731
    box = _Box(sizes, cat("type", torch.int64), torch.float64, dev, 0.5)
    xu, p = cat("x", torch.float64), cat("p", torch.float64)
    x = xu.clone()
    act = [torch.tensor(s["act"], device=dev) for s in states]
    ks = [s["k"].astype(np.int64).copy() for s in states]
    chains = [[list(s["chain"][3 * i:3 * i + 3]) for i in range(3)] for s in states]
    dof = [3.0 * n - 3.0 for n in sizes]

    def active():
        out = []
        for a, k in zip(act, ks):
            kt = torch.tensor(k.T.copy(), dtype=torch.float64, device=dev)
            out.append(torch.where(a[:, None] >= 0, f0 * kt[a.clamp(min=0).long()], torch.zeros(3, dtype=torch.float64, device=dev)))
        return torch.cat(out)

    def per_rep(v):
        return torch.cat([torch.full((n, 1), f, dtype=torch.float64, device=dev) for n, f in zip(sizes, v)])

    def p2():
        return [float((v * v).sum()) for v in p.split(sizes)]

    F = box.forces(x) + active()
    S = p2()
    shuffles = 0
    for step in range(STEPS):
        if tau > 0 and step % tau == 0:
            for k, s in zip(ks, states):
                _shuffle(k, shuffles, s["key"])
            shuffles += 1
            fa = active()
        h = [_nhc_half(S[r], T, dof[r], chains[r]) for r in range(len(sizes))]
        p = p * per_rep([v[0] for v in h]) + F * (0.5 * DT)
        dx = p * DT / box.L
        x = x + dx
        xu = xu + dx
        x = x - torch.floor(x)
        if step < STEPS - 1:
            F = box.forces(x) + fa
        else:
            F, pe, vir = box.forces(x, energy=True)
            F = F + fa
        p = p + F * (0.5 * DT)
        h = [_nhc_half(s, T, dof[r], chains[r]) for r, s in enumerate(p2())]
        p = p * per_rep([v[0] for v in h])
        S = [v[1] for v in h]
    frames = [v.T.contiguous() for v in xu.split(sizes)]
    if case["replicas"] > 1:
        plan, out = _groups(case), []
        for g in range(case["groups"]):
            out += [torch.cat([frames[r] for r in range(len(sizes)) if plan[r] == g], 1), None]
        return out
    eta, pet, q = chains[0]
    ke = 0.5 * S[0]
    heff = ke + pe[0] + eta[0] * T * dof[0] + sum(pet[i] ** 2 / (2.0 * q[i]) for i in range(3)) + T * (eta[1] + eta[2])
    it = 2.0 * ke / dof[0]
    stats = [pe[0], vir[0], ke, it, RHO * it + vir[0] / box.L_of[0] ** 3, float(p[:, 0].sum()), heff, float(STEPS)]
    return [frames[0], np.array(stats)]


# ----------------------------------------------------------------- analysis
def _schedule(origins, gap):
    """Frame steps of the reference's two-level schedule: origins k*gap and
    the lag ladder of each."""
    top = origins * gap / 2.0
    s = set()
    for k in range(origins):
        s.add(k * gap)
        off = 1
        while off < top:
            s.add(k * gap + off)
            off = off + 1 if int(off * FACTOR) == off else int(off * FACTOR)
    return sorted(s)


def _walk(fr, gap, rule):
    """(origin, lag frame, slot) of every pair in the reference's walk order."""
    pos = {f: i for i, f in enumerate(fr)}
    on = 0
    while on * gap + rule in pos:
        on += 1
    top, pairs, k = int(on * gap / 2.0), [], 0
    while k * gap in pos:
        off, slot = 1, 1
        while off < top and k * gap + off in pos:
            pairs.append((pos[k * gap], pos[k * gap + off], slot))
            off = off + 1 if int(off * FACTOR) == off else int(off * FACTOR)
            slot += 1
        k += 1
    return pairs, top


def _walk_of(case):
    fr = _schedule(case["origins"], case["gap"])
    return fr, _walk(fr, case["gap"], 1)[0]


def _trajectory(n, fr, seed):
    """x_u of a glassy trajectory on the device, [3][frames][n]: caged
    particles rattling about their sites and a mobile minority diffusing."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    kw = dict(generator=g, device="cuda", dtype=torch.float64)
    L = (n / RHO) ** (1.0 / 3.0)
    x = torch.empty(3, len(fr), n, dtype=torch.float64, device="cuda")
    mob = torch.where(torch.rand(n, **kw) < 0.3, 0.02, 0.002) / L
    site = torch.rand(3, n, **kw)
    last = 0
    for f, t in enumerate(fr):
        if t > last:
            site = site + torch.randn(3, n, **kw) * (mob * math.sqrt(t - last))
        last = t
        x[:, f] = site + torch.randn(3, n, **kw) * (0.06 / L)
    ty = (torch.rand(n, **kw) < 0.2).to(torch.int32)
    return x, ty, L


def _ana_prepare(case, seed):
    ac4.load()
    fr = _schedule(case["origins"], case["gap"])
    x, ty, L = _trajectory(case["n"], fr, seed)
    torch.cuda.synchronize()
    f = [[x[a, k].data_ptr() for a in range(3)] for k in range(len(fr))]
    return dict(run=_ana_run, case=case, fr=fr, x=x, ty=ty, L=L, ptr=f, tp=ty.data_ptr())


def _ana_run(s):
    c = s["case"]
    an = ac4.Analysis(c["n"], s["L"], s["fr"], gap=c["gap"], factor=FACTOR, a=OVERLAP_A, obs=c["obs"],
                      type_flag=c["flag"])
    push, tp = ac4.lib.ac4_ana_push_frame_device, s["tp"]
    for pos, (px, py, pz) in enumerate(s["ptr"]):
        if push(an.h, pos, px, py, pz, tp) != 0:
            raise ac4.AC4Error(ac4.lib.ac4_last_error().decode())
    an.finalize()
    out = {}
    if c["obs"] & 1:
        r = an.msd()
        out["msd"] = [r["m0"], r["m1"], r["m2"], r["counters"]]
    if c["obs"] & 2:
        r = an.overlap()
        out["overlap"] = [r["c"], r["x4"], r["counters"], an.pairs(ac4.OBS_OVERLAP)]
    for o, name in ((4, "s4"), (8, "fs")):
        if c["obs"] & o:
            r = an.phase(o)
            out[name] = [r["cs"], r["ss"], r["cs2"], r["ss2"], r["counters"]]
    an.close()
    return out


def _qvectors():
    """The 162 lattice vectors of the analyses in their order, with the
    permutations each is averaged over."""
    v = [(1, 0, 0)] + [(0, k, i) for k in (1, 2) for i in range(k, 22)]
    v += [(i, j, j) for i in range(1, 16) for j in range(1, i + 1)]
    q = [1] + [a * a + b * b + c * c for a, b, c in v[1:]]
    n, inc = len(v) - 1, 1
    while True:
        inc = 3 * inc + 1
        if inc > n:
            break
    while True:
        inc //= 3
        for i in range(inc + 1, n + 1):
            qq, vv, j = q[i], v[i], i
            while q[j - inc] > qq:
                q[j], v[j] = q[j - inc], v[j - inc]
                j -= inc
                if j <= inc:
                    break
            q[j], v[j] = qq, vv
        if inc <= 1:
            break
    perms = []
    for a, b, c in v:
        if a == b == c:
            perms.append([(a, b, c)])
        elif len({a, b, c}) == 3:
            perms.append([(a, b, c), (a, c, b), (b, a, c), (b, c, a), (c, a, b), (c, b, a)])
        else:
            perms.append([(a, b, c), (b, c, a), (c, a, b)])
    return perms


def _minimg(d):
    return d - (d >= 0.5).double() + (d < -0.5).double()


def _wrap1(v):
    v = torch.where(v >= 1.0, v - 1.0, v)
    return torch.where(v < 0.0, v + 1.0, v)


def _phase_sums(pts, w, pv):
    """Sums over particles of w * (cos, sin) of 2 pi o.r for every column o:
    pts [n][3], w [rows][n] -> two [rows][columns]."""
    c = torch.zeros(len(w), len(pv), dtype=torch.float64, device=pts.device)
    s = torch.zeros_like(c)
    step = max(1, 40000000 // len(pv))
    for a in range(0, len(pts), step):
        p = pts[a:a + step]
        f = p[:, :1] * pv[:, 0] + p[:, 1:2] * pv[:, 1] + p[:, 2:] * pv[:, 2]
        f = (f - torch.round(f)) * (2.0 * math.pi)
        c += w[:, a:a + step] @ torch.cos(f)
        s += w[:, a:a + step] @ torch.sin(f)
    return c, s


def _ana_exact(case, seed):
    n, obs, flag = case["n"], case["obs"], case["flag"]
    fr = _schedule(case["origins"], case["gap"])
    x, ty, L = _trajectory(n, fr, seed)
    keep = (ty != 1) if flag else torch.ones(n, dtype=torch.bool, device="cuda")
    kd = keep.double()
    tot = 0.8 * n if flag else float(n)
    out = {}
    if obs & 1:
        pairs, top = _walk(fr, case["gap"], 0)
        ns = max(10 + int(math.log(top) / math.log(FACTOR)) + 10, max(p[2] for p in pairs) + 1)
        m = np.zeros((3, ns))
        for o, k, t in pairs:
            d2 = (x[:, k] - x[:, o]) ** 2
            r2 = L * L * d2.sum(0)
            m[:, t] += np.array([float((r2 * kd).sum()), float(((d2 * d2).sum(0) * (L ** 4) * kd).sum()),
                                 float((r2 * r2 * kd).sum())]) / tot
        out["msd"] = [m[0], m[1], m[2], None]
    pairs, top = _walk(fr, case["gap"], 1)
    ns = max(10 + int(math.log(top) / math.log(FACTOR)), len(fr), max(p[2] for p in pairs) + 1)
    if obs & 2:
        c, x4 = np.zeros(ns), np.zeros(ns)
        for o, k, t in pairs:
            d = _minimg(x[:, k] - x[:, o])
            q = float(((L * L * (d * d).sum(0) < OVERLAP_A ** 2) & keep).sum()) / tot
            c[t] += q
            x4[t] += q * q
        out["overlap"] = [c, x4, None, None]
    if not obs & 12:
        return out
    if (obs & 8) and n * len(pairs) > 2e7 or (obs & 4) and n * case["origins"] > 4e6:
        for o, name in ((4, "s4"), (8, "fs")):
            if obs & o:
                out[name] = [None] * 5
        return out
    perms = _qvectors()
    pv = torch.tensor([p for ps in perms for p in ps], dtype=torch.float64, device="cuda")
    avg = torch.zeros(len(pv), len(perms), dtype=torch.float64, device="cuda")
    col = 0
    for q, ps in enumerate(perms):
        avg[col:col + len(ps), q] = 1.0 / len(ps)
        col += len(ps)
    by = {}
    for o, k, t in pairs:
        by.setdefault(o, []).append((k, t))
    for bit, name in ((4, "s4"), (8, "fs")):
        if not obs & bit:
            continue
        acc = torch.zeros(4, ns, len(perms), dtype=torch.float64, device="cuda")
        for o, lags in by.items():
            if bit == 4:
                x0 = _wrap1(x[:, o])
                w = torch.stack([(L * L * (_minimg(_wrap1(x[:, k]) - x0) ** 2).sum(0) < OVERLAP_A ** 2).double()
                                 for k, _ in lags])
                rows = [_phase_sums(x[:, o].T, w, pv)]
            else:
                rows = [_phase_sums(_minimg(_wrap1(x[:, k]) - _wrap1(x[:, o])).T, kd[None], pv) for k, _ in lags]
            c, s = (torch.cat([r[a] for r in rows]) @ avg for a in range(2))
            for i, (_, t) in enumerate(lags):
                acc[:, t] += torch.stack([c[i], s[i], c[i] ** 2, s[i] ** 2])
        out[name] = [*acc, None]
    return out


# ------------------------------------------------------------- frame stores
def _store(n, L, frames, steps):
    fs = ac4.Frames(n, L, len(steps))
    torch.cuda.synchronize()
    for k, t in enumerate(steps):
        h = frames[:, k].cpu().numpy()
        fs.push(h[0], h[1], h[2], t)
    return fs


def _shell_inputs(case, seed):
    steps = [10 * k for k in range(case["pairs"] + 1)]
    x, _, L = _trajectory(case["n"], steps, seed)
    # |q| from 0.05 to about 9 per sigma, the range of the structure factor
    return x, L, steps, list(range(case["pairs"])), [k + 1 for k in range(case["pairs"])], 0.05, 9.0 / case["nshell"]


def _shells_prepare(case, seed):
    ac4.load()
    x, L, steps, orig, lag, q0, dq = _shell_inputs(case, seed)
    fs = _store(case["n"], L, x, steps)
    return dict(run=_shells_run, fs=fs, args=(orig, lag, q0, dq, case["nshell"], case["ndir"], seed))


def _shells_run(s):
    r, d, ph = s["fs"].s4_shells(*s["args"], a=OVERLAP_A, phases=True)
    return [r, d, ph]


def _shells_exact(case, seed):
    n, nsh, nd = case["n"], case["nshell"], case["ndir"]
    if 0.5 * n * case["pairs"] * nsh * nd > 1.2e10:
        return None
    x, L, _, orig, lag, q0, dq = _shell_inputs(case, seed)
    dirs = torch.tensor(_directions(nd, seed), device="cuda")
    q = (q0 + dq * torch.arange(nsh, dtype=torch.float64, device="cuda")) * L
    ph = torch.zeros(len(orig), nd, nsh, 2, dtype=torch.float64, device="cuda")
    for p, (o, k) in enumerate(zip(orig, lag)):
        d = _minimg(x[:, k] - x[:, o])
        pts = x[:, o, L * L * (d * d).sum(0) < OVERLAP_A ** 2]
        pr = dirs @ (pts - torch.floor(pts))
        step = max(1, 60000000 // (nd * nsh))
        for a in range(0, pr.shape[1], step):
            f = pr[:, None, a:a + step] * q[None, :, None]
            ph[p, ..., 0] += torch.cos(f).sum(-1)
            ph[p, ..., 1] += torch.sin(f).sum(-1)
    var = lambda v: (v * v).mean(0) - v.mean(0) ** 2  # noqa: E731
    ref = nd * var(ph.mean(1)).sum(-1) / n
    return [ref, var(ph).sum(-1).mean(0) / n, ph]


def _directions(nd, seed):
    """Unit directions of a seed: Philox words at counters (d, 0x5334, 0, 0)."""
    u = _philox(np.arange(nd), 0x5334, 0, seed)
    z = 1.0 - 2.0 * (u[0] + 0.5) / 4294967296.0
    ph = 6.283185307179586 * (u[1] + 0.5) / 4294967296.0
    r = np.sqrt(np.maximum(0.0, 1.0 - z * z))
    return np.stack([r * np.cos(ph), r * np.sin(ph), z], 1)


def _guu_inputs(case, seed):
    n, gap = case["n"], case["gap"]
    tau_steps = 20
    steps = sorted({k * gap + o for k in range(case["origins"]) for o in (0, 1, 2, 3, 4, 5, 7, 9, 12, 16, 22, 30)})
    x, _, L = _trajectory(n, steps, seed)
    act = np.zeros(n, dtype=np.int32)
    act[np.random.default_rng(seed).permutation(n)[:n // 10]] = 1
    return x, L, steps, act, tau_steps * DT


def _guu_prepare(case, seed):
    ac4.load()
    x, L, steps, act, tau = _guu_inputs(case, seed)
    return dict(run=_guu_run, fs=_store(case["n"], L, x, steps), act=act, gap=case["gap"], tau=tau)


def _guu_run(s):
    h, fn, no = s["fs"].guu(s["act"], s["gap"], s["tau"], factor=FACTOR)
    return [h[0].astype(np.int64), h[1], h[2], fn, no]


def _guu_exact(case, seed):
    x, L, steps, act, tau = _guu_inputs(case, seed)
    pos = {t: i for i, t in enumerate(steps)}
    lag = 22  # the ladder's entry nearest tau: 16 and 22 steps around 20
    a = torch.tensor(np.flatnonzero(act), device="cuda")
    nbin = int(0.5 * L / 0.005)
    h1 = torch.zeros(nbin + 1, dtype=torch.float64, device="cuda")
    h2 = torch.zeros_like(h1)
    for k in range(case["origins"]):
        o, t = pos[k * case["gap"]], pos[k * case["gap"] + lag]
        x0 = x[:, o, a]
        u = L * _minimg(x[:, t, a] - x0)
        r = u.pow(2).sum(0).sqrt()
        x0 = torch.where((x0 >= 1.0) | (x0 < 0.0), x0 - torch.floor(x0), x0)
        for b in range(0, len(a), 2000):
            i, j = torch.meshgrid(torch.arange(b, min(b + 2000, len(a)), device="cuda"),
                                  torch.arange(len(a), device="cuda"), indexing="ij")
            m = j > i
            i, j = i[m], j[m]
            d = _minimg(x0[:, j] - x0[:, i])
            idx = ((L * L * (d * d).sum(0)).sqrt() / 0.005).long().clamp(max=nbin)
            h1 += torch.bincount(idx, weights=2.0 * r[i] * r[j], minlength=nbin + 1)
            h2 += torch.bincount(idx, weights=2.0 * (u[:, i] * u[:, j]).sum(0), minlength=nbin + 1)
    return [None, h1[:nbin], h2[:nbin], None, None]


# --------------------------------------------------------------- frame text
def _text_write_prepare(case, seed):
    ac4.load()
    rng = np.random.default_rng(seed)
    n = case["n"]
    md = ac4.MD([ac4.ReplicaParams(n, RHO, 0.5, 1.0, -1, 200, 7)], precision=ac4.FP32)
    xu = rng.random((3, n)) + np.round(rng.normal(0.0, 0.6, (3, n)))
    x = xu - np.floor(xu)
    x[x >= 1.0] = 0.0
    p = rng.normal(0.0, 0.7, (3, n))
    md.set_state(0, *x, *xu, *p, (rng.random(n) < 0.2).astype(np.int32))
    return dict(run=_text_write_run, md=md, buf=np.zeros(80 * n + 1, dtype=np.uint8))


def _text_write_run(s):
    b = s["buf"]
    k = ac4.lib.ac4_md_format_frame(s["md"].h, 0, b.ctypes.data_as(ctypes.c_char_p), len(b))
    if k < 0:
        raise ac4.AC4Error(ac4.lib.ac4_last_error().decode())
    return [b, int(k)]  # the text and its length; the buffer is zero beyond it


def _text_values(case, seed):
    """x, y, z as whole numbers of 1e-5 and the types, [3][frames][n]."""
    rng = np.random.default_rng(seed)
    k = np.rint(1e5 * (rng.random((3, case["frames"], case["n"])) + np.round(rng.normal(0.0, 0.6, (3, case["frames"], case["n"])))))
    return k.astype(np.int64), (rng.random((case["frames"], case["n"])) < 0.2).astype(np.int32)


class _Device:
    """A device array of the library for torch."""

    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=shape, typestr=typestr, version=3)


def _text_read_prepare(case, seed):
    ac4.load()
    n, nf = case["n"], case["frames"]
    k, t = _text_values(case, seed)
    text = b"".join(ac4.format_frame(*(k[:, f] / 1e5), t[f]) for f in range(nf))
    tf = ac4.TextFrames(n, max(len(text) + 4096, 128 * n))
    ctypes.memmove(tf.buf, text, len(text))
    get = ac4.lib.ac4_textframes_get
    get.argtypes = [ctypes.c_void_p, ctypes.c_int] + [ctypes.POINTER(ctypes.c_void_p)] * 4
    return dict(run=_text_read_run, tf=tf, n=n, nf=nf, len=len(text), get=get)


def _text_read_run(s):
    tf, n = s["tf"], s["n"]
    nf, used = ctypes.c_int(), ctypes.c_longlong()
    if ac4.lib.ac4_textframes_parse(tf.h, s["len"], 1 << 30, ctypes.byref(nf), ctypes.byref(used)) != 0:
        raise ac4.AC4Error(ac4.lib.ac4_last_error().decode())
    ptr = [ctypes.c_void_p() for _ in range(4)]
    if s["get"](tf.h, 0, *[ctypes.byref(p) for p in ptr]) != 0:
        raise ac4.AC4Error(ac4.lib.ac4_last_error().decode())
    # the frames are consecutive: one view of all of them
    out = [torch.as_tensor(_Device(p.value, (nf.value, n), ty), device="cuda")
           for p, ty in zip(ptr, ("<f8", "<f8", "<f8", "<i4"))]
    return out + [int(used.value)]


def _text_read_exact(case, seed):
    k, _ = _text_values(case, seed)
    return [k[0] / 1e5, k[1] / 1e5, k[2] / 1e5, None, None]


_PREPARE = {"md": _md_prepare, "ana": _ana_prepare, "shells": _shells_prepare, "guu": _guu_prepare,
            "text_write": _text_write_prepare, "text_read": _text_read_prepare}
_EXACT = {"md": _md_exact, "ana": _ana_exact, "shells": _shells_exact, "guu": _guu_exact,
          "text_read": _text_read_exact}
