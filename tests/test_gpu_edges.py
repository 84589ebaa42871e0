"""Kernels at the sizes where their tilings can go wrong: edges of tiles,
remainders, the smallest and largest of their ranges, against the oracle or a
64-bit restatement."""
import ctypes
import threading

import numpy as np
import pytest

import oracle_lib as OL
import trajgen

pytestmark = pytest.mark.gpu


# Active counts around the 256-row tile; L = 130 takes 13000 bins, three
# passes of the LDS histogram.
@pytest.mark.parametrize("na,L", [(0, 9.0), (1, 9.0), (255, 9.0), (256, 9.0), (257, 130.0), (513, 9.0), (700, 130.0)])
def test_guu_tile_edges(gpu, na, L):
    n, frames = 700, trajgen.case_frames(5, 40)
    X, Y, Z, _ = trajgen.make_frames(n, frames, 31 + na, 0.3, 1.0)
    act = np.zeros(n, dtype=np.int32)
    act[np.random.default_rng(na).permutation(n)[:na]] = 1
    fr = gpu.Frames(n, L, len(frames))
    for k, t in enumerate(frames):
        fr.push(X[k], Y[k], Z[k], t)
    h, fn, no = fr.guu(act, 40, 0.06)
    fr.close()
    ho, fno, noo = OL.guu(n, L, X, Y, Z, act, frames, 40, 0.06)
    assert (fn, no) == (fno, noo)
    assert np.array_equal(h[0], ho[0])
    # a bin sums at most a few thousand FP64 terms: n_terms * 2^-53 of their absolute sum
    scale = max(1.0, np.abs(ho[1]).max())
    assert np.abs(h[1:] - ho[1:]).max() <= 1e-12 * scale


# Runs of 27 shells about a middle one: part of a run, one, the odd counts
# below and from five, even ones; the widest and the smallest teams; one
# particle, tile remainders, several pairs per launch and more than one batch.
@pytest.mark.parametrize("n,npairs,nshell,ndir", [(1, 1, 1, 1), (511, 3, 9, 5), (513, 40, 28, 7), (700, 2, 81, 85),
                                                  (700, 2, 135, 51), (300, 2, 108, 64), (600, 2, 27, 256),
                                                  (200, 1, 6912, 1), (5000, 20, 54, 3)])
def test_shell_runs_against_direct_sums(gpu, n, npairs, nshell, ndir):
    rng = np.random.default_rng(n + nshell)
    L, a, q0, dq = 9.0, 0.3, 0.11, 0.07
    X = rng.random((3, npairs + 1, n)) + rng.normal(0, 0.08 / L, (3, npairs + 1, n)) * np.arange(npairs + 1)[:, None]
    fr = gpu.Frames(n, L, npairs + 1)
    for k in range(npairs + 1):
        X[:, k] = X[:, 0] + rng.normal(0, 0.1 / L, (3, n)) if k else X[:, 0]
        fr.push(*X[:, k], 10 * k)
    orig, lag = [0] * npairs, list(range(1, npairs + 1))
    _, s4d, ph = fr.s4_shells(orig, lag, q0, dq, nshell, ndir, 99, a=a, phases=True)
    fr.close()
    dirs = gpu.shell_directions(ndir, 99)
    q = (q0 + dq * np.arange(nshell)) * L
    pos = X[:, 0] - np.floor(X[:, 0])
    proj = dirs @ pos
    for p in range(npairs):
        d = X[:, lag[p]] - X[:, 0]
        w = L * L * ((d[0] * d[0] + d[1] * d[1]) + d[2] * d[2]) < a * a
        for k0 in range(0, nshell, 64):
            f = proj[:, None, w] * q[None, k0:k0 + 64, None]
            # a term is off by the rounding of its phase and of 13 products
            tol = (4e-16 * np.abs(f).max() + 4e-14) * max(1, w.sum()) if w.any() else 0.0
            assert np.abs(ph[p, :, k0:k0 + 64, 0] - np.cos(f).sum(-1)).max() <= tol
            assert np.abs(ph[p, :, k0:k0 + 64, 1] - np.sin(f).sum(-1)).max() <= tol
    var = lambda v: (v * v).mean(0) - v.mean(0) ** 2  # noqa: E731
    want = var(ph).sum(-1).mean(0) / n
    assert np.allclose(s4d, want, rtol=1e-9, atol=1e-9 * (ph ** 2).max() / n)


# The fold over the teams, eight and nine of them and more, and part of one run
# of shells: only the lower half of it, the middle one, one above.
@pytest.mark.parametrize("nshell,ndir", [(1, 1), (1, 56), (13, 64), (13, 57), (14, 32), (15, 56), (27, 2), (40, 56)])
def test_shell_teams_and_part_runs(gpu, nshell, ndir):
    test_shell_runs_against_direct_sums(gpu, 700, 2, nshell, ndir)


# Sizes of the automatic force team of 16 and of 4 lanes (those of 8 lanes
# below), with the list layouts of 16, 8, 4 and one nominal lanes, against one
# pinned lane: the same pair terms, summed in FP64 in another order.
@pytest.mark.parametrize("prec,n", [(0, 700), (0, 6000), (0, 9001), (0, 14001), (0, 33001), (1, 700), (1, 6000),
                                    (1, 9001), (1, 14001), (1, 33001), (1, 160001)])
def test_force_team_widths(gpu, prec, n):
    s = gpu.init_lattice(n, 0.5, n)
    rng = np.random.default_rng(n)
    x = [(s[k] + rng.normal(0, 0.02 / n ** (1 / 3), n)) % 1.0 for k in ("x", "y", "z")]
    out = []
    for tpp in (0, 1):
        gpu.set_tuning(tpp)
        try:
            md = gpu.MD([gpu.ReplicaParams(n, 1.2, 0.5, 1.0, -1, 200, 3)], precision=prec)
        finally:
            gpu.set_tuning()
        md.set_state(0, *x, *x, s["px"], s["py"], s["pz"], s["type"], s["act_tag"], s["kx"], s["ky"], s["kz"])
        pv = md.calculate_forces()[0]
        out.append((np.stack(md.forces(0)), pv))
        md.close()
    (fa, pa), (fb, pb) = out
    # about 100 terms of up to a few hundred times the rms force cancel: 100 * 300 * 2^-53
    assert np.abs(fa - fb).max() <= 4e-12 * np.sqrt((fb ** 2).mean())
    # energy and virial: FP32 partial sums of eight pairs in FP32 mode
    assert np.allclose(pa, pb, rtol=1e-11 if prec == 0 else 1e-6)


# The team of 8 lanes, on the list layout of two: the range's edges and a size
# between them.
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n", [16385, 20000, 32768])
def test_force_team_of_eight_lanes(gpu, prec, n):
    test_force_team_widths(gpu, prec, n)


# What the last workgroups of the force pass and of the binning do for a whole
# replica: part of a group of 64 blocks of 16 or 64 particles, a whole one and one
# more, more than 4 groups, cells below and above the limit of the scan in the
# binning pass; several replicas of different sizes in one handle.
@pytest.mark.parametrize("sizes", [(256,), (1024,), (1025,), (16385,), (131073,), (700, 256, 2048, 500)])
def test_sums_and_cells_of_the_last_workgroup(gpu, sizes):
    md = gpu.MD([gpu.ReplicaParams(n, 1.2, 0.5, 1.0, -1, 10, 3 + r) for r, n in enumerate(sizes)])
    for r, n in enumerate(sizes):
        s = gpu.init_lattice(n, 0.5, n)
        xs = [s[k] for k in ("x", "y", "z", "xu", "yu", "zu", "px", "py", "pz")]
        md.set_state(r, *xs, s["type"], s["act_tag"], s["kx"], s["ky"], s["kz"])
    md.relax(20)
    for r in range(len(sizes)):
        md.init_chain(r)
    for k in (1, 40):
        md.step(k)
        seen = [(md.stats(r), md.get_state(r), np.stack(md.forces(r))) for r in range(len(sizes))]
        pv = md.calculate_forces()  # new cells and lists of the same positions
        for r, n in enumerate(sizes):
            st, g, f = seen[r]
            p2 = sum((g[k] ** 2).sum() for k in ("px", "py", "pz"))
            assert np.isclose(st["ke"], 0.5 * p2, rtol=1e-12, atol=0)  # sums of n terms of one sign
            assert abs(st["drift"] - g["px"].sum()) <= 1e-13 * np.abs(g["px"]).sum()
            assert np.allclose((st["pe"], st["virial"]), pv[r], rtol=1e-10, atol=1e-12)
            # about 100 terms of up to a few hundred times the rms force cancel: 100 * 300 * 2^-53
            f2 = np.stack(md.forces(r))
            assert np.abs(f - f2).max() <= 4e-12 * max(1.0, np.sqrt((f2 ** 2).mean()))
    assert all(md.rebuilds(r) > 2 for r in range(len(sizes)))
    md.close()


# Particle counts around the tiles of the frame kernel (256) and of the Fs
# kernel (16, loads of 256), and one large enough for several of each per
# workgroup; with and without the B particles.
@pytest.mark.parametrize("n,flag", [(1, 0), (15, 0), (17, 1), (31, 0), (32, 1), (33, 0), (255, 1), (257, 0), (513, 0),
                                    (70001, 1)])
def test_frame_and_fs_tile_edges(gpu, n, flag):
    frames = [0, 1, 2, 3, 10, 11]
    X, Y, Z, T = trajgen.make_frames(n, frames, 7 + n, 0.08, 1.0)
    L = max(4.0, (n / 1.2) ** (1.0 / 3.0))
    an = gpu.Analysis(n, L, frames, gap=10, obs=11 if n > 1000 else 15, type_flag=flag)
    for f in range(len(frames)):
        an.push(f, X[f], Y[f], Z[f], T[f])
    om = OL.msd(n, L, X, Y, Z, T, frames, 10, flag=flag)
    assert np.allclose(an.pairs(gpu.OBS_MSD), om["pairs"], rtol=1e-12, atol=0)
    oo = OL.overlap(n, L, X, Y, Z, T, frames, 10, flag=flag)
    assert len(oo["pairs"]) == 4 and np.array_equal(an.pairs(gpu.OBS_OVERLAP), oo["pairs"])
    an.finalize()
    ofs = OL.phase("fs", n, L, X, Y, Z, T, frames, 10, flag=flag)
    assert np.abs(an.pairs(gpu.OBS_FS) - ofs["pairs"]).max() < 1e-12 * n  # a term is off by at most a few 1e-14
    if n <= 1000:
        os4 = OL.phase("s4", n, L, X, Y, Z, T, frames, 10)
        v, m = an.pairs(gpu.OBS_S4)
        assert np.array_equal(m, os4["mask"]) and np.abs(v - os4["pairs"]).max() < 1e-12 * n


def test_frames_that_never_arrive(gpu):
    """A lag frame whose origin was left out is refused, an origin's lag frame
    may be left out: the pairs that arrived are those of the full walk."""
    n, frames = 300, trajgen.case_frames(3, 30)
    X, Y, Z, T = trajgen.make_frames(n, frames, 5, 0.08, 1.0)
    L = (n / 1.2) ** (1.0 / 3.0)
    an = gpu.Analysis(n, L, frames, gap=30)
    with pytest.raises(gpu.AC4Error, match="origin frame 0 of pair 0 was not pushed"):
        an.push(1, X[1], Y[1], Z[1], T[1])
    oo = OL.overlap(n, L, X, Y, Z, T, frames, 30)
    om = OL.msd(n, L, X, Y, Z, T, frames, 30)
    an = gpu.Analysis(n, L, frames, gap=30)
    left_out = [k for k in range(len(frames)) if frames[k] % 30 and k % 4 == 1]
    for f in range(len(frames)):
        if f not in left_out:
            an.push(f, X[f], Y[f], Z[f], T[f])
    an.finalize()
    got, want = an.pairs(gpu.OBS_OVERLAP), oo["pairs"]
    lag = np.array([frames.index(o + l) for o, l in _walk(frames, 30)])
    here = ~np.isin(lag, left_out)
    assert 0 < here.sum() < len(want)
    assert np.array_equal(got[here], want[here]) and not got[~here].any()
    assert np.allclose(an.pairs(gpu.OBS_MSD)[:len(here)][here[:len(om["pairs"])]], om["pairs"][here[:len(om["pairs"])]],
                       rtol=1e-12, atol=0)


def _walk(frames, gap):
    """(origin step, lag) of every pair of the overlap walk, in its order."""
    pos, on = set(frames), 0
    while on * gap + 1 in pos:
        on += 1
    out, k = [], 0
    while k * gap in pos:
        off = 1
        while off < int(on * gap / 2.0) and k * gap + off in pos:
            out.append((k * gap, off))
            off = off + 1 if int(off * 1.4) == off else int(off * 1.4)
        k += 1
    return out


# Frames pushed from one set of device arrays that are overwritten as soon as
# the push returns, against host pushes: one workgroup, one and more groups of
# 64, Fs with and without the other observables, more pairs than one reduction
# of Fs takes and a frame left out between them.
@pytest.mark.parametrize("n,obs", [(1, 15), (700, 7), (700, 8), (2049, 15), (70001, 15), (70001, 3)])
def test_device_arrays_reused_after_the_push(gpu, n, obs):
    frames = list(range(60))
    X, Y, Z, T = trajgen.make_frames(n, frames, 5 + n, 0.08, 1.0)
    L = max(4.0, (n / 1.2) ** (1.0 / 3.0))
    hip = ctypes.CDLL("libamdhip64.so")  # the runtime the library has loaded
    dev = ctypes.c_void_p()
    assert hip.hipMalloc(ctypes.byref(dev), ctypes.c_size_t(28 * n)) == 0
    at = [dev.value + 8 * n * k for k in range(4)]  # x, y, z, types
    out = []
    for device in (False, True):
        an = gpu.Analysis(n, L, frames, gap=10, obs=obs)
        for f in range(len(frames)):
            if f == 21:
                continue
            if not device:
                an.push(f, X[f], Y[f], Z[f], T[f])
                continue
            src = [np.ascontiguousarray(v) for v in (X[f], Y[f], Z[f], np.asarray(T[f], dtype=np.int32))]
            for d, v in zip(at, src):
                assert hip.hipMemcpy(ctypes.c_void_p(d), v.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(v.nbytes), 1) == 0
            assert gpu.lib.ac4_ana_push_frame_device(an.h, f, *at) == 0
            assert hip.hipMemset(dev, 255, ctypes.c_size_t(28 * n)) == 0
        an.finalize()
        got = [an.pairs(o) for o in (gpu.OBS_MSD, gpu.OBS_OVERLAP, gpu.OBS_S4, gpu.OBS_FS) if obs & o]
        out.append([v for g in got for v in (g if isinstance(g, tuple) else (g,))])
        an.close()
    hip.hipFree(dev)
    assert not obs & 8 or len(out[0][-1]) > 32
    for a, b in zip(*out):
        assert np.array_equal(a, b)


# S4 by origin with every split of the lags into row tiles of 16 and 4 (and
# two passes), sizes at the line between its two kernels, chunks that end in
# the middle of a mask word, and tiles of less than 32 particles.
@pytest.mark.parametrize("n,nf,nl", [(3073, 5, 2), (3100, 11, 5), (3100, 26, 12), (3073, 30, 14), (3079, 36, 17),
                                     (3072, 46, 22), (3100, 46, 22), (3100, 54, 26), (3100, 64, 31), (3100, 90, 44),
                                     (40001, 11, 5)])
def test_s4_lag_tiles(gpu, n, nf, nl):
    frames = list(range(nf))
    X, Y, Z, T = trajgen.make_frames(n, frames, 11 + n + nf, 0.03, 1.0)
    L = (n / 1.2) ** (1.0 / 3.0)
    an = gpu.Analysis(n, L, frames, gap=nf + 1, factor=1.01, obs=4)
    for f in range(nf):
        an.push(f, X[f], Y[f], Z[f], T[f])
    an.finalize()
    v, m = an.pairs(gpu.OBS_S4)
    an.close()
    o = OL.phase("s4", n, L, X, Y, Z, T, frames, nf + 1, factor=1.01)
    assert len(m) == nl and np.array_equal(m, o["mask"]) and m.max() > 0
    assert np.abs(v - o["pairs"]).max() < 1e-12 * n  # a term is off by at most a few 1e-14


# Columns of the written form (one to three digits and a point and five digits
# between tabs) next to others of nearly that form, in any column; workgroups
# of 256 lines whose text fits the staged 96 bytes a line and whose does not;
# segment and 16-byte edges by the varying lengths.  Bit for bit the host
# reader's values.
@pytest.mark.parametrize("n,blanks", [(1, 0), (255, 0), (257, 0), (3000, 0), (600, 90)])
def test_text_columns_of_every_width(gpu, n, blanks):
    rng = np.random.default_rng(n)
    forms = ["%.5f", "%.5f", "%.5f", "%.5f", "%.4f", "%.6f", "%.0f", "%.5f ", " %.5f", "%+.5f", "%010.5f", "%.9f"]
    lines = []
    for i in range(2 * n):
        v = rng.normal(0.0, 1.0, 3) * 10.0 ** rng.integers(-6, 5, 3)
        f = [forms[k] for k in (rng.integers(0, 4, 3) if i % 3 else rng.integers(0, len(forms), 3))]
        sep = "\t" if i % 5 else "\t " if i % 2 else " "
        t = str(rng.integers(0, 3)) if i % 4 else str(rng.integers(-12, 120))
        lines.append(sep.join([f[k] % v[k] for k in range(3)] + [t]) + " " * (blanks if i % 7 else 0))
    text = ("\n".join(lines) + "\n").encode()
    tf = gpu.TextFrames(n, len(text) + 64)
    k, used = tf.parse(text)
    assert k == 2 and used == len(text)
    pos = 0
    for f in range(2):
        x, y, z, t, u = gpu.parse_frame(text[pos:], n)
        pos += u
        for a, b in zip(tf.frame(f), (x, y, z, t)):
            assert np.array_equal(a, b) and np.array_equal(np.signbit(a), np.signbit(b))
    tf.close()


# Frame text in one, exactly one, two and three pieces of 128 blocks of 256
# lines, a small replica through the buffers of a large one, columns of one to
# twelve digits before the point, and a value the host has to format.
@pytest.mark.parametrize("sizes", [(256, 257), (32768,), (32769, 300), (65793, 256)])
def test_frame_text_pieces(gpu, sizes):
    md = gpu.MD([gpu.ReplicaParams(n, 1.2, 0.5, 1.0, -1, 200, 7) for n in sizes])
    rng = np.random.default_rng(sum(sizes))
    for r, n in enumerate(sizes):
        for big in (0.0, 1e12):
            xu = rng.normal(0.0, 1.0, (3, n)) * 10.0 ** rng.integers(-7, 11, (3, n))
            xu[:, ::3] = np.round(xu[:, ::3], 6) + 5e-6  # halves of the last digit
            xu[0, -1] = big
            x = rng.random((3, n))
            ty = rng.integers(-9, 120, n).astype(np.int32) if big else (rng.random(n) < 0.2).astype(np.int32)
            md.set_state(r, *x, *xu, *x, (ty & 1))
            assert md.format_frame(r) == gpu.format_frame(*xu, ty & 1)
    md.close()


# The list teams' trimmed stencils against the thread-per-particle builder,
# which takes every candidate: two, three and more cells per axis, cells at
# least and less than 0.01 wider than the largest list radius (ordered by x-half
# or not), small and large skins, a dilute box.
@pytest.mark.parametrize("n,rho,skin", [(400, 1.2, 0.35), (753, 1.2, 0.35), (1000, 1.2, 0.35), (1790, 1.2, 0.35),
                                        (4100, 1.2, 0.35), (1500, 0.5, 0.35), (2600, 1.2, 0.2), (2600, 1.2, 0.6)])
def test_trimmed_list_teams(gpu, n, rho, skin):
    out = []
    for mode in (1, 2, 3, 4):
        gpu.set_tuning(0, mode)
        gpu.set_skin(skin)
        try:
            md = gpu.MD([gpu.ReplicaParams(n, rho, 1.0, 1.0, -1, 20, 3)], precision=gpu.FP32)
        finally:
            gpu.set_tuning()
            gpu.set_skin()
        s = gpu.init_lattice(n, 1.0, n)
        md.set_state(0, *[s[k] for k in ("x", "y", "z", "xu", "yu", "zu", "px", "py", "pz")], s["type"], s["act_tag"],
                     s["kx"], s["ky"], s["kz"])
        md.relax(60)
        md.init_chain(0)
        md.step(80)
        assert md.rebuilds(0) > 3
        out.append(md.export_xu()[0])
        md.close()
    for o in out[1:]:
        assert np.array_equal(o, out[0])


# A small handle's steps past the few hundred after which they are replayed
# from a graph, in calls of whole chunks of 25 and remainders, against steps
# launched one by one; the tables change in between (another job in the slot).
@pytest.mark.parametrize("prec,n", [(0, 700), (1, 3000)])
def test_steps_replayed_after_a_while(gpu, prec, n):
    def start(md, seed):
        s = gpu.init_lattice(n, 0.5, seed)
        md.set_state(0, *[s[k] for k in ("x", "y", "z", "xu", "yu", "zu", "px", "py", "pz")], s["type"], s["act_tag"],
                     s["kx"], s["ky"], s["kz"])
        md.relax(40)
        md.init_chain(0)
    out = []
    for calls in ([260, 60, 25, 110, 1, 26], [1] * 24 * 20 + [2]):
        md = gpu.MD([gpu.ReplicaParams(n, 1.2, 0.5, 1.0, -1, 30, 3)], precision=prec)
        start(md, 5)
        for k in calls:
            md.step(k)
        got = [md.get_state(0), md.stats(0), md.get_chain(0)]
        md.set_rebuild_criterion(1)
        for k in calls:
            md.step(k)
        out.append(got + [md.get_state(0), md.stats(0), md.get_chain(0), md.rebuilds(0)])
        md.close()
    assert sum([260, 60, 25, 110, 1, 26]) == 24 * 20 + 2
    for a, b in zip(*out):
        if isinstance(a, dict):
            for k in a:
                assert np.array_equal(a[k], b[k]), k
        else:
            assert np.array_equal(a, b)


# The shuffle inside the half-kick kernel, as its own launch, on the parallel
# path, and both of the last two for a handle whose replicas need them; cells
# scanned by the binning pass and by a kernel of their own.  Each replica alone
# gives what it gives beside the others, direction for direction.
@pytest.mark.parametrize("acts", [(300, 9000), (300, 17000), (16384, 16385), (300, 9000, 17000)])
def test_shuffle_launches_by_the_jobs(gpu, acts):
    def start(r_list):
        gpu.set_tuning(4)
        try:
            md = gpu.MD([gpu.ReplicaParams(120000 if a == 17000 else 20000, 1.2, 0.5, 1.0, a, 5, 3 + a) for a in r_list])
        finally:
            gpu.set_tuning()
        for r, a in enumerate(r_list):
            n = md.n(r)
            s = gpu.init_lattice(n, 0.5, n)
            rng = np.random.default_rng(a)
            tag = np.full(n, -1, np.int32)
            tag[rng.permutation(n)[:a]] = np.arange(a)
            ks = [rng.integers(0, 2, a).astype(np.int32) * 2 - 1 for _ in range(3)]
            md.set_state(r, *[s[k] for k in ("x", "y", "z", "xu", "yu", "zu", "px", "py", "pz")], s["type"], tag, *ks)
        md.step(12)
        out = [md.get_state(r) for r in range(len(r_list))]
        md.close()
        return out
    both = start(acts)
    for r, a in enumerate(acts):
        alone = start([a])[0]
        for k in ("kx", "ky", "kz", "xu", "px"):
            assert np.array_equal(alone[k], both[r][k]), (a, k)


# Another thread's calls on the null stream (copies, the creation of handles)
# while a handle's steps are recorded: they succeed, and the steps are those
# of a handle alone.
def test_steps_recorded_beside_the_null_stream(gpu):
    hip = ctypes.CDLL("libamdhip64.so")
    n, codes, stop = 600, [], threading.Event()
    s = gpu.init_lattice(n, 0.5, 5)

    def steps():
        md = gpu.MD([gpu.ReplicaParams(n, 1.2, 0.5, 1.0, -1, 30, 3)])
        md.set_state(0, *[s[k] for k in ("x", "y", "z", "xu", "yu", "zu", "px", "py", "pz")], s["type"], s["act_tag"],
                     s["kx"], s["ky"], s["kz"])
        md.step(300)
        md.step(50)
        out = md.get_state(0)
        md.close()
        return out

    def copies():
        d, h = ctypes.c_void_p(), np.zeros(16)
        codes.append(hip.hipMalloc(ctypes.byref(d), ctypes.c_size_t(128)))
        while not stop.is_set():
            codes.append(hip.hipMemcpy(h.ctypes.data_as(ctypes.c_void_p), d, ctypes.c_size_t(128), 2))
        hip.hipFree(d)

    alone = steps()
    t = threading.Thread(target=copies)
    t.start()
    try:
        for _ in range(5):
            got = steps()
            assert all(np.array_equal(got[k], alone[k]) for k in ("x", "px", "kx"))
    finally:
        stop.set()
        t.join()
    assert len(codes) > 100 and not any(codes)


# A checkpoint goes on bit for bit in every handle of its layout: capacities at
# both ends of the layout of four lanes, alone and beside another replica.
@pytest.mark.parametrize("prec", [0, 1])
def test_checkpoint_between_capacities_of_a_layout(gpu, prec):
    def relaxed(sizes):
        md = gpu.MD([gpu.ReplicaParams(n, 1.2, 0.5, 1.0, -1, 30, 3) for n in sizes], precision=prec)
        for r, n in enumerate(sizes):
            s = gpu.init_lattice(n, 0.5, 5)
            md.set_state(r, *[s[k] for k in ("x", "y", "z", "xu", "yu", "zu", "px", "py", "pz")], s["type"],
                         s["act_tag"], s["kx"], s["ky"], s["kz"])
        md.relax(40)  # every replica has its forces before the restore
        for r in range(len(sizes)):
            md.init_chain(r)
        return md
    a, b = relaxed([8300]), relaxed([8300, 16384 - 8300])
    a.step(20)
    b.restore(0, a.checkpoint(0))
    for md in (a, b):
        md.step(60)
    x, y = a.get_state(0), b.get_state(0)
    assert all(np.array_equal(x[k], y[k]) for k in x)
    assert np.array_equal(a.get_chain(0), b.get_chain(0))
    a.close()
    b.close()


# A list layout whose chunks of 16 entries times the particles pass 2^24: the
# team builders store the lists the thread-per-particle builder stores.
@pytest.mark.parametrize("n", [1048576, 1048600])
def test_list_addresses_of_large_boxes(gpu, n):
    s = gpu.init_lattice(n, 0.5, 11)
    out = []
    for mode in (1, 2, 3, 4):
        gpu.set_tuning(16, mode)
        try:
            md = gpu.MD([gpu.ReplicaParams(n, 1.2, 1.0, 1.0, -1, 20, 3)], precision=gpu.FP32)
        finally:
            gpu.set_tuning()
        md.set_state(0, *[s[k] for k in ("x", "y", "z", "xu", "yu", "zu", "px", "py", "pz")], s["type"], s["act_tag"],
                     s["kx"], s["ky"], s["kz"])
        md.relax(40)
        assert md.rebuilds(0) > 1
        out.append((md.export_xu()[0], np.stack(md.forces(0))))
        md.close()
    for xu, f in out[1:]:
        assert np.array_equal(xu, out[0][0]) and np.array_equal(f, out[0][1])


# A checkpoint goes on bit for bit in a larger slot of its handle: replicas
# whose force blocks are four groups of 64, in slots of four and of five, at
# force teams of 16, 8 and 4 lanes.
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n,caps", [(4000, (4000, 5000)), (8000, (8000, 9000)), (16000, (16000, 17000))])
def test_checkpoint_between_slot_capacities(gpu, n, caps, prec):
    h = ctypes.c_void_p()
    assert gpu.lib.ac4_md_create_slots(2, (ctypes.c_int * 2)(*caps), prec, ctypes.byref(h)) == 0
    md = gpu.MD.__new__(gpu.MD)
    md.h, md.params = h, [gpu.ReplicaParams(n, 1.2, 0.5, 1.0, -1, 30, 3)] * 2
    for r in range(2):
        assert gpu.lib.ac4_md_assign(h, r, ctypes.byref(md.params[r])) == 0
        s = gpu.init_lattice(n, 0.5, 5)
        md.set_state(r, *[s[k] for k in ("x", "y", "z", "xu", "yu", "zu", "px", "py", "pz")], s["type"], s["act_tag"],
                     s["kx"], s["ky"], s["kz"])
    md.relax(40)
    md.init_chain(0)
    md.step(20)
    md.restore(1, md.checkpoint(0))
    for _ in range(60):  # the sum of p^2 of every step: its last bit seldom survives in the thermostat
        md.step(1)
        assert md.stats(0) == md.stats(1)
    x, y = md.get_state(0), md.get_state(1)
    assert all(np.array_equal(x[k], y[k]) for k in x)
    assert np.array_equal(md.get_chain(0), md.get_chain(1))
    md.close()


# S4 and Fs of an origin whose last lag frame is left out: the lags that came
# are those of the full walk.  The next frame that comes is a lag frame, or an
# origin that takes a place of the resident frames itself, or there is none;
# both S4 kernels.
@pytest.mark.parametrize("n,obs", [(300, 15), (300, 4), (3100, 12)])
def test_origins_without_their_last_lag(gpu, n, obs):
    frames = trajgen.case_frames(3, 30)
    left_out = [frames.index(t) for t in (42, 46, 52, 72, 102)]
    X, Y, Z, T = trajgen.make_frames(n, frames, 5, 0.08, 1.0)
    L = (n / 1.2) ** (1.0 / 3.0)
    an = gpu.Analysis(n, L, frames, gap=30, obs=obs)
    for f in range(len(frames)):
        if f not in left_out:
            an.push(f, X[f], Y[f], Z[f], T[f])
    an.finalize()
    walk = _walk(frames, 30)
    here = ~np.isin([frames.index(o + l) for o, l in walk], left_out)
    last = {o: o + l for o, l in walk}
    assert set(last.values()) <= {frames[k] for k in left_out} and here.sum() > 20
    os4 = OL.phase("s4", n, L, X, Y, Z, T, frames, 30)
    v, m = an.pairs(gpu.OBS_S4)
    assert np.array_equal(m[here], os4["mask"][here]) and m[here].min() > 0 and not m[~here].any()
    # a term is off by at most a few 1e-14
    assert np.abs(v[here] - os4["pairs"][here]).max() < 1e-12 * n and not v[~here].any()
    if obs & 8:
        ofs = OL.phase("fs", n, L, X, Y, Z, T, frames, 30)
        w = an.pairs(gpu.OBS_FS)
        assert np.abs(w[here] - ofs["pairs"][here]).max() < 1e-12 * n and not w[~here].any()
    an.close()


# Boxes of no bin, one bin and two: an empty histogram, and the pairs' counts.
@pytest.mark.parametrize("L,nbin", [(0.004, 0), (0.0101, 1), (0.0201, 2)])
def test_guu_boxes_of_few_bins(gpu, L, nbin):
    n, frames = 300, trajgen.case_frames(5, 40)
    X, Y, Z, _ = trajgen.make_frames(n, frames, 31, 0.3, 1.0)
    act = np.ones(n, dtype=np.int32)
    fr = gpu.Frames(n, L, len(frames))
    for k, t in enumerate(frames):
        fr.push(X[k], Y[k], Z[k], t)
    h, fn, no = fr.guu(act, 40, 0.06)
    fr.close()
    assert h.shape == (3, nbin) and no > 0
    if nbin:
        ho, fno, noo = OL.guu(n, L, X, Y, Z, act, frames, 40, 0.06)
        assert (fn, no) == (fno, noo) and np.array_equal(h[0], ho[0])


# The device push copies arrays that the handle's device may not read where
# they are: pageable and pinned host memory, all of the arrays or one of them,
# overwritten as soon as the push returns.
@pytest.mark.parametrize("n,obs", [(700, 15), (2049, 3)])
@pytest.mark.parametrize("where", ["pageable", "pinned", "types"])
def test_device_push_of_other_memory(gpu, n, obs, where):
    frames = trajgen.case_frames(3, 30)
    X, Y, Z, T = trajgen.make_frames(n, frames, 5 + n, 0.08, 1.0)
    L = (n / 1.2) ** (1.0 / 3.0)
    hip = ctypes.CDLL("libamdhip64.so")  # the runtime the library has loaded
    dev, pin = ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipMalloc(ctypes.byref(dev), ctypes.c_size_t(28 * n)) == 0
    assert hip.hipHostMalloc(ctypes.byref(pin), ctypes.c_size_t(28 * n), 0) == 0
    own = np.zeros(28 * n, dtype=np.uint8)
    base = {"pageable": own.ctypes.data, "pinned": pin.value, "types": dev.value}[where]
    at = [base + 8 * n * k for k in range(4)]  # x, y, z, types
    if where == "types":
        at[3] = own.ctypes.data
    out = []
    for device in (False, True):
        an = gpu.Analysis(n, L, frames, gap=30, obs=obs)
        for f in range(len(frames)):
            if not device:
                an.push(f, X[f], Y[f], Z[f], T[f])
                continue
            src = [np.ascontiguousarray(v) for v in (X[f], Y[f], Z[f], np.asarray(T[f], dtype=np.int32))]
            for d, v in zip(at, src):
                assert hip.hipMemcpy(ctypes.c_void_p(d), v.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(v.nbytes), 4) == 0
            assert gpu.lib.ac4_ana_push_frame_device(an.h, f, *at) == 0
            for d, v in zip(at, src):
                w = np.full(v.nbytes, 255, dtype=np.uint8)
                assert hip.hipMemcpy(ctypes.c_void_p(d), w.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(w.nbytes), 4) == 0
        an.finalize()
        got = [an.pairs(o) for o in (gpu.OBS_MSD, gpu.OBS_OVERLAP, gpu.OBS_S4, gpu.OBS_FS) if obs & o]
        out.append([v for g in got for v in (g if isinstance(g, tuple) else (g,))])
        an.close()
    hip.hipFree(dev)
    hip.hipHostFree(pin)
    for a, b in zip(*out):
        assert np.array_equal(a, b)


# What a handle takes of the device's memory is what ac4_md_slot_bytes says of
# its slots, which the server plans with: the largest slots at the widest team,
# where every block table has its full size.
def test_slot_bytes_cover_the_handle(gpu):
    hip = ctypes.CDLL("libamdhip64.so")  # the runtime the library has loaded

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipDeviceSynchronize() == 0 and hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    caps = [1 << 21] * 4
    gpu.set_tuning(16)
    try:
        for c in ([1000], caps):  # the first loads the code and what else the runtime keeps
            h, f0 = ctypes.c_void_p(), free()
            assert gpu.lib.ac4_md_create_slots(len(c), (ctypes.c_int * len(c))(*c), 0, ctypes.byref(h)) == 0
            used = f0 - free()
            assert gpu.lib.ac4_md_destroy(h) == 0
    finally:
        gpu.set_tuning()
    # the export's arrays are allocated when first used; each of about 70
    # arrays is rounded up to 2 MiB at most
    want = sum(gpu.slot_bytes(c) for c in caps) - 28 * sum(caps)
    assert used <= want + 70 * (2 << 20), (used, want)


# FP32 pair energy of the automatic force team, formed in the order of the list
# layout's team (8, 4, 2 lanes and one), against that team pinned: the same
# FP32 partial sums, added up in FP64 in another order; several replicas, lists
# of few and of many entries.
@pytest.mark.parametrize("sizes,layout", [((5000,), 8), ((8192,), 8), ((3000, 700, 1500), 8), ((8193,), 4), ((14001,), 4),
                                          ((16385,), 2), ((300, 20000, 5001), 2), ((32769,), 1), ((60001, 500), 1),
                                          ((160001,), 1)])
def test_fp32_energy_in_the_layouts_order(gpu, sizes, layout):
    out = []
    for tpp in (0, layout):
        gpu.set_tuning(tpp)
        try:
            md = gpu.MD([gpu.ReplicaParams(n, 1.2, 0.5, 1.0, -1, 200, 3 + r) for r, n in enumerate(sizes)], precision=gpu.FP32)
        finally:
            gpu.set_tuning()
        for r, n in enumerate(sizes):
            s = gpu.init_lattice(n, 0.5, n)
            rng = np.random.default_rng(n)
            x = [(s[k] + rng.normal(0, 0.02 / n ** (1 / 3), n)) % 1.0 for k in ("x", "y", "z")]
            md.set_state(r, *x, *x, s["px"], s["py"], s["pz"], s["type"], s["act_tag"], s["kx"], s["ky"], s["kz"])
        pv = np.array(md.calculate_forces())
        md.step(1)
        out.append((pv, [md.stats(r) for r in range(len(sizes))]))
        md.close()
    (pa, sa), (pb, sb) = out
    # sums of n terms of both signs: a few roundings of the sum of their sizes, about 5 n
    for r, n in enumerate(sizes):
        assert np.abs(pa[r] - pb[r]).max() <= 2.0 ** -53 * 8 * 5 * n
        # after a step the positions differ by the order of the force sums, which an FP32 term can round away from
        assert np.isclose(sa[r]["pe"], sb[r]["pe"], rtol=1e-9) and np.isclose(sa[r]["Heff"], sb[r]["Heff"], rtol=1e-9)


# Energy, virial and Heff after the same steps taken one by one, in calls of
# several, from recorded chunks and from several handles together: bit for bit,
# for every order of the energy and both modes of its last step.
@pytest.mark.parametrize("prec,n", [(0, 700), (1, 700), (1, 5000), (1, 9001), (1, 20000), (1, 40000)])
@pytest.mark.parametrize("nsteps", [1, 25, 26, 49, 50])
def test_energy_after_every_kind_of_call(gpu, prec, n, nsteps):
    mds = []
    for k in range(4):
        md = gpu.MD([gpu.ReplicaParams(n, 1.2, 0.5, 1.0, -1, 7, 3)], precision=prec)
        s = gpu.init_lattice(n, 0.5, n)
        md.set_state(0, *[s[q] for q in ("x", "y", "z", "xu", "yu", "zu", "px", "py", "pz")], s["type"], s["act_tag"],
                     s["kx"], s["ky"], s["kz"])
        md.relax(30)
        md.init_chain(0)
        mds.append(md)
    a, b, c, d = mds
    for rep in range(2):
        for _ in range(nsteps):
            a.step(1)
        b.step(nsteps)
        c.step(nsteps, graph=True)
        gpu.step_multi([d], nsteps)
        want = a.stats(0)
        assert want["pe"] != 0.0
        for md in (b, c, d):
            assert md.stats(0) == want
        x = a.get_state(0)
        for md in (b, c, d):
            y = md.get_state(0)
            assert all(np.array_equal(x[k], y[k]) for k in x)
            assert np.array_equal(np.stack(a.forces(0)), np.stack(md.forces(0)))
    if n <= 32768:  # calls of whole chunks that the plain step replays
        for _ in range(14):
            b.step(25)
            c.step(25, graph=True)
            assert b.stats(0) == c.stats(0)
    for md in mds:
        md.close()


# A slot assigned again while it is occupied, by a job of the same size, of
# another number of active particles, denser and smaller, after steps from
# recorded graphs: it runs as in a handle of its own assignment, and so does
# its neighbour.
def test_slots_assigned_again(gpu):
    def fill(md, r, p):
        md.params[r] = p
        assert gpu.lib.ac4_md_assign(md.h, r, ctypes.byref(p)) == 0
        s = gpu.init_lattice(p.n, 0.5, 5 + r)
        act = s["act_tag"] if p.n_act < 0 else np.where(np.arange(p.n) < p.n_act, np.arange(p.n), -1).astype(np.int32)
        k = [np.resize(s[c], max(p.n_act, 0)) if p.n_act >= 0 else s[c] for c in ("kx", "ky", "kz")]
        md.set_state(r, *[s[c] for c in ("x", "y", "z", "xu", "yu", "zu", "px", "py", "pz")], s["type"], act, *k)
        md.init_chain(r)

    def handle():
        h = ctypes.c_void_p()
        assert gpu.lib.ac4_md_create_slots(2, (ctypes.c_int * 2)(900, 1200), 1, ctypes.byref(h)) == 0
        md = gpu.MD.__new__(gpu.MD)
        md.h, md.params = h, [None] * 2
        return md

    P = gpu.ReplicaParams
    other = P(1100, 1.2, 0.5, 1.0, -1, 10, 4)
    used = handle()
    fill(used, 0, P(900, 1.2, 0.5, 1.0, -1, 10, 3))
    fill(used, 1, other)
    used.step(30, graph=True)
    for p in (P(900, 1.2, 0.6, 1.5, -1, 7, 8), P(900, 1.2, 0.5, 1.0, 250, 10, 3), P(900, 0.9, 0.5, 1.0, -1, 10, 3),
              P(640, 1.2, 0.5, 1.0, -1, 10, 3)):
        fresh = handle()
        for md in (used, fresh):
            fill(md, 0, p)
            fill(md, 1, other)
            md.step(51, graph=True)
        for r in range(2):
            x, y = used.get_state(r), fresh.get_state(r)
            assert all(np.array_equal(x[k], y[k]) for k in x) and used.stats(r) == fresh.stats(r)
        fresh.close()
    used.close()
