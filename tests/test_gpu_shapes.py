"""Kernels at the sizes and inputs where their tiles, remainders and fast paths can go wrong,
against the oracle or the plain statement of the same computation."""
import numpy as np
import pytest

from oracle import oracle as orc
from specfwat_amd import misfit
from specfwat_amd.mesh import BoxMesh
from specfwat_amd.solver import ElasticRun
from specfwat_amd.sources import Receivers, Sources
from test_gpu_parity import KERN_TOL, SEIS_TOL, make_case, oracle_of, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,dt,T,len_fac", [
    ("slow", 0.01, 0.8, 1.0), ("slow", 0.005, 1.0, 1.6), ("fast", 0.02, 2.0, 2.0), ("quiet", 0.02, 2.0, 2.56),
    ("ties", 0.02, 2.0, 2.0), ("zero", 0.02, 2.0, 2.0), ("long", 0.002, 2.0, 4.0)])
def test_sliding_lags_with_many_candidates(kind, dt, T, len_fac):
    """Window selection where single precision cannot tell the lags apart: periods of hundreds of
    samples (neighbouring lags differ by less than the sums' rounding), quiet stretches 1e-9 below
    the trace's maximum, exact ties and data that are zero; windows of 81, 321, 201, 257 and 4,001
    samples.  The same windows as the oracle, which sums every lag in double.  ties: obs repeats
    with opposite sign after 25 samples and syn = -obs f, so that the lags 25 and -25 have the
    same sums wherever f is 1; f grows or decays before and after, so the shift changes sign
    where the tie ends or begins, and the windows' gap there says which lag won.  zero: the lag of
    windows of zeros (the first) is four seconds from its neighbours', which the jump rule shows."""
    rng = np.random.default_rng(3)
    nstep, nrec = (4101, 1) if kind == "long" else (2400, 2)
    print(f"sliding lags: {kind}, {int(len_fac * T / dt) + 1} samples", flush=True)
    t = np.arange(nstep) * dt
    span = nstep * dt
    obs, syn = np.zeros((nstep, nrec, 3), np.float32), np.zeros((nstep, nrec, 3), np.float32)
    tp, dist = (np.array([0.3, 0.25]) * span)[:nrec], (np.array([2.0, 2.2]) * span)[:nrec]
    for r in range(nrec):
        for c in range(3):
            f, env = {"slow": (0.12, 0.06), "long": (8.0, 0.25)}.get(kind, (0.5, 0.25))
            w = lambda s: np.exp(-((t - 0.55 * span - s) * env) ** 2) * np.sin(2 * np.pi * f * (t - s))
            syn[:, r, c] = w(0.0)
            obs[:, r, c] = w(0.04 * (r + 1)) + 1e-3 * rng.standard_normal(nstep) * (kind == "fast")
            if kind == "quiet":
                obs[:nstep // 2, r, c] *= 1e-9
                syn[:nstep // 2, r, c] *= 1e-9
    cfg = dict(sliding_win_len_fac=len_fac, min_peaks_troughs=1, min_snr_window=0.1, min_win_len_fac=0.05)
    if kind in ("ties", "zero"):
        j = np.arange(nstep)
        for r in range(nrec):
            for c in range(3):
                if kind == "ties":
                    f = 1 + (np.maximum(900 - j, 0) + np.maximum(j - 1500, 0)) / 2048.0 * (1 - c)
                    obs[:, r, c] = np.abs((j + 7 * c + 3 * r) % 50 - 25) - 12.5
                    syn[:, r, c] = -obs[:, r, c] * f
                else:
                    syn[:, r, c] = np.sin(2 * np.pi * (0.5 * t + 0.002 * t * t))
                    obs[:, r, c] = np.roll(syn[:, r, c], 2 + 3 * c)
                    obs[:1100 + 9 * r + c, r, c] = 0
        tp, dist = np.array([6.0, 5.0]), np.array([2.4 * 40.0, 2.4 * 41.0])
        cfg.update(min_snr_window=0.0, min_energy_ratio=1e9, threshold_shift_fac=0.4,
                   jump_fac=0.1 if kind == "ties" else 1.5)
    got = misfit.select_windows(obs, syn, dt, 0.0, tp, dist, T, **cfg)
    n = 0
    for r in range(nrec):
        for c in range(3):
            ref, _, _ = orc.win_sel(obs[:, r, c], syn[:, r, c], dt, 0.0, tp[r], dist[r], T, **cfg)
            np.testing.assert_array_equal(got[3 * r + c], ref)
            n += len(ref)
    assert n >= (2 * nrec * 3 - nrec if kind == "ties" else 1)  # a gap in two of three components
    print(f"windows: {n}", flush=True)


@pytest.mark.parametrize("nl", [128, 129, 1024, 1025, 4096, 4097, 8192, 8193])
def test_correlation_shift_by_transforms(nl):
    """xcorr_shift at both ends of the transform path's range and of its lengths (nl 128 and 8193
    take the direct sums), with ties: a periodic window, whose best lags' sums differ by the
    taper only, a square wave against its negative, whose lags 16 and -16 have the same sums, and
    zero data.  The shifts of the oracle's direct sums."""
    nstep, dt = nl + 7, 0.01
    rng = np.random.default_rng(nl)
    t = np.arange(nstep)
    obs, syn = np.zeros((nstep, 2, 3), np.float32), np.zeros((nstep, 2, 3), np.float32)
    wave = np.exp(-((t - 0.5 * nl) / (0.1 * nl)) ** 2) * np.sin(2 * np.pi * t / (0.07 * nl))
    shift = max(1, min(nl // 40, 300))
    for k, (o, s) in enumerate([(np.roll(wave, shift), wave), (1e-12 * np.roll(wave, -shift), wave),
                                (np.sin(2 * np.pi * t / 16.0), np.sin(2 * np.pi * (t - 3) / 16.0)),
                                (np.sign(np.sin(2 * np.pi * t / 32 + 0.1)), -np.sign(np.sin(2 * np.pi * t / 32 + 0.1))),
                                (rng.standard_normal(nstep), rng.standard_normal(nstep)), (0 * t, wave)]):
        obs[:, k // 3, k % 3], syn[:, k // 3, k % 3] = o, s
    win = [[0.03, 0.03 + nl * dt + 0.001]]
    print(f"correlation of {nl} samples", flush=True)
    _, _, meas = misfit.event_cc_adjoint_sources(obs, syn, dt, win, imeas=11)
    for k in range(6):
        _, _, o = orc.cc_adjoint(obs[:, k // 3, k % 3], syn[:, k // 3, k % 3], dt, win, imeas=11)
        if k == 5:  # zero data: the error and the coefficient are not numbers; the shift is the first lag
            assert meas[k, 0, 7] == 1 - (int(win[0][1] / dt) - int(win[0][0] / dt))
            continue
        assert meas[k, 0, 4] == pytest.approx(o["tshift"][0], abs=1e-12), k
        if k == 3:
            assert meas[k, 0, 7] == -16  # the first of the two


def test_more_traces_than_spectra_at_a_time():
    """Spectra of the correlations take at most 512 MiB, 4,095 traces of 4,097 samples: with 4,098
    traces the last three come in a part of their own.  Every trace as in a small call."""
    nl, nrec, dt = 4097, 1366, 0.01
    rng = np.random.default_rng(8)
    obs, syn = (rng.standard_normal((nl + 7, 5, 3)).astype(np.float32) for _ in range(2))
    q = np.arange(nrec) % 5
    win = [[0.03, 0.03 + nl * dt + 0.001]]
    assert misfit.get_window_info(win[0], dt)[2] == nl
    print(f"{3 * nrec} traces", flush=True)
    _, adj0, meas0 = misfit.event_cc_adjoint_sources(obs, syn, dt, win, imeas=12, cc_min=0.0)
    _, adj, meas = misfit.event_cc_adjoint_sources(obs[:, q], syn[:, q], dt, win, imeas=12, cc_min=0.0)
    assert meas0[:, 0, 6].any() and len(set(meas0[:, 0, 7])) == 15
    np.testing.assert_array_equal(meas.reshape(nrec, 3, -1), meas0.reshape(5, 3, -1)[q])
    np.testing.assert_array_equal(adj, adj0[:, q])


@pytest.mark.parametrize("nrec", [1, 3, 4, 5, 7, 8, 9, 17])
def test_many_receivers_in_one_element(nrec):
    """Every receiver in one element on an absorbing side: a point's row then ends in nrec receiver
    terms, read eight terms at a time, after its face and source terms; forward and adjoint runs against
    the FP64 oracle, with the tractions taken inside the assembly."""
    c = make_case(nex=4, ney=3, nez=3, seed=60 + nrec, nstep=140)
    m = c["mesh"]
    rng = np.random.default_rng(nrec)
    c["rxyz"] = np.stack([rng.uniform(0.02, 0.23, nrec) * m.lx, rng.uniform(0.02, 0.31, nrec) * m.ly, np.zeros(nrec)], axis=1)
    c["sxyz"] = [[0.12 * m.lx, 0.2 * m.ly, -0.15 * m.lz]]
    o = oracle_of(c, 64)
    obs = o.forward(save=True)
    adj = (0.5 * obs).astype(np.float32)
    ko = o.adjoint(adj)
    src, rec = Sources(m, c["sxyz"], c["mt"], c["f0"]), Receivers(m, c["rxyz"])
    assert len(set(rec.ispec)) == 1
    f = ElasticRun(m, c["rho"], c["vp"], c["vs"], src, rec, c["dt"], c["nstep"], 1, True)
    f.iterate_time()
    assert rel(f.seismograms(), obs) < SEIS_TOL
    a = ElasticRun(m, c["rho"], c["vp"], c["vs"], src, rec, c["dt"], c["nstep"], 3, False)
    a.take_forward(f)
    a.set_adjoint_sources(adj)
    a.iterate_time()
    k = a.kernels()
    for n in ("rho_kl", "mu_kl", "kappa_kl"):
        assert rel(k[n], ko[n]) < KERN_TOL, n
    f.close()
    a.close()


@pytest.mark.parametrize("mesh,perturb,nfield", [((1, 1, 1), 0.0, 4), ((3, 1, 2), 0.0, 1), ((3, 2, 2), 0.1, 6),
                                                 ((5, 3, 2), 0.0, 21), ((5, 3, 2), 0.1, 24), ((3, 3, 3), 0.0, 25)])
def test_smoothing_of_any_number_of_fields(mesh, perturb, nfield):
    """Diffusion steps of 1 to 25 fields (whole and ragged groups of four, rows of one value and of
    16-byte pieces, a second run for the 25th) on cubes and deformed elements, down to one element,
    all of whose points the element pass finishes; against the loop restatement field by field."""
    from specfwat_amd.smooth import smooth_batch
    print(f"smoothing {nfield} fields on {mesh}, perturb {perturb}", flush=True)
    m = BoxMesh(*mesh, *(1000.0 * v for v in mesh), perturb=perturb)
    rng = np.random.default_rng(nfield)
    fields = rng.standard_normal((nfield, m.nspec, 125)).astype(np.float32)
    out = smooth_batch(m, fields, 800.0, 400.0, faithful=False)[0]
    for q in {0, nfield // 2, nfield - 1}:
        _, ref, _ = orc.smooth_pde(m.smooth_arrays(), fields[q].ravel(), 800.0, 400.0, m.distance_min_glob(), faithful=False)
        assert rel(out[q], ref) < 1e-5, q  # 32-bit steps, the bar of the other smoothing tests


@pytest.mark.parametrize("nrec", [341, 342, 347, 683, 1365, 1366, 1371])
def test_large_results_arrive_whole(nrec):
    """Adjoint sources of 4,096 samples, 48 KiB a receiver: from 16 MiB on results are copied in
    pieces by several threads, of 1 MiB below 64 MiB and 2 MiB above; below, at and above these
    sizes, with ragged last pieces.  The traces repeat those of seven receivers, so each has
    to equal its part of the small call's result."""
    n, dt = 4096, 0.05
    rng = np.random.default_rng(nrec)
    obs, syn = (rng.standard_normal((n, 7, 3)).astype(np.float32) for _ in range(2))
    q = np.arange(nrec) % 7
    small = misfit.event_adjoint_sources(obs, syn, dt, [[1.0, 200.0]])[1]
    large = misfit.event_adjoint_sources(obs[:, q], syn[:, q], dt, [[1.0, 200.0]])[1]
    assert np.abs(small).max() > 0
    np.testing.assert_array_equal(large, small[:, q])


@pytest.mark.parametrize("nstep", [31, 32, 33, 63, 64, 65, 97, 129])
def test_adjoint_filter_at_block_edges(nstep):
    """The bandpass walks blocks of 32 samples, the next one loaded ahead, its second section one
    sample behind: series that end at, before and after a block; against the oracle trace by trace."""
    dt = 0.05
    rng = np.random.default_rng(nstep)
    obs, syn = (rng.standard_normal((nstep, 11, 3)).astype(np.float32) for _ in range(2))
    win = [[0.0, nstep * dt]]
    _, adj = misfit.event_adjoint_sources(obs, syn, dt, win, min_period=0.4, max_period=12.0)
    for r in range(11):
        for c in range(3):
            _, a, _, _ = orc.waveform_adjoint(obs[:, r, c], syn[:, r, c], dt, win)
            a = orc.filter_adj(a, dt, np.float32(1 / 12.0), np.float32(1 / 0.4), win)
            assert np.abs(adj[:, r, c] - a).max() <= 1e-6 * np.abs(a).max(), (r, c)  # single precision, as its other tests


@pytest.mark.parametrize("jump_fac", [-2.0, -0.3, 0.0, 0.1, 3.0])
def test_windows_with_any_jump_rule(jump_fac):
    """The window starts that are computed are those the selection reads: the time range and the
    jump rule's reach, none for a negative factor (the rule is off) and up to the whole trace.  The
    first trace's range ends inside the signal on both sides, so windows reach to its ends."""
    nstep, dt, T = 3000, 0.02, 2.0
    print(f"jump factor {jump_fac}", flush=True)
    t = np.arange(nstep) * dt
    obs, syn = np.zeros((nstep, 2, 3), np.float32), np.zeros((nstep, 2, 3), np.float32)
    for r in range(2):
        for c in range(3):
            syn[:, r, c] = np.sin(2 * np.pi * (0.5 * t + (0.002 + 0.001 * c) * t * t))
            obs[:, r, c] = np.roll(syn[:, r, c], 3 + 2 * c)
    tp, dist = np.array([18.0, 3.0]), np.array([2.4 * 42.0, 2.4 * 60.0])
    cfg = dict(jump_fac=jump_fac, min_peaks_troughs=1, min_snr_window=0.1, min_win_len_fac=0.5)
    got = misfit.select_windows(obs, syn, dt, 0.0, tp, dist, T, **cfg)
    n = 0
    for r in range(2):
        for c in range(3):
            ref, _, _ = orc.win_sel(obs[:, r, c], syn[:, r, c], dt, 0.0, tp[r], dist[r], T, **cfg)
            np.testing.assert_array_equal(got[3 * r + c], ref)
            n += len(ref)
    assert n > 0


def _direct_shift(d, s):
    """The first maximum of every lag's direct sum, the lags in fours over the union of their ranges
    (a sample that is not a number makes a zero product one too); None when no sum is above -inf."""
    n, best, at = len(d), -np.inf, None
    pad = np.concatenate([np.zeros(3), s, np.zeros(3)])
    with np.errstate(invalid="ignore"):
        for mb in range(0, 2 * n - 1, 4):
            lo, hi = max(0, mb - n + 1), min(n - 1, mb + 3)
            for m in range(mb, min(mb + 4, 2 * n - 1)):
                c = np.cumsum(d[lo:hi + 1] * pad[lo + n - 1 - m + 3:hi + n - 1 - m + 4])[-1]
                if c > best:
                    best, at = c, m + 1 - n
    return at


@pytest.mark.filterwarnings("ignore:invalid value")
@pytest.mark.parametrize("nl", [128, 129, 517, 2049])
def test_correlation_shift_of_data_that_are_not_finite(nl):
    """Windows with NaN or infinite samples, whose transforms say nothing: the shift is the direct
    sums' in every path (nl 128 has no other); a window of NaN only is not selected."""
    nstep, dt = nl + 7, 0.01
    rng = np.random.default_rng(nl)
    obs, syn = (rng.standard_normal((nstep, 3, 3)).astype(np.float32) for _ in range(2))
    a, b = 4 + nl // 5, 4 + (7 * nl) // 8
    obs[a, 0, 0], obs[b, 0, 1], syn[a, 0, 2] = np.nan, np.inf, -np.inf
    syn[b, 1, 0], obs[a, 1, 1], obs[b, 1, 1] = np.nan, np.nan, np.nan
    obs[4, 1, 2], syn[nl + 2, 1, 2] = np.nan, np.inf
    obs[:, 2, 0] = np.nan
    win = [[0.03, 0.03 + nl * dt + 0.001]]
    print(f"correlation of {nl} samples that are not finite", flush=True)
    _, adj, meas = misfit.event_cc_adjoint_sources(obs, syn, dt, win, imeas=11)
    first, _, n = misfit.get_window_info(win[0], dt)
    first -= 1
    assert n == nl
    tw = misfit.window_taper(np.ones(n), 0.05, 1)
    for k in range(9):
        d, s = (x[first:first + n, k // 3, k % 3].astype(np.float64) * tw for x in (obs, syn))
        ref = _direct_shift(d, s)
        if k == 6:
            assert ref is None and meas[k, 0, 6] == 0 and not adj[:, 2, 0].any()
        else:
            assert meas[k, 0, 7] == ref, k


@pytest.mark.filterwarnings("ignore:invalid value")
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_windows_of_data_that_are_not_finite(bad):
    """Window starts whose samples are not all finite take every lag's direct sum: their shifts decide
    by the jump rule which starts beside them stay good.  The oracle's shifts and coefficients
    of the clean trace, with those starts' shifts put in, give the windows."""
    nstep, dt, T, thr, max_shift = 1700, 0.02, 2.0, 0.8, 0.3
    t = np.arange(nstep) * dt
    obs, syn = np.zeros((nstep, 1, 3), np.float32), np.zeros((nstep, 1, 3), np.float32)
    for c in range(3):
        syn[:, 0, c] = np.sin(2 * np.pi * (0.5 * t + 0.002 * t * t))
        obs[:, 0, c] = np.roll(syn[:, 0, c], 3 + c)
    hit = (800, 0 if np.isnan(bad) else 1), (1003, 2)  # (sample, component) of obs; the second pair of syn when NaN
    clean = obs.copy(), syn.copy()
    obs[hit[0][0], 0, hit[0][1]] = bad
    (syn if np.isnan(bad) else obs)[hit[1][0], 0, hit[1][1]] = bad
    tp, dist, jump_fac = 6.0, 2.4 * 28.0, 0.1
    print(f"windows with {bad}", flush=True)
    got = misfit.select_windows(obs, syn, dt, 0.0, np.array([tp]), np.array([dist]), T, min_peaks_troughs=0,
                                min_snr_window=0.0, min_energy_ratio=1e9, min_win_len_fac=0.5, jump_fac=jump_fac)
    nlen = int(2.0 * T / dt) + 1
    tw, nw = misfit.window_taper(np.ones(nlen), 1.0, 1), nstep - nlen
    tc = (np.arange(nw) + nlen / 2.0) * dt
    nj, n = int(jump_fac * T / dt + 0.5), 0
    for c in range(3):
        _, cc, ts = orc.win_sel(clean[0][:, 0, c], clean[1][:, 0, c], dt, 0.0, tp, dist, T, min_peaks_troughs=0)
        d, s = (x[:, 0, c].astype(np.float64) / np.abs(clean[1][:, 0, c]).max() for x in (obs, syn))
        for i in range(nw):
            if not (np.isfinite(d[i:i + nlen]).all() and np.isfinite(s[i:i + nlen]).all()):
                dw, sw = d[i:i + nlen] * tw, s[i:i + nlen] * tw
                k = _direct_shift(dw, sw)
                x, y = (dw[k:], sw[:nlen - k]) if k >= 0 else (dw[:k], sw[-k:])  # what overlaps after the shift
                cc[i], ts[i] = (x * y).sum() / np.sqrt((x * x).sum() * (y * y).sum()), k * dt
        good = (cc > thr) & (np.abs(ts) < max_shift * T) & (tc >= tp - 1.5 * T) & (tc <= dist / 2.4 + 1.5 * T)
        for i in np.flatnonzero(np.abs(np.diff(ts)) > jump_fac * T) + 1:
            good[max(0, i - nj):i + nj + 1] = False
        edge = np.flatnonzero(np.diff(np.concatenate([[0], good.astype(int), [0]])))
        ref = [(tc[a], tc[b - 1]) for a, b in zip(edge[::2], edge[1::2]) if (b - 1 - a) * dt >= 0.5 * T]
        np.testing.assert_array_equal(got[c], np.array(ref).reshape(-1, 2))
        n += len(ref)
    assert n >= 4


@pytest.mark.parametrize("nbytes", [1, 7 * 21000, 11 * 21000 + 20999, 36 * 21000])
@pytest.mark.parametrize("aniso", [False, True])
def test_kernels_read_out_in_parts(aniso, nbytes):
    """Kernels leave the device through a bounded piece of memory: one element or point at a time,
    ragged last parts, and exactly all; the same bits as in one piece, for a run and for a batch."""
    from specfwat_amd.batch import EventBatch
    c = make_case(seed=71, nstep=20, aniso=aniso)
    m = c["mesh"]
    src, rec = Sources(m, c["sxyz"], c["mt"], c["f0"]), Receivers(m, c["rxyz"])
    adj = np.random.default_rng(4).standard_normal((2, c["nstep"], rec.nrec, 3)).astype(np.float32)
    f, a = (ElasticRun(m, c["rho"], c["vp"], c["vs"], src, rec, c["dt"], c["nstep"], k, k == 1, cij=c["cij"]) for k in (1, 3))
    f.iterate_time()
    a.take_forward(f)
    a.set_adjoint_sources(adj[0])
    a.iterate_time()
    b = EventBatch(m, c["rho"], c["vp"], c["vs"], [src, src], rec, c["dt"], [c["nstep"]] * 2, cij=c["cij"])
    b.forward()
    b.set_adjoint_sources(adj)
    b.adjoint()
    for run, read in ((a, a.kernels), (b.run, b.kernels)):
        whole = read()
        run.set_readout_bytes(nbytes if aniso else max(nbytes // 10, 1))
        part = read()
        for n in whole:
            assert np.abs(whole[n]).max() > 0
            np.testing.assert_array_equal(part[n], whole[n], err_msg=n)
    b.close()
    f.close()
    a.close()


def test_other_knobs_leave_the_default_element_pass():
    """A new handle takes the library's element pass, which finishes the interior points of cubes;
    setting another knob keeps it, and after another pass -1 brings it back: the same bits throughout."""
    c = make_case(seed=81, nstep=40)
    m = c["mesh"]
    src, rec = Sources(m, c["sxyz"], c["mt"], c["f0"]), Receivers(m, c["rxyz"])
    first = None
    for steps in ([], [{}], [dict(interior=True)], [dict(slab_elems=8), {}], [dict(regular_path=1), dict(regular_path=-1)],
                  [dict(interior=False), dict(blocks_per_cu_adj=4)]):
        f = ElasticRun(m, c["rho"], c["vp"], c["vs"], src, rec, c["dt"], c["nstep"], 1, True)
        for kw in steps:
            f.set_tuning(**kw)
        assert f.interior_info()[2:] == (1, 1), steps
        f.iterate_time()
        syn = f.seismograms()
        f.close()
        first = syn if first is None else first
        np.testing.assert_array_equal(syn, first)
    f = ElasticRun(m, c["rho"], c["vp"], c["vs"], src, rec, c["dt"], c["nstep"], 1, True)
    f.set_tuning(regular_path=1)
    assert f.interior_info()[2:] == (0, 0)
    f.close()


@pytest.mark.parametrize("n", [24, 60])
def test_assemblies_agree_with_many_boundary_points(n):
    """Above 57,344 points with boundary, source or receiver terms (60x60x2: 58,081 at the bottom
    alone) one lane walks the row of each, below eight lanes; slab by slab one lane walks every
    row.  One and two points per lane, and slabs: the same bits, forward and adjoint."""
    nex, ney, lz, h = n, n, 2, 625.0
    m = BoxMesh(nex, ney, lz, nex * h, ney * h, lz * h)
    print(f"assembly with many boundary points, {m.nspec} elements", flush=True)
    rng = np.random.default_rng(n)
    f = (1 + 0.03 * rng.standard_normal(m.nglob))[m.ibool0]
    rho, vp, vs = (np.float32(v) * f.astype(np.float32) for v in (2700, 6000, 3500))
    src = Sources(m, [[0.4 * m.lx, 0.5 * m.ly, -0.5 * m.lz]], [list(1e15 * rng.standard_normal(6))], [6.0])
    rec = Receivers(m, np.stack([rng.uniform(0.35, 0.5, 5) * m.lx, rng.uniform(0.4, 0.6, 5) * m.ly, np.zeros(5)], axis=1))
    steps, first = 24, None
    adj = rng.standard_normal((steps, rec.nrec, 3)).astype(np.float32)
    for lanes, slab in ((1, 0), (2, 0), (0, n * n), (0, 0)):
        out = []
        a = None
        for k in (1, 3):
            r = ElasticRun(m, rho, vp, vs, src, rec, 0.004, steps, k, k == 1)
            r.set_tuning(regular_path=1, slab_elems=slab)
            r.set_assembly_lanes(lanes)
            if k == 1:
                r.iterate_time()
                out.append(r.seismograms())
                out += list(r.fields())
                a = r
                continue
            r.take_forward(a)
            a.close()
            r.set_adjoint_sources(adj)
            r.iterate_time()
            out += list(r.kernels().values())
            r.close()
        assert all(np.abs(x).max() > 0 for x in out)
        first = out if first is None else first
        for x, y in zip(out, first):
            np.testing.assert_array_equal(x, y, err_msg=f"lanes {lanes}, slab {slab}")
