"""xc_fast hot path on the GPU vs the FP64 oracle (oracle/xc.py).

Tolerances (relative L2 against FP64): fp32 <= 1e-5; bf16x3 <= 1e-3 (expected
~1e-5); fp16 <= 1e-3.  Row order (task order) and lag order are exact: every
row is compared with the oracle row of the same task.
"""
import numpy as np
import pytest

from oracle import xc

pytestmark = pytest.mark.gpu

TOL = {"fp32": 1e-5, "bf16x3": 1e-3, "fp16": 1e-3, "fp16x3": 1e-3, "plain": 1e-5}


def _spectra(rng, nstep, nsta, seg, nfft, dt, common=0.5):
    # band-limited noise with a shared component so cross-spectra are correlated
    base = rng.standard_normal((nstep, 1, seg))
    x = common * base + rng.standard_normal((nstep, nsta, seg))
    return (np.fft.rfft(x, n=nfft, axis=-1) * dt).astype(np.complex64)


def _all_pairs(nsta):
    src, rec = np.triu_indices(nsta, k=1)
    return src.astype(np.int32), rec.astype(np.int32)


@pytest.mark.parametrize("precision", ["fp32", "bf16x3", "fp16", "plain"])
@pytest.mark.parametrize("nsta,nstep,seg,nfft,H", [(40, 5, 800, 882 * 2, 100), (9, 24, 1500, 1764, 300),
                                                    (33, 47, 600, 1764, 200), (17, 100, 600, 1764, 200)])
def test_correlate_matches_oracle(gpu, precision, nsta, nstep, seg, nfft, H):
    import torch
    from fastxc_amd.ops import XcPlan

    rng = np.random.default_rng(nsta * 100 + nstep)
    dt = 0.1
    spec = _spectra(rng, nstep, nsta, seg, nfft, dt)
    nspec = nfft // 2 + 1
    src, rec = _all_pairs(nsta)
    plan = XcPlan(nspec, nstep, dt, H, precision)
    plan.set_pairs(nsta, src, rec)
    sd = torch.from_numpy(spec).to(gpu)
    xs = plan.cross_spectra(sd).cpu().numpy()
    want_xs = xc.cross_spectrum(spec, src, rec)
    assert xc.rel_l2(xs, want_xs) < TOL[precision]
    cc = plan.correlate(sd).cpu().numpy()
    want = xc.lags(want_xs, nfft, H, dt)
    err = xc.rel_l2(cc, want)
    print(f"precision={precision} nsta={nsta} rel_l2={err:.3e} maxabs={np.abs(cc - want).max():.3e}")
    assert err < TOL[precision]
    # per-row check: rows are in task order
    row_err = np.linalg.norm(cc - want, axis=1) / np.linalg.norm(want, axis=1)
    assert np.all(row_err < 10 * TOL[precision])


@pytest.mark.parametrize("precision", ["bf16x3", "fp16", "fp16x3"])
@pytest.mark.parametrize("nstep", [1, 12, 20, 28, 36, 44, 60, 90, 128, 200])
def test_every_operand_depth(gpu, precision, nstep):
    """One window count per compiled MFMA operand depth (kh 8, 16, 24, 32, 40,
    48, 64, 96, 128) and one beyond them (200 windows: seven chunks of 32
    accumulated in registers), two station tiles, against FP64."""
    import torch
    from fastxc_amd.ops import XcPlan

    rng = np.random.default_rng(500 + nstep)
    nsta, seg, nfft, H, dt = 37, 600, 1764, 200, 0.1
    spec = _spectra(rng, nstep, nsta, seg, nfft, dt)
    src, rec = _all_pairs(nsta)
    plan = XcPlan(nfft // 2 + 1, nstep, dt, H, precision)
    plan.set_pairs(nsta, src, rec)
    sd = torch.from_numpy(spec).to(gpu)
    xs = plan.cross_spectra(sd).cpu().numpy()
    want_xs = xc.cross_spectrum(spec, src, rec)
    err_xs = xc.rel_l2(xs, want_xs)
    cc = plan.correlate(sd).cpu().numpy()
    want = xc.lags(want_xs, nfft, H, dt)
    err = xc.rel_l2(cc, want)
    print(f"depth test {precision} nstep={nstep} xspec rel_l2={err_xs:.3e} cc rel_l2={err:.3e}")
    assert err_xs < TOL[precision] and err < TOL[precision]
    row_err = np.linalg.norm(cc - want, axis=1) / np.linalg.norm(want, axis=1)
    assert np.all(row_err < 10 * TOL[precision])


def test_production_length_fp32(gpu):
    """nfft = 37044 (2^2 3^3 7^3), H = 1000 at dt = 0.1, a handful of pairs."""
    import torch
    from fastxc_amd.ops import XcPlan

    rng = np.random.default_rng(7)
    nsta, nstep, seg, nfft, H, dt = 5, 3, 36000, 37044, 1000, 0.1
    spec = _spectra(rng, nstep, nsta, seg, nfft, dt)
    src = np.array([0, 0, 1, 3, 2, 4], np.int32)
    rec = np.array([1, 4, 3, 4, 2, 0], np.int32)
    plan = XcPlan(nfft // 2 + 1, nstep, dt, H, "fp32")
    plan.set_pairs(nsta, src, rec)
    cc = plan.correlate(torch.from_numpy(spec).to(gpu)).cpu().numpy()
    want = xc.correlate(spec, src, rec, nfft, H, dt)
    assert xc.rel_l2(cc, want) < 1e-5


def test_delayed_copy_lag_position_exact(gpu):
    import torch
    from fastxc_amd.ops import XcPlan

    rng = np.random.default_rng(3)
    seg, d, H, dt, nfft = 1500, 37, 300, 0.1, 1764
    base = rng.standard_normal(seg + d)
    x = np.stack([base[d:d + seg], base[:seg]])[None]
    spec = (np.fft.rfft(x, n=nfft, axis=-1) * dt).astype(np.complex64)
    plan = XcPlan(nfft // 2 + 1, 1, dt, H, "fp32")
    plan.set_pairs(2, np.array([0], np.int32), np.array([1], np.int32))
    cc = plan.correlate(torch.from_numpy(spec).to(gpu)).cpu().numpy()[0]
    want = xc.correlate(spec, [0], [1], nfft, H, dt)[0]
    # receiver delayed by d (rec(t) = src(t - d)): conj on the source side puts
    # the peak at lag +d, i.e. output index H + d
    assert int(np.argmax(cc)) == int(np.argmax(want)) == H + d


def test_chunked_matches_unchunked(gpu):
    import torch
    from fastxc_amd.ops import XcPlan

    rng = np.random.default_rng(11)
    nsta, nstep, seg, nfft, H, dt = 70, 4, 800, 1764, 200, 0.1
    spec = torch.from_numpy(_spectra(rng, nstep, nsta, seg, nfft, dt)).to(gpu)
    src, rec = _all_pairs(nsta)
    a = XcPlan(nfft // 2 + 1, nstep, dt, H, "fp32")
    a.set_pairs(nsta, src, rec)
    b = XcPlan(nfft // 2 + 1, nstep, dt, H, "fp32", chunk_rows=700)
    b.set_pairs(nsta, src, rec)
    assert b.pairs_info()["nchunks"] > 1
    ca = a.correlate(spec).cpu().numpy()
    cb = b.correlate(spec).cpu().numpy()
    assert np.array_equal(ca, cb)


@pytest.mark.parametrize("precision", ["bf16x3", "fp16x3", "fp16"])
def test_production_length_mfma_forms(gpu, precision):
    """The MFMA forms at nfft 37044: split contraction + the fixed-plan lag
    kernel, against FP64."""
    import torch
    from fastxc_amd.ops import XcPlan

    rng = np.random.default_rng(8)
    nsta, nstep, seg, nfft, H, dt = 40, 6, 36000, 37044, 1000, 0.1
    spec = _spectra(rng, nstep, nsta, seg, nfft, dt)
    src, rec = _all_pairs(nsta)
    plan = XcPlan(nfft // 2 + 1, nstep, dt, H, precision)
    plan.set_pairs(nsta, src, rec)
    cc = plan.correlate(torch.from_numpy(spec).to(gpu)).cpu().numpy()
    want = xc.correlate(spec, src, rec, nfft, H, dt)
    err = xc.rel_l2(cc, want)
    print(f"{precision} nfft 37044 rel_l2={err:.3e}")
    assert err < TOL[precision]


@pytest.mark.parametrize("precision", ["bf16x3", "fp16", "fp16x3", "fp32"])
def test_one_window_product_form(gpu, precision):
    """One window at nfft 37044: the stack of a pair is conj(S[src]) S[rec],
    which the lag kernel forms in FP32 from the two spectra as it reads them
    (no contraction).  Every form then meets the FP32 tolerance against FP64
    and agrees with the PLAIN form (the reference's step order through the
    cross-spectrum); pairs in both orientations, a delayed copy lands at
    exactly H + d."""
    import torch
    from fastxc_amd.ops import XcPlan

    rng = np.random.default_rng(21)
    nsta, seg, nfft, H, dt, d = 40, 36000, 37044, 1000, 0.1, 123
    spec = _spectra(rng, 1, nsta, seg, nfft, dt)
    base = rng.standard_normal(seg + d)
    spec[0, :2] = (np.fft.rfft(np.stack([base[d:d + seg], base[:seg]]), n=nfft, axis=-1)
                   * dt).astype(np.complex64)
    src, rec = _all_pairs(nsta)
    src = np.concatenate([src, rec[:50]]).astype(np.int32)  # 50 pairs reversed
    rec = np.concatenate([rec, src[:50]]).astype(np.int32)
    sd = torch.from_numpy(spec).to(gpu)
    plan = XcPlan(nfft // 2 + 1, 1, dt, H, precision)
    plan.set_pairs(nsta, src, rec)
    cc = plan.correlate(sd).cpu().numpy()
    want = xc.correlate(spec, src, rec, nfft, H, dt)
    err = xc.rel_l2(cc, want)
    print(f"{precision} one window rel_l2={err:.3e} maxabs={np.abs(cc - want).max():.3e}")
    assert err < 1e-5
    ref = XcPlan(nfft // 2 + 1, 1, dt, H, "plain")
    ref.set_pairs(nsta, src, rec)
    assert xc.rel_l2(cc, ref.correlate(sd).cpu().numpy()) < 1e-6
    assert int(np.argmax(cc[0])) == H + d


@pytest.mark.parametrize("precision", ["bf16x3", "fp32"])
def test_one_window_product_form_dt005(gpu, precision):
    """One window at nfft 74088 (dt 0.05 s): the lag synthesis of two half-length
    transforms folds the product conj(S[src]) S[rec] straight from the spectra;
    against FP64 and the PLAIN form, pairs in both orientations."""
    import torch
    from fastxc_amd.ops import XcPlan

    rng = np.random.default_rng(75)
    nsta, seg, nfft, H, dt = 9, 72000, 74088, 2000, 0.05
    spec = _spectra(rng, 1, nsta, seg, nfft, dt)
    src, rec = _all_pairs(nsta)
    src, rec = np.concatenate([src, rec[:5]]), np.concatenate([rec, src[:5]])
    src, rec = src.astype(np.int32), rec.astype(np.int32)
    sd = torch.from_numpy(spec).to(gpu)
    plan = XcPlan(nfft // 2 + 1, 1, dt, H, precision)
    plan.set_pairs(nsta, src, rec)
    cc = plan.correlate(sd).cpu().numpy()
    want = xc.correlate(spec, src, rec, nfft, H, dt)
    err = xc.rel_l2(cc, want)
    print(f"nfft 74088 one window {precision} rel_l2={err:.3e}")
    assert cc.shape == (len(src), 4001) and err < 1e-5
    ref = XcPlan(nfft // 2 + 1, 1, dt, H, "plain")
    ref.set_pairs(nsta, src, rec)
    assert xc.rel_l2(cc, ref.correlate(sd).cpu().numpy()) < 1e-6


@pytest.mark.parametrize("precision", ["bf16x3", "fp32"])
def test_uneven_segments_with_gaps(gpu, precision):
    """Segments of different station and window counts one after another, 10 %
    of station-windows zero-filled (gaps).  As the reference does, a gap
    still counts in the 1/nstep of its segment.  One plan per window count,
    its pair list re-set for every segment."""
    import torch
    from fastxc_amd.ops import XcPlan

    rng = np.random.default_rng(33)
    seg, nfft, H, dt = 600, 1764, 200, 0.1
    plans = {}
    for s in range(8):
        nsta = int(rng.integers(20, 61))
        nstep = int(rng.choice([6, 9, 12]))
        spec = _spectra(rng, nstep, nsta, seg, nfft, dt)
        gaps = rng.random((nstep, nsta)) < 0.1
        spec[gaps] = 0
        src, rec = _all_pairs(nsta)
        plan = plans.setdefault(nstep, XcPlan(nfft // 2 + 1, nstep, dt, H, precision))
        plan.set_pairs(nsta, src, rec)
        cc = plan.correlate(torch.from_numpy(spec).to(gpu)).cpu().numpy()
        want = xc.correlate(spec, src, rec, nfft, H, dt)
        err = xc.rel_l2(cc, want)
        assert err < TOL[precision], (s, nsta, nstep, err)


@pytest.mark.parametrize("precision", ["fp32", "bf16x3"])
def test_long_nfft_dt005(gpu, precision):
    """nfft 74088 (dt 0.05 s, one-hour windows), 4001 lags: the lag synthesis
    runs two half-length transforms in LDS; against FP64, lag order exact."""
    import torch
    from fastxc_amd.ops import XcPlan

    rng = np.random.default_rng(74)
    nsta, nstep, seg, nfft, H, dt = 6, 3, 72000, 74088, 2000, 0.05
    spec = _spectra(rng, nstep, nsta, seg, nfft, dt)
    src, rec = _all_pairs(nsta)
    plan = XcPlan(nfft // 2 + 1, nstep, dt, H, precision)
    plan.set_pairs(nsta, src, rec)
    cc = plan.correlate(torch.from_numpy(spec).to(gpu)).cpu().numpy()
    want = xc.correlate(spec, src, rec, nfft, H, dt)
    err = xc.rel_l2(cc, want)
    print(f"nfft 74088 {precision} rel_l2={err:.3e}")
    assert cc.shape == (len(src), 4001) and err < TOL[precision]
    row_err = np.linalg.norm(cc - want, axis=1) / np.linalg.norm(want, axis=1)
    assert np.all(row_err < 10 * TOL[precision])


@pytest.mark.parametrize("precision", ["fp32", "bf16x3", "fp16x3"])
def test_band_spec_mode(gpu, precision):
    """Spec mode fxc_xc_set_band: the stack is formed for the 16-bin chunks
    holding bins k_lo..k_hi and every other bin is 0.  Spectra that are 0
    outside the band give the parity result exactly; general spectra give the
    FP64 lags of the spectra with the bins outside those chunks zeroed; a
    parity call after a band call (and a band call after it) on the same plan
    and workspace are unaffected by the other mode."""
    import torch
    from fastxc_amd.ops import XcPlan

    rng = np.random.default_rng(31)
    nsta, nstep, seg, nfft, H, dt = 20, 6, 1500, 1764, 300, 0.1
    nspec = nfft // 2 + 1
    spec = _spectra(rng, nstep, nsta, seg, nfft, dt)
    src, rec = _all_pairs(nsta)
    k_lo, k_hi = 70, 611
    c0, c1 = k_lo // 16 * 16, -(-(k_hi + 1) // 16) * 16  # chunk-rounded band [c0, c1)
    inband = spec.copy()
    inband[..., :c0] = 0
    inband[..., c1:] = 0
    plan = XcPlan(nspec, nstep, dt, H, precision)
    plan.set_pairs(nsta, src, rec)
    parity_in = plan.correlate(torch.from_numpy(inband).to(gpu)).cpu().numpy()
    parity_gen = plan.correlate(torch.from_numpy(spec).to(gpu)).cpu().numpy()
    plan.set_band(k_lo, k_hi)
    band_in = plan.correlate(torch.from_numpy(inband).to(gpu)).cpu().numpy()
    assert np.array_equal(band_in, parity_in)
    band_gen = plan.correlate(torch.from_numpy(spec).to(gpu)).cpu().numpy()
    want = xc.lags(xc.cross_spectrum(inband, src, rec), nfft, H, dt)
    err = xc.rel_l2(band_gen, want)
    print(f"precision={precision} band rel_l2={err:.3e}")
    assert err < TOL[precision]
    plan.set_band()
    again = plan.correlate(torch.from_numpy(spec).to(gpu)).cpu().numpy()
    assert np.array_equal(again, parity_gen)
    plan.set_band(k_lo, k_hi)
    assert np.array_equal(plan.correlate(torch.from_numpy(spec).to(gpu)).cpu().numpy(), band_gen)
    plan.close()


def test_band_rejects_bad_ranges(gpu):
    from fastxc_amd.ops import XcPlan

    plan = XcPlan(883, 4, 0.1, 100, "bf16x3")
    with pytest.raises(RuntimeError):
        plan.set_band(10, 5)
    with pytest.raises(RuntimeError):
        plan.set_band(0, 883)
    plan.close()
    plain = XcPlan(883, 4, 0.1, 100, "plain")
    with pytest.raises(RuntimeError):
        plain.set_band(10, 500)
    plain.set_band()  # parity is always accepted
    plain.close()


@pytest.mark.parametrize("nsta,nstep", [(2, 1), (9, 4), (16, 5), (17, 7), (33, 8), (48, 13), (65, 3)])
def test_fp32_matrix_tiles(gpu, nsta, nstep):
    """Edges of the FP32 contraction: window counts around its steps of 4 and 8, station counts
    around its 16- and 32-station blocks, pairs in either order and listed twice, a last bin chunk
    that is not full.  fp32 sums of 2 nstep products: relative error below 2 nstep 2^-24 of
    sum |a||b|, here against the FP64 stack."""
    import torch
    from fastxc_amd.ops import XcPlan

    nspec = 73
    rng = np.random.default_rng(nsta * 100 + nstep)
    spec = (rng.standard_normal((nstep, nsta, nspec)) +
            1j * rng.standard_normal((nstep, nsta, nspec))).astype(np.complex64)
    a, b = np.nonzero(rng.random((nsta, nsta)) < 0.6)
    src = np.concatenate([[0], a, a[:5]]).astype(np.int32)
    rec = np.concatenate([[nsta - 1], b, b[:5]]).astype(np.int32)
    plan = XcPlan(nspec, nstep, 0.1, 20, "fp32")
    plan.set_pairs(nsta, src, rec)
    got = plan.cross_spectra(torch.from_numpy(spec).to(gpu)).cpu().numpy()
    z = spec.astype(np.complex128)
    want = (z[:, src].conj() * z[:, rec]).mean(axis=0)
    bound = (np.abs(z[:, src]) * np.abs(z[:, rec])).mean(axis=0) * (2 * nstep + 2) * 2.0 ** -24
    assert (np.abs(got - want) <= 2 * bound).all()


@pytest.mark.parametrize("nfft,H", [(40000, 1000), (72576, 0), (74088, 2047), (75000, 2500),
                                    (79380, 39689), (80000, 1)])
def test_lag_halves(gpu, nfft, H):
    """Lag transforms of two half-length transforms: the shortest and longest lengths that take
    them, odd and even halves, no lag beside zero to every lag, odd row pitch; and the one-window
    product form.  80000 is just beyond them and takes the four steps over memory.  fp32 transforms of 2^16 points round to about log2(n) 2^-24 relative, 1e-6."""
    import torch
    from fastxc_amd.ops import XcPlan

    nspec, dt, rows = nfft // 2 + 1, 0.05, 5
    rng = np.random.default_rng(nfft)
    X = (rng.standard_normal((rows, nspec)) + 1j * rng.standard_normal((rows, nspec))).astype(np.complex64)
    lag = np.arange(-H, H + 1) % nfft

    def want(x):
        return np.fft.irfft(x.astype(np.complex128), n=nfft, axis=-1)[:, lag] / np.float64(np.float32(dt))

    plan = XcPlan(nspec, 1, dt, H, "fp32")
    got = plan.lags(torch.from_numpy(X).to(gpu)).cpu().numpy()
    ref = want(X)
    assert np.linalg.norm(got - ref) <= 1e-6 * np.linalg.norm(ref)
    src, rec = np.array([0, 3, 2, 4]), np.array([1, 3, 0, 2])
    plan.set_pairs(rows, src, rec)
    got = plan.correlate(torch.from_numpy(X[None]).to(gpu)).cpu().numpy()
    Z = X.astype(np.complex128)
    ref = want(Z[src].conj() * Z[rec])
    assert np.linalg.norm(got - ref) <= 1e-6 * np.linalg.norm(ref)


def test_fp32_few_items_share_the_chip(gpu, monkeypatch):
    """One 32 x 32 station tile of the matrix form has one work item per 16 bins.  Its items go to as many compute
    units as there are items, so it takes well under the time of eight tiles (in runs of eight
    items per workgroup both took the same time)."""
    import torch
    from fastxc_amd.ops import XcPlan

    monkeypatch.setenv("FXC_XC_F32", "matrix")  # whose items these are
    nspec, nstep, nsta = 1876, 64, 320
    g = torch.Generator(device=gpu)
    g.manual_seed(3)
    spec = torch.randn((nstep, nsta, nspec), generator=g, device=gpu, dtype=torch.complex64)
    ms = []
    for ntile in (1, 8):
        rec = np.arange(32, 32 + 32 * ntile)
        plan = XcPlan(nspec, nstep, 1.0, 100, "fp32")
        plan.set_pairs(nsta, np.repeat(np.arange(32), len(rec)), np.tile(rec, 32))
        plan.correlate(spec)
        best = np.inf
        for _ in range(5):
            plan.set_timing(True)
            plan.correlate(spec)
            best = min(best, plan.get_timing()["contract_ms"])
        ms.append(best)
        plan.close()
    print(f"contraction of 1 and 8 tiles: {ms[0]:.4f} {ms[1]:.4f} ms")
    assert ms[0] < 0.7 * ms[1]


@pytest.mark.parametrize("form", ["vector", "matrix"])
@pytest.mark.parametrize("nsta,nstep,pairs", [(70, 1, "all"), (70, 2, "all"), (33, 5, "all"), (130, 7, "one"),
                                              (130, 3, "source"), (97, 13, "random"), (40, 100, "random")])
def test_fp32_both_forms(gpu, monkeypatch, form, nsta, nstep, pairs):
    """The FP32 contraction on the vector ALU and on the matrix instructions, for dense and sparse
    pair lists (duplicates, either order, one station with itself), a band, and row chunks, against
    the FP64 stack.  fp32 sums of 2 nstep products: relative error below 2 nstep 2^-24 of sum
    |a||b|."""
    import torch
    from fastxc_amd.ops import XcPlan

    monkeypatch.setenv("FXC_XC_F32", form)
    nspec = 201
    rng = np.random.default_rng(nsta * 1000 + nstep)
    spec = (rng.standard_normal((nstep, nsta, nspec)) +
            1j * rng.standard_normal((nstep, nsta, nspec))).astype(np.complex64)
    src, rec = {"all": np.triu_indices(nsta), "one": (np.array([nsta - 1]), np.array([3])),
                "source": (np.full(nsta, 37), np.arange(nsta)),
                "random": tuple(rng.integers(0, nsta, (2, 60)))}[pairs]
    src, rec = np.concatenate([src, src[:2]]), np.concatenate([rec, rec[:2]])
    z = spec.astype(np.complex128)
    want = (z[:, src].conj() * z[:, rec]).mean(axis=0)
    bound = (np.abs(z[:, src]) * np.abs(z[:, rec])).mean(axis=0) * (2 * nstep + 2) * 2.0 ** -24
    sd = torch.from_numpy(spec).to(gpu)
    for chunk, band in ((0, None), (17, None), (0, (70, 130))):
        plan = XcPlan(nspec, nstep, 0.1, 20, "fp32", chunk_rows=chunk)
        if band:
            plan.set_band(*band)
        plan.set_pairs(nsta, src, rec)
        got = plan.cross_spectra(sd).cpu().numpy()
        lo, hi = (band[0] // 16 * 16, (band[1] // 16 + 1) * 16) if band else (0, nspec)
        assert (np.abs(got - want) <= 2 * bound)[:, lo:hi].all()
        assert not got[:, :lo].any() and not got[:, hi:].any()
        plan.close()


def test_fp32_sparse_pairs_need_no_operand(gpu):
    """A few pairs of many stations are contracted from the spectra themselves: the call holds no
    transposed copy of them (whose cost is that of every station)."""
    import torch
    from fastxc_amd.ops import XcPlan

    nspec, nstep, nsta = 9262, 8, 200
    spec = torch.zeros((nstep, nsta, nspec), device=gpu, dtype=torch.complex64)
    plan = XcPlan(nspec, nstep, 0.2, 100, "fp32")
    plan.set_pairs(nsta, [3, 150], [190, 20])
    out = torch.empty((2, 201), device=gpu)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    plan.correlate(spec, out)
    torch.cuda.synchronize()
    held = free - torch.cuda.mem_get_info()[0]
    print(f"held {held} of {spec.numel() * 8} bytes of spectra")
    assert held < spec.numel() * 8 // 4


@pytest.mark.parametrize("grid", [8, 256])
@pytest.mark.parametrize("nstep", [1, 4, 8, 12, 16, 17, 20, 24, 28, 32, 36, 40, 41, 44, 48, 49, 52, 64])
def test_fp32_every_depth(gpu, monkeypatch, grid, nstep):
    """Every compiled depth of the FP32 matrix form (1 to 12 steps of 4 windows, and any depth
    beyond), with its sources kept over runs of tiles and exchanged between them (8 workgroups, whose
    runs are of 8 items) and with runs of one, tiles that list no pair of a receiver half or of a
    source half, and a last bin chunk that is not full.  Bound as in test_fp32_matrix_tiles."""
    import torch
    from fastxc_amd.ops import XcPlan

    monkeypatch.setenv("FXC_XC_F32", "matrix")
    monkeypatch.setenv("FXC_XC_MFMA_GRID", str(grid))
    nspec, nsta = 321, 110
    rng = np.random.default_rng(nstep)
    spec = (rng.standard_normal((nstep, nsta, nspec)) +
            1j * rng.standard_normal((nstep, nsta, nspec))).astype(np.complex64)
    src, rec = np.triu_indices(nsta, k=1)
    keep = ~((rec >= 48) & (rec < 64)) & ~((src >= 64) & (src < 80))
    src, rec = src[keep], rec[keep]
    plan = XcPlan(nspec, nstep, 0.1, 20, "fp32")
    plan.set_pairs(nsta, src, rec)
    got = plan.cross_spectra(torch.from_numpy(spec).to(gpu)).cpu().numpy()
    z = spec.astype(np.complex128)
    for lo in range(0, len(src), 1000):
        a, b = src[lo:lo + 1000], rec[lo:lo + 1000]
        want = (z[:, a].conj() * z[:, b]).mean(axis=0)
        bound = (np.abs(z[:, a]) * np.abs(z[:, b])).mean(axis=0) * (2 * nstep + 2) * 2.0 ** -24
        assert (np.abs(got[lo:lo + 1000] - want) <= 2 * bound).all()


@pytest.mark.parametrize("nfft", [72576, 72900, 73500, 74088, 75000])
def test_long_lags_keep_their_precision(gpu, nfft):
    """Lags of lengths beyond one workgroup (20 Hz windows with 25 to 110 s of lags): two half-length
    transforms of five or six passes round to 1.8 to 2.0e-7 of white spectra's lags with powers of at
    most three products of table values; powers chained from one value give 2.6 to 3.1e-7, the four
    steps they replace 1.7 to 2.7e-7."""
    import torch
    from fastxc_amd.ops import XcPlan

    H, dt = 2000, 0.05
    g = torch.Generator(device=gpu)
    g.manual_seed(nfft)
    X = torch.randn((48, nfft // 2 + 1), generator=g, device=gpu, dtype=torch.complex64)
    got = XcPlan(nfft // 2 + 1, 2, dt, H, "fp32").lags(X).double()
    lag = torch.arange(-H, H + 1, device=gpu) % nfft
    want = torch.fft.irfft(X.to(torch.complex128), n=nfft)[:, lag] / float(np.float32(dt))
    err = float(torch.linalg.vector_norm(got - want) / torch.linalg.vector_norm(want))
    print(f"nfft {nfft} rel_l2={err:.3e}")
    assert err < 2.3e-7


@pytest.mark.parametrize("nstep", [4, 24, 36, 47, 100])
def test_fp32_matrix_form_rounds_as_the_vector_form(gpu, monkeypatch, nstep):
    """The matrix instructions' sums are no further from 64 bits than the vector form's: a sum takes
    one rounding per window in both (two per window would be 1.2 to 1.4 times as far)."""
    import torch
    from fastxc_amd.ops import XcPlan

    nspec, nsta = 641, 48
    g = torch.Generator(device=gpu)
    g.manual_seed(nstep)
    spec = torch.randn((nstep, nsta, nspec), generator=g, device=gpu, dtype=torch.complex64)
    src, rec = _all_pairs(nsta)
    z = spec.to(torch.complex128)
    want = (z[:, src].conj() * z[:, rec]).mean(dim=0)
    err = {}
    for form in ("vector", "matrix"):
        monkeypatch.setenv("FXC_XC_F32", form)
        plan = XcPlan(nspec, nstep, 0.1, 20, "fp32")
        plan.set_pairs(nsta, src, rec)
        d = plan.cross_spectra(spec).to(torch.complex128) - want
        err[form] = float(torch.linalg.vector_norm(d) / torch.linalg.vector_norm(want))
        plan.close()
    print(f"{nstep} windows: {err}")
    assert err["matrix"] <= 1.04 * err["vector"]
