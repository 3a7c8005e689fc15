"""Isolated samples far above the signal's noise (a telemetry glitch, the last
sample of a loud stretch) and runs of infinities: windows beside them keep the
accuracy they have without them.  Correlations against the FP64 two-pass
oracle."""
import numpy as np
import pytest

import oracle as O
from mflib_amd import capi

pytestmark = pytest.mark.gpu


def _rows(tpls, x, dtype, nfft=0, variant=0):
    h = capi.Handle(dtype, "batched")
    h.set_templates(tpls)
    h.set_batch_layout([x.size], [0] * len(tpls), [0] * len(tpls), 1)
    if nfft:
        h.set_fft_length(nfft)
    if variant:
        h.set_kernel_variant(variant)
    h.initialize()
    h.set_signal(0, x)
    h.apply()
    out = [h.rho(r) for r in range(len(tpls))]
    stats = h.window_stats()
    h.close()
    return out, stats


def _templates(rng, lengths):
    return [rng.standard_normal(L) * np.hanning(L) for L in lengths]


def _spiked(rng, tpls, at, amp, n):
    """Unit noise, a spike of `amp` at every position of `at`, and right after
    each a copy of one template four times the noise (|rho| about 0.9, where an
    error of the window's norm shows in full)."""
    x = rng.standard_normal(n)
    for k, p in enumerate(at):
        t = tpls[k % len(tpls)]
        x[p + 1 + k % 5:][:t.size] += 4.0 * t
    x[at] = amp * np.where(np.arange(len(at)) % 2, -0.9, 1.0)
    return x


@pytest.mark.parametrize("amp", [3.0e4, 3.0e5, 1.0e6, 1.0e7])
@pytest.mark.parametrize("variant", [3, 4])
@pytest.mark.parametrize("lengths", [(200,) * 24, tuple(range(230, 257)), (60,) * 20])
def test_time_domain_windows_beside_a_spike(variant, lengths, amp):
    """Spikes at every position within a tile of 16 outputs: the windows after
    one are quiet beside their block and are recomputed, whole tiles of them."""
    rng = np.random.default_rng(61)
    tpls = _templates(rng, lengths)
    n = 40_000
    at = 1_000 + 1_201 * np.arange(32)  # 1201 = 1 modulo 16
    x = _spiked(rng, tpls, at, amp, n).astype(np.float32)
    out, _ = _rows(tpls, x, np.float32, variant=variant)
    for r, t in enumerate(tpls):
        ref = O.pearson(t, x)[:out[r].size]
        err = np.abs(out[r].astype(np.float64) - ref)
        assert err.max() < 1e-5, (r, int(err.argmax()), err.max())


@pytest.mark.parametrize("nfft", [1024, 2048])
@pytest.mark.parametrize("lengths", [(300,), (300,) * 5, (300, 250, 120)])
def test_fp64_windows_far_from_a_spike(nfft, lengths):
    """Spikes at multiples of 1/64 of a block and as the last sample of a short
    last block.  The anchor moves by amp / nfft, and window sums about it lose
    (amp / nfft)^2 2^-53 of the noise's: under 1e-12 with the other roundings.
    The windows that a spike has left fewer than 24 outputs before are not
    compared here (a sliding sum keeps 2^-53 amp^2 of it over a run of outputs)."""
    rng = np.random.default_rng(67)
    tpls = _templates(rng, lengths)
    nb = max(lengths)
    step = (nfft - nb + 1) & ~1
    for amp in (1.0e4, 3.0e4):
        n = 4 * step + nfft // 8 + nb
        at = np.array([0, nfft // 2, step + 5 * nfft // 64, 3 * step + 40 * nfft // 64, n - 1])
        x = rng.standard_normal(n)
        x[at] = amp
        out, _ = _rows(tpls, x, np.float64, nfft=nfft, variant=2)
        far = np.ones(out[0].size, dtype=bool)
        for p in at:
            far[p + 1:p + 25] = False
        for r, t in enumerate(tpls):
            ref = O.pearson(t, x)[:out[r].size]
            err = np.abs(out[r] - ref)[far]
            assert err.max() < 1e-12, (amp, r, err.max())


@pytest.mark.parametrize("rows", [1, 5])
def test_server_runs_of_infinities(rows):
    """A run of equal infinities has no finite mean, so its windows are NaN, as
    are all that touch it, for rows that share a scale and for a row alone; a
    run of equal finite samples stays 0 and the other windows exact."""
    rng = np.random.default_rng(71)
    tpls = _templates(rng, (100,) * rows)
    n = 3_000
    x = rng.standard_normal(n).astype(np.float32)
    x[700:1_000] = np.inf
    x[1_600:1_900] = np.float32(2.5)
    srv = capi.Server(np.float32, budget_bytes=1 << 28, max_batch=4, max_inflight=1)
    ids = srv.add_templates(tpls)
    rid = srv.submit([x], ids)
    srv.wait(rid)
    clean = np.where(np.isinf(x), np.float32(0), x)
    for r, t in enumerate(tpls):
        row = srv.rho(rid, r, 0)
        i = np.arange(row.size)
        touched = (i + 99 >= 700) & (i < 1_000)
        assert np.isnan(row[touched]).all(), np.flatnonzero(~np.isnan(row) & touched)
        assert not row[1_600:1_801].any()
        ref = O.pearson(t, clean)[:row.size]
        assert np.abs(row[~touched] - ref[~touched]).max() < 1e-5
    srv.release(rid)
    srv.close()


@pytest.mark.parametrize("variant", [3, 4])
@pytest.mark.parametrize("rows", [2, 17, 18, 40])
def test_time_domain_most_tiles_noisy(variant, rows):
    """A level that steps by 60 times the noise every 400 samples puts the noise
    bound of the windows between steps above the tolerance, so most tiles of two
    rows or more are recorded for recomputation, the same way in every pass."""
    rng = np.random.default_rng(73)
    tpls = _templates(rng, rng.integers(100, 129, size=rows))
    n = 6_000
    x = (rng.standard_normal(n) + 60.0 * (np.arange(n) // 400 % 2) + 500.0).astype(np.float32)
    h = capi.Handle(np.float32, "batched")
    h.set_templates(tpls)
    h.set_batch_layout([n], [0] * rows, [0] * rows, 1)
    h.set_kernel_variant(variant)
    h.initialize()
    h.set_signal(0, x)
    h.apply()
    out = [h.rho(r) for r in range(rows)]
    ws = h.window_stats()
    assert ws["flagged"] > 0.5 * ws["windows"] and ws["full"] == 0, ws
    for r, t in enumerate(tpls):
        ref = O.pearson(t, x)[:out[r].size]
        assert np.abs(out[r].astype(np.float64) - ref).max() < 1e-5, r
    h.apply()
    for r in range(rows):
        assert np.array_equal(h.rho(r), out[r]), r
    h.close()


@pytest.mark.parametrize("variant", [3, 4])
@pytest.mark.parametrize("lt", [128, 256])
@pytest.mark.parametrize("bad", [np.nan, np.inf, 1.0e9])
def test_sample_just_past_a_tile(variant, lt, bad):
    """The recorded tiles at the end of an item of 512 outputs, whose windows end
    just before a bad sample that the item does not read."""
    rng = np.random.default_rng(79)
    tpls = _templates(rng, (lt,) * 16)
    n, end = 3_000, 512 + lt  # the item's samples are [0, 512 + lt)
    x = (rng.standard_normal(n) + 60.0 * (np.arange(n) >= 400)).astype(np.float32)
    x[end:end + 3] = bad
    out, _ = _rows(tpls, x, np.float32, variant=variant)
    i = np.arange(out[0].size)
    touched = (i + lt > end) & (i < end + 3)
    assert not touched[:512].any() and touched[513]
    if np.isfinite(bad):
        touched[:] = False
    clean = np.where(np.isfinite(x), x, np.float32(0))
    for r, t in enumerate(tpls):
        assert not np.isnan(bad) or np.isnan(out[r][touched]).all()
        ref = O.pearson(t, clean)[:out[r].size]
        err = np.abs(out[r].astype(np.float64) - ref)[~touched]
        assert err.max() < 1e-5, (r, np.flatnonzero(~touched)[err.argmax()], err.max())


@pytest.mark.parametrize("variant,lt,nfft", [(3, 200, 0), (4, 200, 0), (2, 300, 2048), (2, 300, 1024)])
def test_last_sample_of_a_short_block_flags_no_block(variant, lt, nfft):
    """A last sample of 200 times the noise in a short last block is one sample
    of its anchor at most, and no reason to recompute the block's windows."""
    rng = np.random.default_rng(83)
    tpls = _templates(rng, (lt,) * 5)
    step = ((nfft - lt + 1) & ~1) if nfft else 512
    n = 5 * step + (nfft // 8 if nfft else 64) + lt
    x = rng.standard_normal(n).astype(np.float32)
    x[-1] = 200.0
    out, ws = _rows(tpls, x, np.float32, nfft=nfft, variant=variant)
    assert ws["flagged"] == 0, ws
    for r, t in enumerate(tpls):
        assert np.abs(out[r].astype(np.float64) - O.pearson(t, x)[:out[r].size]).max() < 1e-5, r


@pytest.mark.parametrize("variant,lt", [(3, 200), (4, 200), (3, 60), (4, 100)])
def test_one_outlier_flags_no_item(variant, lt):
    """A spike of 200 times the noise on a sample that a time-domain item takes
    its anchor from is no reason to recompute the item's windows."""
    rng = np.random.default_rng(89)
    tpls = _templates(rng, (lt,) * 5)
    kt = 256 if lt > 128 else 128 if lt > 64 else 64
    n = 512 * 41 + lt
    x = rng.standard_normal(n).astype(np.float32)
    x[2_048 * np.arange(10) + 20 * (512 + kt) // 64] = 200.0
    out, ws = _rows(tpls, x, np.float32, variant=variant)
    assert ws["flagged"] == 0, ws
    for r, t in enumerate(tpls):
        assert np.abs(out[r].astype(np.float64) - O.pearson(t, x)[:out[r].size]).max() < 1e-5, r


@pytest.mark.parametrize("variant", [3, 4])
def test_time_domain_one_sample_templates(variant):
    """A window of one sample is constant, so 0, also where the sample is a NaN
    or an infinity."""
    rng = np.random.default_rng(97)
    x = rng.standard_normal(1_300).astype(np.float32)
    x[[3, 600]] = np.nan, np.inf
    out, _ = _rows([np.array([1.0]), np.array([1.0, -1.0])], x, np.float32, variant=variant)
    assert not out[0].any()
    assert np.isnan(out[1][2:4]).all()
