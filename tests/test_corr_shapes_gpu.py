"""The correlation kernels at the sizes where their block shapes can go wrong:
every FFT size and kernel, one row and rows of one and of many lengths, row
ends around a block's end and around the groups of outputs the epilogue
takes, exactly constant stretches, a NaN sample, and the time-domain tiles.
Correlations against the FP64 two-pass oracle; constant windows are 0."""
import numpy as np
import pytest

import oracle as O
from mflib_amd import capi

pytestmark = pytest.mark.gpu

# unflagged FP32 windows stay below 4e-6 and flagged ones are exact, inside the
# 1e-5 contract; FP64 windows within 1e-11
TOL = {np.float32: 1e-5, np.float64: 1e-11}


def _rows(lengths, n, dtype, nfft=0, variant=0, x=None, seed=5):
    rng = np.random.default_rng(seed)
    tpls = [rng.standard_normal(L) * np.hanning(L) for L in lengths]
    if x is None:
        x = (rng.standard_normal(n) + 30.0).astype(dtype)
    h = capi.Handle(dtype, "batched")
    h.set_templates(tpls)
    h.set_batch_layout([n], [0] * len(tpls), [0] * len(tpls), 1)
    if nfft:
        h.set_fft_length(nfft)
    if variant:
        h.set_kernel_variant(variant)
    h.initialize()
    h.set_signal(0, x)
    h.apply()
    out = [h.rho(r) for r in range(len(tpls))]
    ref = [O.pearson(t, x)[:n - max(lengths) + 1] for t in tpls]
    h.close()
    return x, out, ref


def _check(out, ref, tol, ctx):
    for r, (a, b) in enumerate(zip(out, ref)):
        assert a.shape == b.shape and np.abs(a.astype(np.float64) - b).max() < tol, (ctx, r)


SHAPES = [(np.float32, 1024, 2), (np.float32, 2048, 2), (np.float32, 4096, 2), (np.float32, 1024, 1),
          (np.float32, 8192, 1), (np.float64, 1024, 2), (np.float64, 2048, 2), (np.float64, 4096, 1)]


@pytest.mark.parametrize("dtype,nfft,variant", SHAPES)
@pytest.mark.parametrize("lengths", [(250,), (250,) * 5, (250, 249, 100), (250,) * 4 + (77, 31)])
def test_rows_around_block_ends(dtype, nfft, variant, lengths):
    nb = max(lengths)
    block = (nfft - nb + 1) & ~1
    # one output, a group of 64 or 128 outputs and its neighbours, both halves of
    # a block, a whole block, one more, and a ragged last block
    for outs in (1, 63, 64, 129, nfft // 2 - 1, nfft // 2 + 1, block - 1, block, block + 1, 2 * block + 77):
        n = outs + nb - 1
        if n <= 1:
            continue
        _, out, ref = _rows(lengths, n, dtype, nfft, variant)
        _check(out, ref, TOL[dtype], (nfft, variant, lengths, outs))


@pytest.mark.parametrize("dtype,nfft,variant", SHAPES[:3] + SHAPES[5:7])
@pytest.mark.parametrize("lengths", [(200,), (200,) * 5, (200, 150, 120)])
def test_constant_stretches_and_a_nan(dtype, nfft, variant, lengths):
    """Windows inside a constant stretch are 0, also where it crosses a
    block's end: exactly in FP32; in FP64, whose two-pass mean of Lt equal
    samples may be off by an ulp of 1e3 (1.2e-13), within that times the taps'
    rounded sum (about 1e-16) over the norm's floor 2.2e-16, below 1e-12.
    Windows that touch a NaN are NaN and no others."""
    rng = np.random.default_rng(11)
    n = 3 * nfft
    x = (rng.standard_normal(n) + 1.0e3).astype(dtype)
    x[300:700] = x[300]
    x[nfft - 90:nfft + 700] = dtype(1000.25)
    _, out, ref = _rows(lengths, n, dtype, nfft, variant, x=x)
    _check(out, ref, TOL[dtype], (nfft, lengths))
    for L, row in zip(lengths, out):
        flat = np.concatenate([row[300:701 - L], row[nfft - 90:nfft + 701 - L]])
        assert np.abs(flat).max() <= (0.0 if dtype == np.float32 else 1e-12)
    x = x.copy()
    at = 2 * nfft + 17
    x[at] = np.nan
    clean = x.copy()
    clean[at] = 0
    _, out, _ = _rows(lengths, n, dtype, nfft, variant, x=x)
    for t, (L, row) in enumerate(zip(lengths, out)):
        i = np.arange(row.size)
        touched = (i <= at) & (at < i + L)
        assert np.isnan(row[touched]).all() and np.isfinite(row[~touched]).all(), (nfft, lengths, t)
        want = ref[t].copy()
        far = ~touched
        assert np.abs(row[far] - want[far]).max() < TOL[dtype]


@pytest.mark.parametrize("variant", [3, 4])
@pytest.mark.parametrize("lengths", [(64,), (40,) * 16 + (33,), tuple(range(100, 250)), (256,) * 200])
def test_time_domain_items_and_dense_tiles(variant, lengths):
    """Row counts around the groups of 16 and the items' even split, outputs
    around the tiles of 16 and items of 512; a loud burst beside quiet noise
    flags whole tiles, a gap gives constant windows."""
    rng = np.random.default_rng(3)
    nb = max(lengths)
    for outs in (1, 17, 511, 513, 1_024 + 15):
        n = outs + nb - 1
        x = (rng.standard_normal(n) + 50.0).astype(np.float32)
        if outs > 500:
            x[outs // 2:outs // 2 + 9] += np.float32(3.0e4)
        _, out, ref = _rows(lengths, n, np.float32, 0, variant, x=x)
        _check(out, ref, 1e-5, (variant, len(lengths), outs))
    n = 2_500
    x = (rng.standard_normal(n) + 1.0e4).astype(np.float32)
    x[700:1_900] = np.float32(10_031.0)
    _, out, ref = _rows(lengths, n, np.float32, 0, variant, x=x)
    _check(out, ref, 1e-5, (variant, len(lengths), "gap"))
    for L, row in zip(lengths, out):
        assert not row[700:1_901 - L].any()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_device_signal_copies_and_dead_traces(dtype):
    """mf_set_signal_device at lengths and alignments around its 16-byte
    vectors, and its dead-trace rule |min| == |max| when flags change."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(9)
    for n in (65, 127, 4_099, 70_001):
        buf = torch.from_numpy(rng.standard_normal(n + 3).astype(dtype)).cuda()
        torch.cuda.synchronize()
        t = rng.standard_normal(40)
        h = capi.Handle(dtype, "single")
        h.set_templates([t])
        h.set_signal_size(n)
        h.initialize()
        for off in range(3):
            x = buf[off:off + n]
            h.set_signal_device(0, x.data_ptr(), n)
            assert np.array_equal(h.get_signal(0, n), x.cpu().numpy())
            h.apply()
            assert np.abs(h.rho(0) - O.pearson(t, x.cpu().numpy())[:n - 39]).max() < TOL[dtype]
        dead = torch.full((n,), -2.5, dtype=buf.dtype, device="cuda")
        dead[n // 2:] = 2.5
        torch.cuda.synchronize()
        h.set_signal_device(0, dead.data_ptr(), n)
        h.apply()
        assert not h.rho(0).any()
        h.set_signal_device(0, buf.data_ptr(), n)
        h.apply()
        assert h.rho(0).any()
        h.close()


@pytest.mark.parametrize("alpha", [1, 3, 51, 511, 512])
def test_lanczos_table_against_a_sine_per_tap(alpha):
    """Windows on either side of the table's size, and the interpolant's own
    maximum against the oracle's profile (1e-12 of it)."""
    rng = np.random.default_rng(21)
    n, L = 4_000, 60
    x = rng.standard_normal(n)
    t = rng.standard_normal(L)
    h = capi.Handle(np.float64, "single")
    h.set_templates([t])
    h.set_signal_size(n)
    h.initialize()
    h.set_signal(0, x)
    h.apply()
    row = h.rho(0)
    peaks = [0, 1, 2, 500, 1_777, row.size - 2, row.size - 1]
    points = 40
    got = h.detection_products(peaks, [0] * len(peaks), [1.0], interpolation=capi.INTERP_LANCZOS,
                               lanczos_alpha=alpha, lanczos_points=points)["shift"]
    for k, p in enumerate(peaks):
        ref, prof = O.lanczos_shift(row, p, 1.0, False, alpha, points)
        top = prof.max()
        j = int(round((got[k] + 0.5) * points)) - 1
        assert prof[j] >= top - 1e-12 * max(1.0, abs(top)), (alpha, p)
        if np.sort(prof)[-2] < top - 1e-9:
            assert got[k] == pytest.approx(ref, abs=1e-12), (alpha, p)
    h.close()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("slen", [511, 512, 513, 1025, 383 * 2048, 383 * 2048 + 1])
def test_stacks_on_either_side_of_the_chunk_rule(dtype, slen):
    """Stacks cut into chunks of 512 outputs (383 chunks of 2048 and fewer) and
    of 2048: both entry points equal the oracle's stack bit for bit, and every
    local maximum is found, the chunk edges' included."""
    rng = np.random.default_rng(slen)
    C, L = 2, 40
    shifts, weights = [0, 5], [0.625, 0.375]
    n = L - 1 + slen + max(shifts)
    h = capi.Handle(dtype, "batched")
    h.set_templates([rng.standard_normal(L) for _ in range(C)], shifts=shifts, weights=weights)
    h.set_batch_layout([n] * C, list(range(C)), [0] * C, 1)
    h.initialize()
    for c in range(C):
        h.set_signal(c, rng.standard_normal(n).astype(dtype))
    h.apply()
    ref = O.shift_and_stack(np.stack([h.rho(r) for r in range(C)]), shifts, weights)
    assert ref.size == slen
    assert np.array_equal(h.detect(0.0, 0)[0], O.peak_finder(ref, 0.0, 0))
    assert np.array_equal(h.shift_and_stack(0), ref)
    h.close()


def test_device_signal_of_almost_2_31_samples():
    """A signal handed over in device memory, so long that its length plus a
    block's share leaves the range of int."""
    torch = pytest.importorskip("torch")
    n = 2 ** 31 - 1_000
    x = torch.zeros(n, dtype=torch.float32, device="cuda")
    x[-3:] = torch.tensor([1.0, -2.0, 0.5], device="cuda")
    torch.cuda.synchronize()
    h = capi.Handle(np.float32, "single")
    h.set_templates([np.hanning(60)])
    h.set_signal_size(n)
    h.initialize()
    h.set_signal_device(0, x.data_ptr(), n)
    got = h.get_signal(0, n)[-4:]
    assert np.array_equal(got, np.array([0.0, 1.0, -2.0, 0.5], dtype=np.float32))
    h.close()


def test_plans_of_few_and_of_many_blocks():
    """FP64 rows of 400 to 500 samples: blocks of 2048 where they fill the
    device, blocks of 1024 where fewer blocks than compute units are all the
    work there is (a launch then takes one block's time)."""
    rng = np.random.default_rng(25)
    tpls = [rng.standard_normal(L) for L in range(400, 500, 5)]
    for n, nfft in ((100_000, 1024), (8_000_000, 2048)):
        h = capi.Handle(np.float64, "batched")
        h.set_templates(tpls)
        h.set_batch_layout([n], [0] * len(tpls), [0] * len(tpls), 1)
        h.initialize()
        assert {h.plan(r)[0] for r in range(len(tpls))} == {nfft}, n
        h.close()


@pytest.mark.parametrize("rows", [192, 193])
def test_time_domain_rows_on_either_side_of_the_item_split(rows):
    """192 rows are one item, 193 two of 112 and 81."""
    rng = np.random.default_rng(27)
    lengths = tuple(int(v) for v in rng.integers(20, 129, size=rows))
    for variant in (3, 4):
        _, out, ref = _rows(lengths, 1_500, np.float32, 0, variant)
        _check(out, ref, 1e-5, (variant, rows))
