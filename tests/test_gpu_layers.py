"""The layers' kernels at the edges of their tiles and launches, against the
CPU oracle (1e-12 of the largest value, as in the parity tests)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _tf(gpu, orc, n, seed):
    orc.seed(seed)
    tf = orc.transform_draw(n)
    return tf, gpu.transform_make(n, int(tf[0]), int(tf[1]), int(tf[2]))


@pytest.mark.parametrize("n,bins,m", [(4099, 3, 1), (1 << 12, 4095, 64), (1 << 16, 101, 256),
                                      (1 << 18, 2001, 257), (1000003, 501, 1025)])
def test_bin_in_freq_edges(gpu, orc, n, bins, m):
    """One thread per (mode, bit): mode counts at and beyond a workgroup,
    bits from 1 (n / B < 2) up; calls in a row on one plan, one of them with
    zero coefficients (no grid) and one of tiny ones, share its scratch."""
    rng = np.random.default_rng(n + m)
    bits = orc.num_bits(n, bins)
    tf_o, tf = _tf(gpu, orc, n, m)
    keys = rng.choice(n, m, replace=False).astype(np.int64)
    plan = gpu.Plan(n, bins, 1e-6, bits)
    for scale in (1.0, 0.0, 1e-30, 1.0):
        coefs = scale * (rng.standard_normal(m) + 1j * rng.standard_normal(m))
        base = scale * (rng.standard_normal((1 + 2 * bits, bins)) + 1j)
        ref, got = base.copy(), base.copy()
        orc.bin_in_freq(keys.astype(np.int32), coefs, n, bins, 1e-6, bits, tf_o, 77, ref, version=1)
        plan.bin_in_freq(keys, coefs, tf, 77, got)
        assert np.abs(got - ref).max() <= TOL * np.abs(ref).max()


# the second: more modes than the exponent pass has threads, more sums too
@pytest.mark.parametrize("n,bins,m", [(1 << 14, 101, 50), (1 << 18, 4095, 140000)])
def test_bin_in_freq_first_call_on_a_stream(gpu, orc, n, bins, m):
    """A fresh plan's first BinInFreq on a non-blocking stream."""
    rng = np.random.default_rng(m)
    bits = orc.num_bits(n, bins)
    tf_o, tf = _tf(gpu, orc, n, m)
    keys = rng.choice(n, m, replace=False).astype(np.int64)
    coefs = rng.standard_normal(m) + 1j * rng.standard_normal(m)
    base = rng.standard_normal((1 + 2 * bits, bins)) + 1j
    ref = base.copy()
    orc.bin_in_freq(keys.astype(np.int32), coefs, n, bins, 1e-6, bits, tf_o, 77, ref, version=1)
    stream = C.c_void_p()
    assert gpu.lib().mpsft_stream_create(C.byref(stream)) == 0
    kd, cd, od = (gpu.DeviceArray.from_numpy(v) for v in (keys, coefs, base))
    plan = gpu.Plan(n, bins, 1e-6, bits)
    plan.bin_in_freq_dev(kd, cd, m, tf, 77, od, stream)
    assert gpu.lib().mpsft_stream_synchronize(stream) == 0
    got = od.to_numpy(np.complex128, base.shape)
    assert np.abs(got - ref).max() <= TOL * np.abs(ref).max()
    assert gpu.lib().mpsft_stream_destroy(stream) == 0


@pytest.mark.parametrize("special", [np.inf, np.nan, 1.3e308 * (1 + 1j)])
def test_bin_in_freq_beyond_the_finite(gpu, orc, special):
    """A coefficient that is not finite, or whose modulus is not: its own bins
    are as the oracle's (finite or not), and the others' sums are right."""
    n, bins, m = 1 << 14, 301, 40
    rng = np.random.default_rng(3)
    bits = orc.num_bits(n, bins)
    tf_o, tf = _tf(gpu, orc, n, 21)
    keys = rng.choice(n, m, replace=False).astype(np.int64)
    coefs = rng.standard_normal(m) + 1j * rng.standard_normal(m)
    # the mode nearest a bin's centre, where the window is 1
    k1 = (int(tf_o[0]) * keys + int(tf_o[1])) % n
    at = int(np.argmin(np.abs((k1 * bins / n) % 1 - 0.5)))
    coefs[at] = special
    base = rng.standard_normal((1 + 2 * bits, bins)) + 1j
    ref, got = base.copy(), base.copy()
    orc.bin_in_freq(keys.astype(np.int32), coefs, n, bins, 1e-6, bits, tf_o, 77, ref, version=1)
    gpu.Plan(n, bins, 1e-6, bits).bin_in_freq(keys, coefs, tf, 77, got)
    own = np.arange(bins) == k1[at] * bins // n
    # beside a term of 2^1025 the sums resolve 2^-94 of it
    tol = TOL * np.abs(ref[:, ~own]).max() if not np.isfinite(special) else 2.0 ** (1025 - 94) * m
    assert np.abs(got[:, ~own] - ref[:, ~own]).max() <= tol
    a, b = (np.concatenate([v[:, own].real, v[:, own].imag]) for v in (got, ref))
    # on the edge of the range the oracle's products may pass it where ours do not
    assert (np.isfinite(a) == np.isfinite(b)).mean() >= 0.9
    both = np.isfinite(a) & np.isfinite(b)
    assert (np.abs(a[both] / 1e308 - b[both] / 1e308) <= TOL).all()
    assert both.any() == np.isfinite(special)


def test_iterate_after_overflow_changes_nothing(gpu):
    """A map that overflowed its capacity stays as it is: the one-launch
    parameters of Iterate carry the stop to the later kernels."""
    from mpsft_amd.signals import make_signal
    n, k = 1 << 14, 40
    x, _ = make_signal(n, k, 1e-6, seed=3)
    s = gpu.Solver(n, gpu.solve_options(k, 1e-6), capacity=4)
    opt = gpu.iterate_options(101, trials=1, bin_threshold=3e-7, window_threshold=0.1,
                              sv_threshold=1e-7)
    xd = s.upload(x)
    for rep in range(2):
        tf = gpu.transform_make(n, 2 * rep + 5, 1, 2)
        with pytest.raises(gpu.MpsftError) as e:
            s.iterate(xd, opt, tf, [7])
        assert e.value.status == 6
        got = s.modes_dict()
        assert len(got) == 4 and (rep == 0 or got == first)
        first = got


@pytest.mark.parametrize("n,ks,precision,trials", [
    # first bins 2 k + 1 on both sides of the sorted order's 256; ragged last
    # tiles (B mod 8 = 1 .. 7) and wide ones (8 residues); three trials
    (1 << 20, (127, 128), "FP64", 1), (1 << 21, (600, 303, 140), "MIXED", 1),
    (1 << 21, (150, 130, 129, 131), "MIXED", 3), (1 << 20, (500, 451), "FP64", 3)])
def test_batch_sorted_tiles_match_single(gpu, n, ks, precision, trials):
    """Signals of 16 MB and more take the sorted gather order in a batch
    (and XCD order); a signal alone takes neither.  Same decisions, and
    coefficients to rounding (the sums are split differently)."""
    from mpsft_amd.signals import make_signal, quantization_sigma
    prec = gpu.MPSFT_FP64 if precision == "FP64" else gpu.MPSFT_MIXED
    xs, opts = [], []
    for i, k in enumerate(ks):
        x, _ = make_signal(n, k, 1e-6, seed=50 + i)
        sig = 1e-6
        if precision == "MIXED":
            x64 = x.astype(np.complex64)
            sig = float(np.hypot(sig, quantization_sigma(x, x64)))
            x = x64
        xs.append(x)
        opts.append(gpu.solve_options(k, sig, trials=trials))
    seeds = [9 + i for i in range(len(ks))]
    batch = gpu.Batch([n] * len(ks), opts, prec)
    iters, status = batch.solve(batch.upload(xs), seeds)
    assert all(v == 0 for v in status)
    for i, x in enumerate(xs):
        s = gpu.Solver(n, opts[i], prec)
        assert s.solve(s.upload(x), seeds[i]) == iters[i]
        want, got = s.modes_dict(), batch.modes_dict(i)
        assert set(got) == set(want)
        top = max(abs(v) for v in want.values())
        for key, v in want.items():
            assert abs(got[key] - v) <= TOL * max(abs(v), 1e-2 * top)


def test_batch_sorted_tiles_of_every_width(gpu):
    """Autotuning solves sorted signals with tiles of 1, 2, 4 and 8 residues; the
    width it leaves gives the modes that the default gave."""
    from mpsft_amd.signals import make_signal
    n, ks = 1 << 20, (150, 130)
    xs = [make_signal(n, k, 1e-6, seed=80 + k)[0] for k in ks]
    batch = gpu.Batch([n] * 2, [gpu.solve_options(k, 1e-6) for k in ks])
    xd = batch.upload(xs)
    iters, status = batch.solve(xd, [3, 4])
    want = [batch.modes_dict(i) for i in range(2)]
    assert status == [0, 0] and batch.autotune(xd, [3, 4]) in (0, 1, 2, 4, 8)
    assert batch.solve(xd, [3, 4]) == (iters, status)
    for i, m in enumerate(want):
        got = batch.modes_dict(i)
        assert set(got) == set(m)
        assert max(abs(got[q] - v) for q, v in m.items()) <= TOL


@pytest.mark.parametrize("bins", [1, 3, 125, 127, 129, 131, 253, 255, 257, 511, 513])
def test_bin_in_time_dft_paths(gpu, orc, bins):
    """The bin DFT's forms and their edges: direct with one (B <= 127) or two
    (B <= 255) outputs per thread, radix-4 passes (B <= 511), Stockham."""
    n = 1 << 14
    rng = np.random.default_rng(bins)
    x = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    bits = orc.num_bits(n, bins)
    tf_o, tf = _tf(gpu, orc, n, bins)
    ref = orc.bin_in_time(x, bins, 1e-6, bits, tf_o, 4321, version=0)
    got = gpu.Plan(n, bins, 1e-6, bits).bin_in_time(x, tf, 4321)
    for r in range(ref.shape[0]):
        assert np.abs(got[r] - ref[r]).max() <= TOL * np.abs(ref[r]).max(), r


@pytest.mark.parametrize("k", [40, 1100, 1300])
def test_solve_many_modes_at_min_bins(gpu, orc, k):
    """Late iterations (B = 101) with more modes than a bin-FFT workgroup
    prefetches terms of (4 x 256): S = 1100, 1300, and few."""
    from mpsft_amd.signals import make_signal
    n = 1 << 18
    x, _ = make_signal(n, k, 1e-6, seed=k)
    s = gpu.Solver(n, gpu.solve_options(k, 1e-6))
    s.solve(s.upload(x), 5)
    orc.seed(5)
    mm, _, _ = orc.demo1_run(x, k, 1e-6)
    want, got = mm.to_dict(), s.modes_dict()
    assert set(got) == set(want)
    assert max(abs(got[q] - v) for q, v in want.items()) <= 1e-11


def test_mode_counts_follow_every_call(gpu):
    """The host keeps the map's size between calls: it is right after solves,
    Iterate, modes_set, a replay, and for a batch's signals."""
    from mpsft_amd.signals import make_signal
    n, k = 1 << 14, 30
    xs = [make_signal(n, k, 1e-6, seed=s)[0] for s in (1, 2)]
    s = gpu.Solver(n, gpu.solve_options(k, 1e-6))
    s.set_record(True)
    xd = [s.upload(x) for x in xs]
    maps = []
    for x in xd + xd:
        s.solve(x, 4)
        maps.append(s.modes_dict())
    assert [len(m) for m in maps[:2]] == [len(m) for m in maps[2:]]
    assert maps[0] == maps[2] and maps[1] == maps[3]
    s.replay(xd[1])
    assert set(s.modes_dict()) == set(maps[1])
    some = dict(list(maps[0].items())[:7])
    s.set_modes(some)
    assert s.modes_dict() == some
    opt = gpu.iterate_options(101, trials=1, bin_threshold=3e-7, window_threshold=0.1,
                              sv_threshold=1e-7)
    assert s.iterate(xd[0], opt, gpu.transform_make(n, 5, 1, 2), [3])
    assert len(s.modes_dict()) > 7
    s.set_modes({})
    assert s.modes_dict() == {}
    b = gpu.Batch([n, n], [s.opt, s.opt])
    for seeds in ([4, 4], [5, 5], [4, 4]):
        b.solve(xd, seeds)
        sizes = [len(b.modes_dict(i)) for i in range(2)]
    assert sizes == [len(maps[0]), len(maps[1])]


def test_replay_with_another_tile_width(gpu):
    """A tile width set between a recorded solve and its replay."""
    from mpsft_amd.signals import make_signal
    n, k = 1 << 16, 60
    s = gpu.Solver(n, gpu.solve_options(k, 1e-6))
    s.set_record(True)
    xd = s.upload(make_signal(n, k, 1e-6, seed=3)[0])
    s.solve(xd, 4)
    want = s.modes_dict()
    for residues in (8, 1, 2):
        s.set_tile_residues(residues)
        s.replay(xd)
        got = s.modes_dict()
        assert set(got) == set(want)
        assert max(abs(got[q] - v) for q, v in want.items()) <= TOL


def test_modes_after_the_stream_ends(gpu):
    """A solve's stream may be destroyed once the solve has returned."""
    from mpsft_amd.signals import make_signal
    n, k = 1 << 16, 60
    s = gpu.Solver(n, gpu.solve_options(k, 1e-6))
    xd = s.upload(make_signal(n, k, 1e-6, seed=3)[0])
    s.solve(xd, 4)
    want = s.modes_dict()
    for _ in range(3):
        stream = C.c_void_p()
        assert gpu.lib().mpsft_stream_create(C.byref(stream)) == 0
        s.solve(xd, 4, stream=stream)
        assert gpu.lib().mpsft_stream_destroy(stream) == 0
        assert s.modes_dict() == want
    s.solve(xd, 4)
    assert s.modes_dict() == want


@pytest.mark.parametrize("n,k,min_bins,precision", [
    (1 << 16, 50, 101, 0),  # 2^(bits-1) B + f B below n: offsets have one positive lag
    (1 << 16, 50, 127, 0),  # above n: offsets below f B have two
    (1 << 16, 50, 129, 1),
    (1 << 9, 3, 7, 0),      # fewer samples than a workgroup's threads x 4
])
def test_adjoint_gather_ranges(gpu, n, k, min_bins, precision):
    """<F d, g> = <d, F^H g> on both forms of the adjoint's table gather."""
    from mpsft_amd.signals import make_signal
    x, _ = make_signal(n, k, 1e-6, seed=3)
    s = gpu.Solver(n, gpu.solve_options(k, 1e-5, min_bins=min_bins),
                   gpu.MPSFT_MIXED if precision else gpu.MPSFT_FP64)
    s.set_record(True)
    s.solve(s.upload(x.astype(np.complex64) if precision else x), 5)
    keys, _ = s.modes()
    rng = np.random.default_rng(13)
    d = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    s.replay(gpu.DeviceArray.from_numpy(d), precision=gpu.MPSFT_FP64)
    fd = s.modes_dict()
    fd = np.array([fd[int(q)] for q in keys])
    g = rng.standard_normal(keys.size) + 1j * rng.standard_normal(keys.size)
    adj = s.adjoint(keys, g)
    assert keys.size >= k // 2
    tol = TOL * (np.linalg.norm(g) * np.linalg.norm(fd) + np.linalg.norm(adj) * np.linalg.norm(d))
    assert abs(np.vdot(g, fd) - np.vdot(adj, d)) <= tol
