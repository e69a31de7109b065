"""GPU parity of the RFI clipper with the oracle: identical outputs (bit for
bit), identical spectrum flags and running statistics, across chunk
boundaries, through the learning phase into the steady state, with narrowband
and broadband RFI."""
import numpy as np
import pytest
import torch

from synth import bandpass_values, stokes_noise

pytestmark = pytest.mark.gpu


def _stream(n_t, n_sub, n_ch, seed, n_pol=1):
    n_bins = n_sub * n_ch
    v = 150.0 - 0.0122 * np.arange(n_bins)
    level = 1000.0 + 6.0 * (v - 145.0)
    x = stokes_noise(n_t, n_sub, n_ch, level, seed, n_pol=n_pol)
    rng = np.random.default_rng(seed + 1)
    # narrowband RFI: 3 channels bright in most spectra, 2 in every spectrum
    # (their last-good slots never fill)
    for k, b in enumerate(rng.choice(n_bins, 5, replace=False)):
        on = rng.random(n_t) < (0.7 if k < 3 else 1.0)
        x[on, b // n_ch, :, b % n_ch] *= 30.0
    # broadband impulses in 1% of spectra
    imp = rng.random(n_t) < 0.01
    x[imp] *= 5.0
    return x


def _bp(n_sub, n_ch):
    return bandpass_values(n_sub * n_ch, 150.0, -0.0122, 1000.0, 40.0, poly=(6.0, 0.001))


@pytest.mark.parametrize("zero_dm,n_pol,history", [(True, 1, 1200), (False, 1, 1200), (True, 2, 1100)])
def test_clipper_bit_exact(orc, ppl, zero_dm, n_pol, history):
    n_sub, n_ch = 8, 16
    x = _stream(2800, n_sub, n_ch, seed=21, n_pol=n_pol)
    bp = _bp(n_sub, n_ch)
    oc = orc.Clipper(bp, 10.0, 4.0, history, zero_dm)
    gc = ppl.Clipper(bp, 10.0, 4.0, history, zero_dm)
    for a in range(0, x.shape[0], 256):
        chunk = np.ascontiguousarray(x[a:a + 256])
        ref = chunk.copy()
        W = np.ones_like(ref)  # WeightedSpectrumDataSet::reset sets every weight to 1
        oc.run(ref, W)
        good_o, _ = oc.last_flags(chunk.shape[0])
        d = torch.from_numpy(chunk).cuda()
        dw = torch.zeros_like(d)
        gc.run(d, dw)
        out = d.cpu().numpy()
        good_g = gc.flags(chunk.shape[0])
        assert np.array_equal(good_g, good_o), (a, np.nonzero(good_g != good_o)[0][:5])
        bad = np.nonzero(~((out == ref) | (np.isnan(out) & np.isnan(ref))))
        assert bad[0].size == 0, (a, bad[0][:5], out[bad][:5], ref[bad][:5])
        assert np.all(dw.cpu().numpy() == 1.0) and np.all(W == 1.0)
        st_o, _ = oc.state()
        m, r = gc.stats()
        assert (np.float32(m), np.float32(r)) == (st_o[0], st_o[1])
    # the run went through the warm-up into steady state and kept spectra
    assert good_o.sum() > 0


def test_clipper_first_1000_clipped(orc, ppl):
    n_sub, n_ch = 4, 16
    x = _stream(600, n_sub, n_ch, seed=5)
    gc = ppl.Clipper(_bp(n_sub, n_ch), history=10000)
    d = torch.from_numpy(x).cuda()
    gc.run(d)
    assert gc.flags(600).sum() == 0
    bpv = orc.Clipper(_bp(n_sub, n_ch), history=10000)
    ref = x.copy()
    bpv.run(ref)
    # a rejected spectrum is -0.2 minus (bandpass + data model): never normalised
    assert np.array_equal(d.cpu().numpy(), ref)


def test_clipper_rejects_bad_shapes(ppl):
    gc = ppl.Clipper(_bp(4, 16))
    with pytest.raises(ppl.PPLError):
        gc.run(torch.zeros((10, 3, 1, 5), device="cuda"))  # 15 bins: not a multiple of 8


def test_clipper_long_steady_state_3968_bins(orc, ppl):
    """The LOFAR-beam width (62 x 64 bins) through learning into a long steady
    state, where most spectra take the precomputed-mask path."""
    n_sub, n_ch = 62, 64
    x = _stream(4200, n_sub, n_ch, seed=33)
    bp = _bp(n_sub, n_ch)
    oc = orc.Clipper(bp, 10.0, 4.0, 1000, True)
    gc = ppl.Clipper(bp, 10.0, 4.0, 1000, True)
    for a in range(0, x.shape[0], 700):
        chunk = np.ascontiguousarray(x[a:a + 700])
        ref = chunk.copy()
        oc.run(ref)
        d = torch.from_numpy(chunk).cuda()
        gc.run(d)
        assert np.array_equal(gc.flags(chunk.shape[0]), oc.last_flags(chunk.shape[0])[0]), a
        out = d.cpu().numpy()
        assert np.array_equal(out, ref), (a, np.argwhere(out != ref)[:5])
    st_o, sizes = oc.state()
    assert sizes[0] == 1000 and sizes[1] == 1000
    cnt = gc.counters()
    assert cnt["fast"] + cnt["slow"] == x.shape[0] and cnt["fast"] > 1000, cnt  # steady state mostly fast
    assert cnt["learn"] + cnt["box"] + cnt["undecided"] + cnt["fill"] + cnt["ver"] == cnt["slow"], cnt
    assert (np.float32(gc.stats()[0]), np.float32(gc.stats()[1])) == (st_o[0], st_o[1])


def test_clipper_sub_chunks_and_drift(orc, ppl):
    """Runs longer than one walk sub-chunk (4096 spectra), with a slow rise
    of the whole band by 3% that carries the state out of the speculation
    box: sub-chunks end early and re-centre, and every output still matches
    the oracle bit for bit."""
    n_sub, n_ch, n_t = 8, 16, 14000
    x = _stream(n_t, n_sub, n_ch, seed=77)
    ramp = np.clip((np.arange(n_t) - 6000) / 3000.0, 0.0, 1.0) * 0.03 + 1.0
    x = (x * ramp[:, None, None, None]).astype(np.float32)
    bp = _bp(n_sub, n_ch)
    oc = orc.Clipper(bp, 10.0, 4.0, 1000, True)
    gc = ppl.Clipper(bp, 10.0, 4.0, 1000, True)
    for a in range(0, n_t, 7000):
        chunk = np.ascontiguousarray(x[a:a + 7000])
        ref = chunk.copy()
        oc.run(ref)
        d = torch.from_numpy(chunk).cuda()
        gc.run(d)
        assert np.array_equal(gc.flags(chunk.shape[0]), oc.last_flags(chunk.shape[0])[0]), a
        out = d.cpu().numpy()
        bad = np.nonzero(~((out == ref) | (np.isnan(out) & np.isnan(ref))))
        assert bad[0].size == 0, (a, bad[0][:5], out[bad][:5], ref[bad][:5])
    cnt = gc.counters()
    assert cnt["fast"] + cnt["slow"] == n_t, cnt
    assert cnt["stop"] >= 1 and cnt["fast"] > n_t // 2, cnt
    st_o, _ = oc.state()
    assert (np.float32(gc.stats()[0]), np.float32(gc.stats()[1])) == (st_o[0], st_o[1])


def test_split_run_equals_run(orc, ppl):
    """A run split over two streams (front and back on one, the walk on
    another, ordered by events) gives what run() gives, bit for bit: through
    the learning phase, the steady state and a drift that carries the state
    out of the box (the split run's whole-chunk box ends early and the walk
    continues from a fresh one); calls out of order are refused."""
    n_sub, n_ch, n_t = 8, 16, 14000
    x = _stream(n_t, n_sub, n_ch, seed=79)
    ramp = np.clip((np.arange(n_t) - 6000) / 3000.0, 0.0, 1.0) * 0.03 + 1.0
    x = (x * ramp[:, None, None, None]).astype(np.float32)
    bp = _bp(n_sub, n_ch)
    a, b = ppl.Clipper(bp, 10.0, 4.0, 1000, True), ppl.Clipper(bp, 10.0, 4.0, 1000, True)
    walk = torch.cuda.Stream()
    main = torch.cuda.current_stream()
    for t0 in range(0, n_t, 3500):
        chunk = np.ascontiguousarray(x[t0:t0 + 3500])
        da, db = torch.from_numpy(chunk).cuda(), torch.from_numpy(chunk).cuda()
        a.run(da)
        b.run_front(db)
        ev = torch.cuda.Event()
        ev.record(main)
        walk.wait_event(ev)
        b.run_walk(stream=walk)
        ev2 = torch.cuda.Event()
        ev2.record(walk)
        main.wait_event(ev2)
        b.run_back()
        assert torch.equal(torch.nan_to_num(da, nan=-1e30), torch.nan_to_num(db, nan=-1e30)), t0
        assert np.array_equal(a.flags(chunk.shape[0]), b.flags(chunk.shape[0])), t0
        assert a.stats() == b.stats(), t0
    ca, cb = a.counters(), b.counters()
    assert ca["fast"] + ca["slow"] == cb["fast"] + cb["slow"] == n_t
    with pytest.raises(ppl.PPLError, match="without a front"):
        b.run_walk()
    with pytest.raises(ppl.PPLError, match="without a walk"):
        b.run_back()
    d = torch.from_numpy(np.ascontiguousarray(x[:100])).cuda()
    b.run_front(d)
    with pytest.raises(ppl.PPLError, match="front called twice"):
        b.run_front(d)
    b.run_walk()
    b.run_back()


def test_run_after_a_refused_one(orc, ppl):
    """A run of more spectra than the card has memory for records of is
    refused; the next one makes its records anew and gives the oracle's
    outputs, flags and statistics."""
    n_sub, n_ch = 8, 16
    x = _stream(3000, n_sub, n_ch, seed=81)
    bp = _bp(n_sub, n_ch)
    oc = orc.Clipper(bp, 10.0, 4.0, 1000, True)
    gc = ppl.Clipper(bp, 10.0, 4.0, 1000, True)
    for chunk in (x[:2000], x[2000:]):
        ref = np.ascontiguousarray(chunk)
        d = torch.from_numpy(ref.copy()).cuda()
        oc.run(ref)
        if chunk.shape[0] < 2000:
            n_max = (1 << 31) - 1  # 136 bytes each: more than the card holds
            assert ppl.lib().ppl_clipper_run(gc.h, d.data_ptr(), None, n_max, n_sub, 1, n_ch, None) != 0
        gc.run(d)
        assert np.array_equal(gc.flags(chunk.shape[0]), oc.last_flags(chunk.shape[0])[0])
        assert np.array_equal(d.cpu().numpy(), ref, equal_nan=True)


@pytest.mark.parametrize("n_und,every", [(2, 40), (16, 40), (17, 40), (5, 9)])
def test_clipper_rejected_with_undecided_channels(orc, ppl, n_und, every):
    """Every 40th (9th) spectrum loses half its channels to interference, so
    it is rejected whatever n_und further channels do that lie within 2e-4 of
    the channel threshold.  Up to 16 such channels are counted in the walk's
    speculative blocks, for up to 32 spectra a stage of 512; more go to the
    workgroup.  Outputs, flags and state are the oracle's bit for bit."""
    n_sub, n_ch, n_t = 8, 16, 3000
    x = _stream(1500 + n_t, n_sub, n_ch, seed=60 + n_und)
    bp = _bp(n_sub, n_ch)
    oc = orc.Clipper(bp, 10.0, 4.0, 1000, True)
    gc = ppl.Clipper(bp, 10.0, 4.0, 1000, True)

    def both(chunk):
        ref = chunk.copy()
        oc.run(ref)
        d = torch.from_numpy(chunk).cuda()
        gc.run(d)
        assert np.array_equal(gc.flags(chunk.shape[0]), oc.last_flags(chunk.shape[0])[0])
        assert np.array_equal(d.cpu().numpy(), ref, equal_nan=True)
        st_o, _ = oc.state()
        assert (np.float32(gc.stats()[0]), np.float32(gc.stats()[1])) == (st_o[0], st_o[1])

    both(np.ascontiguousarray(x[:1500]))
    before = gc.counters()
    vals = gc.model(n_sub * n_ch)[3]
    rng = np.random.default_rng(n_und)
    y = np.ascontiguousarray(x[1500:])
    flat = y.reshape(n_t, n_sub * n_ch)
    for t in range(5, n_t, every):
        bins = rng.permutation(n_sub * n_ch)
        flat[t, bins[:64]] *= 50.0
        near = bins[64:64 + n_und]
        flat[t, near] = vals[near] + 10.0 * gc.stats()[1] * (1.0 + rng.uniform(-2e-4, 2e-4, n_und))
    both(y)
    after = gc.counters()
    hit = len(range(5, n_t, every))
    took = {k: after[k] - before[k] for k in after}
    # (the noise itself adds spectra of both kinds)
    if n_und > 16 or every < 10:
        assert took["undecided"] > hit // 4, took
    if n_und <= 16:
        assert took["resolved"] > hit // 4, took


def test_clipper_batch_equals_separate_runs(orc, ppl):
    """Beams of different shapes and spectrum counts in one batched run give
    the same outputs, flags and running statistics as separate runs, through
    the learning phase into the steady state."""
    shapes = [(8, 16, 1), (4, 16, 2), (62, 64, 1)]
    hist = 1000
    streams = [_stream(3600, ns, nc, seed=50 + k, n_pol=npol) for k, (ns, nc, npol) in enumerate(shapes)]
    bps = [_bp(ns, nc) for ns, nc, _ in shapes]
    single = [ppl.Clipper(bp, 10.0, 4.0, hist, True) for bp in bps]
    batch = [ppl.Clipper(bp, 10.0, 4.0, hist, True) for bp in bps]
    oracle = orc.Clipper(bps[0], 10.0, 4.0, hist, True)
    lens = [(700, 900, 500), (1300, 700, 900), (1600, 2000, 2200)]  # spectra per call, per beam
    pos = [0, 0, 0]
    for call in range(3):
        xs = []
        for k in range(3):
            n = lens[call][k]
            xs.append(np.ascontiguousarray(streams[k][pos[k]:pos[k] + n]))
            pos[k] += n
        ds = [torch.from_numpy(x).cuda() for x in xs]
        dw = [torch.zeros_like(d) for d in ds]
        ppl.clipper_run_batch(batch, ds, dw)
        for k in range(3):
            ref = torch.from_numpy(xs[k]).cuda()
            single[k].run(ref)
            got = ds[k].cpu().numpy()
            want = ref.cpu().numpy()
            assert np.array_equal(got, want, equal_nan=True), (call, k)
            assert np.array_equal(batch[k].flags(lens[call][k]), single[k].flags(lens[call][k])), (call, k)
            assert batch[k].stats() == single[k].stats(), (call, k)
            assert np.all(dw[k].cpu().numpy() == 1.0)
        # beam 0 also against the oracle
        o = xs[0].copy()
        oracle.run(o)
        got0 = ds[0].cpu().numpy()
        assert np.array_equal(got0, o, equal_nan=True), call
    cnt = batch[2].counters()
    assert cnt["fast"] > 0 and cnt["learn"] == hist, cnt


def test_clipper_reference_bandpass_file(orc, ppl):
    """The reference's own band31.bp (31 x 64 bins), read as the reference
    reads it, through learning into the steady state with narrowband spikes
    and broadband impulses: identical outputs, flags and state."""
    from test_oracle_clipper import _band31_stream
    impulses = list(range(1500, 3000, 100))
    v, x = _band31_stream(orc, 3000, seed=12, spikes=(17, 900, 1700), impulses=impulses)
    oc = orc.Clipper(v, 10.0, 4.0, 1000, True)
    gc = ppl.Clipper(v, 10.0, 4.0, 1000, True)
    for a in range(0, 3000, 1000):
        chunk = np.ascontiguousarray(x[a:a + 1000])
        ref = chunk.copy()
        oc.run(ref)
        d = torch.from_numpy(chunk).cuda()
        gc.run(d)
        assert np.array_equal(gc.flags(1000), oc.last_flags(1000)[0]), a
        assert np.array_equal(d.cpu().numpy(), ref, equal_nan=True), a
    st_o, _ = oc.state()
    assert (np.float32(gc.stats()[0]), np.float32(gc.stats()[1])) == (st_o[0], st_o[1])


@pytest.mark.parametrize("per_spectrum", [1, 2])
def test_clipper_near_margin_channels(orc, ppl, per_spectrum):
    """Channels a little below and above the clipping margin (8-12 rms
    above the bandpass, one or two per spectrum, and whole spectra at 3x):
    the steady state's undecided channels.  With one, the precompute keeps a
    second record with that channel kept and the walk picks one by the
    channel's exact decision (in the fast run, or by prediction in a
    speculative block); with two, the workgroup takes the spectrum and the
    kept mean comes from the ordered sum, the precomputed mean, or is not
    needed (a spectrum rejected for certain)."""
    n_sub, n_ch, n_t = 62, 64, 5200
    nb = n_sub * n_ch
    level, hist = 1000.0, 1000
    sig = level * np.sqrt(2 / 16)
    bp = bandpass_values(nb, 150.0, -0.1953125 / 64, level, sig)
    x = stokes_noise(n_t, n_sub, n_ch, level, seed=41)
    rng = np.random.default_rng(42)
    flat = x.reshape(n_t, nb)
    for _ in range(per_spectrum):
        cols = rng.integers(0, nb, n_t)
        flat[np.arange(n_t), cols] += (8.0 + 4.0 * rng.random(n_t)) * sig
    imp = rng.random(n_t) < 0.01
    x[imp] *= 3.0
    oc = orc.Clipper(bp, 10.0, 4.0, hist, True)
    gc = ppl.Clipper(bp, 10.0, 4.0, hist, True)
    for a in range(0, n_t, 1300):
        chunk = np.ascontiguousarray(x[a:a + 1300])
        ref = chunk.copy()
        oc.run(ref)
        d = torch.from_numpy(chunk).cuda()
        gc.run(d)
        assert np.array_equal(gc.flags(chunk.shape[0]), oc.last_flags(chunk.shape[0])[0]), a
        assert np.array_equal(d.cpu().numpy(), ref, equal_nan=True), a
    cnt = gc.counters()
    if per_spectrum == 1:
        assert cnt["resolved"] > 50 and cnt["fast"] > 2000, cnt
    else:
        assert cnt["undecided"] > 50 and cnt["fast"] > 1000, cnt
    st_o, _ = oc.state()
    assert (np.float32(gc.stats()[0]), np.float32(gc.stats()[1])) == (st_o[0], st_o[1])


@pytest.mark.parametrize("dtype", ["f32", "u8"])
def test_run_into_equals_run_then_add(ppl, dtype):
    """ppl_clipper_run_into (the clipper, then DedispersionBuffer::addSamples
    of its output, in one call) leaves the same clipped spectra, flags and
    dedispersion buffer, chunk by chunk through the learning phase and
    carries, as Clipper.run followed by DDBuffer.add.  The 1000-sample
    buffer with a 200-sample overlap fills part way through 256-spectrum
    chunks: run_into reports how many spectra it took, and the rest of the
    chunk goes into the rotated buffer."""
    n_sub, n_ch = 8, 16
    n_chan = n_sub * n_ch
    x = _stream(2304, n_sub, n_ch, seed=33)
    bp = _bp(n_sub, n_ch)
    ca, cb = ppl.Clipper(bp, 10.0, 4.0, 1000, True), ppl.Clipper(bp, 10.0, 4.0, 1000, True)
    ba = ppl.DDBuffer(n_chan, 1000, 200, dtype, 12.7)
    bb = ppl.DDBuffer(n_chan, 1000, 200, dtype, 12.7)
    mid_chunk_fills = 0
    for a in range(0, x.shape[0], 256):
        chunk = np.ascontiguousarray(x[a:a + 256])
        n_t = chunk.shape[0]
        da, db = torch.from_numpy(chunk).cuda(), torch.from_numpy(chunk.copy()).cuda()
        ca.run(da)
        used_a, full_a = ba.add(da.view(n_t, n_chan))
        used_b, full_b = cb.run_into(db, bb)
        assert (used_a, full_a) == (used_b, full_b), a
        assert torch.equal(da, db), a
        assert np.array_equal(ca.flags(n_t), cb.flags(n_t)), a
        n = ba.fill()  # samples written so far (the rest of the buffer is not initialised)
        assert n == bb.fill()
        assert torch.equal(ba.tensor()[:, :n], bb.tensor()[:, :n]), a
        first = used_a
        while first < n_t or full_a:
            assert full_a, a
            mid_chunk_fills += first < n_t
            ba.rotate()
            bb.rotate()
            assert ba.fill() == bb.fill() == 200
            assert torch.equal(ba.tensor()[:, :200], bb.tensor()[:, :200]), a
            if first == n_t:
                break
            used_a, full_a = ba.add(da.view(n_t, n_chan), first)
            used_b, full_b = bb.add(db.view(n_t, n_chan), first)
            assert (used_a, full_a) == (used_b, full_b), a
            first += used_a
            n = ba.fill()
            assert torch.equal(ba.tensor()[:, :n], bb.tensor()[:, :n]), a
    assert mid_chunk_fills >= 2


def test_run_into_rejects_a_mismatched_buffer(ppl):
    """A buffer whose channel count differs from nSub*nCh is refused before
    the clipper runs: the clipper state is untouched, so a later run equals
    a fresh clipper's."""
    n_sub, n_ch = 8, 16
    x = _stream(256, n_sub, n_ch, seed=34)
    bp = _bp(n_sub, n_ch)
    ca, cb = ppl.Clipper(bp, 10.0, 4.0, 1000, True), ppl.Clipper(bp, 10.0, 4.0, 1000, True)
    for n_chan in (n_sub * n_ch + 8, n_sub * n_ch - 8):
        bad = ppl.DDBuffer(n_chan, 1024, 0, "f32", 1.0)
        d = torch.from_numpy(x.copy()).cuda()
        with pytest.raises(ppl.PPLError, match="does not match buffer sample size"):
            cb.run_into(d, bad)
        assert torch.equal(d, torch.from_numpy(x).cuda())
        assert bad.fill() == 0
    da, db = torch.from_numpy(x.copy()).cuda(), torch.from_numpy(x.copy()).cuda()
    ca.run(da)
    cb.run(db)
    assert torch.equal(da, db)
    assert ca.stats() == cb.stats()


@pytest.mark.parametrize("case", ["mean +35", "mean +36", "25% bright in 3 bands", "25% bright in 4 bands",
                                  "one band all bright", "26 bright channels", "25 bright channels"])
def test_clipper_steady_state_known_answers(orc, ppl, case):
    """The hand-worked steady-state cases of the oracle tests (tolerance
    edge, history rollback, bad-band and total-kept rules) through the
    device clipper: outputs, flags and running statistics as the oracle's."""
    from test_oracle_clipper import KA_HIST, _ka_bp, ka_stream
    x = ka_stream(case)
    ref = x.copy()
    oc = orc.Clipper(_ka_bp(), 10.0, 4.0, KA_HIST, True)
    oc.run(ref)
    gc = ppl.Clipper(_ka_bp(), 10.0, 4.0, KA_HIST, True)
    d = torch.from_numpy(x).cuda()
    gc.run(d)
    assert np.array_equal(gc.flags(x.shape[0]), oc.last_flags(x.shape[0])[0])
    assert np.array_equal(d.cpu().numpy(), ref)
    st_o, _ = oc.state()
    assert (np.float32(gc.stats()[0]), np.float32(gc.stats()[1])) == (st_o[0], st_o[1])


def test_clipper_kill_lines_bit_exact(orc, ppl, tmp_path):
    """A .bp file with kill lines (BandPassAdapter.cpp:58-71,101-106): the
    killed bins hold 0.0 in every model the clipper builds (BandPass.cpp:
    101-157); outputs, flags, statistics and the live model equal the
    oracle's through learning into the steady state."""
    from test_oracle_clipper import write_bp
    path = write_bp(str(tmp_path / "k.bp"), 128, 0.0, 1.0, 40.0, 1000.0, [0.0, 0.5], ["K 5 5", "K 77 77"])
    v, kills = orc.read_bp(path, with_kills=True)
    x = _stream(2600, 8, 16, seed=61)
    oc = orc.Clipper(v, 10.0, 4.0, 1000, True, kill=kills)
    gc = ppl.Clipper(v, 10.0, 4.0, 1000, True, kill=kills)
    for a in range(0, x.shape[0], 650):
        chunk = np.ascontiguousarray(x[a:a + 650])
        ref = chunk.copy()
        oc.run(ref)
        d = torch.from_numpy(chunk).cuda()
        gc.run(d)
        assert np.array_equal(gc.flags(chunk.shape[0]), oc.last_flags(chunk.shape[0])[0]), a
        assert np.array_equal(d.cpu().numpy(), ref, equal_nan=True), a
    p0, mean, rms, vals = gc.model(128)
    st, _ = oc.state()
    assert (np.float32(p0), np.float32(mean), np.float32(rms)) == (st[2], st[3], st[1])
    assert np.array_equal(vals, oc.bandpass(128))
    assert np.all(vals[[5, 6, 77, 78]] == 0.0) and np.count_nonzero(vals == 0.0) == 4


def test_clipper_kill_mismatch_refused(ppl, orc, tmp_path):
    from test_oracle_clipper import write_bp
    path = write_bp(str(tmp_path / "m.bp"), 128, 141.5, -0.0122, 40.0, 1000.0, [0.0], ["K 5 141.44"])
    v, kills = orc.read_bp(path, with_kills=True)
    with pytest.raises(ppl.PPLError, match="kill mismatch"):
        ppl.Clipper(v, kill=kills)


def test_clipper_live_model(orc, ppl):
    """RFI_Clipper::bandPass() after every run is the model setMean / setRMS
    left (RFI_Clipper.cpp:562-563): constant coefficient, mean, RMS and
    values as the oracle's, before and after the steady state."""
    n_sub, n_ch = 8, 16
    x = _stream(2400, n_sub, n_ch, seed=8)
    bp = _bp(n_sub, n_ch)
    oc = orc.Clipper(bp, 10.0, 4.0, 1000, True)
    gc = ppl.Clipper(bp, 10.0, 4.0, 1000, True)
    p0, mean, rms = gc.model()
    for a in range(0, x.shape[0], 800):
        chunk = np.ascontiguousarray(x[a:a + 800])
        ref = chunk.copy()
        oc.run(ref)
        gc.run(torch.from_numpy(chunk).cuda())
        p0, mean, rms, vals = gc.model(n_sub * n_ch)
        st, _ = oc.state()
        assert (np.float32(p0), np.float32(mean), np.float32(rms)) == (st[2], st[3], st[1]), a
        assert np.array_equal(vals, oc.bandpass(n_sub * n_ch)), a


def test_clipper_module_bandpass_is_live(orc, tmp_path):
    """The C++ RFI_Clipper module (ppl_bandpass clip) on the reference's
    band31.bp: clipped spectra and its bandPass() after the run (the live
    model on the run map) as the oracle's."""
    import json
    import os
    import subprocess
    from test_oracle_clipper import _band31_stream
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    exe = os.path.join(root, "pelican-lofar_amd", "ppl_bandpass")
    bp_path = os.path.join(root, "tests", "golden", "band31.bp")
    v, x = _band31_stream(orc, 2500, seed=14, spikes=(9, 700), impulses=list(range(1200, 2500, 150)))
    x = np.ascontiguousarray(x, np.float32)
    f = tmp_path / "s.f32"
    x.tofile(f)
    r = subprocess.run([exe, "-", "clip", bp_path, "1000", str(f), str(x.shape[0]), "31", "64", "700"],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    out = json.loads(r.stdout)
    oc = orc.Clipper(v, 10.0, 4.0, 1000, True)
    ref = x.copy()
    for a in range(0, x.shape[0], 700):
        chunk = np.ascontiguousarray(ref[a:a + 700])
        oc.run(chunk)
        ref[a:a + 700] = chunk
    got = np.fromfile(str(f) + ".out", np.float32).reshape(x.shape)
    assert np.array_equal(got, ref, equal_nan=True)
    st, _ = oc.state()
    assert (np.float32(out["p0"]), np.float32(out["mean"]), np.float32(out["rms"])) == (st[2], st[3], st[1])
    vals = np.fromfile(str(f) + ".bp", np.float32)
    assert out["bins"] == 1984 and np.array_equal(vals, oc.bandpass(1984))


def test_clipper_steady_cases_in_speculative_blocks(orc, ppl):
    """The hand-worked steady-state cases scattered through a long steady
    stream (past the first 4096-spectrum sub-chunk, where the walk runs
    speculative blocks): spectra rejected by the tolerance test, by bad
    bands or by the total-kept rule, runs of consecutive rejections, and
    kept offsets, at varying distances.  Outputs, flags and statistics as
    the oracle's, and most spectra on the fast paths."""
    from test_oracle_clipper import KA_CASES, KA_HIST, _ka_bp, _ka_normal
    rng = np.random.default_rng(77)
    n_t = KA_HIST + 9000
    x = _ka_normal(n_t)
    names = sorted(KA_CASES)
    t = KA_HIST + 30
    while t < n_t - 10:
        run = 1 + int(rng.integers(0, 3)) if rng.random() < 0.2 else 1
        for j in range(run):
            x[t + j] = KA_CASES[names[int(rng.integers(len(names)))]][0][0]
        t += run + int(rng.integers(5, 140))
    # small noise so that spectra differ (multiples of 1/8: exact sums)
    x += (rng.integers(-8, 9, size=x.shape) / 8.0).astype(np.float32)
    ref = x.copy()
    oc = orc.Clipper(_ka_bp(), 10.0, 4.0, KA_HIST, True)
    gc = ppl.Clipper(_ka_bp(), 10.0, 4.0, KA_HIST, True)
    for a in range(0, n_t, 5000):
        r = np.ascontiguousarray(ref[a:a + 5000])
        oc.run(r)
        ref[a:a + 5000] = r
        d = torch.from_numpy(np.ascontiguousarray(x[a:a + 5000])).cuda()
        gc.run(d)
        assert np.array_equal(gc.flags(r.shape[0]), oc.last_flags(r.shape[0])[0]), a
        assert np.array_equal(d.cpu().numpy(), r), a
    st_o, _ = oc.state()
    assert (np.float32(gc.stats()[0]), np.float32(gc.stats()[1])) == (st_o[0], st_o[1])
    cnt = gc.counters()
    assert cnt["fast"] > 5000, cnt
