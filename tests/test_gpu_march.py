"""The split march: rays among scattered pixels, what it takes beside the
one-sample march, and the calls that share its kernels."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rc():
    import radiancecascade_amd as rc
    if rc.device_count() < 1:
        pytest.skip("no HIP device")
    return rc


def _scattered(W, H, share, wall=False, seed=0):
    """Flat depth and emitters on a share of the pixels; wall: a lit column and
    row too, along which rays repeat their step."""
    rng = np.random.RandomState(seed)
    e = (rng.uniform(0.5, 2.0, (3, H, W)) * (rng.uniform(size=(H, W)) < share)).astype(np.float32)
    if wall:
        e[0, :, W // 3] = 1.0
        e[1, H // 2, W // 2:] = 1.0
    return np.full((H, W), 0.5, np.float32), e


def _us(fn, n=20, reps=5):
    """Best mean time of a pass in microseconds."""
    best = float("inf")
    for _ in range(reps):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(n):
            fn()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) * 1e3 / n)
    return best


@pytest.mark.parametrize("share,wall", [(0.0005, False), (0.002, True), (0.02, True), (0.0, True)])
@pytest.mark.parametrize("W,H", [(511, 300), (90, 901)])
def test_rays_among_scattered_pixels(rc, oracle, W, H, share, wall):
    """Rays longer than the march's first samples, with steps that differ, that
    repeat, and both in one wave: every code is the oracle's.  Another scene's
    codes are in the buffer before each frame."""
    L = 5
    d, e = _scattered(W, H, share, wall)
    other = _scattered(W, H, 0.1, seed=1)
    field = oracle.sdf_from_d2(oracle.edt_d2(oracle.seed_init(d, e)))
    ref = [oracle.march_level(field, e, i)[1].ravel() for i in range(L)]
    irr = torch.empty((3, H, W), device="cuda:0")
    with rc.RadianceCascadeStage(W, H, levels=L) as st:
        for order in (0, 2, 5):
            for i in range(1, L):
                st.set_march_order(i, order)
            for dd, ee in (other, (d, e)):
                st.run_device(torch.from_numpy(dd).cuda(), torch.from_numpy(ee).cuda(), irr)
            for i in range(1, L):
                h = torch.empty(rc.level_rays(W, H, i), dtype=torch.int32, device="cuda:0")
                st.debug_march(i, h)
                assert np.array_equal(h.cpu().numpy(), ref[i]), (order, i)


def test_scattered_pixels_are_no_slower_than_one_sample_a_step(rc):
    """Where every step differs, guessing the next samples only costs loads:
    the frame then took 1.28 times the in-place march, which takes one sample
    a step; it takes 0.82 times as long when the waves notice."""
    W, H = 1920, 1080
    d, e = (torch.from_numpy(x).cuda() for x in _scattered(W, H, 0.001))
    irr = torch.empty((3, H, W), device="cuda:0")
    us = {}
    with rc.RadianceCascadeStage(W, H) as st:
        for split in (0, 1):
            st.set_march(split, 1, 1)
            us[split] = _us(lambda: st.run_device(d, e, irr))
    assert us[1] <= us[0], us


def _boxes(rc, W, H, seed):
    d, a, e = (torch.empty(s, device="cuda:0") for s in ((H, W), (3, H, W), (3, H, W)))
    rc.gbuffer_raster(rc.scene_generate(seed, 32, 4), W, H, d, a, e)
    return d, e


@pytest.mark.parametrize("W,H,L", [(1366, 768, 6), (1921, 1079, 3), (3840, 2160, 7)])
def test_fallback_march_of_several_packets_a_wave(rc, W, H, L):
    """A fallback launch of more packets than its waves may be (and of more than
    512 K, where a plain frame's waves form groups): flagged tiles equal the plain level 1 bit for bit, the others the learned one, with
    another scene's codes left in the buffer."""
    irr = torch.empty((3, H, W), device="cuda:0")
    with rc.RadianceCascadeStage(W, H, levels=L) as plain, rc.RadianceCascadeStage(W, H, levels=L) as st:
        st.load_weights()
        py, px = plain.level_shape(1)[:2]
        a1 = {k: torch.empty(plain.level_shape(1), device="cuda:0") for k in "plf"}
        terr = torch.empty(st.surrogate_shapes()["tiles"], device="cuda:0")
        for seed in (2, 3):
            d, e = _boxes(rc, W, H, seed)
            plain.run_device(d, e, irr)
            plain.debug_level(1, a1["p"])
            st.set_surrogate(True)
            st.run_device(d, e, irr)
            st.debug_level(1, a1["l"])
            st.debug_surrogate(tile_err=terr)
            thr = float(terr.median())
            st.set_surrogate(True, threshold=thr)
            st.run_device(d, e, irr)
            st.debug_level(1, a1["f"])
            torch.cuda.synchronize()
            flag = np.repeat(np.repeat(~(terr.cpu().numpy() <= thr), 16, axis=0), 16, axis=1)[:py, :px]
            assert 0 < flag.sum() < flag.size
            f, p, l = (a1[k].cpu().numpy().view(np.uint32) for k in "fpl")
            assert np.array_equal(f[flag], p[flag]) and np.array_equal(f[~flag], l[~flag]), seed


def test_an_unused_fallback_costs_its_launches(rc):
    """A learned frame with the fallback on and no tile flagged: 1.31 times the
    frame without it where the fallback marched level by level, 1.30 now, 1.47
    when its march handed out a workgroup per wave of the whole frame."""
    W, H = 1920, 1080
    d, e = _boxes(rc, W, H, 3)
    irr = torch.empty((3, H, W), device="cuda:0")
    us = {}
    with rc.RadianceCascadeStage(W, H) as st:
        st.load_weights()
        for thr in (float("inf"), 1e30):
            st.set_surrogate(True, threshold=thr)
            us[thr] = _us(lambda: st.run_device(d, e, irr))
        assert st.stats().flagged_tiles == 0
    assert us[1e30] <= 1.4 * us[float("inf")], us


_FORMS = [(1, 1, 1), (1, 2, 1), (1, 4, 1), (1, 1, 2), (1, 2, 4), (1, 1, 8), (2, 1, 1)]


@pytest.mark.parametrize("W,H,L,march", [(W, H, L, m) for W, H, L in ((413, 211, 6), (97, 61, 4), (1030, 17, 3),
                                                                      (1366, 768, 6)) for m in _FORMS] +
                         [(3801, 1900, 6, (1, 1, 1)), (3801, 1900, 6, (1, 2, 1))])
def test_every_form_and_order_marches_every_ray(rc, oracle, W, H, L, march):
    """Each form of the split march in each order of its lanes, after another
    form left the codes and levels of a frame in which every ray hits: codes
    and irradiance are the oracle's, and the march's own packets place every
    ray in one slot.  The two larger sizes take several packets a wave, the
    largest 4 that are 4,096 apart in canonical order and 8 in the others."""
    e_lit = torch.ones((3, H, W), device="cuda:0")
    d, e = _boxes(rc, W, H, 4)
    dn, en = d.cpu().numpy(), e.cpu().numpy()
    want = oracle.run(dn, en, L, np.float32)
    field = oracle.sdf_from_d2(oracle.edt_d2(oracle.seed_init(dn, en)))
    codes = [oracle.march_level(field, en, i)[1].ravel() for i in range(L)]
    irr = torch.empty((3, H, W), device="cuda:0")
    before = (1, 1, 4) if march[2] == 1 else (1, 1, 1)
    with rc.RadianceCascadeStage(W, H, levels=L) as st:
        for order in range(6 if march[0] == 1 else 1):
            st.set_march(*before)
            for i in range(1, L):
                st.set_march_order(i, 0)
            st.run_device(d, e_lit, irr)
            st.set_march(*march)
            for i in range(1, L):
                legal = not (order == 1 and 4 * 4 ** i < 16 or order == 4 and 4 * 4 ** i < 32)
                st.set_march_order(i, order if legal else 0)
            st.run_device(d, e, irr)
            assert np.array_equal(irr.cpu().numpy().view(np.uint32), want.view(np.uint32)), order
            for i in range(1, L):
                n = rc.level_rays(W, H, i)
                h = torch.empty(n, dtype=torch.int32, device="cuda:0")
                ix = torch.empty(n, dtype=torch.int64, device="cuda:0")
                st.debug_march(i, h, ix)
                assert np.array_equal(h.cpu().numpy(), codes[i]), (order, i)
                assert ix.min().item() >= 0 and torch.unique(ix).numel() == n, (order, i)
                if st.march_order()[i] == 0:
                    assert torch.equal(ix, torch.arange(n, device="cuda:0")), (order, i)


@pytest.mark.parametrize("march,order", [((2, 1, 1), 0), ((1, 1, 2), 0), ((1, 1, 1), 5)])
@pytest.mark.parametrize("storage", ["f32", "f16"])
def test_every_tiling_of_an_unmerged_top_level(rc, march, order, storage):
    """The level kernel that reads stored codes runs only for a top level the
    march does not merge: each of its tiles and rays per lane gives the frame
    of the in-place march, after a frame in which every ray hits."""
    W, H, L = 331, 190, 4
    d, e = _boxes(rc, W, H, 6)
    e_lit = torch.ones((3, H, W), device="cuda:0")
    irr = torch.empty((3, H, W), device="cuda:0")
    with rc.RadianceCascadeStage(W, H, levels=L, storage=storage) as st:
        st.set_march(0, 1, 1)
        st.run_device(d, e, irr)
        want = irr.clone()
        top = torch.empty(st.level_shape(L - 1), device="cuda:0")
        st.debug_level(L - 1, top)
        st.set_march_order(L - 1, order)
        for shape in rc._abi.TILE_SHAPES:
            for rpt in (1, 2, 4):
                st.set_march(0, 1, 1)
                st.run_device(d, e_lit, irr)
                st.set_march(*march)
                st.set_tiling(L - 1, shape, rpt)
                st.run_device(d, e, irr)
                got = torch.empty_like(top)
                st.debug_level(L - 1, got)
                assert torch.equal(got, top) and torch.equal(irr, want), (shape, rpt)


def test_readbacks_follow_a_replayed_frame(rc):
    """Training rows between two replays of a learned frame with a fallback:
    the fallback's march has overwritten the rows' codes, so the readback
    refuses them, as after a frame that is launched directly; and after a
    replayed plain frame it returns that frame's levels."""
    W, H, L = 240, 160, 4
    d, e = _boxes(rc, W, H, 5)
    d2, e2 = _boxes(rc, W, H, 6)
    irr = torch.empty((3, H, W), device="cuda:0")
    qy, qx = rc.probe_grid(W, H, 2)[::-1]
    rows = torch.empty((qx * qy, 64), device="cuda:0"), torch.empty((qx * qy, 48), device="cuda:0")
    codes = torch.empty(rc.level_rays(W, H, 2), dtype=torch.int32, device="cuda:0")
    with rc.RadianceCascadeStage(W, H, levels=L, graph=True) as st, rc.RadianceCascadeStage(W, H, levels=L) as plain:
        a2, want = torch.empty(st.level_shape(2), device="cuda:0"), torch.empty(st.level_shape(2), device="cuda:0")
        plain.run_device(d, e, irr)
        plain.debug_level(2, want)
        st.load_weights()
        st.set_surrogate(True, threshold=-1e30)
        st.run_device(d, e, irr)
        st.surrogate_samples(d2, e2, *rows)
        st.run_device(d, e, irr)
        with pytest.raises(rc.RcError):
            st.debug_march(2, codes)
        st.set_surrogate(False)
        for _ in range(2):
            st.run_device(d, e, irr)
            st.debug_march(2, codes)
            st.debug_level(2, a2)
            assert torch.equal(a2, want)
