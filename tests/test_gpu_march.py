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
