"""The raster's two routes: a box list that travels with the launch, and one in
device memory."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [41, 42, 43, 44])
@pytest.mark.parametrize("W,H", [(1, 1), (65, 17), (203, 90)])
def test_raster_either_side_of_the_launch_arguments(n, W, H):
    """Bit for bit the oracle's where the list last fits the launch's arguments
    and where it first does not."""
    import radiancecascade_amd as rc
    from oracle import rco
    if rc.device_count() < 1:
        pytest.skip("no HIP device")
    boxes = rc.scene_generate(60 + n, n, 4)
    out = [torch.empty(s, device="cuda:0") for s in ((H, W), (3, H, W), (3, H, W))]
    rc.gbuffer_raster(boxes, W, H, *out)
    for got, ref in zip(out, rco.raster(boxes, W, H)):
        assert np.array_equal(got.cpu().numpy().view(np.uint32), ref.view(np.uint32))
