"""The rows a training epoch takes, where half of them are left out."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,batch,seed", [(63, 32, 1), (127, 64, 2), (511, 256, 3), (66000, 33024, 326)])
def test_an_epoch_takes_the_head_of_the_order(n, batch, seed):
    """One batch of the epoch's order and no more fits, so a row on the wrong
    side of the order's middle shows in the epoch's loss (rows of unlike loss,
    a step too small to move a weight).  The last case's first epoch has a list
    of 26 steps, beyond the sorted buffer's 24."""
    import radiancecascade_amd as rc
    from oracle import mlp
    from oracle import surrogate as so
    from test_shuffle import fisher_yates
    if rc.device_count() < 1:
        pytest.skip("no HIP device")
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, 64)).astype(np.float32)
    t = (rng.standard_normal((n, 48)) * np.exp(rng.normal(0.0, 1.5, (n, 1)))).astype(np.float32)
    with rc.RadianceCascadeStage(64, 64, levels=3) as st:
        rep = st.train_surrogate_rows(torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda(), epochs=1, batch=batch,
                                      lr=1e-30, seed=seed)
        net = st.mlp_get()
    z, _ = mlp.forward(so.params_to_layers(net["params"]),
                       (x.astype(np.float64) - net["in_mean"]) * net["in_istd"], emulate_bf16=True)
    rows = ((z[:, :48] - t.astype(np.float64) / net["out_scale"]) ** 2).mean(axis=1)
    rows = rows + mlp.ERR_WEIGHT * (z[:, 48] - np.log(rows + mlp.ERR_EPS)) ** 2
    order = np.array(fisher_yates(n, seed ^ 0x5DEECE66D))
    want = rows[order[:batch]].mean()
    # fp32 sums, and bf16 activations on the other side of a rounding boundary
    # (2^-8 of one of a row's 192, each row's own loss moves by some 1e-4)
    assert abs(rep["epoch_loss"][0] - want) <= 1e-4 * want
    # a row on the wrong side moves the mean by more, for most rows
    if n < 1000:
        moved = np.abs(np.subtract.outer(rows[order[:batch]], rows[order[batch:]])) / batch
        assert np.mean(moved > 2e-4 * want) > 0.7
