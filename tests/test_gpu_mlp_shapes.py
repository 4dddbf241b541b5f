"""The surrogate network's kernels at the edges of their tiles: batches of one row,
one below and above a 16-row group and a 64-row pad; widths of one pad, the widest
the one-launch forward pass takes, and one beyond it (layer by layer).  Against the
CPU FP64 restatement at 3e-2 relative L2, the bound that BF16 activations set."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(3, 5), (13, 64, 5), (70, 960, 33), (40, 961, 200, 20)])
@pytest.mark.parametrize("B", [1, 15, 17, 64, 65, 200])
def test_forward_and_gradients_at_tile_edges(dims, B):
    from mpifdtd_amd import surrogate as S
    from oracle import mlp as om
    print(dims, B, flush=True)
    rng = np.random.default_rng(B)
    net = S.MLP(list(dims), batch_max=200, seed=1)
    params = [((rng.standard_normal((o, i)) / np.sqrt(i)).astype(np.float32), (0.1 * rng.standard_normal(o)).astype(np.float32))
              for i, o in zip(dims[:-1], dims[1:])]
    for l, (w, b) in enumerate(params):
        net.set_params(l, w, b)
    x, t = rng.random((B, dims[0])).astype(np.float32), rng.standard_normal((B, dims[-1])).astype(np.float32)
    assert rel_l2(net.forward(x), om.forward(params, x)[0]) <= 3e-2
    loss = net.grads(x, t)
    ref, ref_loss = om.grads(params, x, t)
    assert abs(loss - ref_loss) <= 3e-2 * ref_loss
    for l, (dw, db) in enumerate(ref):
        gw, gb = net.layer_grads(l)
        assert rel_l2(gw, dw) <= 3e-2 and rel_l2(gb, db) <= 3e-2, l
