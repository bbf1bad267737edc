"""The network's passes over the PPE graph at the edges of their batches (32 entries of a row in the
aggregation, 8 in the matrix product, 16 blocks of partial gradients, 16 x 1,024 rows of a column sum):
gradients of a drum with fewer rows than one batch of each and of one with more, with the matrix in
FP64 and in FP32, against the FP64 oracle network (bounds as for BF16 activations and messages)."""
import numpy as np
import pytest

from simulation_project_amd import Solver, abi, cases, load_library
from oracle import mpnn
from test_gpu_mpnn import active_graph, oracle_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver", [abi.MPSR_PCG_FP64, abi.MPSR_PCG_MIXED])
@pytest.mark.parametrize("l0", [1.6e-2, 5e-3])
def test_gradients_below_and_above_the_batches(l0, solver):
    case = cases.drum(load_library(), l0=l0)
    ppe = abi.PpeOptions(solver, 1e-8, 20000, abi.MPSR_WARM_LEARNED, 0.0, 0.0)
    g = Solver(case, pressure_mode=abi.MPSR_PRESSURE_PPE, ppe=ppe)
    p = mpnn.init_params(5)
    g.mpnn_set_weights(mpnn.flatten(p).astype(np.float32))
    g.step_many(0, 2)
    X, _, s = g.mpnn_rows()
    G, act, sol = active_graph(g)
    print(f"[mpnn-rows] particles={case.n} active={G.n}", flush=True)
    parts, grads = g.mpnn_train_step(update=False, want_grads=True)
    po = oracle_params(p)
    y, cache = mpnn.forward(po, X[act].astype(np.float64), G)
    loss, dy, _ = mpnn.loss_and_dy(y, G, s, sol)
    assert abs(parts[0] - loss) <= 2e-2 * abs(loss), (parts, loss)
    go, gg = mpnn.backward(po, cache, dy, G), mpnn.unflatten(grads.astype(np.float64))
    for k in mpnn.PARAM_ORDER:
        a, b = gg[k].ravel(), go[k].ravel()
        nb = np.linalg.norm(b)
        if nb == 0:
            continue
        assert np.linalg.norm(a - b) < 6e-2 * nb, k
