"""The scorer's matrix-core training kernels and its two inference kernels at
the edges of their tiles, against the FP64 oracle.  Tolerance: FP32 sums of 256
terms through three layers (6e-8 * 16 * 3, about 3e-6 of the largest value),
with a factor of 7 to spare."""
import numpy as np
import pytest

import lighttraffic_amd as lt
from oracle import mlp_ref as M
from test_gpu_scorer import _part, _partition_handle, _sample

pytestmark = pytest.mark.gpu
TOL = 2e-5


def _scorer(P, rng):
    node, edge = _part(P, rng)
    part = _partition_handle(node, edge)
    sc = lt.Scorer(part, seed=3)
    sc.set_params((rng.normal(0, 0.1, lt.Scorer.NUM_PARAMS)).astype(np.float32))
    return sc, part, M.shares(node, edge)


# rows: one, a tile less one, a tile, one more, two tiles; more than one tile a
# workgroup (over 16384 rows); rows that straddle decisions
@pytest.mark.parametrize("n,P", [(1, 1), (1, 31), (1, 32), (3, 11), (2, 32), (13, 5), (33, 449), (37, 449), (70, 300)])
def test_gradient_at_tile_edges(n, P):
    print(f"scorer gradient n={n} P={P}", flush=True)
    rng = np.random.default_rng(n * 1000 + P)
    sc, part, (vsh, esh) = _scorer(P, rng)
    samples = [_sample(rng, P, with_next=i % 3 != 2) for i in range(n)]
    loss, grad = sc.loss_grad(samples)
    rloss, rgrad = M.loss_and_grad(sc.get_params().astype(np.float64), samples, vsh, esh)
    assert np.allclose(loss, rloss, rtol=TOL, atol=1e-7), (loss, rloss)
    off = 0
    for name, shape in M.SIZES:
        k = int(np.prod(shape))
        g, r = grad[off:off + k], rgrad[off:off + k]
        assert np.abs(g - r).max() <= TOL * max(np.abs(r).max(), 1e-2 * np.abs(rgrad).max()), name
        off += k


@pytest.mark.parametrize("P", [1, 2, 3, 1023, 1024, 1025, 1031])
def test_inference_at_row_edges_and_after_an_update(P):
    print(f"scorer inference P={P}", flush=True)
    rng = np.random.default_rng(P)
    sc, part, (vsh, esh) = _scorer(P, rng)

    def check():
        s = _sample(rng, P)
        st = (s["counts"], s["resident"], s["age"], s["recent"], s["cur"], s["w_total"])
        out = sc.infer(*st)
        Wb = {k: M.bf16_round(v) for k, v in M.unpack(sc.get_params().astype(np.float64)).items()}
        Y = M.forward(Wb, M.features(*st, vsh, esh))[2]
        assert np.abs(out - Y).max() <= TOL * np.abs(Y).max()

    check()
    sc.train([_sample(rng, P) for _ in range(4)], epochs=2, batch=2, lr=1e-2)
    check()  # the update's own copy of the weights
