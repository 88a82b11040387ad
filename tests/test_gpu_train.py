"""The training gradient (k_mlp_grad, k_mlp_fold_adam) at the edges of its
units of 32 samples, 4 wavefronts and 256 workgroups, against the FP64 CPU
oracle: one sample, one short of, exactly and one past a unit, past a
workgroup, and more samples than one unit per wavefront holds (32 x 4 x 256).

FP32 sums of n terms of either sign: the error grows as the square root of n
roundings of 2^-24 of a term, against a result that shrinks against its terms
in the same way, so 1e-5 of each parameter block's norm is some 100 roundings;
a lane, unit or wavefront left out or counted twice is 1/n of it at least,
and n <= 33000 samples of one block's norm."""
import numpy as np
import pytest

import pyoracle
from tlbm_amd.gpu import MLP_NPARAM, MlpTrainer, mlp_init

pytestmark = pytest.mark.gpu

BLOCKS = {"W1": (0, 224), "b1": (224, 256), "W2": (256, 1280), "b2": (1280, 1312), "w3": (1312, 1344),
          "b3": (1344, 1345)}


@pytest.mark.parametrize("count", [1, 31, 32, 33, 127, 128, 129, 32 * 4 * 256 + 1])
def test_gradient_at_unit_edges_matches_oracle(gpu_lib, count):
    rng = np.random.default_rng(count)
    n = count + 5
    x = rng.normal(0, 1, (n, 7)).astype(np.float32)
    t = np.abs(rng.normal(0.3, 0.5, n)).astype(np.float32)
    p = mlp_init(3)
    p[224:256] = rng.normal(0, 0.2, 32)
    p[1280:1312] = rng.normal(0, 0.2, 32)
    print(f"count {count}", flush=True)
    with MlpTrainer(x, t, p, seed=1, max_batch=count) as tr:
        loss, g = tr.loss_grad(3, count)
    loss_ref, ref = pyoracle.mlp_loss_grad(p.astype(np.float64), x[3:3 + count], t[3:3 + count])
    assert g.size == MLP_NPARAM and loss == pytest.approx(loss_ref, rel=1e-5)
    for name, (a, b) in BLOCKS.items():
        assert np.linalg.norm(g[a:b] - ref[a:b]) <= 1e-5 * np.linalg.norm(ref[a:b]), name


@pytest.mark.parametrize("count", [100, 4096, 65536, 65537, 1 << 17, 1 << 20])
def test_sums_keep_their_precision_at_any_batch(gpu_lib, count):
    """`count` copies of one sample.  The mean loss is that sample's, to the
    rounding of a double, because every sum of losses is one.  With a power of
    two each sample's share of the gradient is the one sample's, scaled
    exactly (another quotient rounds, and sums that nearly cancel within the
    sample magnify that); a partial gradient is an FP32 sum: a wavefront's
    units of 32 samples (one for each 32 x 4 x 256 of the batch), added one
    after the other, then 4 wavefronts, so so many roundings of at most 2^-24
    of the sum each."""
    rng = np.random.default_rng(7)
    x = np.repeat(rng.normal(0, 1, (1, 7)).astype(np.float32), count, axis=0)
    t = np.full(count, 0.37, np.float32)
    p = mlp_init(3)
    p[224:256] = rng.normal(0, 0.2, 32)
    p[1280:1312] = rng.normal(0, 0.2, 32)
    print(f"count {count}", flush=True)
    with MlpTrainer(x, t, p, seed=1, max_batch=count) as tr:
        one, g1 = tr.loss_grad(0, 1)
        loss, g = tr.loss_grad(0, count)
    assert loss == pytest.approx(one, rel=1e-14)
    if count & (count - 1) == 0:
        assert np.all(np.abs(g - g1) <= (max(32, count // 1024) + 4) * 2.0 ** -24 * np.abs(g1))
