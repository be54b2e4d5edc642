"""The network's loss and gradient at the edges of its chunks of 128 samples
and of its grid of 1024 workgroups, against the float64 CPU reference.

Tolerance: every sample's FP32 forward and backward pass is a chain of under
100 operations (relative error below 1e-5), and the sums add at most n / 1024
+ 1024 + 128 rounded terms of like size, whose errors stay below 1e-4 of the
sum of magnitudes; the entries are compared with the largest one."""
import numpy as np
import pytest

import cpsd_amd
import mlp_ref as M
from test_gpu_learned import sample_set, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 127, 128, 129, 1000, 1023 * 128, 1024 * 128, 1024 * 128 + 1, 300001])
def test_mlp_loss_grad_sizes_vs_cpu(gpu, n):
    say("mlp loss/grad, %d samples" % n)
    X, A, B = sample_set(n, n % 97)
    p = (M.init_params(3) + np.random.default_rng(4).normal(0, 0.1, size=M.NP)).astype(np.float32)
    L, g = cpsd_amd.mlp_loss_grad(X, A, B, p)
    Lr, gr = M.loss_grad(X.astype(np.float64), A.astype(np.float32).astype(np.float64),
                         B.astype(np.float32).astype(np.float64), p.astype(np.float64))
    assert abs(L - Lr) < 1e-4 * abs(Lr)
    assert np.max(np.abs(g - gr)) < 1e-4 * np.max(np.abs(gr))
