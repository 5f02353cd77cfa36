"""Predictions and input gradients of the register-resident network kernel
against the NumPy oracle at ragged ends: less than a wave's 16 rows, around a
workgroup's 64, and the two-fragment kernel (32 rows per wave) that large
batches take; before and after a training step, which must refresh the packed
weights.  Tolerances are those of the other network tests (BF16 activations:
2e-3 of the largest value, 2e-2 in the norm of the gradient)."""
import numpy as np
import pytest
import torch

import mlp_oracle as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 15, 17, 64, 65, 129, 49159])
def test_network_kernel(cuda, rows):
    print(f"[gpu] network kernel, {rows} rows", flush=True)
    from acehip.mlp import MLPEnsemble
    rng = np.random.default_rng(rows)
    ens = MLPEnsemble(nmemb=2, nin=152, seed=5)
    X = np.zeros((rows, 160))
    X[:, :152] = rng.normal(size=(rows, 152))
    Xt = torch.as_tensor(M.bf16(X).astype(np.float32)).to(torch.bfloat16).cuda()
    sel = np.unique(np.concatenate([np.arange(min(rows, 70)), np.arange(max(0, rows - 70), rows)]))
    for step in range(2):
        P = ens.get_params()
        y0, (y, dX) = ens.predict(Xt), ens.predict_grad(Xt)
        assert torch.equal(y0, y)
        for m in range(2):
            yr, cache = M.forward(P[m], X[sel])
            _, dXr = M.backward(P[m], cache, np.ones(len(sel)))
            assert np.max(np.abs(y[m].cpu().numpy()[sel] - yr)) < 2e-3 * max(1.0, np.max(np.abs(yr)))
            d = dX[m].cpu().numpy()[sel]
            assert np.linalg.norm(d - dXr) / np.linalg.norm(dXr) < 2e-2
        ens.train_step(Xt[:64], torch.zeros(min(rows, 64), device="cuda"), 0.05)
