"""The gradients of act(X) W from a float32 dY (dtc_gcn_input_grad,
dtc_gcn_weight_grad) against the float64 products of the operands as the
kernels round them to bf16."""
import numpy as np
import pytest
import torch

from helpers import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("x_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("relu", [False, True])
# partial 64-row tiles and 32-row steps, one and several partials of dW, a K
# that ends inside a 64-wide tile, one and several tiles each way
@pytest.mark.parametrize("M,K,F", [(1, 32, 64), (33, 96, 64), (100, 64, 192), (1000, 288, 128), (5003, 256, 256),
                                   (70001, 32, 64)])
def test_gradients_vs_float64(x_dtype, relu, M, K, F):
    """Float32 accumulation: within (terms) 2^-24 of the sum of magnitudes,
    terms = F or M; the rounding to bf16 adds 2^-8 of the value."""
    from dtc import load_extension
    ext = load_extension()
    g = torch.Generator().manual_seed(M + K)
    X = torch.randn(M, K, generator=g).to(x_dtype).cuda()
    W = (torch.randn(K, F, generator=g) / 8).to(torch.bfloat16).cuda()
    dY = torch.randn(M, F, generator=g).cuda()
    say("gcn gradients", M, K, F, x_dtype, relu)
    dX, dW = ext.gcn_gradients(dY, X, W, relu, True, True)
    assert dX.dtype == x_dtype and dX.shape == X.shape and dW.dtype == torch.bfloat16 and dW.shape == W.shape
    y = dY.to(torch.bfloat16).double().cpu().numpy()
    w = W.double().cpu().numpy()
    x = X.double().cpu()
    a = (torch.relu(x) if relu else x).to(torch.bfloat16).double().numpy()
    mask = (x.numpy() > 0) if relu else 1.0
    ref, mag = (y @ w.T) * mask, np.abs(y) @ np.abs(w).T
    assert np.all(np.abs(dX.double().cpu().numpy() - ref) <= F * 2.0 ** -24 * mag + 2.0 ** -8 * np.abs(ref))
    ref, mag = a.T @ y, np.abs(a).T @ np.abs(y)
    assert np.all(np.abs(dW.double().cpu().numpy() - ref) <= M * 2.0 ** -24 * mag + 2.0 ** -8 * np.abs(ref))
    again = ext.gcn_gradients(dY, X, W, relu, False, True)
    assert again[0] is None and torch.equal(again[1], dW)
