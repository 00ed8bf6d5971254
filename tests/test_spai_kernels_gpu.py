"""The learned preconditioner's dense and reduction kernels past the sizes where
their launch changes: 131,072 rows (tiles per wavefront), 512 tiles of 256 rows
(partials of the weight gradients)."""
import os
import sys

import numpy as np
import pytest
import torch

from tnl_amd import spai

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import spai_oracle as SO  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 63, 65, 131071, 131072, 131073, 131072 + 255, 300001])
def test_dense_layer(rows):
    g = torch.Generator(device="cuda").manual_seed(rows)
    X = torch.randn(rows, 64, generator=g, device="cuda").bfloat16()
    W = torch.randn(64, 64, generator=g, device="cuda").bfloat16()
    want = X.double() @ W.double()
    # exact products, 64 of them added in FP32
    assert float((spai.bf16_gemm64(X, W) - want).abs().max()) <= 64 * 2 ** -24 * float((X.double().abs() @ W.double().abs()).max())


def test_gradients_of_many_edges():
    m = 164  # 133,824 edges: 523 tiles, 4 tiles per wavefront
    A, _ = spai.convdiff_matrix(m, 3)
    off, cols, vals, _ = spai.convdiff(m, 3)
    p = spai.init_parameters(5)
    p[-65:] = 0.05 * np.random.default_rng(6).standard_normal(65)
    net = spai.Network(p)
    Z = np.random.default_rng(7).integers(0, 2, (1, m * m)) * 2.0 - 1.0
    loss, _ = net.loss_grad(A, torch.from_numpy(Z).cuda())
    want_loss, want, _ = SO.loss_and_grad(p.astype(np.float64), off, cols, vals, Z, bf=True)
    assert abs(loss - want_loss) <= 1e-3 * want_loss
    got, k = net.gradients().astype(np.float64), 0
    for name, shape in SO.param_shapes():
        size = int(np.prod(shape))
        a, b = got[k:k + size], want[k:k + size]
        k += size
        # BF16 activations: values near a tie or zero fall either way (as tests/test_spai_gpu.py)
        assert np.linalg.norm(a - b) <= 3e-2 * max(np.linalg.norm(b), 1e-12), name
