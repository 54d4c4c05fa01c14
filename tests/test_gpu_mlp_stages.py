"""The network's stage kernel at the edges of its tiles, against the fp64 reference MLP
(oracle/mlp_ref.py): ragged widths and batches (tiles of 32, k steps of 16, passes of 304
or 608 k), one layer only, the four-tile blocks of large products (1,280 tiles and more), and
batches that shrink on one handle (the padding a larger batch left must not be read).

Tolerances: weights and activations are bf16 (relative rounding 2^-9 each), as in
test_gpu_mlp.py: 3e-2 for outputs and loss, 8e-2 for each gradient block, by relative L2 norm.
An Adam step is checked against the handle's own gradients: its result passes through fewer
than 16 fp32 roundings (2^-24 each) and is stored in fp32.
"""
import ctypes

import numpy as np
import pytest

import epirust_amd as G
from oracle import mlp_ref as M
from tests.gpu_helpers import say
from tests.test_gpu_mlp import make_mlp, params_of, rel

pytestmark = pytest.mark.gpu

CASES = [
    ([1, 1], [1]),
    ([9, 33, 31], [33, 1]),
    ([17, 130, 640, 5], [257, 64, 31]),
    ([9, 512, 600], [512, 500, 16]),
    ([3, 1280, 1056, 7], [1040, 1000]),  # 33 x 40 and 33 x 33 tiles forward, 40 x 33 for the weights
]


@pytest.mark.parametrize("widths,batches", CASES)
def test_stages_at_tile_edges(widths, batches):
    say("[mlp stages] %s batches %s" % (widths, batches))
    rng = np.random.default_rng(sum(widths))
    h = make_mlp(widths, max(batches))
    lr = 1e-3
    for B in batches:
        p = params_of(h)
        x = rng.uniform(0, 1, (B, widths[0])).astype(np.float32)
        t = rng.uniform(0, 1, (B, widths[-1])).astype(np.float32)
        y = np.zeros((B, widths[-1]), dtype=np.float32)
        assert G.lib().epi_mlp_forward(h, x.ctypes.data, B, y.ctypes.data) == 0
        y_ref, _ = M.forward(p, widths, x)
        assert rel(y, y_ref) < 3e-2
        g = np.zeros_like(p)
        loss = ctypes.c_float()
        assert G.lib().epi_mlp_gradients(h, x.ctypes.data, t.ctypes.data, B, g.ctypes.data, ctypes.byref(loss)) == 0
        l_ref, g_ref = M.loss_and_grad(p, widths, x, t)
        assert abs(loss.value - l_ref) / l_ref < 3e-2
        o = 0
        for k, n in zip(widths[:-1], widths[1:]):
            for size in (k * n, n):
                assert rel(g[o:o + size], g_ref[o:o + size]) < 8e-2, "batch %d, layer block at %d" % (B, o)
                o += size
        assert np.array_equal(params_of(h), p)  # gradients leave the parameters alone
        # the first Adam step after the parameters are set: p - lr g / (|g| + eps)
        assert G.lib().epi_mlp_set_params(h, p.ctypes.data, len(p)) == 0
        assert G.lib().epi_mlp_train_step(h, x.ctypes.data, t.ctypes.data, B, lr, None) == 0
        g64, p64 = g.astype(np.float64), p.astype(np.float64)
        want = p64 - lr * g64 / (np.abs(g64) + 1e-8)
        ok = np.abs(g64) > 1e-15  # the square of a smaller one leaves fp32's normal range
        err = np.abs(params_of(h) - want)[ok]
        assert np.all(err <= 16 * 2.0 ** -24 * lr + 2.0 ** -24 * np.abs(want[ok]))
    G.lib().epi_mlp_destroy(h)
