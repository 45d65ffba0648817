"""The single-pass quantizer kernels (rows of 32-, 64- and 128-value groups, either layout) at the
edges of their tiles, bit for bit against the oracle: fewer columns than a tile, a ragged last
tile in both directions, values on rounding ties, constant groups, and scales so small or large
that the reciprocal of the scale is no longer a normal number."""
import numpy as np
import pytest

from oracle import gptq

pytestmark = pytest.mark.gpu


def weights(K, N, seed):
    g = np.random.default_rng(seed)
    W = g.standard_normal((K, N)).astype(np.float32)
    W[:, 0] = 0.25                                       # constant: scale 1e-8
    W[:, 1] = np.round(W[:, 1] * 4) / 2                  # quotients on ties
    W[:, 2] = np.linspace(0, 15, K).astype(np.float32)
    W[:, 3] += 300.0                                     # far from zero: the zero point clips
    W[:, 4] = 0.0
    return W


@pytest.mark.parametrize("dt", [np.float16, np.float32])
@pytest.mark.parametrize("from_out_in", [False, True])
@pytest.mark.parametrize("K,N,gs,bits", [(32, 8, 32, 4), (288, 72, 32, 8), (64, 136, 64, 4), (320, 264, 64, 8),
                                         (128, 8, 128, 8), (640, 1000, 128, 4), (96, 56, 96, 4)])
def test_quantizer_tiles_bit_exact(gpu, K, N, gs, bits, from_out_in, dt):
    import torch
    from webpytorch_amd import core
    W = weights(K, N, K + N).astype(dt)
    if dt == np.float32:
        W[:, 5] *= np.float32(2.0 ** -120)               # 1 / scale past the normal range
        W[:, 6] *= np.float32(2.0 ** 118)
    want = gptq.gptq_quantize(W.astype(np.float32), gs, bits)
    src = torch.from_numpy(np.ascontiguousarray(W.T if from_out_in else W)).cuda()
    for t in (src, torch.cat([src.reshape(-1)[:1], src.reshape(-1)])[1:].view(src.shape)):  # aligned, then not
        got = core.gptq_quantize(t, gs, bits, from_out_in=from_out_in)
        for a, b in zip(got[:3], want[:3]):
            np.testing.assert_array_equal(a.cpu().numpy(), b)
