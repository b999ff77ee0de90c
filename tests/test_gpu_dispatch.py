"""Kernels and dispatch rules at the sizes where they can go wrong: one test per kernel,
over the edges of its tiles, remainders, and the smallest and largest of its range."""
import numpy as np
import pytest

import k2t  # noqa: F401

pytestmark = pytest.mark.gpu


def _t(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _act_buffers(ntok, K):
    import torch
    new = lambda s, t: torch.empty(s, dtype=t, device="cuda")  # noqa: E731
    return new((ntok, K), torch.int8), new((ntok, K // 64), torch.float32), new((ntok, K // 64), torch.int32)


def _inv_rms_tree(x, eps):
    """rmsnorm_quant_kernel's sum of squares: 256 chains of fmaf (one rounding each; the
    product of two floats is exact in float64), butterflies inside the 32-lane halves, the
    halves, then the four waves pairwise."""
    K = x.shape[1]
    pad = -K % 256
    v = np.pad(x, ((0, 0), (0, pad))).astype(np.float64).reshape(x.shape[0], -1, 256)
    s = np.zeros((x.shape[0], 256), np.float32)
    for i in range(v.shape[1]):
        s = (v[:, i] * v[:, i] + s.astype(np.float64)).astype(np.float32)
    s = s.reshape(-1, 4, 2, 32)
    for m in (1, 2, 4, 8, 16):
        s = s + s[..., np.arange(32) ^ m]
    w = s[..., 0, 0] + s[..., 1, 0]
    tot = (w[:, 0] + w[:, 1]) + (w[:, 2] + w[:, 3])
    one = np.float32(1.0)
    return one / np.sqrt(tot / np.float32(K) + np.float32(eps), dtype=np.float32)


# one chunk; partial and whole groups of eight loads; several chunks per wave (many tokens);
# more chunks than the Hadamard sign table holds (512)
@pytest.mark.parametrize("K,ntok", [(64, 1), (576, 3), (2048, 1), (2112, 200), (4160, 2), (1920, 1100), (32832, 2)])
def test_rmsnorm_quant_equals_split_form(gpu_ctx, K, ntok):
    """k2t_act_quant_rmsnorm gives, bit for bit, what k2t_act_quant gives for the inv_rms of
    its own summation order; a zero row gives zero codes and scales."""
    rng = np.random.default_rng(K + ntok)
    x = rng.standard_normal((ntok, K)).astype(np.float32)
    x[:, rng.integers(0, K)] *= 30.0
    if ntok > 1:
        x[1] = 0.0
    w = (1 + 0.1 * rng.standard_normal(K)).astype(np.float32)
    got, want = _act_buffers(ntok, K), _act_buffers(ntok, K)
    gpu_ctx.act_quant_rmsnorm(_t(x), _t(w), 1e-5, *got, K, ntok)
    gpu_ctx.act_quant(_t(x), *want, K, ntok, norm_w=_t(w), inv_rms=_t(_inv_rms_tree(x, 1e-5)))
    gpu_ctx.sync()
    for a, b in zip(got, want):
        assert np.array_equal(a.cpu().numpy(), b.cpu().numpy())
    if ntok > 1:
        assert not got[0][1].any() and not got[1][1].any()
