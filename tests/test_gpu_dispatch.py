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


def _gemv(ctx, m, xq, xs, xsum, rows, exact=False):
    import torch
    ntok = xq.shape[0]
    out = torch.full((ntok, rows), float("nan"), dtype=torch.float32, device="cuda")
    ctx.set_exact(exact)
    try:
        ctx.gemv(m, _t(xq), _t(xs), _t(xsum), out, ntok=ntok, out_stride=rows)
        ctx.sync()
    finally:
        ctx.set_exact(False)
    return out.cpu().numpy()


# one and several 16-token blocks per wave, partial blocks, a tail stripe, rows past the end of
# the last stripe, scale groups of one, two and four chunks with a ragged last group
@pytest.mark.parametrize("rows,cols,sgc,ntok", [(16, 64, 1, 16), (48, 320, 2, 17), (1030, 2048, 2, 64),
                                                (2048, 576, 4, 200), (5000, 192, 2, 130)])
@pytest.mark.parametrize("lane", [True, False])
def test_mfma_nf3_equals_reference_chain(gpu_ctx, rows, cols, sgc, ntok, lane):
    """NF3 batches of 16 or more tokens, stripe-chunks in lane order and in the reference's:
    every output bit-identical to the oracle's per-token chain in chunk order, both modes."""
    import oracle as O
    from helpers import acts, random_nf_streams
    rng = np.random.default_rng(rows + cols + ntok)
    idx, sc, pair, tail = random_nf_streams(rng, rows, cols, sgc, bits=3)
    cb = np.array([-127, -79, -45, -14, 14, 45, 79, 127] + 8 * [0], np.int8)
    dp, dt = _t(pair if pair.size else np.zeros(16, np.uint8)), _t(tail if tail.size else np.zeros(16, np.uint8))
    m = gpu_ctx.wrap_nf(rows, cols, 3, sgc, cb, dp, pair.size, dt if tail.size else None, tail.size)
    if lane:
        m.nf3_lane_order()
    base = [acts(rng, cols, 20, outlier_frac=0.001, outlier_scale=30.0)]
    xq, xs, xsum = (np.concatenate([a] * -(-ntok // 20))[:ntok] for a in base[0])
    xs[3, 0] = 0.0
    xq[3, :64] = 0
    ref = np.stack([O.nf_gemv(pair, tail, rows, cols, 3, sgc, cb, xq[t], xs[t]) for t in range(min(ntok, 24))])
    for exact in (False, True):
        out = _gemv(gpu_ctx, m, xq, xs, xsum, rows, exact)
        assert np.array_equal(out[:ref.shape[0]].view(np.uint32), ref.view(np.uint32))
        assert np.array_equal(out[24:].view(np.uint32), out[4:][np.arange(ntok - 24) % 20].view(np.uint32)) \
            if ntok > 24 else True
    m.close()
