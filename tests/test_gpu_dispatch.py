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
                                                (2048, 576, 4, 200), (5000, 192, 2, 130), (1030, 4160, 2, 40)])
@pytest.mark.parametrize("lane", [True, False])
def test_mfma_nf3_equals_reference_chain(gpu_ctx, rows, cols, sgc, ntok, lane):
    """NF3 batches of 16 or more tokens, stripe-chunks in lane order and in the reference's:
    in exact mode every output is bit-identical to the oracle's per-token chain in chunk order,
    otherwise to the one-token GEMV's."""
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
        want = ref
        if not exact:
            want = np.concatenate([_gemv(gpu_ctx, m, xq[t:t + 1], xs[t:t + 1], xsum[t:t + 1], rows) for t in range(min(ntok, 24))])
        assert np.array_equal(out[:want.shape[0]].view(np.uint32), want.view(np.uint32))
        assert np.array_equal(out[24:].view(np.uint32), out[4:][np.arange(ntok - 24) % 20].view(np.uint32)) \
            if ntok > 24 else True
    m.close()


def _matrix(ctx, rng, fmt, rows, cols, sgc=2):
    """A matrix of random codes in any format (bit planes b4 .. b6, NF4, NF3)."""
    from helpers import random_nf_streams, random_nibble4_streams
    if fmt[0] == "b":
        pair, tail = random_nibble4_streams(rng, rows, cols, int(fmt[1]) - 4)
        return ctx.upload_nibble4(rows, cols, int(fmt[1]) - 4, pair, tail)
    bits = int(fmt[2])
    _, _, pair, tail = random_nf_streams(rng, rows, cols, sgc, bits=bits)
    cb = np.sort(rng.choice(np.arange(-127, 128), 16, replace=False)).astype(np.int8)
    return ctx.upload_nf(rows, cols, bits, sgc, cb, pair, tail)


# stripe mode and pair mode (512 or more stripes), one and several rounds of a wave's chunks,
# ragged last rounds, a tail stripe, rows past the last stripe's end, 2 and 15 tokens
@pytest.mark.parametrize("fmt", ["nf4", "nf3", "b4", "b5", "b6"])
@pytest.mark.parametrize("rows,cols,ntok", [(16, 64, 2), (40, 576, 15), (1030, 4160, 5), (8208, 192, 3),
                                            (8300, 2112, 11), (9000, 8256, 4)])
def test_small_batch_gemv_equals_one_token(gpu_ctx, fmt, rows, cols, ntok):
    """2 .. 15 tokens: each token's outputs are the one-token GEMV's bit for bit (the same
    exact chunk dots, summed in the same order), also for a stripe range and with the number
    of K segments capped; outputs outside the range stay untouched."""
    import torch
    from helpers import acts
    rng = np.random.default_rng(rows + cols + ntok)
    m = _matrix(gpu_ctx, rng, fmt, rows, cols)
    xq, xs, xsum = acts(rng, cols, ntok, outlier_frac=0.001, outlier_scale=30.0)
    xs[ntok - 1, 0] = 0.0
    xq[ntok - 1, :64] = 0
    xsum[ntok - 1, 0] = 0
    out = _gemv(gpu_ctx, m, xq, xs, xsum, rows)
    one = np.concatenate([_gemv(gpu_ctx, m, xq[t:t + 1], xs[t:t + 1], xsum[t:t + 1], rows) for t in range(ntok)])
    assert np.array_equal(out.view(np.uint32), one.view(np.uint32))
    s0, s1 = m.info()[2] // 3, -(-2 * m.info()[2] // 3)
    part = [torch.full((ntok, rows + 3), 7.0, device="cuda") for _ in range(2)]
    args = _t(xq), _t(xs), _t(xsum)
    gpu_ctx.set_splitk(3)
    try:
        gpu_ctx.gemv(m, *args, part[0], ntok=ntok, s0=s0, s1=s1, out_stride=rows + 3)
        for t in range(ntok):
            gpu_ctx.gemv(m, args[0][t], args[1][t], args[2][t], part[1][t], s0=s0, s1=s1)
        gpu_ctx.sync()
    finally:
        gpu_ctx.set_splitk(0)
    a, b = (p.cpu().numpy() for p in part)
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    assert np.all(a[:, s1 * 16:] == 7.0) and np.all(a[:, :s0 * 16] == 7.0)
    m.close()


# the activation in LDS: stripe and pair mode, segments of 16 chunks, of a round and a few, of less than a
# round; 2, 3 and 4 tokens, more of them dealt to several workgroups; the shortest rows that take it
@pytest.mark.parametrize("fmt", ["nf4", "nf3", "b4", "b5", "b6"])
@pytest.mark.parametrize("rows,cols,ntok", [(1030, 4160, 4), (1040, 16384, 7), (8300, 8256, 3), (8208, 16320, 2), (40, 1600, 4),
                                            (48, 1088, 3), (64, 12288, 13)])
def test_few_tokens_equal_one_token(gpu_ctx, fmt, rows, cols, ntok):
    """The same bits with up to four tokens a workgroup."""
    test_small_batch_gemv_equals_one_token(gpu_ctx, fmt, rows, cols, ntok)


# the batched GEMV's kernels at their edges: K dealt over a workgroup with 1, 2 and 4 blocks of
# tokens, from rows and from tiles, ragged rounds and a tail stripe; a wave per stripe (512 or more
# stripes, up to 32 tokens); 64-token and 128-token tiles, partial ones, a last stage of one chunk,
# stripe counts that end inside a pair
@pytest.mark.parametrize("fmt", ["nf4", "nf3", "b4", "b5", "b6"])
@pytest.mark.parametrize("rows,cols,ntok", [(40, 64, 16), (1030, 1088, 17), (1040, 4160, 40), (2064, 1984, 130),
                                            (8200, 320, 16), (8200, 576, 31), (8200, 448, 33), (8300, 1088, 129),
                                            (16400, 320, 200)])
def test_batched_gemv_equals_exact_passes(gpu_ctx, fmt, rows, cols, ntok):
    """16 or more tokens on the matrix cores: every output equals the exact-order 4-token passes
    bit for bit (the same chain in chunk order), and nothing outside the outputs is written."""
    import torch
    from helpers import acts
    rng = np.random.default_rng(rows + cols + ntok)
    m = _matrix(gpu_ctx, rng, fmt, rows, cols)
    xq, xs, xsum = acts(rng, cols, ntok, outlier_frac=0.001, outlier_scale=30.0)
    xs[ntok - 1, 0] = 0.0
    xq[ntok - 1, :64] = 0
    xsum[ntok - 1, 0] = 0
    args = _t(xq), _t(xs), _t(xsum)
    out = [torch.full((ntok + 1, rows + 3), 7.0, device="cuda") for _ in range(2)]
    gpu_ctx.set_exact(True)
    try:
        for k, mfma in enumerate((True, False)):
            gpu_ctx.set_mfma(mfma)
            gpu_ctx.gemv(m, *args, out[k], ntok=ntok, out_stride=rows + 3)
        gpu_ctx.sync()
    finally:
        gpu_ctx.set_mfma(True)
        gpu_ctx.set_exact(False)
    a, b = (o.cpu().numpy() for o in out)
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    assert np.all(a[ntok:] == 7.0) and np.all(a[:, rows:] == 7.0)
    m.close()


# three and more blocks of tokens on a wave per stripe and block: K dealt over a workgroup would be a
# round and a few workgroups (313 and 626 of them), or mostly padding (nine chunks); more tiles than CUs
@pytest.mark.parametrize("fmt", ["nf4", "nf3", "b4", "b6"])
@pytest.mark.parametrize("rows,cols,ntok", [(5000, 2112, 48), (5000, 2112, 90), (3080, 576, 70), (6160, 1088, 65)])
def test_batched_gemv_of_a_wave_per_block(gpu_ctx, fmt, rows, cols, ntok):
    """The same bits on the wave-per-stripe kernel beyond 32 tokens."""
    test_batched_gemv_equals_exact_passes(gpu_ctx, fmt, rows, cols, ntok)


# the ordered kernel with 1, 2 and 4 blocks of tokens, stripe and pair mode, partial blocks, ragged
# segments, a tail stripe; the 16-token passes of small products, one block over many stripes, short
# rows; K segments capped at 3 (more visits per accumulator than one) and at 1
@pytest.mark.parametrize("rows,cols,ntok", [(4000, 9280, 16), (2064, 8960, 20), (1030, 4160, 200), (8208, 1088, 130),
                                            (8300, 2112, 70), (8300, 4160, 16), (8200, 576, 37), (40, 64, 17)])
@pytest.mark.parametrize("cap", [0, 3, 1])
def test_nf3_batch_equals_one_token(gpu_ctx, rows, cols, ntok, cap):
    """NF3 batches of 16 or more tokens: each token's outputs are the one-token GEMV's bit for bit,
    and nothing outside the outputs is written."""
    import torch
    from helpers import acts
    rng = np.random.default_rng(rows + cols + ntok)
    m = _matrix(gpu_ctx, rng, "nf3", rows, cols)
    m.nf3_lane_order()
    xq, xs, xsum = acts(rng, cols, ntok, outlier_frac=0.001, outlier_scale=30.0)
    xs[ntok - 1, 0] = 0.0
    xq[ntok - 1, :64] = 0
    args = _t(xq), _t(xs), _t(xsum)
    out = [torch.full((ntok + 1, rows + 3), 7.0, device="cuda") for _ in range(2)]
    gpu_ctx.set_splitk(cap)
    try:
        gpu_ctx.gemv(m, *args, out[0], ntok=ntok, out_stride=rows + 3)
        for t in range(ntok):
            gpu_ctx.gemv(m, args[0][t], args[1][t], args[2][t], out[1][t])
        gpu_ctx.sync()
    finally:
        gpu_ctx.set_splitk(0)
    a, b = (o.cpu().numpy() for o in out)
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    assert np.all(a[ntok:] == 7.0) and np.all(a[:, rows:] == 7.0)
    m.close()


# gate_up with the SwiGLU epilogue in 64-token (n 250) and 128-token tiles (n 300), qkv's epilogue in
# 64-token tiles (28 heads x 19 token blocks, int8 cache) and 16-token ones, partial tiles in each
@pytest.mark.parametrize("fmt,planes,kv_bits,n", [("nf4", None, 8, 250), ("nf4", None, 4, 300), ("n4", "p55454", 8, 300)])
def test_prefill_epilogues_equal_separate_kernels(gpu_ctx, fmt, planes, kv_bits, n):
    """A prefill whose qkv and gate_up products end in the fused epilogues gives the logits of
    the one with separate kernels (mode 2), bit for bit, and so does a decode step after it."""
    from model_oracle import random_model
    from test_gpu_model import P55454, _gpu_model
    cfg = dict(n_layers=2, hidden=256, n_heads=20, n_kv_heads=4, head_dim=64, intermediate=8192, vocab=520, max_seq=400,
               rms_eps=1e-5, rope_theta=10000.0)
    layers, head, fn = random_model(cfg, seed=43, fmt=fmt, planes=P55454 if planes else None)
    gm, mats = _gpu_model(gpu_ctx, cfg, layers, head, fn, max_batch=320)
    gm.set_kv_bits(kv_bits)
    toks = np.random.default_rng(44).integers(0, cfg["vocab"], n).astype(np.int32)
    got = {}
    try:
        for mode in (1, 2):
            gpu_ctx.set_mfma(mode)
            gm.reset()
            got[mode] = gm.prefill(toks, want_logits=True), gm.decode(3)
    finally:
        gpu_ctx.set_mfma(True)
        gm.close()
        for m in mats:
            m.close()
    for a, b in zip(got[1], got[2]):
        assert np.isfinite(a).all() and np.array_equal(a.view(np.uint32), b.view(np.uint32))


# the NF4 cache: 100 heads x 25 token blocks are 16-token workgroups, x 26 are 64-token tiles
@pytest.mark.parametrize("n", [400, 401])
def test_qkv_epilogue_of_the_nf4_cache(gpu_ctx, n):
    """The fused epilogue of many heads gives the logits of the separate kernel (mode 2), bit for
    bit, and so does a decode step after it (which reads the stored cache)."""
    from model_oracle import random_model
    from test_gpu_model import _gpu_model
    cfg = dict(n_layers=1, hidden=256, n_heads=92, n_kv_heads=4, head_dim=64, intermediate=256, vocab=128, max_seq=416,
               rms_eps=1e-5, rope_theta=10000.0)
    layers, head, fn = random_model(cfg, seed=45, fmt="nf4")
    gm, mats = _gpu_model(gpu_ctx, cfg, layers, head, fn, max_batch=416)
    gm.set_kv_bits(4)
    toks = np.random.default_rng(46).integers(0, cfg["vocab"], n).astype(np.int32)
    got = {}
    try:
        for mode in (1, 2):
            gpu_ctx.set_mfma(mode)
            gm.reset()
            got[mode] = gm.prefill(toks, want_logits=True), gm.decode(3)
    finally:
        gpu_ctx.set_mfma(True)
        gm.close()
        for m in mats:
            m.close()
    for a, b in zip(got[1], got[2]):
        assert np.isfinite(a).all() and np.array_equal(a.view(np.uint32), b.view(np.uint32))


# all experts used by every token (items of 16 and a remainder), and few tokens over many
# experts; the wide router (d > 2048); a shared expert (its width), on the 4-token passes (three-chunk
# scale groups) and with 2-chunk ones on the matrix cores, at fewer and more than 16 tokens a call;
# more tokens than one MoE call takes; enough pairs per expert for a workgroup to take several stripes
@pytest.mark.parametrize("bits,E,k,d,ntok,max_batch,shared", [(3, 4, 4, 256, 40, 64, 0), (4, 16, 3, 256, 2, 8, 0),
                                                              (3, 32, 6, 256, 15, 15, 128), (4, 8, 2, 2112, 9, 16, 0),
                                                              (3, 4, 2, 256, 37, 8, 128), (3, 4, 4, 320, 500, 500, 0),
                                                              (4, 4, 4, 576, 500, 500, 0), (3, 4, 2, 256, 40, 64, 1024),
                                                              (4, 4, 2, 320, 150, 160, 1088), (3, 4, 2, 256, 20, 12, 1024)])
def test_moe_prompt_equals_token_by_token(gpu_ctx, bits, E, k, d, ntok, max_batch, shared):
    """A prompt through sparse-MoE layers (tokens grouped by expert) gives the logits of
    decoding its tokens one by one, bit for bit.  (Three-chunk scale groups and the NF4 KV
    cache keep the attention half on kernels with that property at any batch size.)"""
    import oracle as O
    from k2tb_writer import random_moe_layer, write_k2tm
    cfg = dict(n_layers=2, hidden=d, n_heads=4, n_kv_heads=2, head_dim=64, intermediate=64, vocab=300, max_seq=512,
               rms_eps=1e-6, rope_theta=10000.0)
    rng = np.random.default_rng(E * 100 + ntok)
    dff, hd = 192 if ntok < 500 else 1088, 64
    w = lambda r, c: (rng.standard_normal((r, c)) * 0.02).astype(np.float32)  # noqa: E731
    moe = [random_moe_layer(rng, d, dff, E, bits=bits) for _ in range(2)]
    bank = k2t.ExpertBank.upload(gpu_ctx, write_k2tm([m[0] for m in moe], d, dff, bits, 2))
    m = k2t.Model(gpu_ctx, cfg, max_batch=max_batch)
    mats = []

    def up(rows, cols, sgc=3, b=4):
        W = w(rows, cols)
        cb, mu = O.nf_fit_codebook(W, b, sgc)
        idx, sc = O.nf_rtn(W, b, sgc, cb, mu)
        mats.append(gpu_ctx.upload_nf(rows, cols, b, sgc, cb, *O.nf_from_indices(idx, sc, rows, cols, b, sgc)))
        return mats[-1]

    for i in range(2):
        m.set_layer(i, up((4 + 4) * hd, d), up(d, 4 * hd), None, None, 1 + w(1, d)[0], 1 + w(1, d)[0])
        m.set_moe(i, bank, i, moe[i][1], k, True, i, router_bias=w(1, E)[0] if i else None)
        if shared:
            sgc = 3 if shared == 128 else 2
            m.set_moe_shared(i, up(2 * shared, d, sgc), up(d, shared, sgc, 4 if i else bits), w(1, d)[0] if i else None)
    m.set_head(up(300, d), np.ones(d, np.float32))
    m.set_kv_bits(4)
    toks = rng.integers(0, 300, ntok).astype(np.int32)
    a = m.prefill(toks)
    m.reset()
    for t in toks:
        b = m.decode(int(t))
    assert np.isfinite(a).all() and np.array_equal(a.view(np.uint32), b.view(np.uint32))
    m.close()
    for x in mats:
        x.close()
    bank.close()


# more heads than may wait in one launch (half the CUs): split partials and a merge
@pytest.mark.parametrize("nq,nkv,hd,seq,window", [(136, 136, 64, 1100, 0), (512, 64, 64, 300, 0), (600, 150, 128, 700, 300)])
@pytest.mark.parametrize("bits", [8, 4])
def test_attention_of_many_heads(gpu_ctx, nq, nkv, hd, bits, seq, window):
    """A call of many heads gives each group of them what a call of its own gives (4e-5 of the
    largest output: two fp32 orders), and never waits for workgroups that have no place to run."""
    import torch
    rng = np.random.default_rng(nq + seq)
    cap, sinks = (window + 512, 4) if window else (seq, 0)
    codes = [torch.empty((nkv, cap, hd if bits == 8 else hd // 2), dtype=torch.int8, device="cuda") for _ in range(2)]
    scales = [torch.empty((nkv, cap, 1 if bits == 8 else hd // 64), device="cuda",
                          dtype=torch.float32 if bits == 8 else torch.bfloat16) for _ in range(2)]
    for c, s in zip(codes, scales):
        gpu_ctx.kv_store(bits, _t(rng.standard_normal((nkv * cap, hd)).astype(np.float32)), nkv * cap, hd, c, s)
    q = _t((2 * rng.standard_normal((nq, hd))).astype(np.float32))
    out, own = torch.full((nq, hd), float("nan"), device="cuda"), torch.full((nq, hd), float("nan"), device="cuda")
    for call in (gpu_ctx.attn_decode, gpu_ctx.attn_decode_noalloc):
        call(bits, q, nq, nkv, hd, codes[0], scales[0], codes[1], scales[1], cap, seq, hd ** -0.5, out, window, sinks)
        gpu_ctx.sync()
        g = nq // nkv
        for k in range(0, nkv, 10):
            n = min(10, nkv - k)
            gpu_ctx.attn_decode(bits, q[k * g:], n * g, n, hd, codes[0][k:], scales[0][k:], codes[1][k:], scales[1][k:], cap,
                                seq, hd ** -0.5, own[k * g:], window, sinks)
        assert (out - own).abs().max() <= 4e-5 * own.abs().max()


# one span (128- and 256-position form) and its edges, several spans, more spans than a merge
# thread polls at once; 1 .. 8 q heads per KV head; windows not yet full, full and wrapped
@pytest.mark.parametrize("nq,nkv,hd", [(3, 3, 64), (6, 2, 128), (8, 2, 64), (10, 2, 128), (8, 1, 64)])
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("seq,window,sinks", [(1, 0, 0), (127, 0, 0), (128, 0, 0), (129, 0, 0), (257, 0, 0), (1100, 0, 0),
                                              (9000, 0, 0), (90, 100, 4), (1300, 300, 4), (2777, 1001, 0)])
def test_span_attention_matches_reference(gpu_ctx, nq, nkv, hd, bits, seq, window, sinks):
    """Decode attention against float64 softmax attention over the cache as stored (codes times
    scales): 2e-5 of the largest output, about 40 ulp of fp32 for sums of up to 9000 terms."""
    import torch
    import oracle as O
    rng = np.random.default_rng(nq * 1000 + seq + bits)
    cap = window + 512 if window else seq + 3
    heads = rng.standard_normal((2, nkv * cap, hd)).astype(np.float32)
    q = (2 * rng.standard_normal((nq, hd))).astype(np.float32)
    codes = [torch.empty((nkv * cap, hd if bits == 8 else hd // 2), dtype=torch.int8, device="cuda") for _ in range(2)]
    scales = [torch.empty((nkv * cap, 1 if bits == 8 else hd // 64), device="cuda",
                          dtype=torch.float32 if bits == 8 else torch.bfloat16) for _ in range(2)]
    for i in range(2):
        gpu_ctx.kv_store(bits, _t(heads[i]), nkv * cap, hd, codes[i], scales[i])
    out = [torch.full((nq, hd), float("nan"), device="cuda") for _ in range(2)]
    args = (bits, _t(q), nq, nkv, hd, codes[0], scales[0], codes[1], scales[1], cap, seq, hd ** -0.5)
    gpu_ctx.attn_decode(*args, out[0], window, sinks)
    gpu_ctx.attn_decode_noalloc(*args, out[1], window, sinks)
    gpu_ctx.sync()
    # the stored values
    dense = []
    for i in range(2):
        c, s = codes[i].cpu().numpy(), scales[i].float().cpu().numpy().astype(np.float64)
        if bits == 8:
            v = c.astype(np.float64) * s
        else:
            cb = np.array([-127, -96, -75, -58, -44, -31, -18, -6, 6, 18, 31, 44, 58, 75, 96, 127], np.float64)
            b = c.view(np.uint8).reshape(-1, hd // 64, 2, 1, 16)  # [block][half][nibble][16]
            v = cb[np.concatenate([b & 15, b >> 4], axis=3)].reshape(-1, hd // 64, 64) * s[:, :, None]
        dense.append(v.reshape(nkv, cap, hd))
    pos = np.arange(seq)
    if window and seq > window:
        pos = np.concatenate([np.arange(sinks), np.arange(seq - (window - sinks), seq)])
    if window:
        pos = np.where(pos < sinks, pos, sinks + (pos - sinks) % (cap - sinks))
    ref = np.zeros((nq, hd))
    for h in range(nq):
        qi, qs = O.kv_quant_head(q[h])
        k, v = (d[h // (nq // nkv)][pos] for d in dense)
        s = k @ (qi.astype(np.float64) * float(qs)) * hd ** -0.5
        p = np.exp(s - s.max())
        ref[h] = O.ifwht64(((p / p.sum()) @ v).astype(np.float32))
    for o in out:
        assert np.abs(o.cpu().numpy() - ref).max() <= 2e-5 * np.abs(ref).max()


@pytest.mark.parametrize("nq,nkv,hd", [(4, 4, 64), (8, 2, 128), (8, 1, 64)])
@pytest.mark.parametrize("bits,window", [(8, 0), (4, 0), (8, 1100), (4, 1100)])
def test_span_attention_in_decode_steps(gpu_ctx, nq, nkv, hd, bits, window):
    """Decode steps of a model whose cache is sized for the span kernel (more than 1024
    positions) against the same model with a short cache (one workgroup per head): the
    current position's K / V built and stored in the launch, one span and several."""
    from model_oracle import random_model
    cfg = dict(n_layers=2, hidden=256, n_heads=nq, n_kv_heads=nkv, head_dim=hd, intermediate=256, vocab=200,
               rms_eps=1e-5, rope_theta=10000.0)
    layers, head, fn = random_model(cfg, seed=nq + hd, fmt="nf4")
    up = lambda m: gpu_ctx.upload_nf(m.rows, m.cols, 4, m.sgc, m.cb, m.pair, m.tail)  # noqa: E731
    mats = [[up(L[k]) for k in ("qkv", "o", "gu", "down")] for L in layers]
    hm = up(head)
    logits = []
    for max_seq, win in ((2048, window), (1000, 0)):
        m = k2t.Model(gpu_ctx, dict(cfg, max_seq=max_seq), max_batch=300)
        for i, L in enumerate(layers):
            m.set_layer(i, *mats[i], L["in_norm"], L["post_norm"])
        m.set_head(hm, fn)
        m.set_persistent(False)
        m.set_kv_bits(bits)
        if win:
            m.set_kv_window(win, 4)
        toks = np.random.default_rng(1).integers(0, 200, 300)
        got = [m.decode(int(t)) for t in toks[:3]]
        m.prefill(toks[3:254].astype(np.int32), want_logits=False)
        got += [m.decode(int(t)) for t in toks[254:260]]
        logits.append(np.stack(got))
        m.close()
    a, b = logits
    cos = (a * b).sum(1) / (np.linalg.norm(a, axis=1) * np.linalg.norm(b, axis=1))
    assert cos.min() > 0.9998 and np.isfinite(a).all()
    for x in [hm] + [x for r in mats for x in r]:
        x.close()


# spans of 128 positions (up to four q heads a group, and eight) and of 256; the last place of a span,
# then a span of one position; one span, then two; a full window whose ring wraps between the steps
@pytest.mark.parametrize("nq,nkv,hd,window,pos", [(4, 4, 64, 0, 1279), (32, 32, 64, 0, 1279), (8, 1, 128, 0, 1279),
                                                  (8, 2, 128, 0, 126), (8, 2, 128, 1100, 1611), (32, 32, 64, 1100, 1610)])
@pytest.mark.parametrize("bits", [8, 4])
def test_span_attention_stores_and_reads_the_current_position(gpu_ctx, nq, nkv, hd, window, pos, bits):
    """Decode steps through the span kernel against the same tokens as a batch of two (K / V stored
    by a launch of their own, split partials and a merge).  One layer, so the cache depends on
    the tokens alone and a batch has the one-token bits: a later step's logits are equal bit for
    bit only if the stored K / V are.  The steps' own logits agree to 5e-3 of their norm, a few
    moved int8 codes of the attention output (one is about 1.5e-3 of 256 elements); the first q head
    of each group has its K's projection, so the current position takes about half of the weight
    there, and a stale or missing row would move them by far more."""
    rng = np.random.default_rng(nq + hd + pos + bits)
    d, V = 256, 64
    up = lambda W: (lambda c: gpu_ctx.upload_nf(*W.shape, 4, 2, c[0], c[2], c[3]))(k2t.compile_nf4(W, 2))  # noqa: E731
    dense = lambda r, c: (0.1 * rng.standard_normal((r, c))).astype(np.float32)  # noqa: E731
    W = dense((nq + 2 * nkv) * hd, d)
    for g in range(nkv):
        q0 = g * (nq // nkv) * hd
        W[q0:q0 + hd] = W[(nq + g) * hd:(nq + g + 1) * hd]
    mats = [up(w) for w in (W, dense(d, nq * hd), dense(256, d), dense(d, 128), dense(V, d))]
    m = k2t.Model(gpu_ctx, dict(n_layers=1, hidden=d, n_heads=nq, n_kv_heads=nkv, head_dim=hd, intermediate=128, vocab=V,
                                rms_eps=1e-5, rope_theta=10000.0, max_seq=2048), max_batch=300)
    ones = np.ones(d, np.float32)
    m.set_layer(0, *mats[:4], ones, ones)
    m.set_qk_norm(0, np.ones(hd, np.float32), np.ones(hd, np.float32))
    m.set_head(mats[4], ones)
    m.set_persistent(False)
    m.set_kv_bits(bits)
    if window:
        m.set_kv_window(window, 4)
    toks = rng.integers(0, V, pos + 3).astype(np.int32)
    got = []
    for batch in (False, True):
        m.reset()
        m.prefill(toks[:pos], want_logits=False)
        if batch:
            last = m.prefill(toks[pos:pos + 2])
        else:
            m.decode(int(toks[pos]), want_logits=False)
            last = m.decode(int(toks[pos + 1]))
        got.append((last, m.decode(int(toks[pos + 2]))))
    (a, a3), (b, b3) = got
    assert np.linalg.norm(a - b) <= 5e-3 * np.linalg.norm(b) and np.isfinite(a).all()
    assert np.array_equal(a3.view(np.uint32), b3.view(np.uint32))
    m.close()
    for x in mats:
        x.close()


# banks of different expert counts on one context (its hand-off words are shared), calls with and
# without the route's outputs, the wide router (d > 2048)
def test_moe_ffn_calls_share_the_context_state(gpu_ctx):
    """Each call's hidden state and route equal those of the same call on a fresh context."""
    import torch
    from k2tb_writer import random_moe_layer, write_k2tm
    rng = np.random.default_rng(77)
    shapes = [(256, 128, 128, 8), (2112, 64, 8, 2), (256, 64, 16, 3)]
    banks, calls = [], []
    for d, dff, E, k in shapes:
        exp, router = random_moe_layer(rng, d, dff, E, bits=3)
        banks.append((write_k2tm([exp], d, dff, 3, 2), _t(np.asarray(router, np.float32)), d, k))

    def run(ctx, bank, i, x, outs):
        _, router, d, k = banks[i]
        h, ids, wts = x.clone(), torch.full((k,), -1, dtype=torch.int32, device="cuda"), torch.full((k,), -1.0, device="cuda")
        kw = dict(route_ids=ids, route_weights=wts) if outs else {}
        ctx.moe_ffn(bank, 0, router, h, torch.ones(d, device="cuda"), 1e-5, k, **kw)
        ctx.sync()
        return h, ids, wts

    shared = [k2t.ExpertBank.upload(gpu_ctx, b[0]) for b in banks]
    xs = [_t(rng.standard_normal(b[2]).astype(np.float32)) for b in banks]
    for i, outs in ((0, True), (1, True), (2, False), (0, False), (2, True), (1, False), (0, True)):
        calls.append((i, outs, run(gpu_ctx, shared[i], i, xs[i], outs)))
    want = []
    for i, b in enumerate(banks):
        ctx = k2t.Ctx(0)
        bank = k2t.ExpertBank.upload(ctx, b[0])
        want.append(run(ctx, bank, i, xs[i], True))
        bank.close()
        ctx.close()
    for i, outs, got in calls:
        assert torch.isfinite(got[0]).all() and torch.equal(got[0], want[i][0])
        if outs:
            assert torch.equal(got[1], want[i][1]) and torch.equal(got[2], want[i][2])
        else:
            assert (got[1] == -1).all() and (got[2] == -1).all()
    for bank in shared:
        bank.close()


# the router in the gate_up launch (d <= 2048) and in its own (above); one token and a batch
@pytest.mark.parametrize("d,E,k,scoring", [(256, 8, 4, 0), (256, 128, 8, 0), (256, 16, 16, 1), (256, 16, 3, 2), (2112, 8, 4, 0)])
@pytest.mark.parametrize("bad", ["bias", "hidden"])
def test_moe_routes_without_a_finite_logit(gpu_ctx, d, E, k, scoring, bad):
    """Logits that are all -inf (bias) or NaN (hidden state): softmax scores are NaN then.  The
    route is still k different experts of the bank in ascending order, a prompt with such a
    token ends, and the model's next prompts are those of a model that never saw one."""
    import torch
    from k2tb_writer import random_moe_layer, write_k2tm
    from model_oracle import quantize_matrix
    rng = np.random.default_rng(d + E + scoring)
    dff = 64
    exp, router = random_moe_layer(rng, d, dff, E, bits=3)
    bank = k2t.ExpertBank.upload(gpu_ctx, write_k2tm([exp], d, dff, 3, 2))
    bias = np.full(E, -np.inf if bad == "bias" else 0.0, np.float32)
    h = _t(rng.standard_normal(d).astype(np.float32))
    if bad == "hidden":
        h[5] = float("nan")
    ids = torch.full((k,), -1, dtype=torch.int32, device="cuda")
    for exact in (False, True):
        gpu_ctx.set_exact(exact)
        try:
            gpu_ctx.moe_ffn(bank, 0, _t(np.asarray(router, np.float32)), h, torch.ones(d, device="cuda"), 1e-5, k,
                            scoring=scoring, router_bias=_t(bias), route_ids=ids)
            gpu_ctx.sync()
        finally:
            gpu_ctx.set_exact(False)
        got = ids.cpu().numpy()
        assert (np.diff(got) > 0).all() and got[0] >= 0 and got[-1] < E
    cfg = dict(n_layers=1, hidden=d, n_heads=2, n_kv_heads=1, head_dim=64, intermediate=64, vocab=64, max_seq=64,
               rms_eps=1e-6, rope_theta=10000.0)
    m = k2t.Model(gpu_ctx, cfg, max_batch=32)
    w = lambda r, c: (rng.standard_normal((r, c)) * 0.02).astype(np.float32)  # noqa: E731
    mats = []
    for r, c in ((4 * 64, d), (d, 2 * 64), (64, d)):
        q = quantize_matrix(w(r, c), "nf4")
        mats.append(gpu_ctx.upload_nf(r, c, 4, q.sgc, q.cb, q.pair, q.tail))
    m.set_layer(0, mats[0], mats[1], None, None, np.ones(d, np.float32), np.ones(d, np.float32))
    m.set_moe(0, bank, 0, np.asarray(router, np.float32), k, True, scoring, router_bias=bias if bad == "bias" else None)
    m.set_head(mats[2], np.ones(d, np.float32))
    rows = rng.standard_normal((64, d)).astype(np.float32)
    if bad == "hidden":
        rows[63] = np.nan
    m.set_embedding(k2t.EMBED_F32, rows)
    toks = np.arange(20, dtype=np.int32)
    first = m.prefill(toks)
    m.reset()
    m.prefill(np.append(toks, 63).astype(np.int32))
    m.decode(63)
    m.reset()
    again = m.prefill(toks)
    assert np.array_equal(first.view(np.uint32), again.view(np.uint32))
    assert bad == "bias" or np.isfinite(first).all()
    m.close()
    for x in mats:
        x.close()
    bank.close()


def test_moe_layer_unchanged_by_a_failed_allocation(gpu_ctx):
    """k2t_model_set_moe / _shared whose batch workspace does not fit in the GPU's memory raise
    and leave the layer as it was: its prompts give the same logits as before, and the same
    calls succeed once there is memory."""
    import torch
    from k2tb_writer import random_moe_layer, write_k2tm
    rng = np.random.default_rng(5)
    d, dff, E, inter = 2048, 1024, 8, 8192
    exp, router = random_moe_layer(rng, d, dff, 1, bits=3)
    bank = k2t.ExpertBank.upload(gpu_ctx, write_k2tm([exp * E], d, dff, 3, 2))
    router = (0.05 * rng.standard_normal((E, d))).astype(np.float32)
    cfg = dict(n_layers=1, hidden=d, n_heads=2, n_kv_heads=1, head_dim=64, intermediate=64, vocab=64, max_seq=512,
               rms_eps=1e-6, rope_theta=10000.0)
    m = k2t.Model(gpu_ctx, cfg, max_batch=512)
    mats = [_matrix(gpu_ctx, rng, "nf4", r, c) for r, c in ((4 * 64, d), (d, 2 * 64), (64, d), (2 * inter, d), (d, inter))]
    m.set_layer(0, mats[0], mats[1], None, None, np.ones(d, np.float32), np.ones(d, np.float32))
    m.set_head(mats[2], np.ones(d, np.float32))
    m.set_moe(0, bank, 0, router, 2, False)
    toks = rng.integers(0, 64, 300).astype(np.int32)

    def logits():
        m.reset()
        return m.prefill(toks).view(np.uint32).copy()

    before = logits()
    room = torch.empty(1 << 25, dtype=torch.uint8, device="cuda")
    hold, size = [], 1 << 36
    while size >= 1 << 24:  # all but 32 .. 48 MiB; the workspaces need 59 (shared) and 73 MiB (top 8)
        try:
            hold.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
        except torch.OutOfMemoryError:
            size //= 2
    del room
    torch.cuda.empty_cache()
    try:
        for call in (lambda: m.set_moe_shared(0, mats[3], mats[4]), lambda: m.set_moe(0, bank, 0, router, 8, False)):
            with pytest.raises(k2t.K2TError, match="hipMalloc"):
                call()
            assert np.array_equal(logits(), before)
    finally:
        hold.clear()
        torch.cuda.empty_cache()
    m.set_moe(0, bank, 0, router, 8, False)
    top8 = logits()
    m.set_moe_shared(0, mats[3], mats[4])
    shared = logits()
    assert not np.array_equal(top8, before) and not np.array_equal(shared, top8)
    m.set_moe(0, bank, 0, router, 2, False)
    assert np.array_equal(logits(), before)
    m.close()
    for x in mats:
        x.close()
    bank.close()


# a product that the matrix cores take after a copy into tiles, and one that they take as its
# rows lie (no copy)
@pytest.mark.parametrize("rows,cols,ntok", [(1030, 4160, 64), (1040, 576, 80)])
def test_captured_nf3_batch_needs_no_scratch(rows, cols, ntok):
    """A captured NF3 batch keeps its outputs over replays while other calls use, and grow (so
    free), the context's scratch: the graph holds none of it.  Its bits are those of the same
    capture on a context that has not been used before."""
    import torch
    from helpers import acts
    rng = np.random.default_rng(rows)
    outs = []
    for used in (False, True):
        ctx, s = k2t.Ctx(0), torch.cuda.Stream()
        ctx.set_stream(s.cuda_stream)
        rng2 = np.random.default_rng(rows + 1)
        m, big = _matrix(ctx, rng2, "nf3", rows, cols), _matrix(ctx, rng2, "nf4", 64, 4160)
        a = [_t(x) for x in acts(rng2, cols, ntok)]
        n = 16 * ntok
        b = [_t(x) for x in acts(rng, 4160, 16)]
        b = [x.repeat(n // 16, 1) for x in b]
        out, bout = torch.zeros((ntok, rows), device="cuda"), torch.zeros((n, 64), device="cuda")
        torch.cuda.synchronize()
        if used:  # the scratch now holds the tiles of either product
            ctx.gemv(m, *a, out, ntok=ntok, out_stride=rows)
            ctx.gemv(big, *[x[:ntok] for x in b], bout, ntok=ntok, out_stride=64)
        ctx.sync()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            ctx.gemv(m, *a, out, ntok=ntok, out_stride=rows)
        for k in range(3):
            ctx.gemv(big, *[x[:(4 + 6 * k) * ntok] for x in b], bout, ntok=(4 + 6 * k) * ntok, out_stride=64)
            ctx.sync()
            out.zero_()
            torch.cuda.synchronize()
            with torch.cuda.stream(s):
                g.replay()
            torch.cuda.synchronize()
            outs.append(out.cpu().numpy().view(np.uint32))
        m.close()
        big.close()
        ctx.close()
    assert outs[0].any() and all(np.array_equal(outs[0], o) for o in outs[1:])


@pytest.mark.parametrize("fmt", ["nf3", "nf4", "b5"])
def test_batch_past_two_gib_of_activations(gpu_ctx, fmt):
    """Tokens past the first 2 GiB of int8 activations: their outputs are those of a call of their
    own (1e-5 of the largest: another order of fp32 sums over 512 chunks)."""
    import torch
    rng = np.random.default_rng(3)
    rows, cols, n, last = 16, 32768, 65536 + 20, 24
    m = _matrix(gpu_ctx, rng, fmt, rows, cols)
    g = torch.Generator(device="cuda").manual_seed(1)
    xq = torch.empty((n, cols), dtype=torch.int8, device="cuda").random_(-127, 128, generator=g)
    xs = torch.rand((n, cols // 64), device="cuda", generator=g) * 0.01
    xsum = torch.empty((n, cols // 64), dtype=torch.int32, device="cuda")
    for i in range(0, n, 4096):
        xsum[i:i + 4096] = xq[i:i + 4096].view(-1, cols // 64, 64).sum(2, dtype=torch.int32)
    out, own = torch.zeros((n, rows), device="cuda"), torch.zeros((last, rows), device="cuda")
    gpu_ctx.gemv(m, xq, xs, xsum, out, ntok=n, out_stride=rows)
    gpu_ctx.gemv(m, xq[-last:], xs[-last:], xsum[-last:], own, ntok=last, out_stride=rows)
    gpu_ctx.sync()
    assert own.any() and (out[-last:] - own).abs().max() <= 1e-5 * own.abs().max()
    m.close()


@pytest.mark.parametrize("noalloc", [False, True])
def test_attention_wait_that_gives_up_is_reported(gpu_ctx, noalloc):
    """A merge that stops waiting before its spans are there (32 polls, a context whose spans take
    ten times as long) makes k2t_attn_decode, or the sync after the no-alloc variant, raise; the
    next call, with the usual bound, is right again."""
    import torch
    rng = np.random.default_rng(9)
    nq, hd, seq = (128, 64, 40000) if not noalloc else (32, 64, 31000)
    code = [torch.from_numpy(rng.integers(-100, 100, (nq, seq, hd), np.int8)).cuda() for _ in range(2)]
    scale = [torch.full((nq, seq), 0.01, device="cuda") for _ in range(2)]
    q, out = _t(rng.standard_normal((nq, hd)).astype(np.float32)), [torch.zeros((nq, hd), device="cuda") for _ in range(2)]
    call = gpu_ctx.attn_decode_noalloc if noalloc else gpu_ctx.attn_decode
    args = (8, q, nq, nq, hd, code[0], scale[0], code[1], scale[1], seq, seq, hd ** -0.5)
    call(*args, out[0])
    gpu_ctx.sync()
    gpu_ctx.set_span_wait(1)
    try:
        with pytest.raises(k2t.K2TError, match="timed out"):
            call(*args, out[1])
            gpu_ctx.sync()
    finally:
        gpu_ctx.set_span_wait(0)
    call(*args, out[1])
    gpu_ctx.sync()
    assert out[0].any() and torch.equal(out[0], out[1])


def test_attention_of_a_growing_context_allocates_a_few_times():
    """A decode loop over a growing cache: the context's span workspace (2 MB per 2048 positions of
    these heads, which the free memory shows) doubles instead of growing with every call, and
    every call equals the same call on a context whose workspace was large from the start."""
    import torch
    nq, hd, cap = 128, 128, 32768
    g = torch.Generator(device="cuda").manual_seed(4)
    code = [torch.empty((nq, cap, hd), dtype=torch.int8, device="cuda").random_(-100, 100, generator=g) for _ in range(2)]
    scale = [torch.full((nq, cap), 0.01, device="cuda") for _ in range(2)]
    q, out = torch.randn((nq, hd), device="cuda", generator=g), [torch.zeros((nq, hd), device="cuda") for _ in range(2)]
    grown, large = k2t.Ctx(0), k2t.Ctx(0)
    args = lambda n: (8, q, nq, nq, hd, code[0], scale[0], code[1], scale[1], cap, n, hd ** -0.5)  # noqa: E731
    large.attn_decode(*args(cap), out[1])
    grown.attn_decode(*args(1), out[0])
    torch.cuda.synchronize()
    free, steps = torch.cuda.mem_get_info()[0], 0
    for n in range(300, cap, 2048):
        grown.attn_decode(*args(n), out[0])
        large.attn_decode(*args(n), out[1])
        assert torch.equal(out[0], out[1])
        now = torch.cuda.mem_get_info()[0]
        steps += now != free
        free = now
    assert 2 <= steps <= 7  # 16 calls
    grown.close()
    large.close()


@pytest.mark.parametrize("bits,hd,seq", [(8, 64, 1500), (8, 128, 300), (4, 64, 700), (4, 128, 1500)])
def test_attention_of_a_cache_at_any_address(gpu_ctx, bits, hd, seq):
    """V codes at a 4-byte address and, for the NF4 cache, scales at a 2-byte one: the output is
    that of the aligned cache (4e-5 of the largest: two fp32 orders)."""
    import torch
    rng = np.random.default_rng(seq + bits)
    nq, nkv = 8, 4
    code, scale = [], []
    for _ in range(2):
        code.append(torch.empty((nkv, seq, hd if bits == 8 else hd // 2), dtype=torch.int8, device="cuda"))
        scale.append(torch.empty((nkv, seq, 1 if bits == 8 else hd // 64), device="cuda",
                                 dtype=torch.float32 if bits == 8 else torch.bfloat16))
        gpu_ctx.kv_store(bits, _t(rng.standard_normal((nkv * seq, hd)).astype(np.float32)), nkv * seq, hd, code[-1], scale[-1])

    def moved(t, n):
        """A copy of t, n bytes past an aligned address."""
        raw = t.reshape(-1).view(torch.uint8)
        buf = torch.zeros(raw.numel() + n, dtype=torch.uint8, device="cuda")
        buf[n:] = raw
        return buf[n:]

    q = _t(rng.standard_normal((nq, hd)).astype(np.float32))
    out = torch.zeros((3, nq, hd), device="cuda")
    v = moved(code[1], 4)
    ks, vs = (moved(s, 2) if bits == 4 else s for s in scale)
    gpu_ctx.attn_decode(bits, q, nq, nkv, hd, code[0], scale[0], code[1], scale[1], seq, seq, hd ** -0.5, out[0])
    gpu_ctx.attn_decode(bits, q, nq, nkv, hd, code[0], ks, v, vs, seq, seq, hd ** -0.5, out[1])
    gpu_ctx.attn_decode_noalloc(bits, q, nq, nkv, hd, code[0], ks, v, vs, seq, seq, hd ** -0.5, out[2])
    gpu_ctx.sync()
    assert out[0].any() and (out[1:] - out[0]).abs().max() <= 4e-5 * out[0].abs().max()
    assert torch.equal(out[1], out[2])


# every kernel of batches whose passes skip a chunk of zero activation: 2 .. 15 tokens, NF3 on the
# small-batch kernel, the K-split one (ordered and chain) and the tiles; rows 0 and 33 have an
# infinite and a NaN scale in the first chunk
@pytest.mark.parametrize("fmt,ntok,rows,cols", [("nf4", 5, 64, 576), ("b4", 7, 64, 576), ("b6", 15, 64, 576), ("nf3", 5, 64, 576),
                                                ("nf4", 3, 64, 2112), ("b6", 4, 64, 2112), ("nf3", 4, 64, 2112),
                                                ("nf3", 20, 64, 576), ("nf3", 200, 1040, 4160), ("nf3", 40, 8200, 1088),
                                                ("nf3", 16, 8200, 2112), ("nf3", 130, 8200, 576)])
@pytest.mark.parametrize("exact", [False, True])
def test_chunk_of_zero_activation_is_skipped(gpu_ctx, fmt, ntok, rows, cols, exact):
    """A chunk whose activation scale is 0 takes no part whatever the row's scale, as in the
    4-token passes, whose outputs every batch equals."""
    import torch
    from helpers import acts, random_nf_streams, random_nibble4_streams
    rng = np.random.default_rng(rows + ntok)
    if fmt[0] == "b":
        hp = int(fmt[1]) - 4
        pair, tail = random_nibble4_streams(rng, rows, cols, hp)
        per, at = pair.size // (rows // 32), 1024 + 256 * hp
    else:
        _, _, pair, tail = random_nf_streams(rng, rows, cols, 2, bits=int(fmt[2]))
        per, at = pair.size // (rows // 32), 0
    pair[at:at + 2] = np.frombuffer(b"\x80\x7f", np.uint8)  # row 0: inf
    pair[per + at + 2:per + at + 4] = np.frombuffer(b"\xc0\x7f", np.uint8)  # row 33: NaN
    if fmt[0] == "b":
        m = gpu_ctx.upload_nibble4(rows, cols, hp, pair, tail)
    else:
        cb = np.sort(rng.choice(np.arange(-127, 128), 16, replace=False)).astype(np.int8)
        m = gpu_ctx.upload_nf(rows, cols, int(fmt[2]), 2, cb, pair, tail)
    xq, xs, xsum = acts(rng, cols, ntok, outlier_frac=0.001, outlier_scale=30.0)
    n = 2 if fmt[0] != "b" else 1  # the chunks of that scale
    for t in (0, ntok - 1):
        xq[t, :64 * n], xs[t, :n], xsum[t, :n] = 0, 0.0, 0
    got = _gemv(gpu_ctx, m, xq, xs, xsum, rows, exact)
    gpu_ctx.set_mfma(False)
    try:
        want = _gemv(gpu_ctx, m, xq, xs, xsum, rows, exact)
    finally:
        gpu_ctx.set_mfma(True)
    assert np.array_equal(got, want, equal_nan=True)
    assert np.isfinite(got[[0, ntok - 1]]).all() and not np.isfinite(got[1, [0, 33]]).any()
    m.close()
