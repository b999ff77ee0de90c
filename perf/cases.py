"""The work that a user of this framework has it do, as measurable cases.

Five kinds, each through the public entry points of kronos-2t_amd/k2t.py:

  proj  one quantized linear layer: activation rotation + int8 (with or without the RMSNorm
        in front) and the GEMV of 1 .. 1024 tokens; bit planes b4 / b5 / b6, NF4, NF3
  attn  one token's attention over a Hadamard KV cache (int8 or NF4, full or a sliding
        window with sinks), grouped or plain heads
  moe   one token through one sparse-MoE feed-forward
  turn  a stack of two decoder layers serving one request: a prompt, then decode steps over
        a given continuation; the prompt's logits and the last step's come back
  moe_turn  the same with sparse-MoE layers

Weights are drawn as quantizer codes of N(0, 0.02) matrices and packed here into the
streams that the C ABI takes, so that preparing them is quick and exact() knows them.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "kronos-2t_amd"))
import k2t  # noqa: E402

DEV = "cuda"
F64 = torch.float64
# Lloyd-Max levels of N(0, 1) as int8 codebooks (16 entries; NF3 uses the first 8)
NF4_CB = [-127, -96, -75, -58, -44, -31, -18, -6, 6, 18, 31, 44, 58, 75, 96, 127]
NF3_CB = [-127, -79, -45, -14, 14, 45, 79, 127, 0, 0, 0, 0, 0, 0, 0, 0]
NF_TOP = {"nf4": 2.7326, "nf3": 2.1520}  # the level of code 127, in standard deviations
STD = 0.02
PLANES = {"b4": 4, "b5": 5, "b6": 6}

# decoder shapes: hidden, heads, KV heads, head size, feed-forward width, rope base
SHAPES = {
    "135m": dict(hidden=576, n_heads=9, n_kv_heads=3, head_dim=64, intermediate=1536, rope_theta=100000.0),
    "1.7b": dict(hidden=2048, n_heads=32, n_kv_heads=32, head_dim=64, intermediate=8192, rope_theta=130000.0),
    "gqa128": dict(hidden=1024, n_heads=8, n_kv_heads=2, head_dim=128, intermediate=2816, rope_theta=1000000.0),
    "30b-a3b": dict(hidden=2048, n_heads=32, n_kv_heads=4, head_dim=128, intermediate=64, rope_theta=1000000.0),
}
# matrix formats of a model: qkv, o, gate_up, down, head (p55454: 5 planes but for gate_up and head)
FORMATS = {"nf4": ("nf4",) * 5, "b4": ("b4",) * 5, "b6": ("b6",) * 5, "p55454": ("b5", "b5", "b4", "b5", "b4"),
           "nf3nf4": ("nf3", "nf3", "nf3", "nf3", "nf4")}
LAYERS, VOCAB, EPS = 2, 8192, 1e-5


def listed():
    return [
        # the qkv projection of a 135M decoder for one token: the smallest call of a decode step
        dict(name="proj_b5_qkv_small", kind="proj", fmt="b5", rows=960, cols=576, ntok=1, norm=True),
        # one token through a large NF4 matrix: weight streaming
        dict(name="proj_nf4_one_token", kind="proj", fmt="nf4", rows=14336, cols=4096, ntok=1, norm=True),
        # four tokens through a 6-plane down projection (four sequences decoding, or a drafted continuation)
        dict(name="proj_b6_four_tokens", kind="proj", fmt="b6", rows=4096, cols=14336, ntok=4, norm=False),
        # a short user turn of eleven tokens through a qkv projection
        dict(name="proj_nf4_short_turn", kind="proj", fmt="nf4", rows=6144, cols=2048, ntok=11, norm=True),
        # a 200-token prompt through a dense NF3 matrix of odd sizes
        dict(name="proj_nf3_prompt", kind="proj", fmt="nf3", rows=5000, cols=2112, ntok=200, norm=True),
        # grouped-query attention of a long context, int8 cache
        dict(name="attn_gqa_long", kind="attn", bits=8, nq=32, nkv=4, hd=128, seq=6600, window=0),
        # plain multi-head attention over the compact NF4 cache
        dict(name="attn_mha_nf4_cache", kind="attn", bits=4, nq=32, nkv=32, hd=64, seq=4100, window=0),
        # one token through a sparse-MoE layer, 128 NF3 experts, top 8
        dict(name="moe_one_token", kind="moe", d=2048, dff=768, experts=128, top_k=8, bits=3),
        # a short request to a small mixed-plane model: decode steps dominate
        dict(name="turn_135m", kind="turn", shape="135m", fmt="p55454", prompt=45, steps=16, kv=8, window=0),
        # a request to the 1.7B-shaped NF4 model: a 256-token prompt, then decode
        dict(name="turn_1.7b", kind="turn", shape="1.7b", fmt="nf4", prompt=256, steps=32, kv=8, window=0),
        # reading a longer document: prefill alone, in batches of 512
        dict(name="prefill_1.7b", kind="turn", shape="1.7b", fmt="nf4", prompt=777, steps=0, kv=8, window=0),
        # a 96-token prompt to the sparse-MoE model
        dict(name="prefill_moe", kind="moe_turn", shape="30b-a3b", dff=768, experts=128, top_k=8, bits=3,
             prompt=96, steps=0, kv=8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["proj", "proj", "proj", "attn", "attn", "moe", "turn", "turn", "moe_turn"])
    if kind == "proj":
        ntok = rng.choice([1, 1, rng.randint(2, 4), rng.randint(5, 15), _log(rng, 16, 1024)])
        rows, cols = _log(rng, 200, 16384), 64 * _log(rng, 8, 224)
        while rows * cols * ntok > 3e10:
            rows = max(200, rows * 3 // 4)
            ntok = max(16, ntok * 3 // 4)
        return dict(kind=kind, fmt=rng.choice(["b4", "b5", "b6", "nf4", "nf4", "nf3"]), rows=rows, cols=cols,
                    ntok=ntok, norm=rng.random() < 0.5)
    if kind == "attn":
        nq, nkv, hd = rng.choice([(32, 4, 128), (32, 32, 64), (9, 3, 64), (32, 8, 128), (16, 16, 128)])
        seq = _log(rng, 64, 12000)
        return dict(kind=kind, bits=rng.choice([8, 8, 4]), nq=nq, nkv=nkv, hd=hd, seq=seq,
                    window=rng.choice([0, 0, 0, _log(rng, 256, 4096)]))
    if kind == "moe":
        e = rng.choice([16, 64, 128])
        return dict(kind=kind, d=64 * rng.randint(8, 32), dff=64 * rng.randint(4, 24), experts=e,
                    top_k=rng.choice([2, 4, 8]), bits=rng.choice([3, 3, 4]))
    if kind == "turn":
        shape = rng.choice(["135m", "1.7b", "gqa128"])
        return dict(kind=kind, shape=shape, fmt=rng.choice(["nf4", "nf4", "p55454", "b4", "b6", "nf3nf4"]),
                    prompt=_log(rng, 4, 700), steps=rng.randint(0, 24), kv=rng.choice([8, 8, 8, 4]),
                    window=rng.choice([0, 0, 0, _log(rng, 64, 600)]))
    return dict(kind=kind, shape="30b-a3b", dff=64 * rng.randint(6, 12), experts=rng.choice([32, 64, 128]),
                top_k=rng.choice([4, 8]), bits=rng.choice([3, 3, 4]), prompt=_log(rng, 4, 96),
                steps=rng.randint(0, 8), kv=8)


# ---------------------------------------------------------------- matrices
class _Q:
    """One quantized matrix: codes [rows][cols] (uint8) and BF16 scales [rows][groups]."""

    def __init__(self, g, fmt, rows, cols, sgc=2):
        self.fmt, self.rows, self.cols, self.nc = fmt, rows, cols, cols // 64
        self.sgc = 1 if fmt in PLANES else sgc
        self.nsg = -(-self.nc // self.sgc)
        w = torch.randn(rows, cols, generator=g, device=DEV)
        if fmt in PLANES:
            top = (1 << PLANES[fmt]) - 1
            delta = 2.2 / top  # odd levels (2u - top) * delta reach 2.2 deviations
            self.codes = (w * (0.5 / delta) + 0.5 * top).round_().clamp_(0, top).to(torch.uint8)
        else:
            cb = torch.tensor(NF4_CB if fmt == "nf4" else NF3_CB[:8], dtype=torch.float32, device=DEV)
            delta = NF_TOP[fmt] / 127.0
            self.codes = torch.bucketize(w, (cb[1:] + cb[:-1]) * (0.5 * delta), out_int32=True).to(torch.uint8)
        del w
        spread = 1.0 + 0.06 * torch.randn(rows, self.nsg, generator=g, device=DEV)
        self.scales = (STD * delta * spread).to(torch.bfloat16)

    def dense(self, rows=None):
        """The matrix (rotated domain) in 64 bits."""
        codes = self.codes if rows is None else self.codes[rows]
        scales = self.scales if rows is None else self.scales[rows]
        if self.fmt in PLANES:
            v = 2.0 * codes.to(F64) - ((1 << PLANES[self.fmt]) - 1)
        else:
            cb = torch.tensor(NF4_CB if self.fmt == "nf4" else NF3_CB, dtype=F64, device=DEV)
            v = cb[codes.to(torch.int32)]
        s = scales.to(F64).repeat_interleave(64 * self.sgc, dim=1)[:, :self.cols]
        return v * s

    def _chunks(self):
        """Packed stripe-chunks [stripes][nc][bytes]; bit planes: nibbles and hi-plane bytes apart."""
        s = -(-self.rows // 16)
        c = torch.zeros(s * 16, self.cols, dtype=torch.uint8, device=DEV)
        c[:self.rows] = self.codes
        if self.fmt == "nf3":
            # [s, nc, kp, g, piece, j, t] from columns (2 kp + k) * 16 + quad * 4 + t
            c = c.view(s, 4, 4, self.nc, 2, 2, 4, 4).permute(5, 6, 0, 3, 4, 1, 2, 7).reshape(
                8, s, self.nc, 2, 4, 4, 4)
            b = [c[0] | (c[1] << 3) | ((c[2] & 3) << 6), c[3] | (c[4] << 3) | ((c[5] & 3) << 6),
                 c[6] | (c[7] << 3) | ((c[2] >> 2) << 6) | ((c[5] >> 2) << 7)]
            return torch.stack(b, dim=4).reshape(s, self.nc, 384), None
        # columns k * 16 + half * 8 + nibble * 4 + t, rows 4 g + j -> [k, g, half, j, t]
        v = c.view(s, 4, 4, self.nc, 4, 2, 2, 4).permute(6, 0, 3, 4, 1, 5, 2, 7)
        low = ((v[0] & 15) | (v[1] << 4)).reshape(s, self.nc, 512)
        hp = PLANES.get(self.fmt, 4) - 4
        if hp == 0:
            return low, None
        u = (c >> 4).view(s, 4, 4, self.nc, 4, 4, 4).permute(5, 0, 3, 4, 1, 2, 6)  # [sub, s, nc, k, g, j, t]
        if hp == 2:
            hi = (u[0] << 4) | (u[1] << 6) | (u[2] << 2) | u[3]
        else:
            h = u[0] | (u[1] << 1) | (u[2] << 2) | (u[3] << 3)
            hi = (h[:, :, 0::2] << 4) | h[:, :, 1::2]
        return low, hi.reshape(s, self.nc, 128 * hp)

    def streams(self):
        """(pair bytes, tail bytes) on the GPU, in the layout of k2t_mat_wrap_*."""
        s = -(-self.rows // 16)
        pairs = s // 2
        low, hi = self._chunks()
        sc = torch.zeros(s * 16, self.nsg, dtype=torch.bfloat16, device=DEV)
        sc[:self.rows] = self.scales
        sc = sc.view(s, 16, self.nsg).transpose(1, 2).contiguous().view(torch.uint8)  # [s][nsg][32]

        def cut(per, n):  # n groups of `per` stripes: the stripes' pieces side by side
            first = 0 if per == 2 else 2 * pairs
            take = lambda a: None if a is None else a[first:first + n * per].reshape(  # noqa: E731
                n, per, a.shape[1], -1).transpose(1, 2).reshape(n, a.shape[1], -1)
            lo, hh, ss = take(low), take(hi), take(sc)
            if self.fmt in PLANES:
                return torch.cat([x for x in (lo, hh, ss) if x is not None], dim=2).reshape(-1)
            full, cb = self.nc // self.sgc, lo.shape[2]
            body = lo[:, :full * self.sgc].reshape(n, full, self.sgc * cb)
            parts = [torch.cat([ss[:, :full], body], dim=2).reshape(n, -1)]
            if self.nsg > full:
                parts += [ss[:, full], lo[:, full * self.sgc:].reshape(n, -1)]
            return torch.cat(parts, dim=1).reshape(-1)

        return cut(2, pairs), cut(1, 1) if s & 1 else torch.empty(0, dtype=torch.uint8, device=DEV)

    def upload(self, ctx):
        pair, tail = self.streams()
        t = tail if tail.numel() else None
        if self.fmt in PLANES:
            return ctx.wrap_nibble4(self.rows, self.cols, PLANES[self.fmt] - 4, pair, pair.numel(), t, tail.numel())
        cb = np.array(NF4_CB if self.fmt == "nf4" else NF3_CB, np.int8)
        m = ctx.wrap_nf(self.rows, self.cols, 4 if self.fmt == "nf4" else 3, self.sgc, cb, pair, pair.numel(), t,
                        tail.numel())
        m.nf3_lane_order()  # NF3 in the order that an upload stores; nothing to do for NF4
        return m


def _q_bytes(fmt, rows, cols):
    per = {"b4": 4.25, "b5": 5.25, "b6": 6.25, "nf4": 4.125, "nf3": 3.125}[fmt]
    return rows * cols * per / 8


# ---------------------------------------------------------------- inputs
def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFF)


def _acts(g, ntok, cols):
    """Rows ~N(0, 1) with 0.1% outlier channels, 30 times as large."""
    x = torch.randn(ntok, cols, generator=g, device=DEV)
    hot = torch.randperm(cols, generator=g, device=DEV)[:max(1, cols // 1000)]
    x[:, hot] *= 30.0
    return x


def _norm_w(g, n):
    return 1.0 + 0.1 * torch.randn(n, generator=g, device=DEV)


def _proj_inputs(case, seed):
    g = _gen(seed, 1)
    w = _Q(g, case["fmt"], case["rows"], case["cols"])
    return w, _acts(g, case["ntok"], case["cols"]), _norm_w(g, case["cols"])


def _attn_inputs(case, seed):
    g = _gen(seed, 2)
    nq, nkv, hd, seq, win = case["nq"], case["nkv"], case["hd"], case["seq"], case["window"]
    sinks = min(4, win // 2)
    cap = win + 512 if win else seq + 32
    k = torch.randn(nkv * cap, hd, generator=g, device=DEV)
    v = torch.randn(nkv * cap, hd, generator=g, device=DEV)
    q = 2.0 * torch.randn(nq, hd, generator=g, device=DEV)
    return q, k, v, cap, sinks


def _experts(g, n, d, dff, bits):
    """n experts: one code matrix of all gate_up rows, one of all down rows."""
    fmt = "nf%d" % bits
    return _Q(g, fmt, n * 2 * dff, d), _Q(g, fmt, n * d, dff)


def _bank(ctx, layers, experts, d, dff, bits):
    lay = k2t.k2tm_expert_layout(d, dff, bits, 2)
    rec = lay["aligned_expert_bytes"]
    page = np.zeros(16384, np.uint8)
    page[:12] = np.frombuffer(b"K2TM800B_V1\0", np.uint8)
    page[16:72] = np.array([len(layers), experts, d, dff, 2, rec, bits], np.uint64).view(np.uint8)
    buf = torch.zeros(16384 + len(layers) * experts * rec, dtype=torch.uint8, device=DEV)
    buf[:16384] = torch.from_numpy(page)
    recs = buf[16384:].view(len(layers), experts, rec)
    cb = torch.tensor(NF4_CB if bits == 4 else NF3_CB, dtype=torch.int8).view(torch.uint8).to(DEV)
    for li, (gu, dn) in enumerate(layers):
        for m, cb_off, off in ((gu, "gu_codebook_off", "gu_pair_off"), (dn, "dn_codebook_off", "dn_pair_off")):
            pair, _ = m.streams()
            n = pair.numel() // experts
            recs[li, :, lay[cb_off]:lay[cb_off] + 16] = cb
            recs[li, :, lay[off]:lay[off] + n] = pair.view(experts, n)
    bank = k2t.ExpertBank.wrap(ctx, buf, buf.numel(), page)
    bank.nf3_lane_order()
    return bank


def _moe_inputs(case, seed):
    g = _gen(seed, 3)
    ex = _experts(g, case["experts"], case["d"], case["dff"], case["bits"])
    router = 0.05 * torch.randn(case["experts"], case["d"], generator=g, device=DEV)
    return ex, router, torch.randn(case["d"], generator=g, device=DEV), _norm_w(g, case["d"])


def _turn_inputs(case, seed):
    g = _gen(seed, 4)
    c = SHAPES[case["shape"]]
    d, hd, inter = c["hidden"], c["head_dim"], c["intermediate"]
    moe = case["kind"] == "moe_turn"
    f = FORMATS["nf4" if moe else case["fmt"]]
    layers = []
    for _ in range(LAYERS):
        lay = dict(qkv=_Q(g, f[0], (c["n_heads"] + 2 * c["n_kv_heads"]) * hd, d),
                   o=_Q(g, f[1], d, c["n_heads"] * hd), in_norm=_norm_w(g, d), post_norm=_norm_w(g, d))
        if moe:
            lay["experts"] = _experts(g, case["experts"], d, case["dff"], case["bits"])
            lay["router"] = 0.05 * torch.randn(case["experts"], d, generator=g, device=DEV)
            lay["qn"], lay["kn"] = _norm_w(g, hd), _norm_w(g, hd)
        else:
            lay["gu"], lay["down"] = _Q(g, f[2], 2 * inter, d), _Q(g, f[3], d, inter)
        layers.append(lay)
    head, fn = _Q(g, f[4], VOCAB, d), _norm_w(g, d)
    toks = torch.randint(0, VOCAB, (case["prompt"] + case["steps"],), generator=g, device=DEV).cpu().numpy()
    return layers, head, fn, toks.astype(np.int32)


def prepare(case, seed):
    ctx = k2t.Ctx(0)
    if case["kind"] == "proj":
        w, x, nw = _proj_inputs(case, seed)
        t, k, r = case["ntok"], case["cols"], case["rows"]
        new = functools.partial(torch.empty, device=DEV)
        return dict(case=case, ctx=ctx, m=w.upload(ctx), x=x, nw=nw, q=new((t, k), dtype=torch.int8),
                    s=new((t, k // 64), dtype=torch.float32), sums=new((t, k // 64), dtype=torch.int32),
                    out=new((t, r), dtype=torch.float32))
    if case["kind"] == "attn":
        q, k, v, cap, sinks = _attn_inputs(case, seed)
        hd, bits, n = case["hd"], case["bits"], k.shape[0]
        st = dict(case=case, ctx=ctx, qh=q, cap=cap, sinks=sinks, out=torch.empty_like(q))
        for name, heads in (("k", k), ("v", v)):
            codes = torch.empty((n, hd if bits == 8 else hd // 2), dtype=torch.int8, device=DEV)
            sc = torch.empty((n, 1 if bits == 8 else hd // 64), device=DEV,
                             dtype=torch.float32 if bits == 8 else torch.bfloat16)
            ctx.kv_store(bits, heads, n, hd, codes, sc)
            st[name + "q"], st[name + "s"] = codes, sc
        ctx.sync()
        return st
    if case["kind"] == "moe":
        ex, router, h, nw = _moe_inputs(case, seed)
        bank = _bank(ctx, [ex], case["experts"], case["d"], case["dff"], case["bits"])
        return dict(case=case, ctx=ctx, bank=bank, router=router, x=h, h=torch.empty_like(h), nw=nw,
                    ids=torch.empty(case["top_k"], dtype=torch.int32, device=DEV),
                    wts=torch.empty(case["top_k"], dtype=torch.float32, device=DEV))
    layers, head, fn, toks = _turn_inputs(case, seed)
    cfg = dict(SHAPES[case["shape"]], n_layers=LAYERS, vocab=VOCAB, rms_eps=EPS,
               max_seq=max(1024, len(toks) + 8, case.get("window", 0) + 520))
    m = k2t.Model(ctx, cfg, max_batch=min(512, max(16, case["prompt"])))
    if case["kv"] == 4:
        m.set_kv_bits(4)
    if case.get("window"):
        m.set_kv_window(case["window"], 4)
    host = lambda a: a.cpu().numpy()  # noqa: E731
    bank = None
    if case["kind"] == "moe_turn":
        bank = _bank(ctx, [la["experts"] for la in layers], case["experts"], cfg["hidden"], case["dff"], case["bits"])
    for i, la in enumerate(layers):
        gu, dn = (la["gu"].upload(ctx), la["down"].upload(ctx)) if bank is None else (None, None)
        m.set_layer(i, la["qkv"].upload(ctx), la["o"].upload(ctx), gu, dn, host(la["in_norm"]), host(la["post_norm"]))
        if bank is not None:
            m.set_qk_norm(i, host(la["qn"]), host(la["kn"]))
            m.set_moe(i, bank, i, host(la["router"]), case["top_k"], True, k2t.MOE_SOFTMAX)
    m.set_head(head.upload(ctx), host(fn))
    torch.cuda.synchronize()  # the streams are packed before the model's own stream reads them
    return dict(case=case, ctx=ctx, m=m, bank=bank, toks=toks)


def run(state):
    case, ctx = state["case"], state["ctx"]
    if case["kind"] == "proj":
        x, q, s, sums, out = state["x"], state["q"], state["s"], state["sums"], state["out"]
        if case["norm"]:
            ctx.act_quant_rmsnorm(x, state["nw"], EPS, q, s, sums, case["cols"], case["ntok"])
        else:
            ctx.act_quant(x, q, s, sums, case["cols"], case["ntok"])
        ctx.gemv(state["m"], q, s, sums, out, ntok=case["ntok"], out_stride=case["rows"])
        return dict(q=q, s=s, sums=sums, y=out)
    if case["kind"] == "attn":
        ctx.attn_decode_noalloc(case["bits"], state["qh"], case["nq"], case["nkv"], case["hd"], state["kq"],
                                state["ks"], state["vq"], state["vs"], state["cap"], case["seq"],
                                case["hd"] ** -0.5, state["out"], case["window"], state["sinks"])
        return state["out"]
    if case["kind"] == "moe":
        state["h"].copy_(state["x"])  # the feed-forward adds to the residual stream in place
        ctx.moe_ffn(state["bank"], 0, state["router"], state["h"], state["nw"], EPS, case["top_k"],
                    route_ids=state["ids"], route_weights=state["wts"])
        return dict(h=state["h"], ids=state["ids"], wts=state["wts"])
    m, toks, n = state["m"], state["toks"], case["prompt"]
    m.reset()
    out = [m.prefill(toks[:n])]
    if case["steps"]:
        for t in toks[n:-1]:
            m.decode(t, want_logits=False)
        out.append(m.decode(toks[-1]))
    return out


def work(case):
    if case["kind"] == "proj":
        t, k, r = case["ntok"], case["cols"], case["rows"]
        return dict(bytes=_q_bytes(case["fmt"], r, k) + t * (4 * k + k + k // 8 + 4 * r), flops=2.0 * t * k * r)
    if case["kind"] == "attn":
        n = min(case["seq"], case["window"] or case["seq"])
        per = case["hd"] + 4 if case["bits"] == 8 else case["hd"] / 2 + case["hd"] / 32
        return dict(bytes=2.0 * n * case["nkv"] * per + 8 * case["nq"] * case["hd"],
                    flops=4.0 * n * case["nq"] * case["hd"])
    if case["kind"] == "moe":
        w = case["top_k"] * 3 * case["dff"] * case["d"]
        return dict(bytes=_q_bytes("nf%d" % case["bits"], 1, w) + 4 * case["experts"] * case["d"] + 12 * case["d"],
                    flops=2.0 * w + 2.0 * case["experts"] * case["d"])
    c = SHAPES[case["shape"]]
    d, hd, nq, nkv = c["hidden"], c["head_dim"], c["n_heads"], c["n_kv_heads"]
    moe = case["kind"] == "moe_turn"
    f = FORMATS["nf4" if moe else case["fmt"]]
    mats = [(f[0], (nq + 2 * nkv) * hd * d), (f[1], d * nq * hd)]
    if not moe:
        mats += [(f[2], 2 * c["intermediate"] * d), (f[3], c["intermediate"] * d)]
    layer, head = sum(_q_bytes(a, 1, n) for a, n in mats), _q_bytes(f[4], VOCAB, d)
    macs = sum(n for _, n in mats)
    n, steps = case["prompt"], case["steps"]
    total, kv = n + steps, 2 * nkv * (hd + 4 if case["kv"] == 8 else hd / 2 + hd / 32)
    win = case.get("window") or total
    seen = [min(i + 1, win) for i in range(total)]
    b = (1 + steps) * (LAYERS * layer + head) + LAYERS * kv * (total + sum(seen[n:]) + seen[n - 1])
    fl = 2.0 * (LAYERS * macs * total + (1 + steps) * VOCAB * d) + 4.0 * LAYERS * nq * hd * sum(seen)
    if moe:
        one = 3 * case["dff"] * d
        used = case["experts"] * (1 - (1 - case["top_k"] / case["experts"]) ** n) + steps * case["top_k"]
        b += LAYERS * (_q_bytes("nf%d" % case["bits"], 1, one) * used + (1 + steps) * 4 * case["experts"] * d)
        fl += 2.0 * LAYERS * total * (case["top_k"] * one + case["experts"] * d)
    return dict(bytes=float(b), flops=fl)


def tolerance(case):
    # proj: fp32 sums of 8 .. 224 chunk terms in another order; a code of the int8 activation
    # can move where the RMSNorm's sum is taken in another order
    if case["kind"] == "proj":
        return dict(rel=2e-4, max=2e-3, differ=1e-4) if case["norm"] else dict(rel=5e-6, max=1e-4)
    # attn: fp32 softmax and weighted sums over up to 12000 positions
    if case["kind"] == "attn":
        return dict(rel=2e-5, max=4e-4)
    # moe: the SwiGLU output is quantized to int8 again, so single codes can move (one moved
    # code of one expert is about 1e-5 of the residual stream)
    if case["kind"] == "moe":
        return dict(rel=5e-5, max=1e-3)
    # two layers: a moved code of one layer travels through the int8 activations of all that follow
    return dict(rel=0.03, max=0.3)


# ---------------------------------------------------------------- the same in 64 bits
@functools.lru_cache(None)
def _signs(block):
    """Sign of each element of Hadamard block `block` (SplitMix64 of the block's seed)."""
    mask, out = (1 << 64) - 1, []
    for i in range(64):
        z = (0x9E3779B97F4A7C15 + block * 0xBF58476D1CE4E5B9 + (i + 1) * 0x9E3779B97F4A7C15) & mask
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & mask
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
        out.append(-1.0 if (z ^ (z >> 31)) & 1 else 1.0)
    return out


def _sign_rows(n):
    return torch.tensor([_signs(b) for b in range(n)], dtype=F64, device=DEV)


def _hadamard():
    h = torch.ones(1, 1, dtype=F64, device=DEV)
    for _ in range(6):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / 8.0


def _rot(x):
    """Signed Hadamard-64 of the last dimension's blocks."""
    b = x.to(F64).unflatten(-1, (-1, 64))
    return ((b * _sign_rows(b.shape[-2])) @ _hadamard()).flatten(-2)


def _unrot(x):
    b = x.unflatten(-1, (-1, 64))
    return ((b @ _hadamard()) * _sign_rows(b.shape[-2])).flatten(-2)


def _int8(x, block):
    """Codes and scale per `block` values of the last dimension."""
    b = x.unflatten(-1, (-1, block))
    mx = b.abs().amax(-1, keepdim=True)
    q = torch.where(mx > 0, (b * (127.0 / mx.clamp_min(1e-300))).round(), torch.zeros_like(b))
    return q, mx / 127.0


def _act(x):
    """The activation a GEMV reads, dequantized."""
    q, s = _int8(_rot(x), 64)
    return (q * s).flatten(-2)


def _rms(x, w, eps=EPS):
    x = x.to(F64)
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.to(F64)


def _kv(x, bits):
    """Rotated, quantized and dequantized KV heads (last dimension: one head)."""
    r = _rot(x)
    if bits == 8:
        q, s = _int8(r, x.shape[-1])
        return (q * s).flatten(-2)
    cb = torch.tensor(NF4_CB, dtype=F64, device=DEV)
    mid = (cb[1:] + cb[:-1]) / 2
    b = r.unflatten(-1, (-1, 64))
    c = cb[torch.bucketize(b * (127.0 / b.abs().amax(-1, keepdim=True)), mid, right=True)]
    s = ((b * c).sum(-1, keepdim=True) / (c * c).sum(-1, keepdim=True)).to(torch.bfloat16).to(F64)
    return (cb[torch.bucketize(b / s, mid, right=True)] * s).flatten(-2)


def _qrot(q):
    c, s = _int8(_rot(q), q.shape[-1])
    return (c * s).flatten(-2)


def _active(seq, window, sinks):
    if window and seq > window:
        return list(range(sinks)) + list(range(seq - (window - sinks), seq))
    return list(range(seq))


def _route(xn, router, top_k):
    p, ids = torch.softmax(xn @ router.to(F64).T, -1).topk(top_k, -1)
    return p / p.sum(-1, keepdim=True), ids


def _swiglu(gate, up):
    return gate / (1.0 + torch.exp(-gate)) * up


def _moe(xn, router, ex, experts, top_k):
    """(sum over routes [t][d], ids, weights) for normalized rows xn [t][d]."""
    gu, dn = ex
    d, dff = xn.shape[1], gu.rows // experts // 2
    p, ids = _route(xn, router, top_k)
    a, out = _act(xn), torch.zeros_like(xn)
    for e in ids.unique().tolist():
        t, z = (ids == e).nonzero(as_tuple=True)
        y = a[t] @ gu.dense(slice(e * 2 * dff, (e + 1) * 2 * dff)).T
        y = _act(_swiglu(y[:, :dff], y[:, dff:])) @ dn.dense(slice(e * d, (e + 1) * d)).T
        out.index_add_(0, t, p[t, z, None] * y)
    return out, ids, p


def _exact_turn(case, seed):
    layers, head, fn, toks = _turn_inputs(case, seed)
    c = SHAPES[case["shape"]]
    d, nq, nkv, hd = c["hidden"], c["n_heads"], c["n_kv_heads"], c["head_dim"]
    n, win = len(toks), case.get("window", 0)
    inv = torch.tensor([1.0 / c["rope_theta"] ** (2 * i / hd) for i in range(hd // 2)], dtype=torch.float32)
    ang = (torch.arange(n, dtype=torch.float32)[:, None] * inv[None, :]).to(DEV).to(F64)  # angles are fp32
    cos, sin = ang.cos()[:, None, :], ang.sin()[:, None, :]
    mask = torch.full((n, n), -math.inf, dtype=F64, device=DEV)
    for i in range(n):
        mask[i, _active(i + 1, win, min(4, win // 2))] = 0.0
    x = _unrot(head.dense(torch.from_numpy(toks.astype(np.int64)).to(DEV)))

    def rope(v):
        a, b = v[..., :hd // 2], v[..., hd // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    for la in layers:
        y = (_act(_rms(x, la["in_norm"])) @ la["qkv"].dense().T).view(n, nq + 2 * nkv, hd)
        q, k, v = y[:, :nq], y[:, nq:nq + nkv], y[:, nq + nkv:]
        if "qn" in la:
            q, k = _rms(q, la["qn"]), _rms(k, la["kn"])
        q, k, v = _qrot(rope(q)), _kv(rope(k), case["kv"]), _kv(v, case["kv"])
        k, v = (t.repeat_interleave(nq // nkv, 1).transpose(0, 1) for t in (k, v))
        p = torch.softmax(q.transpose(0, 1) @ k.transpose(1, 2) * hd ** -0.5 + mask, -1)
        o = _unrot((p @ v).transpose(0, 1)).reshape(n, nq * hd)
        x = x + _act(o) @ la["o"].dense().T
        xn = _rms(x, la["post_norm"])
        if "router" in la:
            x = x + _moe(xn, la["router"], la["experts"], case["experts"], case["top_k"])[0]
        else:
            y = (_act(xn) @ la["gu"].dense().T).view(n, -1, 2, 64)
            x = x + _act(_swiglu(y[:, :, 0], y[:, :, 1]).flatten(1)) @ la["down"].dense().T
    rows = [case["prompt"] - 1] + ([n - 1] if case["steps"] else [])
    logits = _act(_rms(x[rows], fn)) @ head.dense().T
    return [r.cpu().numpy() for r in logits]


def exact(case, seed):
    if case["kind"] == "proj":
        w, x, nw = _proj_inputs(case, seed)
        r = _rot(_rms(x, nw) if case["norm"] else x)
        q, s = _int8(r, 64)
        return dict(q=None, s=s.squeeze(-1), sums=None, y=(q * s).flatten(-2) @ w.dense().T)
    if case["kind"] == "attn":
        q, k, v, cap, sinks = _attn_inputs(case, seed)
        nq, nkv, hd, win = case["nq"], case["nkv"], case["hd"], case["window"]
        pos = torch.tensor(_active(case["seq"], win, sinks), device=DEV)
        if win:  # the ring's slot of each position
            pos = torch.where(pos < sinks, pos, sinks + (pos - sinks) % (cap - sinks))
        k, v = (_kv(t, case["bits"]).view(nkv, cap, hd)[:, pos].repeat_interleave(nq // nkv, 0) for t in (k, v))
        p = torch.softmax((k @ _qrot(q)[:, :, None]).squeeze(-1) * hd ** -0.5, -1)
        return _unrot((p[:, None, :] @ v).squeeze(1))
    if case["kind"] == "moe":
        ex, router, h, nw = _moe_inputs(case, seed)
        y, _, p = _moe(_rms(h, nw)[None], router, ex, case["experts"], case["top_k"])
        order = _route(_rms(h, nw)[None], router, case["top_k"])[1][0].argsort()
        return dict(h=h.to(F64) + y[0], ids=None, wts=p[0][order])
    return _exact_turn(case, seed)
