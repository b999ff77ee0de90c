// Decode attention of one token over spans of the KV cache, one launch: the int8 and the
// NF4 Hadamard cache, full or a sliding-window ring, plain or grouped query heads.
//
// Span workgroups, one per (KV head, span of positions), score all G = nq / nkv q heads of
// the group, so each K / V tile is read from memory once instead of once per q head.  The
// tile goes to LDS (int8: direct-to-LDS loads; NF4: through registers, decoded to the
// codebook's int8 values once for all heads); meanwhile each wave applies bias / QK-norm /
// RoPE and the Hadamard int8 quantization to one q head (and, in the span holding the
// current position, waves 6 and 7 build that position's K / V and store them in the cache).
// Per head: s_t = float(q8 . k8_t) * ks_t * (qs * scale) as causal_gqa_group_q8
// (real_llm.rs:8471-8594), or the sum of such terms per 64-block for the NF4 cache and
// windows (causal_gqa_group_q4_or_window, 8794-8937); the span's maximum m and sum of
// exp(s_t - m), and o = sum_t (exp(s_t - m) * vs_t) * v8_t.
//
// A context of one span ends in its span workgroups.  Otherwise a span workgroup publishes
// its partials as {payload, epoch} words (one agent-scope atomic store each: the value and
// its ready mark arrive together, no fence or counter).  Merge workgroups, one per q head,
// come first in dispatch order and poll (bounded) the words of their head's spans until
// every one carries this launch's epoch, then combine the spans (global maximum,
// exp-weighted sums in span order), apply ifwht64 (real_llm.rs:8588-8592), and write the
// o_proj activation (populate_chunk_fwht_raw(None), real_llm.rs:7060-7084).  The epoch is one
// more than the last launch's; the last merge workgroup to finish advances it, so the
// words never need clearing.
//
// What bounds it is latency: a context of one span takes 5.5 us, the hand-off and the merge 2
// to 4 more; 9 MB of K / V at copy rate are 1.8 us.  Against one workgroup per q head and
// 256-position span with a merge launch (which had the position stored by a launch of its
// own), back to back: 32 heads x 64, 4100 positions, NF4 cache 15.4 -> 12.3 us, int8 12.1 -> 13.0 (waited
// for 26.1 -> 25.0; 12000 positions 30.6 -> 21.7); 32 / 4 heads x 128, 12000 positions, NF4 49.0 -> 13.7, int8
// (grouped before too) 21.0 -> 14.2; a 1000-position window of it 18.4 -> 9.9.
#include <float.h>
#include <math.h>

#include <algorithm>

#include "k2t_device.h"
#include "k2t_internal.h"
#include "k2t_kv_dev.h"

namespace k2t {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kSpanThreads = 512, kSpanWaves = kSpanThreads / 64;
constexpr int kSpanMaxGroup = 8;  // q heads per KV head: one per wave

struct SpanArgs {
    const float *q;
    int8_t *kq, *vq;
    float *ks, *vs;
    const int *pos_dev;  // the token's position, or NULL: pos
    int pos;
    int layer, nq, nkv;
    KvRing kr;
    float attn_scale;
    int nspan;  // spans the words have room for
    AttnPost post;
    unsigned long long *words;  // [q head][nspan][2 + hd] {payload, epoch} span words
    unsigned int *cnt;          // {epoch of the last launch, merge workgroups done}
    int *err;
    unsigned int spin_limit;
    float *out_f;
    int8_t *aq;
    float *as;
    int32_t *asum;
};

// LDS of a workgroup: the int8 K and V tiles [position][HD], and the waves' partial o
// [wave][head][o_stride(HD)]: behind the tiles in the kernel of more than four heads over 128-position
// spans, which saves it the barrier before their first store, else in the tiles' place once
// those are read.  The stride: heads HD floats apart lie in the same banks, and the stores of
// eight heads took 0.6 us longer.
constexpr int o_stride(int hd) { return hd + 4; }
constexpr bool o_behind(int tiles_per_wave, bool g8) { return g8 && tiles_per_wave == 1; }
size_t span_lds(int hd, int positions, int group) {
    const size_t t = (size_t)2 * positions * hd, o = (size_t)kSpanWaves * group * o_stride(hd) * sizeof(float);
    return o_behind(positions / 128, group > 4) ? t + o : std::max(t, o);
}

// o (this wave's 64-block b of q head `head`, one element per lane, rotated domain) through
// ifwht64 into out_f and / or the o_proj activation.
__device__ __forceinline__ void finish_head(const SpanArgs &A, float rotated, int head, int b, int nb, uint32_t lane) {
    const float o = ifwht_lane(rotated, (uint64_t)b, lane);
    const size_t c = (size_t)head * nb + b;
    if (A.out_f) A.out_f[c * 64 + lane] = o;
    if (A.aq) quant_chunk_store(fwht_lane(o, c, lane), lane, A.aq + c * 64, A.as + c, A.asum + c);
}

// TPW: 16-position tiles per wave; a span is 128 * TPW positions.
// G8: more than 4 q heads per KV head.
template <int HD, int BITS, bool RING, int TPW, bool G8>
__global__ __launch_bounds__(kSpanThreads, HD == 128 && G8 ? 4 : 6) void attn_span_kernel(SpanArgs A) {
    constexpr int NTH = kSpanThreads, NW = kSpanWaves, P = 16 * NW * TPW, nb = HD / 64, DB = HD / 16;
    constexpr int HP = G8 ? 2 : 1, GC = 4 * HP;  // passes of four heads; score columns repeat every GC
    constexpr int SB = BITS == 4 ? nb : 1;  // scales per position
    extern __shared__ __align__(16) int8_t tiles[];
    __shared__ float kst[P * SB], vst[P * SB];
    __shared__ __align__(16) int8_t qi[kSpanMaxGroup * HD];
    __shared__ float qas[kSpanMaxGroup];
    __shared__ float red_m[kSpanMaxGroup][NW], red_l[kSpanMaxGroup][NW];
    __shared__ __align__(16) int8_t kcur[HD], vcur[HD];
    __shared__ __align__(8) float cur_k[2], cur_v[2];
    __shared__ float fin[kSpanMaxGroup * HD];  // one-span contexts: o / L
    const int nq = A.nq, nkv = A.nkv, G = nq / nkv, layer = A.layer;
    const int kvh = (int)blockIdx.x;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const int wv = __builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const int seq = (A.pos_dev ? A.pos_dev[0] : A.pos) + 1;
    const KvRing kr = A.kr;
    const int act = RING ? active_len(kr, seq) : seq;  // attended positions
    const int nact = (act + P - 1) / P;
    // this launch's epoch: one more than the last launch's (advanced by its last merge
    // workgroup, after every span workgroup of that launch had read it)
    const uint32_t ep = __hip_atomic_load(A.cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u;
    const size_t pstride = (size_t)A.nspan * (2 + HD);
    if ((int)blockIdx.y < G) {
        // ------------------------------------------------------------ merge workgroup
        if (nact == 1) return;
        // thread (span subset sub, 4-column group cg): spans sub, sub + nsub, ... ascending;
        // per span it polls the words {m, L, o[4 columns]} until they carry this epoch
        const int head = kvh * G + (int)blockIdx.y;
        const unsigned long long *pp = A.words + (size_t)head * pstride;
        constexpr int ncg = HD / 4, nsub = NTH / ncg;
        const int cg = (int)tid % ncg, sub = (int)tid / ncg;
        // spans per thread polled together; the large kernel has the registers for 3 (30B-A3B
        // decode at 6600 positions, 52 spans: 422 tok/s with 3, 420 with 4 at 127 VGPRs)
        constexpr int kPre = HD == 128 && G8 ? 3 : 2;
        bool ok = true;
        auto poll = [&](int s, unsigned long long (&w)[6]) {
            // (the caller keeps s < nact)
            const unsigned long long *ps = pp + (size_t)s * (2 + HD);
            w[0] = ll_word_load(ps);
            w[1] = ll_word_load(ps + 1);
#pragma unroll
            for (int k = 0; k < 4; k++) w[2 + k] = ll_word_load(ps + 2 + cg * 4 + k);
        };
        // Every slot's words are requested before any is examined (a slot past nact reads
        // span nact - 1's and is then replaced by the empty span {-inf, 0, 0}): under a
        // per-slot branch the compiler waited for each slot's loads before issuing the
        // next slot's.
        unsigned long long wv6[kPre][6];
#pragma unroll
        for (int j = 0; j < kPre; j++) poll(min(sub + j * nsub, nact - 1), wv6[j]);
        uint32_t pending = 0;
#pragma unroll
        for (int j = 0; j < kPre; j++) {
            const bool live = sub + j * nsub < nact;
#pragma unroll
            for (int k = 0; k < 6; k++) {
                if (live && (uint32_t)(wv6[j][k] >> 32) != ep) pending |= 1u << (6 * j + k);
                if (!live) wv6[j][k] = k == 0 ? (unsigned long long)__float_as_uint(-INFINITY) : 0ull;
            }
        }
        for (uint32_t spins = 0; pending != 0 && ok; spins++) {
            if ((spins & 31u) == 31u) {
                if (spins > A.spin_limit) {
                    __hip_atomic_store(A.err, 3, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    ok = false;
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
#pragma unroll
            for (int j = 0; j < kPre; j++) {
                const unsigned long long *ps = pp + (size_t)(sub + j * nsub) * (2 + HD);
#pragma unroll
                for (int k = 0; k < 6; k++)
                    if (pending & (1u << (6 * j + k)))
                        wv6[j][k] = ll_word_load(ps + (k < 2 ? k : 2 + cg * 4 + (k - 2)));
            }
#pragma unroll
            for (int j = 0; j < kPre; j++)
#pragma unroll
                for (int k = 0; k < 6; k++)
                    if ((pending & (1u << (6 * j + k))) && (uint32_t)(wv6[j][k] >> 32) == ep)
                        pending &= ~(1u << (6 * j + k));
        }
        // spans past kPre per thread (contexts above nsub * kPre * P positions): one by one, the
        // first of them kept (read again after the maximum, it cost another 0.3 us)
        auto wait6 = [&](int s, unsigned long long (&w)[6]) {
            poll(s, w);
            for (uint32_t spins = 0; ok; spins++) {
                bool cur = true;
#pragma unroll
                for (int k = 0; k < 6; k++) cur = cur && (uint32_t)(w[k] >> 32) == ep;
                if (cur) break;
                if (spins > A.spin_limit) {
                    __hip_atomic_store(A.err, 3, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    ok = false;
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
                poll(s, w);
            }
        };
        const int sx = sub + kPre * nsub;
        unsigned long long wx[6] = {(unsigned long long)__float_as_uint(-INFINITY)};
        if (sx < nact) wait6(sx, wx);
        auto wf = [](unsigned long long w) { return __uint_as_float((uint32_t)w); };
        float *mred = reinterpret_cast<float *>(tiles);  // [NW] wave maxima
        // global maximum of the span maxima
        float M = -INFINITY;
#pragma unroll
        for (int j = 0; j < kPre; j++) M = fmaxf(M, wf(wv6[j][0]));
        M = fmaxf(M, wf(wx[0]));
        for (int s = sx + nsub; s < nact; s += nsub) {
            unsigned long long w[6];
            wait6(s, w);
            M = fmaxf(M, wf(w[0]));
        }
        M = wave_max_f(M);
        if (lane == 0) mred[wv] = M;
        __syncthreads();
        M = mred[0];
        for (int w = 1; w < NW; w++) M = fmaxf(M, mred[w]);
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
        float L = 0.0f;
        auto add_span = [&](const unsigned long long (&w)[6]) {
            const float e = expf(wf(w[0]) - M);
            L = fmaf(wf(w[1]), e, L);
            acc.x = fmaf(wf(w[2]), e, acc.x);
            acc.y = fmaf(wf(w[3]), e, acc.y);
            acc.z = fmaf(wf(w[4]), e, acc.z);
            acc.w = fmaf(wf(w[5]), e, acc.w);
        };
#pragma unroll
        for (int j = 0; j < kPre; j++)
            if (sub + j * nsub < nact) add_span(wv6[j]);
        if (sx < nact) add_span(wx);
        for (int s = sx + nsub; s < nact; s += nsub) {
            unsigned long long w[6];
            wait6(s, w);
            add_span(w);
        }
        // subsets added in order
        float *osub = reinterpret_cast<float *>(tiles) + 64;  // [nsub][HD]
        float *lsub = osub + nsub * HD;                      // [nsub]
        *reinterpret_cast<float4 *>(osub + sub * HD + cg * 4) = acc;
        if (cg == 0) lsub[sub] = L;
        __syncthreads();
        if ((int)tid < HD) {
            float Lt = lsub[0], o = osub[tid];
            for (int u = 1; u < nsub; u++) {
                Lt += lsub[u];
                o += osub[u * HD + tid];
            }
            fin[tid] = o * (1.0f / Lt);
        }
        __syncthreads();
        if (wv < nb) finish_head(A, fin[wv * 64 + (int)lane], head, wv, nb, lane);
        // the last merge workgroup of the launch advances the epoch (every span workgroup
        // of this launch has published, so all have read the epoch already)
        if (tid == 0) {
            const unsigned int total = gridDim.x * (unsigned int)G;
            if (__hip_atomic_fetch_add(A.cnt + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == total - 1u) {
                __hip_atomic_store(A.cnt + 1, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(A.cnt, ep, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        return;
    }
    // ---------------------------------------------------------------- span workgroup
    const int span = (int)blockIdx.y - G;
    const int t0 = span * P, n = min(act - t0, P);
    if (n <= 0) return;  // spans past the context take no part
    const size_t base = ((size_t)layer * nkv + kvh) * kr.cap;
    int8_t *kt = tiles, *vt = tiles + P * HD;
    // Slot of the idx-th attended position: the sinks keep theirs; later positions follow the
    // ring from the first one's place (`first`), wrapping at most once.
    int first = 0;
    if constexpr (RING) first = (seq > kr.window ? seq - kr.window : 0) % kr.ring;
    auto slot_of = [&](int idx) -> size_t {
        if constexpr (!RING) return base + (size_t)idx;
        int s = idx;
        if (idx >= kr.sinks) {
            s = first + (idx - kr.sinks);
            s = kr.sinks + (s >= kr.ring ? s - kr.ring : s);
        }
        return base + (size_t)s;
    };
    // 1. K / V rows of positions t0 .. t0 + P - 1 (rows past n re-read row n - 1), 16 bytes a
    //    lane, and their scales
    constexpr int row_bytes = BITS == 4 ? HD / 2 : HD, per_row = row_bytes / 16, pieces = P * per_row;
    constexpr int PT = (pieces + NTH - 1) / NTH;  // (past the last piece: row n - 1 again, not stored)
    static_assert(BITS == 4 || pieces % NTH == 0, "direct-to-LDS copies by whole waves");
    uint4 kreg[BITS == 4 ? PT : 1], vreg[BITS == 4 ? PT : 1];
    uint32_t ksc = 0, vsc = 0;
    if constexpr (BITS == 8) {
        const uint32_t mk = lds_offset(kt), mvv = lds_offset(vt);
#pragma unroll
        for (int j = 0; j < PT; j++) {
            const int i = j * NTH + (int)tid;
            const size_t off = slot_of(t0 + min(i / per_row, n - 1)) * row_bytes + (size_t)(i % per_row) * 16;
            const uint32_t m0 = (uint32_t)(j * NTH + wv * 64) * 16u;
            lds_dma16(A.kq + off, mk + m0);
            lds_dma16(A.vq + off, mvv + m0);
        }
        // scales, 64 positions a load: K's P / 64 groups, then V's
        for (int u = wv; u < 2 * P / 64; u += NW) {
            const int w = u % (P / 64);
            const size_t sl = slot_of(t0 + min(w * 64 + (int)lane, n - 1));
            const uint32_t m0 = (uint32_t)__builtin_amdgcn_readfirstlane(
                (int)(lds_offset(u < P / 64 ? kst : vst) + (uint32_t)w * 256u));
            lds_dma4((u < P / 64 ? A.ks : A.vs) + sl, m0);
        }
    } else {
#pragma unroll
        for (int j = 0; j < PT; j++) {
            const int i = j * NTH + (int)tid;
            const size_t off = slot_of(t0 + min(i / per_row, n - 1)) * row_bytes + (size_t)(i % per_row) * 16;
            kreg[j] = ld_global(reinterpret_cast<const uint4 *>(A.kq + off));
            vreg[j] = ld_global(reinterpret_cast<const uint4 *>(A.vq + off));
        }
        // scales: one position a thread (BF16, one per 64-block)
        static_assert(P <= NTH, "a thread per position");
        const size_t sl = slot_of(t0 + min((int)tid, n - 1));
        if constexpr (nb == 2) {
            ksc = ld_global(reinterpret_cast<const uint32_t *>(A.ks) + sl);
            vsc = ld_global(reinterpret_cast<const uint32_t *>(A.vs) + sl);
        } else {
            ksc = ld_global(reinterpret_cast<const uint16_t *>(A.ks) + sl);
            vsc = ld_global(reinterpret_cast<const uint16_t *>(A.vs) + sl);
        }
    }
    // 2. q head wv (and the current position's K / V where this span holds it)
    const AttnPost &post = A.post;
    const int cur = act - 1;  // the current position's place among the attended ones
    const bool covers = post.on && t0 <= cur && cur < t0 + n;
    if (wv < G) {
        const int head = kvh * G + wv;
        const float *qh = A.q + (size_t)head * HD;
        float qv0, qv1;
        if (post.on) {
            head_post(qh, head, nq, nkv, HD, post.bias, post.qn, post.kn, post.eps, post.rope, seq - 1, lane, qv0, qv1);
        } else {
            qv0 = qh[lane];
            qv1 = nb > 1 ? qh[64 + lane] : 0.0f;
        }
        const float r0 = fwht_lane(qv0, 0, lane);
        const float r1 = nb > 1 ? fwht_lane(qv1, 1, lane) : 0.0f;
        const float mx = wave_max_f(fmaxf(fabsf(r0), fabsf(r1)));
        int8_t *qd = qi + wv * HD;
        if (mx <= FLT_EPSILON) {
            qd[lane] = 0;
            if (nb > 1) qd[64 + lane] = 0;
            if (lane == 0) qas[wv] = 0.0f;
        } else {
            const float inv = 127.0f / mx;
            qd[lane] = (int8_t)(int)rintf(r0 * inv);
            if (nb > 1) qd[64 + lane] = (int8_t)(int)rintf(r1 * inv);
            if (lane == 0) qas[wv] = (mx / 127.0f) * A.attn_scale;
        }
    }
    if (covers && wv >= 6) {
        const bool is_k = wv == 6;
        const int hh = is_k ? nq + kvh : nq + nkv + kvh;
        float a0, a1;
        head_post(A.q + (size_t)hh * HD, hh, nq, nkv, HD, post.bias, post.qn, post.kn, post.eps, post.rope, seq - 1, lane,
                  a0, a1);
        const float r0 = fwht_lane(a0, 0, lane);
        const float r1 = nb > 1 ? fwht_lane(a1, 1, lane) : 0.0f;
        kv_store_head(r0, r1, nb, lane, BITS, HD, 0, is_k ? kcur : vcur, is_k ? cur_k : cur_v);
        kv_store_head(r0, r1, nb, lane, BITS, HD, slot_of(cur), is_k ? A.kq : A.vq, is_k ? A.ks : A.vs);
    }
    // NF4: 16 packed bytes (32 codes of one row) to int8 codebook values: low nibbles are 16
    // consecutive elements, high nibbles the next 16
    auto unpack = [](const uint4 &p, int8_t *dst) {
        uint32_t T0, T1, U0, U1;
        nf4_xor_tables(kNf4Cb0, kNf4Cb1, kNf4Cb2, kNf4Cb3, T0, T1, U0, U1);
        const uint32_t d[4] = {p.x, p.y, p.z, p.w};
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            lo[j] = nf4_xlut(d[j] & 0x0F0F0F0Fu, T0, T1, U0, U1);
            hi[j] = nf4_xlut((d[j] >> 4) & 0x0F0F0F0Fu, T0, T1, U0, U1);
        }
        reinterpret_cast<uint4 *>(dst)[0] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
        reinterpret_cast<uint4 *>(dst)[1] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    };
    if constexpr (BITS == 4) {
#pragma unroll
        for (int j = 0; j < PT; j++) {
            const int i = j * NTH + (int)tid;
            if (i >= pieces) break;
            unpack(kreg[j], kt + (size_t)i * 32);
            unpack(vreg[j], vt + (size_t)i * 32);
        }
        if ((int)tid < P)
#pragma unroll
            for (int g = 0; g < nb; g++) {
                kst[tid * nb + g] = g ? bf16_hi(ksc) : bf16_lo(ksc);
                vst[tid * nb + g] = g ? bf16_hi(vsc) : bf16_lo(vsc);
            }
    } else {
        wait_vmcnt<0>();  // this wave's tile copies have landed
    }
    __syncthreads();
    if (covers) {  // the current position's row (its tile copy read the slot before it was written)
        const int r = cur - t0;
        if constexpr (BITS == 8) {
            if ((int)tid < HD) {
                kt[r * HD + tid] = kcur[tid];
                vt[r * HD + tid] = vcur[tid];
            }
            if (tid == 0) {
                kst[r] = cur_k[0];
                vst[r] = cur_v[0];
            }
        } else {
            if ((int)tid < 2 * per_row) {
                const int c = (int)tid % per_row;
                const bool is_k = (int)tid < per_row;
                unpack(*reinterpret_cast<const uint4 *>((is_k ? kcur : vcur) + 16 * c), (is_k ? kt : vt) + r * HD + 32 * c);
            }
            if ((int)tid < 2 * nb) {
                const int g = (int)tid % nb;
                const bool is_k = (int)tid < nb;
                const uint16_t s = reinterpret_cast<const uint16_t *>(is_k ? cur_k : cur_v)[g];
                (is_k ? kst : vst)[r * nb + g] = __uint_as_float((uint32_t)s << 16);
            }
        }
        __syncthreads();
    }
    // 3. scores and o on the matrix cores.  Wave w takes the 16-position tiles w, w + 8, ...:
    //  - scores: v_mfma_i32_16x16x64_i8 with A = K (lane l: position l%16 of the tile) and
    //    B = the int8 q heads, repeated over the 16 columns (lane l: head l%16%GC; heads past G
    //    are zero): exact integer dots, lane l holding positions 4(l/16) + r of its head;
    //  - the span's maximum and sum per head: each wave's over its positions, then the
    //    waves' in wave order;
    //  - o^T += V^T (p vs)^T by v_mfma_f32_4x4x1 (16 blocks of 4 dims x 4 heads, one position
    //    each): the step for register r and V byte k takes the positions 4g + r of the four
    //    lane rows g at once, with A = the row's V values (lane l: dims DB (l%16) + k) and
    //    B = the score registers as they stand, because the heads repeat every four lanes.
    //    Four heads cost 8 cycles a step; 16x16x4 steps with mostly empty columns cost four
    //    times that (one head x 64 dims x 16 positions: 512 cycles, 128 here).
    //    Lane l ends with the dims of block l/4 for head l%4, over its row's positions: the
    //    rows are added by lane swaps, after which row g holds dims of accumulator row g.
    //    (The NF4 cache's V scale depends on the dim: it goes with V, where code times
    //    scale is exact.)
    const uint32_t li = lane & 15u, lg = lane >> 4;
    const int hq = (int)(li % GC);
    const bool hl = hq < G;
    const float qs = hl ? qas[hq] : 0.0f;
    float sc4[TPW][4];
    float tmax = -INFINITY;
#pragma unroll
    for (int t = 0; t < TPW; t++) {
        const int pw0 = 16 * (wv + NW * t), pr = pw0 + 4 * (int)lg;  // this lane's first position
        v4i acc[nb];
#pragma unroll
        for (int k = 0; k < nb; k++) {
            const int4 kv = *reinterpret_cast<const int4 *>(kt + (pw0 + (int)li) * HD + 64 * k + 16 * (int)lg);
            const int4 qv = hl ? *reinterpret_cast<const int4 *>(qi + hq * HD + 64 * k + 16 * lg) : make_int4(0, 0, 0, 0);
            const v4i zero = {0, 0, 0, 0};
            // one dot per head, or one per 64-block where each block has its own term
            acc[k] = __builtin_amdgcn_mfma_i32_16x16x64_i8(v4i{kv.x, kv.y, kv.z, kv.w}, v4i{qv.x, qv.y, qv.z, qv.w},
                                                            (BITS == 8 && !RING && k > 0) ? acc[k - 1] : zero, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            float s = 0.0f;
            if constexpr (BITS == 8 && !RING) {
                s = ((float)acc[nb - 1][r] * kst[pr + r]) * qs;
            } else {
#pragma unroll
                for (int k = 0; k < nb; k++) {
                    const float term = ((float)acc[k][r] * kst[(pr + r) * SB + (SB > 1 ? k : 0)]) * qs;
                    s = k == 0 ? term : s + term;
                }
            }
            sc4[t][r] = hl && pr + r < n ? s : -INFINITY;
            tmax = fmaxf(tmax, sc4[t][r]);
        }
    }
    tmax = fmaxf(tmax, xor_lane(tmax, 16));
    tmax = fmaxf(tmax, xor_lane(tmax, 32));
    if (lane < (uint32_t)GC && hl) red_m[lane][wv] = tmax;
    __syncthreads();
    float m = -INFINITY;
    if (hl) {
        m = red_m[hq][0];
#pragma unroll
        for (int u = 1; u < NW; u++) m = fmaxf(m, red_m[hq][u]);
    }
    float psum = 0.0f;
    v4f o[HP][DB];
#pragma unroll
    for (int h = 0; h < HP; h++)
#pragma unroll
        for (int k = 0; k < DB; k++) o[h][k] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < TPW; t++) {
        const int pr = 16 * (wv + NW * t) + 4 * (int)lg;
        if (16 * (wv + NW * t) >= n) break;  // wave-uniform: no position left
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float pe = sc4[t][r] == -INFINITY ? 0.0f : expf(sc4[t][r] - m);
            psum += pe;
            // (a row past the span's end may hold the scale of a slot not yet written, any bits)
            const bool in = pr + r < n;
            const float w = BITS == 4 ? pe : in ? pe * vst[pr + r] : 0.0f;
            const float vsg = BITS == 4 && in ? vst[(pr + r) * SB + (SB > 1 ? (int)(li >> 3) : 0)] : 0.0f;
            float wh[HP];
            if constexpr (G8) {  // this lane's own head and the one four columns on
                const float x = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(w), 0x124, 0xF, 0xF, true));
                wh[0] = (li & 4u) ? x : w;
                wh[1] = (li & 4u) ? w : x;
            } else {
                wh[0] = w;
            }
            uint32_t vw[DB / 4];
            const int8_t *vp = vt + (pr + r) * HD + DB * (int)li;
            if constexpr (DB == 8) {
                const uint2 u = *reinterpret_cast<const uint2 *>(vp);
                vw[0] = u.x;
                vw[1] = u.y;
            } else {
                vw[0] = *reinterpret_cast<const uint32_t *>(vp);
            }
#pragma unroll
            for (int k = 0; k < DB; k++) {
                float a = (float)(int8_t)((vw[k / 4] >> (8 * (k & 3))) & 0xFFu);
                if constexpr (BITS == 4) a *= vsg;
#pragma unroll
                for (int h = 0; h < HP; h++) o[h][k] = __builtin_amdgcn_mfma_f32_4x4x1f32(a, wh[h], o[h][k], 0, 0, 0);
            }
        }
    }
    psum += xor_lane(psum, 16);
    psum += xor_lane(psum, 32);
    if (lane < (uint32_t)GC && hl) red_l[lane][wv] = psum;
    constexpr int OS = o_stride(HD);
    constexpr bool kBehind = o_behind(TPW, G8);
    if constexpr (!kBehind) __syncthreads();  // the tiles are read
    float *opw = reinterpret_cast<float *>(tiles + (kBehind ? 2 * P * HD : 0));  // [wave][head][OS]
#pragma unroll
    for (int h = 0; h < HP; h++) {
        // Rows added: a swap of odd and even 16-lane rows of two values and an add leave
        // each value's row pairs side by side, the swap of 32-lane halves the totals.
        // Accumulator row i of byte k (dim DB (4 (l%16/4) + i) + k) ends in lane row i.
        float v[DB];
#pragma unroll
        for (int k = 0; k < DB; k++) {
            const auto p01 = __builtin_amdgcn_permlane16_swap(__float_as_uint(o[h][k][0]), __float_as_uint(o[h][k][1]), false, false);
            const auto p23 = __builtin_amdgcn_permlane16_swap(__float_as_uint(o[h][k][2]), __float_as_uint(o[h][k][3]), false, false);
            const float s01 = __uint_as_float(p01[0]) + __uint_as_float(p01[1]);
            const float s23 = __uint_as_float(p23[0]) + __uint_as_float(p23[1]);
            const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(s01), __float_as_uint(s23), false, false);
            v[k] = __uint_as_float(q[0]) + __uint_as_float(q[1]);
        }
        const int head = 4 * h + (int)(lane & 3u);
        if (head < G) {
            float *dst = opw + ((size_t)wv * G + head) * OS + DB * (4 * (int)(li >> 2) + (int)lg);
#pragma unroll
            for (int k = 0; k < DB; k += 4) *reinterpret_cast<float4 *>(dst + k) = make_float4(v[k], v[k + 1], v[k + 2], v[k + 3]);
        }
    }
    __syncthreads();
    // 4. the waves' sums in wave order, published (or, with one span, finished here)
    unsigned long long *pbase = A.words + (size_t)(kvh * G) * pstride + (size_t)span * (2 + HD);
    for (int i = (int)tid; i < G * HD; i += NTH) {
        const int h = i / HD, c = i % HD;
        float ov = opw[(size_t)h * OS + c];
        for (int u = 1; u < NW; u++) ov += opw[((size_t)u * G + h) * OS + c];
        unsigned long long *pp = pbase + (size_t)h * pstride;
        if (nact != 1) {
            ll_word_store(pp + 2 + c, __float_as_uint(ov), ep);
            if (c != 0) continue;
        }
        float mm = red_m[h][0], l = red_l[h][0];
        for (int u = 1; u < NW; u++) {
            mm = fmaxf(mm, red_m[h][u]);
            l += red_l[h][u];
        }
        if (nact == 1) {
            fin[i] = ov * (1.0f / l);
        } else {
            ll_word_store(pp, __float_as_uint(mm), ep);
            ll_word_store(pp + 1, __float_as_uint(l), ep);
        }
    }
    if (nact != 1) return;
    __syncthreads();
    for (int i = wv; i < G * nb; i += NW) finish_head(A, fin[i * 64 + (int)lane], kvh * G + i / nb, i % nb, nb, lane);
}

// Tiles per wave (spans of 128 or 256 positions): one span where the context fits in one
// (no hand-off; 200 positions, 32 heads x 64: 7.3 us in two spans, 5.5 in one), else 128-position
// spans until their workgroups are more than the CUs, then 256 (8 KV heads x 128, 4100 positions:
// 264 workgroups 14.4 us, 136 of twice the length 11.1 us; 32 KV heads x 64, 1024 positions:
// 256 workgroups 8.7 us, 128 8.3 us).
int span_tiles(int num_cus, int nkv, int positions) {
    if (positions <= 256) return positions <= 128 ? 1 : 2;
    return (long)nkv * ((positions + 127) / 128) > num_cus ? 2 : 1;
}

template <int HD, int BITS, bool RING>
void launch_span(hipStream_t st, int tpw, bool g8, dim3 grid, size_t lds, const SpanArgs &A) {
    const dim3 blk(kSpanThreads);
    if (tpw == 2 && g8) hipLaunchKernelGGL((attn_span_kernel<HD, BITS, RING, 2, true>), grid, blk, lds, st, A);
    else if (tpw == 2) hipLaunchKernelGGL((attn_span_kernel<HD, BITS, RING, 2, false>), grid, blk, lds, st, A);
    else if (g8) hipLaunchKernelGGL((attn_span_kernel<HD, BITS, RING, 1, true>), grid, blk, lds, st, A);
    else hipLaunchKernelGGL((attn_span_kernel<HD, BITS, RING, 1, false>), grid, blk, lds, st, A);
}

}  // namespace

// The nq merge workgroups come first in dispatch order and wait for the span workgroups', so
// those must find room beside them.  At least two workgroups fit on a CU (at most 76 KB of LDS,
// 8 waves of 128 VGPRs): with one merge workgroup per two CUs a launch uses at most a quarter of
// the places for waiting, and up to three launches on streams of their own still end.
bool attn_span_supported(int num_cus, int nq, int nkv, int hd, const KvRing &kr) {
    return nq / nkv <= kSpanMaxGroup && nq <= num_cus / 2 && (hd == 64 || hd == 128) &&
           (kr.bits == 8 || kr.bits == 4) && (kr.window == 0 || kr.ring >= kr.window - kr.sinks);
}

size_t attn_span_words(int positions, int nq, int hd) { return (size_t)((positions + 127) / 128) * nq * (2 + hd); }

void launch_attn_span(hipStream_t st, const float *q, int8_t *kq, int8_t *vq, float *ks, float *vs, const AttnPost &post,
                      const int *pos_dev, int pos, int layer, int nq, int nkv, int hd, KvRing kr, float attn_scale,
                      int max_positions, float *out_f, int8_t *aq, float *as, int32_t *asum, const SpanWork &w) {
    const int tpw = span_tiles(w.num_cus, nkv, max_positions), P = 128 * tpw, G = nq / nkv;
    const int nspan = (max_positions + P - 1) / P;
    SpanArgs A{q, kq, vq, ks, vs, pos_dev, pos, layer, nq, nkv, kr, attn_scale, nspan, post, w.words,
               w.cnt, w.err, w.wait, out_f, aq, as, asum};
    const dim3 grid(nkv, G + nspan);
    const size_t lds = std::max(span_lds(hd, P, G), (size_t)(64 + 4 * kSpanThreads + 64) * sizeof(float));
    const bool ring = kr.window > 0;
    if (hd == 128 && kr.bits == 8 && !ring) launch_span<128, 8, false>(st, tpw, G > 4, grid, lds, A);
    else if (hd == 128 && kr.bits == 8) launch_span<128, 8, true>(st, tpw, G > 4, grid, lds, A);
    else if (hd == 128 && !ring) launch_span<128, 4, false>(st, tpw, G > 4, grid, lds, A);
    else if (hd == 128) launch_span<128, 4, true>(st, tpw, G > 4, grid, lds, A);
    else if (kr.bits == 8 && !ring) launch_span<64, 8, false>(st, tpw, G > 4, grid, lds, A);
    else if (kr.bits == 8) launch_span<64, 8, true>(st, tpw, G > 4, grid, lds, A);
    else if (!ring) launch_span<64, 4, false>(st, tpw, G > 4, grid, lds, A);
    else launch_span<64, 4, true>(st, tpw, G > 4, grid, lds, A);
    hip_check(hipGetLastError(), "attn_span launch");
}

}  // namespace k2t
