// Batched quantized GEMV (prefill) on the int8 matrix cores of gfx950: out[t][r] =
// sum_c fmaf(float(dot_{r,c,t}) * sx[t][c], ws[r][c], ...), the chunk dots from v_mfma_i32_16x16x64_i8.  NF4 and NF3 (NfSdotMatrix) and the bit-plane
// formats b4 / b5 / b6 (Nibble4SdotMatrix) share the kernel (FMT 1, 2, 0).
//
// The reference runs prefill through the same kernels as decode, four tokens per weight
// pass (nf_sdot_decode_neon's 4-token tile, simd_lut.rs:6074-6364, and the Nibble4 tile
// nibble4_sdot_batch_stripe_range, 4101-4320).  Here a 16-row stripe's codes of a 64-column
// chunk are decoded to int8 once per up to 128 tokens, with one MFMA per 16-token block
// (A: 16 rows x 64 codes, B: 64 activation bytes x 16 tokens).  Three kernels share that step and
// differ in how stripes, tokens and chunks are dealt to waves (plain_form's rule).
//  - NF4: the codebook value of each code (the codebook as two v_perm XOR tables,
//    nf4_xlut); the MFMA gives the chunk dot.
//  - NF3: the same through one v_perm per four codes, from the row's triplet of dwords, in
//    the device's lane order or the reference's.  With the fast epilogue its sums keep the
//    one-token GEMV's order (launch_gemm_ordered).
//  - bit planes: the unsigned code u (4 + hp bits: the nibble and the hi-plane bits); the
//    MFMA gives sum(u * x), and the chunk dot of the odd weights 2u - (2^(4+hp) - 1) is
//    2 * sum(u * x) - (2^(4+hp) - 1) * sum(x), as the reference computes it (simd_lut.rs:
//    4030-4045 and 4304-4309: the sdot of the codes acc, then 2 * acc - max_odd * xsum).
// The epilogue is the reference's per-row chain in chunk order (simd_lut.rs:4030-4059,
// 6334-6335: f = fmaf(float(dot) * sx, scale, f), chunks with sx == 0 skipped), so every
// output (but NF3's with the fast epilogue) equals the exact-order GEMV's (k2t_ctx_set_exact) bit
// for bit.
//
// Operand layouts of v_mfma_i32_16x16x64_i8 (checked on the GPU): lane l holds 16 bytes of
// A row l % 16 and of B column l % 16; the products pair lane l's byte b of A with lane
// l's byte b of B over the four lane groups l / 16, so any one assignment of the 64
// columns to (l / 16, b) used for both operands gives the dot.  Here byte b of group g is
// column 16g + b.  The 16 x 16 int32 result: lane l holds rows 4 (l / 16) + r, r = 0..3,
// of column l % 16.
//
// Nibble bytes of a stripe-chunk (512 per stripe, the same order in both formats:
// NfSdotMatrix, simd_lut.rs:4796-5023; Nibble4SdotMatrix, 3331-3385): byte e of dword j at
// kk*128 + g*32 + half*16 + 4j holds the codes of row 4g + j, columns kk*16 + half*8 + e
// (low nibble) and kk*16 + half*8 + 4 + e (high nibble).  Row i's columns 16kk .. 16kk+15
// are therefore the dwords at kk*128 + (i/4)*32 + 4(i%4) and 16 bytes further: low / high
// nibbles of the first give columns 0-3 / 4-7, of the second 8-11 / 12-15.  Bit-plane hi
// planes: for 16-byte piece p of a stripe's hi bytes (64 bytes apart), dword j of row
// group g (g*16 + 4j) holds the bits of row 4g + j for columns kk*16 .. kk*16+15, kk = 2p
// and 2p + 1 (one hi plane) or kk = p (two), in the bit positions the decode kernels'
// rotations select (chunk_dots in k2t_gemv_core.h).
#include <type_traits>

#include "../../include/k2t_hip.h"
#include "k2t_device.h"
#include "k2t_internal.h"
#include "k2t_kv_dev.h"

namespace k2t {

namespace {

constexpr int kMfmaDepth = 4;  // chunks in flight per wave (gemm_mfma_kernel)

typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));

struct MfArgs {
    const uint8_t *pair, *tail;
    size_t ptot;  // bytes per pair stream
    int rows, nc, np, stripes, sgc_log2;  // NF scale group = 1 << sgc_log2 chunks
    uint32_t t0, t1, u0, u1;  // NF4 codebook XOR tables (nf4_xor_tables); NF3: t0, t1 the codebook
    int lane;                 // NF3: stripe-chunks in lane order
    const int8_t *xt;  // activations tile-major: [16-token block][chunk][64 lanes][16 bytes]
    const float *st;   // their scales: [16-token block][chunk][16 tokens]
    const int32_t *ut;  // their code sums (bit planes): [16-token block][chunk][16 tokens]
    int K, ntok, nblk;  // nblk: 16-token blocks
    int tiled;          // gemm_ks_kernel: 0 = xt / st / ut are the [token] rows themselves
    int nseg, cps, g_log2;  // gemm_ks_kernel, one-token order: plan_gemv's K segments and accumulators
    float *out;
    size_t out_stride;
    int accum;
    // SwiGLU epilogue (gate_up with interleaved [gate64, up64] blocks): the down input as
    // int8 chunks, scales and sums ([token][nci]) and its tile-major copy
    int8_t *sq;
    float *ss;
    int32_t *ssum;
    ActTiles stiles;
    int nci;
    QkvPostDev qp;  // q / k / v epilogue (the qkv projection at head size 64)
};

// Everything one chunk needs (one ring stage): the stripe-chunk's codes and scales, the
// activation blocks and their scales.
template <int FMT, int NB>
struct MfChunk {
    uint32_t d0, d1;
    uint32_t hv;  // bit planes with hi planes: this lane's hi-plane dword; NF3: its third dword
    uint2 sw;
    int4 x[NB];
    float sx[NB];
    int32_t su[FMT == 0 ? NB : 1];  // bit planes: the tokens' code sums
};

// Buffer resource of a wave-uniform base (raw, no stride; dword 3 as gfx950 wants it).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t mf_rsrc(const void *base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, 0x7FFFFFFF, 0x00020000);
}

struct MfSrc {
    __amdgpu_buffer_rsrc_t w, x, s, u;  // the stripe's stream (pair or tail), the tiles, scales, sums
};

// Per-lane offsets of a stripe-chunk record, fixed for the wave's life.
struct MfLane {
    uint32_t a_off, b_off;  // the lane's first and second code dword
    uint32_t h_off;  // its hi-plane dword (bit planes), its third code dword (NF3)
    uint32_t s_off;  // its rows' BF16 scale pair
    uint32_t x_off, sx_off;
};

// A lane's 16 bytes of the A operand: the int8 values (NF: codebook entries; bit planes: the
// unsigned codes) of its row's columns 16 (lane / 16) .. + 15, from its code dwords.
template <int FMT, int HP>
__device__ __forceinline__ v4i mf_decode(uint32_t d0, uint32_t d1, uint32_t hv, uint32_t t0, uint32_t t1, uint32_t u0,
                                         uint32_t u1, uint32_t lane) {
    v4i a;
    if constexpr (FMT == 0) {
        // the unsigned codes: nibble, then the hi-plane bits (as chunk_dots places them for
        // kk = lane group, half 0 for the first dword and half 1 for the second)
        uint32_t lo0 = d0 & 0x0F0F0F0Fu, hi0 = (d0 >> 4) & 0x0F0F0F0Fu;
        uint32_t lo1 = d1 & 0x0F0F0F0Fu, hi1 = (d1 >> 4) & 0x0F0F0F0Fu;
        if constexpr (HP == 2) {
            lo0 |= hv & 0x30303030u;
            hi0 |= __builtin_rotateright32(hv, 2u) & 0x30303030u;
            lo1 |= __builtin_rotateright32(hv, 30u) & 0x30303030u;
            hi1 |= __builtin_rotateright32(hv, 28u) & 0x30303030u;
        } else if constexpr (HP == 1) {
            // odd lane groups: the piece's upper bits
            const uint32_t h = __builtin_rotateright32(hv, (lane & 16u) ? 28u : 0u);
            lo0 |= h & 0x10101010u;
            hi0 |= __builtin_rotateright32(h, 1u) & 0x10101010u;
            lo1 |= __builtin_rotateright32(h, 2u) & 0x10101010u;
            hi1 |= __builtin_rotateright32(h, 3u) & 0x10101010u;
        }
        a[0] = (int)lo0;
        a[1] = (int)hi0;
        a[2] = (int)lo1;
        a[3] = (int)hi1;
    } else if constexpr (FMT == 2) {
        // NF3 triplet (v0, v1, v2) of this row and 32-column half: codes 0-3 (even lane
        // group) or 4-7 (odd) are this lane's four column quads; code 2 / 5 has its third
        // bit in v2.  v0 = i0 | i1 << 3 | i2 << 6, v1 = i3 | i4 << 3 | i5 << 6, v2 = i6 | i7 << 3
        // | third bits of i2, i5.  One v_perm looks four codes up in the 8-entry codebook.
        const bool odd = (lane & 16u) != 0u;
        const uint32_t p = odd ? d1 : d0, r = odd ? hv : d1;
        const uint32_t e = (odd ? hv >> 3 : d0) & 0x07070707u;              // i0 / i7
        const uint32_t n = (p >> 3) & 0x07070707u;                              // i1 / i4
        const uint32_t m = ((p >> 6) & 0x03030303u) | ((hv >> (odd ? 5 : 4)) & 0x04040404u);  // i2 / i5
        const uint32_t l = r & 0x07070707u;                                     // i3 / i6
        a[0] = (int)__builtin_amdgcn_perm(t1, t0, odd ? n : e);
        a[1] = (int)__builtin_amdgcn_perm(t1, t0, odd ? m : n);
        a[2] = (int)__builtin_amdgcn_perm(t1, t0, odd ? l : m);
        a[3] = (int)__builtin_amdgcn_perm(t1, t0, odd ? e : l);
    } else {
        a[0] = (int)nf4_xlut(d0 & 0x0F0F0F0Fu, t0, t1, u0, u1);
        a[1] = (int)nf4_xlut((d0 >> 4) & 0x0F0F0F0Fu, t0, t1, u0, u1);
        a[2] = (int)nf4_xlut(d1 & 0x0F0F0F0Fu, t0, t1, u0, u1);
        a[3] = (int)nf4_xlut((d1 >> 4) & 0x0F0F0F0Fu, t0, t1, u0, u1);
    }
    return a;
}

// Per-lane offsets inside the records of a stripe (side 0 / 1 of its pair, or the tail).
template <int FMT, int HP>
__device__ __forceinline__ MfLane mf_lane(uint32_t lane, bool is_tail, uint32_t side, int lane_order) {
    MfLane L;
    const uint32_t li = lane & 15u, lg = lane >> 4;
    if constexpr (FMT == 2) {
        // block (g, half): 16-byte pieces 128 bytes apart in lane order, 16 in the reference's
        const uint32_t g = li >> 2, half = lg >> 1, ps = lane_order ? 128u : 16u;
        L.a_off = (is_tail ? 0u : side * 384u) + (lane_order ? (2u * g + half) * 16u : half * 192u + g * 48u) +
                  4u * (li & 3u);
        L.b_off = L.a_off + ps;
        L.h_off = L.a_off + 2u * ps;
        L.s_off = (is_tail ? 0u : side * 32u) + 8u * lg;
    } else {
        L.a_off = (is_tail ? 0u : side * 512u) + lg * 128u + (li >> 2) * 32u + 4u * (li & 3u);
        L.b_off = L.a_off + 16u;
    }
    if constexpr (FMT == 0) {
        const uint32_t hib = is_tail ? 512u : 1024u + side * 128u * HP;  // the stripe's hi bytes
        L.h_off = hib + (HP == 2 ? lg : lg >> 1) * 64u + (li >> 2) * 16u + 4u * (li & 3u);
        L.s_off = (is_tail ? 512u + 128u * HP : 1024u + 256u * HP + side * 32u) + 8u * lg;  // rows 4lg .. 4lg+3
    } else if constexpr (FMT == 1) {
        L.h_off = 0;
        L.s_off = (is_tail ? 0u : side * 32u) + 8u * lg;
    }
    return L;
}

// Every load is a buffer load: the wave-uniform part of its offset in an SGPR, the
// per-lane part (fixed for the wave's life) in one VGPR, so no 64-bit address adds.
//  - NF: group sg = c / sgc starts at sg * gsz + sg * sgc * cs (gsz = 64 bytes of scales,
//    32 in the tail; cs = 1024 bytes of codes per chunk, 512 in the tail), the chunk's
//    codes at that + gsz + (c - sg * sgc) * cs.
//  - bit planes: chunk c's record at c * REC (REC = 1024 + 256 hp + 64, the tail's
//    512 + 128 hp + 32): codes, hi bytes, scales; the lane offsets point inside it.
template <int FMT, int HP>
__device__ __forceinline__ void mf_record(int sgc_log2, bool is_tail, int c, uint32_t &rec, uint32_t &sgb) {
    if constexpr (FMT == 0) {
        rec = (uint32_t)c * (is_tail ? 512u + 128u * HP + 32u : 1024u + 256u * HP + 64u);
        sgb = rec;
    } else {
        const uint32_t sg = (uint32_t)c >> sgc_log2, sb = (uint32_t)c - (sg << sgc_log2);
        constexpr uint32_t CB = FMT == 2 ? 384u : 512u;  // bytes per stripe-chunk
        const uint32_t cs = is_tail ? CB : 2u * CB, gsz = is_tail ? 32u : 64u;
        sgb = sg * gsz + (sg << sgc_log2) * cs;  // scale-group base
        rec = sgb + gsz + sb * cs;
    }
}

template <int FMT, int HP, int NB>
__device__ __forceinline__ void mf_fetch(const MfArgs &A, const MfSrc &R, const MfLane &L, bool is_tail, int tb0,
                                         int c, MfChunk<FMT, NB> &f) {
    uint32_t rec, sgb;
    mf_record<FMT, HP>(A.sgc_log2, is_tail, c, rec, sgb);
    f.d0 = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(R.w, L.a_off, rec, 0);
    f.d1 = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(R.w, L.b_off, rec, 0);
    if constexpr ((FMT == 0 && HP > 0) || FMT == 2) f.hv = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(R.w, L.h_off, rec, 0);
    const v2u sw = __builtin_amdgcn_raw_buffer_load_b64(R.w, L.s_off, sgb, 0);
    f.sw = make_uint2(sw[0], sw[1]);
#pragma unroll
    for (int b = 0; b < NB; b++) {
        // blocks past the last repeat it; their outputs are never stored
        const uint32_t tile = (uint32_t)min(tb0 + b, A.nblk - 1) * (uint32_t)A.nc + (uint32_t)c;
        const v4u x = __builtin_amdgcn_raw_buffer_load_b128(R.x, L.x_off, tile * 1024u, 0);
        f.x[b] = make_int4((int)x[0], (int)x[1], (int)x[2], (int)x[3]);
        f.sx[b] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(R.s, L.sx_off, tile * 64u, 0));
        if constexpr (FMT == 0) f.su[b] = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(R.u, L.sx_off, tile * 64u, 0);
    }
}

// One chunk's decode, MFMAs and epilogue steps.  A chunk whose activation scale is 0
// needs no select (NF4, bit planes) where ws is finite: its term float(d) * 0 * ws is +-0, and
// adding +-0 leaves every accumulator unchanged (each starts at +0 and a round-to-nearest sum is
// -0 only when both addends are -0, so no accumulator is ever -0).  Where the passes before these
// kernels skipped such a chunk whatever ws (NF3, 2 .. 15 tokens, experts), its ws is taken as 0.
template <int FMT, int HP, int NB>
__device__ __forceinline__ void mf_step(const MfArgs &A, const MfChunk<FMT, NB> &f, float (&acc)[NB][4], uint32_t lane) {
    const v4i a = mf_decode<FMT, HP>(f.d0, f.d1, f.hv, A.t0, A.t1, A.u0, A.u1, lane);
    const float ws[4] = {bf16_lo(f.sw.x), bf16_hi(f.sw.x), bf16_lo(f.sw.y), bf16_hi(f.sw.y)};
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const v4i bv = {f.x[b].x, f.x[b].y, f.x[b].z, f.x[b].w};
        const v4i zero = {0, 0, 0, 0};
        const v4i d = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, bv, zero, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            int dot = d[r];
            if constexpr (FMT == 0) dot = 2 * dot - ((1 << (4 + HP)) - 1) * f.su[b];
            acc[b][r] = fmaf((float)dot * f.sx[b], FMT == 2 && f.sx[b] == 0.0f ? 0.0f : ws[r], acc[b][r]);
        }
    }
}

// qkv (head size 64): qkv_post_kernel's work on a head's 64 rows of up to 64 tokens in LDS
// (ep[token][row], RP floats a token): bias, q / k RMSNorm and RoPE, then q into the qkv
// rows, k and v rotated and stored in the cache slot of their position.  The same arithmetic
// on the same values, so the cache and q equal the separate kernel's.
template <int RP, int W, int TOK>
__device__ __forceinline__ void mf_qkv_epilogue(const MfArgs &A, const float *ep, int tokb, int wave, uint32_t lane) {
    const QkvPostDev &Q = A.qp;
    const int head = (int)blockIdx.x, pos0 = Q.pos_dev[0];
    const uint32_t lg = lane >> 4;
    if (Q.kr.bits == 8) {
        // Four tokens per wave pass: lanes 16k .. 16k + 15 hold token 4 (pass * W + w) + k,
        // four consecutive elements each (head_post4; the K / V rotation and int8 by
        // rotate_quant4 with block 0's signs: fwht_lane + kv_store_head's int8 branch).
        const uint32_t sl = lane & 15u;
        const uint64_t m0 = __ballot(hadamard_sign_bit(0, lane) != 0u);
        for (int tl0 = 4 * wave; tl0 < TOK; tl0 += 4 * W) {
            if (tokb + tl0 >= A.ntok) break;  // wave-uniform
            const int t = tokb + tl0 + (int)lg;
            const bool live = t < A.ntok;
            const float4 e4 = *reinterpret_cast<const float4 *>(ep + (tl0 + (int)lg) * RP + 4 * sl);
            float v[4] = {e4.x, e4.y, e4.z, e4.w};
            head_post4(head, Q.nq, Q.nkv, Q.bias, Q.qn, Q.kn, Q.eps, Q.rope, pos0 + min(t, A.ntok - 1), sl, v);
            if (head < Q.nq) {
                if (live)
                    *reinterpret_cast<float4 *>(A.out + (size_t)t * A.out_stride + (size_t)head * 64 + 4 * sl) =
                        make_float4(v[0], v[1], v[2], v[3]);
                continue;
            }
            const Chunk4 r = rotate_quant4(v, m0, sl);
            if (live) {
                const bool is_k = head < Q.nq + Q.nkv;
                const int kvh = is_k ? head - Q.nq : head - Q.nq - Q.nkv;
                const size_t slot = ((size_t)Q.layer * Q.nkv + kvh) * Q.kr.cap + ring_slot(Q.kr, pos0 + t);
                *reinterpret_cast<uint32_t *>((is_k ? Q.kq : Q.vq) + slot * 64 + 4 * sl) = r.w;
                if (sl == 0) (is_k ? Q.ks : Q.vs)[slot] = r.scale;
            }
        }
        return;
    }
    for (int tl = wave; tl < TOK; tl += W) {
        const int t = tokb + tl;
        if (t >= A.ntok) break;  // wave-uniform
        float v0 = ep[tl * RP + (int)lane], v1 = 0.0f;
        head_post_vals(head, Q.nq, Q.nkv, 64, Q.bias, Q.qn, Q.kn, Q.eps, Q.rope, pos0 + t, lane, v0, v1);
        if (head < Q.nq) {
            A.out[(size_t)t * A.out_stride + (size_t)head * 64 + lane] = v0;
            continue;
        }
        const bool is_k = head < Q.nq + Q.nkv;
        const int kvh = is_k ? head - Q.nq : head - Q.nq - Q.nkv;
        const size_t slot = ((size_t)Q.layer * Q.nkv + kvh) * Q.kr.cap + ring_slot(Q.kr, pos0 + t);
        kv_store_head(fwht_lane(v0, 0, lane), 0.0f, 1, lane, Q.kr.bits, 64, slot, is_k ? Q.kq : Q.vq,
                      is_k ? Q.ks : Q.vs);
    }
}

// gate_up: swiglu_act_kernel's work on an interleaved block of 128 rows ([gate64(ic), up64(ic)],
// simd_lut.rs:3310-3325) of up to 64 tokens in LDS: per token v = (g / (1 + exp(-g))) * u
// (swiglu_activate_scalar, real_llm.rs:9801-9805), the FWHT of chunk ic and the int8
// quantization (populate_chunk_fwht_raw) of the down input, with its tile-major copy.  The
// same arithmetic in the same order as that kernel, so the outputs are the same.
template <int RP, int W, int TOK>
__device__ __forceinline__ void mf_swiglu_epilogue(const MfArgs &A, const float *ep, int tokb, int wave, uint32_t lane) {
    const int ic = (int)blockIdx.x;
    // Four tokens per wave at a time: lanes 16k .. 16k + 15 hold token tl0 + k, four
    // consecutive elements each (rotate_quant4: the arithmetic of fwht_lane +
    // quant_chunk_store in that layout, so the codes, scales and sums are the same).
    const uint64_t smask = __ballot(hadamard_sign_bit((uint64_t)ic, lane) != 0u);
    const uint32_t sl = lane & 15u;
    for (int tl0 = 4 * wave; tl0 < TOK; tl0 += 4 * W) {
        if (tokb + tl0 >= A.ntok) break;  // wave-uniform
        const int tl = tl0 + (int)(lane >> 4), t = tokb + tl;
        const float4 g4 = *reinterpret_cast<const float4 *>(ep + tl * RP + 4 * sl);
        const float4 u4 = *reinterpret_cast<const float4 *>(ep + tl * RP + 64 + 4 * sl);
        const float gs[4] = {g4.x, g4.y, g4.z, g4.w}, us[4] = {u4.x, u4.y, u4.z, u4.w};
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = (gs[j] / (1.0f + expf(-gs[j]))) * us[j];
        const Chunk4 r = rotate_quant4(v, smask, sl);
        if (t < A.ntok)
            chunk4_store(r, sl, t, ic, A.nci, A.sq, A.ss, A.ssum, A.stiles.xt, A.stiles.st, A.stiles.ut);
    }
}

// Many stripes, up to 32 tokens: a wave per stripe and NB 16-token blocks, which walks the
// stripe's K; bound by the weight stream and the latency of each wave's chain.
// P chunks in flight per wave: a register ring of P stages, unrolled so that each stage
// is a fixed set of registers (no copies, so the compiler's load waits count only the
// stages issued after the one consumed).  Stage i holds chunks i, i + P, i + 2P, ...;
// fetches past the last chunk re-read the last chunk and are never consumed.  Scheduling
// barriers keep each refill right after the step that frees its stage: left to itself,
// the compiler sank every load of a round below the round's last MFMA and a wait for all
// loads, so no load was in flight during compute.
template <int FMT, int HP, int NB, int P, bool QP = false>
__global__ __launch_bounds__(256) void gemm_mfma_kernel(MfArgs A) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: stripe math on SGPRs
    const int stripe = (int)blockIdx.x * 4 + (int)wave;
    if (stripe >= A.stripes) return;
    const bool is_tail = stripe >= 2 * A.np;
    const uint32_t side = is_tail ? 0u : (uint32_t)(stripe & 1);
    const uint8_t *mbase = is_tail ? A.tail : A.pair + (size_t)(stripe >> 1) * A.ptot;
    const uint32_t li = lane & 15u, lg = lane >> 4;
    MfLane L = mf_lane<FMT, HP>(lane, is_tail, side, A.lane);
    L.x_off = lane * 16u;
    L.sx_off = li * 4u;
    const MfSrc R{mf_rsrc(mbase), mf_rsrc(A.xt), mf_rsrc(A.st), mf_rsrc(FMT == 0 ? (const void *)A.ut : A.st)};
    const int tb0 = (int)blockIdx.y * NB;
    float acc[NB][4];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[b][r] = 0.0f;
    const int nc = A.nc, last = nc - 1;
    MfChunk<FMT, NB> ring[P];
#pragma unroll
    for (int i = 0; i < P; i++) mf_fetch<FMT, HP, NB>(A, R, L, is_tail, tb0, min(i, last), ring[i]);
    int c0 = 0;
    for (; c0 + P <= nc; c0 += P) {
#pragma unroll
        for (int i = 0; i < P; i++) {
            mf_step<FMT, HP, NB>(A, ring[i], acc, lane);
            __builtin_amdgcn_sched_barrier(0);
            mf_fetch<FMT, HP, NB>(A, R, L, is_tail, tb0, min(c0 + P + i, last), ring[i]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int i = 0; i < P - 1; i++)
        if (c0 + i < nc) mf_step<FMT, HP, NB>(A, ring[i], acc, lane);
    if constexpr (QP) {
        __shared__ __align__(16) float ep[16 * NB * 68];
#pragma unroll
        for (int b = 0; b < NB; b++)
            *reinterpret_cast<float4 *>(ep + (16 * b + (int)li) * 68 + 16 * (int)wave + 4 * (int)lg) =
                make_float4(acc[b][0], acc[b][1], acc[b][2], acc[b][3]);
        __syncthreads();
        mf_qkv_epilogue<68, 4, 16 * NB>(A, ep, tb0 * 16, (int)wave, lane);
        return;
    }
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int t = (tb0 + b) * 16 + (int)li;
        if (t >= A.ntok) continue;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = stripe * 16 + 4 * (int)lg + r;
            if (row >= A.rows) continue;
            float *o = A.out + (size_t)t * A.out_stride + row;
            *o = A.accum ? *o + acc[b][r] : acc[b][r];
        }
    }
}

// ---------------------------------------------------------------- few waves: K dealt over a workgroup
// One stripe and up to 64 tokens per workgroup of 8 waves.  gemm_mfma_kernel gives a wave its
// stripe's whole K, so a matrix with few stripes leaves SIMDs idle while each wave walks its
// chunks one after the other (NF4 4096 x 14336, 16 tokens: 40.5 us for 30 MB).  Here the waves
// take the chunks of a round of 8 side by side: decode, MFMA and the terms float(dot) * sx go
// to LDS, one barrier a round (two buffers), and the chain f = fmaf(term, scale, f) runs over
// the round's terms in chunk order, each wave owning one (block, row mod 4) part of the
// outputs.  The same operations in the same order, so the outputs equal gemm_mfma_kernel's;
// 16.5 us for that shape.  Bound by the exchange (2 KB of LDS traffic per tile of 16 x 16
// outputs and chunk) and the issue rate of the chain.
// ORD (NF3 with the fast epilogue): the sums in the order of gemv_kernel's fast epilogue, so a batch
// gives each token the bits of the one-token GEMV, as its 4-token passes did, and their error (one
// chain over K has up to three times it).  A wave holds one accumulator of a K segment in
// registers; the exchange is one value per output, accumulator and segment, added pairwise and
// then segment by segment by the outputs' owners.  NF3 5000 x 2112, 200 tokens 128.5 us as 4-token
// passes, 23.1 here (one chain over K in tiles: 18.1); 14336 x 4096, 200 tokens 277 and 74 (46);
// 4096 x 14336, 64 tokens 127 and 25 (30).
constexpr int kKsWaves = 8;

template <int FMT, int NB>
struct KsFrag {
    uint32_t d0, d1, hv;
    uint2 sw;
    v4i x[NB];
    float sx[NB];
    int32_t su[FMT == 0 ? NB : 1];
};

template <int FMT, int HP, int NB, bool ORD = false>
__global__ __launch_bounds__(64 * kKsWaves, 4) void gemm_ks_kernel(MfArgs A) {
    constexpr int W = kKsWaves, P = NB == 4 ? 2 : NB == 2 ? 3 : 4;  // rounds in flight
    constexpr int OWN = NB == 4 ? 2 : 1;              // chains per wave
    __shared__ float tt[2][W][NB][4][64];             // terms [chunk of the round][block][row mod 4][lane]
    __shared__ __align__(16) float wss[2][W][16];     // the chunks' row scales (not ORD)
    const uint32_t lane = threadIdx.x & 63u, li = lane & 15u, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    int stripe = (int)blockIdx.x;
    if ((gridDim.x & 15u) == 0) {  // both stripes of a pair on one XCD, as in gemv_kernel
        const int a = stripe >> 4, s8 = (stripe >> 3) & 1, j = stripe & 7;
        stripe = 2 * (8 * a + j) + s8;
    }
    const bool is_tail = stripe >= 2 * A.np;
    const MfLane L = mf_lane<FMT, HP>(lane, is_tail, is_tail ? 0u : (uint32_t)(stripe & 1), A.lane);
    const __amdgpu_buffer_rsrc_t rw = mf_rsrc(is_tail ? A.tail : A.pair + (size_t)(stripe >> 1) * A.ptot),
                                 rx = mf_rsrc(A.xt), rs = mf_rsrc(A.st), ru = mf_rsrc(FMT == 0 ? (const void *)A.ut : A.st);
    const int tokb = (int)blockIdx.y * 16 * NB;
    uint32_t xo[NB], so[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) {  // (blocks and tokens past the end repeat the last one, not stored)
        if (A.tiled) {
            const uint32_t t = (uint32_t)min((int)blockIdx.y * NB + b, A.nblk - 1) * (uint32_t)A.nc;
            xo[b] = t * 1024u + lane * 16u;
            so[b] = t * 64u + li * 4u;
        } else {
            const uint32_t t = (uint32_t)min(tokb + 16 * b + (int)li, A.ntok - 1);
            xo[b] = t * (uint32_t)A.K + lg * 16u;
            so[b] = t * (uint32_t)A.nc * 4u;
        }
    }
    const uint32_t xstep = A.tiled ? 1024u : 64u, sstep = A.tiled ? 64u : 4u;
    auto fetch = [&](KsFrag<FMT, NB> &f, int c) {
        uint32_t rec, sgb;
        mf_record<FMT, HP>(A.sgc_log2, is_tail, c, rec, sgb);
        f.d0 = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rw, L.a_off, rec, 0);
        f.d1 = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rw, L.b_off, rec, 0);
        if constexpr ((FMT == 0 && HP > 0) || FMT == 2)
            f.hv = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rw, L.h_off, rec, 0);
        const v2u sw = __builtin_amdgcn_raw_buffer_load_b64(rw, L.s_off, sgb, 0);
        f.sw = make_uint2(sw[0], sw[1]);
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const v4u x = __builtin_amdgcn_raw_buffer_load_b128(rx, xo[b], (uint32_t)c * xstep, 0);
            f.x[b] = v4i{(int)x[0], (int)x[1], (int)x[2], (int)x[3]};
            f.sx[b] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, so[b], (uint32_t)c * sstep, 0));
            if constexpr (FMT == 0)
                f.su[b] = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(ru, so[b], (uint32_t)c * sstep, 0);
        }
    };
    // this wave's chains: row 4 lg + r of token li, blocks ob, ob + 2
    const int r_own = wave & 3, ob = wave >> 2;
    float acc[OWN];
#pragma unroll
    for (int k = 0; k < OWN; k++) acc[k] = ORD ? -0.0f : 0.0f;  // (-0 + v is v)
    const int nc = A.nc, last = nc - 1;
    auto round = [&](const KsFrag<FMT, NB> &f, int i) {
        const int buf = i & 1;
        const v4i a = mf_decode<FMT, HP>(f.d0, f.d1, f.hv, A.t0, A.t1, A.u0, A.u1, lane);
        if (li == 0)
            *reinterpret_cast<float4 *>(&wss[buf][wave][4 * lg]) =
                make_float4(bf16_lo(f.sw.x), bf16_hi(f.sw.x), bf16_lo(f.sw.y), bf16_hi(f.sw.y));
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const v4i zero = {0, 0, 0, 0};
            const v4i d = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, f.x[b], zero, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                int dot = d[r];
                if constexpr (FMT == 0) dot = 2 * dot - ((1 << (4 + HP)) - 1) * f.su[b];
                // (NF3: -0 marks a chunk to skip, mf_step's note)
                tt[buf][wave][b][r][lane] = FMT == 2 && f.sx[b] == 0.0f ? -0.0f : (float)dot * f.sx[b];
            }
        }
        __syncthreads();
        if (NB > 1 || ob == 0) {
            const int n = min(W, nc - i * W);  // (a wave past the last chunk repeated it; not added)
#pragma unroll
            for (int h = 0; h < W; h += 4) {
                float ws[4], t[OWN][4];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    ws[k] = wss[buf][h + k][4 * lg + r_own];
#pragma unroll
                    for (int o = 0; o < OWN; o++) t[o][k] = tt[buf][h + k][NB == 1 ? 0 : ob + 2 * o][r_own][lane];
                }
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (h + k < n)
#pragma unroll
                        for (int o = 0; o < OWN; o++)
                            acc[o] = fmaf(t[o][k], FMT == 2 && __float_as_uint(t[o][k]) == 0x80000000u ? 0.0f : ws[k], acc[o]);
            }
        }
    };
    // ORD: this wave's accumulator u of segment h, h + 8 / G, ...; `len` visits per segment
    const int G = ORD ? 1 << A.g_log2 : W, u = wave & (G - 1), h = ORD ? wave >> A.g_log2 : 0;
    const int len = ORD ? (A.cps + G - 1) >> A.g_log2 : 1, seg_step = W / G;
    const int rounds = ORD ? (A.nseg + seg_step - 1) / seg_step * len : (nc + W - 1) / W;
    struct At {  // a round's place: first segment of the step, visit within it, parity of the step
        int seg, v, buf;
    };
    auto next = [&](At &a) {
        if (++a.v < len) return;
        a.v = 0;
        a.seg += seg_step;
        a.buf ^= 1;
    };
    auto chunk_of = [&](const At &a, bool &live) {
        const int off = u + a.v * G, c = (a.seg + h) * A.cps + off;
        live = off < A.cps && c < nc;
        return min(c, last);
    };
    float po[ORD ? NB : 1][4];
    auto round_ord = [&](const KsFrag<FMT, NB> &f, const At &at) {
        bool live;
        (void)chunk_of(at, live);
        if (at.v == 0)
#pragma unroll
            for (int b = 0; b < NB; b++)
#pragma unroll
                for (int r = 0; r < 4; r++) po[ORD ? b : 0][r] = 0.0f;
        if (live) {
            const v4i a = mf_decode<FMT, HP>(f.d0, f.d1, f.hv, A.t0, A.t1, A.u0, A.u1, lane);
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const uint2 sw = f.sx[b] == 0.0f ? make_uint2(0u, 0u) : f.sw;  // (mf_step's note)
                const float ws[4] = {bf16_lo(sw.x), bf16_hi(sw.x), bf16_lo(sw.y), bf16_hi(sw.y)};
                const v4i zero = {0, 0, 0, 0};
                const v4i d = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, f.x[b], zero, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    int dot = d[r];
                    if constexpr (FMT == 0) dot = 2 * dot - ((1 << (4 + HP)) - 1) * f.su[b];
                    float &o = po[ORD ? b : 0][r];
                    o = fmaf((float)dot * f.sx[b], ws[r], o);
                }
            }
        }
        if (at.v != len - 1) return;
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int r = 0; r < 4; r++) tt[at.buf][wave][b][r][lane] = po[ORD ? b : 0][r];
        __syncthreads();
        if (NB > 1 || ob == 0) {
#pragma unroll
            for (int o = 0; o < OWN; o++) {
                float t[W];
#pragma unroll
                for (int k = 0; k < W; k++) t[k] = tt[at.buf][k][NB == 1 ? 0 : ob + 2 * o][r_own][lane];
                const float lo = (t[0] + t[1]) + (t[2] + t[3]), hi = (t[4] + t[5]) + (t[6] + t[7]);
                if (A.g_log2 == 3) {
                    acc[o] += lo + hi;
                } else {
                    acc[o] += lo;
                    if (at.seg + 1 < A.nseg) acc[o] += hi;
                }
            }
        }
    };
    KsFrag<FMT, NB> ring[P];
    At now{0, 0, 0}, ahead{0, 0, 0};
    auto refill = [&](KsFrag<FMT, NB> &f, int i) {  // round i's chunk
        if constexpr (ORD) {
            bool live;
            fetch(f, chunk_of(ahead, live));
            next(ahead);
        } else {
            fetch(f, min(W * i + wave, last));
        }
    };
    auto take = [&](const KsFrag<FMT, NB> &f, int i) {
        if constexpr (ORD) {
            round_ord(f, now);
            next(now);
        } else {
            round(f, i);
        }
    };
#pragma unroll
    for (int k = 0; k < P; k++) refill(ring[k], k);
    int i = 0;
    for (; i + P <= rounds; i += P) {
#pragma unroll
        for (int k = 0; k < P; k++) {
            take(ring[k], i + k);
            __builtin_amdgcn_sched_barrier(0);
            refill(ring[k], i + k + P);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int k = 0; k < P - 1; k++)
        if (i + k < rounds) take(ring[k], i + k);
    // through LDS, so that a token's 16 rows are stored together
    __syncthreads();
    float *ot = &tt[0][0][0][0][0];  // [16 NB tokens][17]
    if (NB > 1 || ob == 0)
#pragma unroll
        for (int o = 0; o < OWN; o++)
            ot[(16 * (NB == 1 ? 0 : ob + 2 * o) + (int)li) * 17 + 4 * lg + r_own] = acc[o];
    __syncthreads();
    for (int k = (int)threadIdx.x; k < 16 * NB * 16; k += 64 * W) {
        const int t = tokb + k / 16, row = stripe * 16 + k % 16;
        if (t >= A.ntok || row >= A.rows) continue;
        const float v = ot[(k / 16) * 17 + k % 16];
        float *o = A.out + (size_t)t * A.out_stride + row;
        *o = A.accum ? *o + v : v;
    }
}

// ---------------------------------------------------------------- tile kernel
// NP stripe pairs x 64 tokens per workgroup of 4 waves, 4 chunks per stage:
//  - wave w loads and decodes chunk 4 i + w of the NP pairs into LDS (A operands and row
//    scales as floats; two buffers, one barrier per stage), so a decode serves 4 token blocks
//    whatever the number of waves the launch has;
//  - wave w then runs the stage's 4 chunks over all 2 NP stripes for its own token block w
//    (TB: its TB blocks) whose activation it loads straight in B order, while stage i + 1 is
//    decoded into the other buffer.
// Per output tile (16 x 16, one chunk) that is 12 instructions of epilogue (convert, multiply,
// fma per output, the reference's chain) and 6 / TB of decode next to an MFMA of 16 cycles
// that the other instructions do not overlap: the issue rate bounds the kernel (NF4 14336 x
// 4096, 512 tokens: 81 us for 1.8 M tiles, 94 us when a wave decoded for its own blocks).
// Weights and activations of the next D stages are in flight in registers.
// MODE 0 stores the outputs; 1 (gate_up, NP 4: one interleaved block of 128 rows) has
// swiglu_act_kernel's work as its epilogue; 2 (qkv at head size 64, NP 2: one head of 64 rows)
// qkv_post_kernel's.
template <int FMT, int HP, int NP, int TB, int D, int MODE>
__global__ __launch_bounds__(256, NP* TB >= 4 ? 1 : 2) void gemm_tile_kernel(MfArgs A) {
    constexpr int W = 4, NS = 2 * NP, TOK = 16 * W * TB;
    constexpr uint32_t CB = FMT == 2 ? 384u : 512u;  // bytes per stripe-chunk
    extern __shared__ __align__(16) unsigned char tile_lds[];
    int4(*al)[W][NS][64] = reinterpret_cast<int4(*)[W][NS][64]>(tile_lds);                          // [2] decoded A
    float(*wl)[W][NS][16] = reinterpret_cast<float(*)[W][NS][16]>(tile_lds + 2 * W * NS * 1024);  // [2] row scales
    const uint32_t lane = threadIdx.x & 63u, li = lane & 15u, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int npt = (A.stripes + 1) >> 1, p0 = (int)blockIdx.x * NP;  // pairs, the odd last stripe among them
    bool tail[NP];
    __amdgpu_buffer_rsrc_t rw[NP];
#pragma unroll
    for (int k = 0; k < NP; k++) {  // (pairs past the last repeat it, not stored)
        const int pk = min(p0 + k, npt - 1);
        tail[k] = pk >= A.np;
        rw[k] = mf_rsrc(tail[k] ? A.tail : A.pair + (size_t)pk * A.ptot);
    }
    const __amdgpu_buffer_rsrc_t rx = mf_rsrc(A.xt), rs = mf_rsrc(A.st), ru = mf_rsrc(FMT == 0 ? (const void *)A.ut : A.st);
    const MfLane L = mf_lane<FMT, HP>(lane, true, 0u, A.lane);  // offsets from the stripe's codes, hi bytes, scales
    const uint32_t ah = FMT == 0 ? L.h_off - 512u : L.h_off, as = 8u * lg;
    struct Wt {
        uint32_t d0[NS], d1[NS], hv[NS];
        uint2 sw[NS];
    };
    struct Bt {
        v4i x[TB];
        float sx[TB];
        int32_t su[TB];
    };
    const int nc = A.nc, last = nc - 1;
    auto fetch_w = [&](Wt &f, int stage) {
        const int c = min(W * stage + wave, last);
#pragma unroll
        for (int k = 0; k < NP; k++) {
            uint32_t rec, sgb;
            mf_record<FMT, HP>(A.sgc_log2, tail[k], c, rec, sgb);
#pragma unroll
            for (int s = 0; s < 2; s++) {  // (side 1 of the tail stripe repeats side 0, not stored)
                const uint32_t sd = tail[k] ? 0u : (uint32_t)s;
                const uint32_t code = rec + sd * CB;
                uint32_t sc = sgb + sd * 32u;
                if constexpr (FMT == 0) sc = rec + (tail[k] ? 512u + 128u * HP : 1024u + 256u * HP + sd * 32u);
                f.d0[2 * k + s] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rw[k], L.a_off, code, 0);
                f.d1[2 * k + s] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rw[k], L.b_off, code, 0);
                if constexpr (FMT == 2)
                    f.hv[2 * k + s] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rw[k], ah, code, 0);
                if constexpr (FMT == 0 && HP > 0)
                    f.hv[2 * k + s] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(
                        rw[k], ah, rec + (tail[k] ? 512u : 1024u + sd * 128u * HP), 0);
                const v2u sw = __builtin_amdgcn_raw_buffer_load_b64(rw[k], as, sc, 0);
                f.sw[2 * k + s] = make_uint2(sw[0], sw[1]);
            }
        }
    };
    const int tb = ((int)blockIdx.y * W + wave) * TB, tokb = (int)blockIdx.y * TOK;
    uint32_t t0[TB];
#pragma unroll
    for (int b = 0; b < TB; b++) t0[b] = (uint32_t)min(tb + b, A.nblk - 1) * (uint32_t)nc;
    auto fetch_b = [&](Bt &f, int c) {
#pragma unroll
        for (int b = 0; b < TB; b++) {
            const uint32_t t = t0[b] + (uint32_t)min(c, last);
            const v4u x = __builtin_amdgcn_raw_buffer_load_b128(rx, lane * 16u, t * 1024u, 0);
            f.x[b] = v4i{(int)x[0], (int)x[1], (int)x[2], (int)x[3]};
            f.sx[b] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, li * 4u, t * 64u, 0));
            if constexpr (FMT == 0) f.su[b] = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(ru, li * 4u, t * 64u, 0);
        }
    };
    float acc[NS][TB][4];
#pragma unroll
    for (int s = 0; s < NS; s++)
#pragma unroll
        for (int b = 0; b < TB; b++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[s][b][r] = 0.0f;
    const int stages = (nc + W - 1) / W;
    auto decode = [&](const Wt &f, int buf) {
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const v4i a = mf_decode<FMT, HP>(f.d0[s], f.d1[s], f.hv[s], A.t0, A.t1, A.u0, A.u1, lane);
            al[buf][wave][s][lane] = make_int4(a[0], a[1], a[2], a[3]);
            // (every lane of a group of 16 writes the same 16 bytes)
            *reinterpret_cast<float4 *>(&wl[buf][wave][s][4 * lg]) =
                make_float4(bf16_lo(f.sw[s].x), bf16_hi(f.sw[s].x), bf16_lo(f.sw[s].y), bf16_hi(f.sw[s].y));
        }
    };
    struct Ld {
        int4 a[2];
        float4 w[2];
    };
    auto read = [&](Ld &f, int buf, int g) {  // group g: chunk g / NP, pair g % NP
#pragma unroll
        for (int s = 0; s < 2; s++) {
            f.a[s] = al[buf][g / NP][2 * (g % NP) + s][lane];
            f.w[s] = *reinterpret_cast<const float4 *>(&wl[buf][g / NP][2 * (g % NP) + s][4 * lg]);
        }
    };
    auto mul = [&](const Ld &f, const Bt &x, int k) {
        v4i d[2][TB];
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int b = 0; b < TB; b++) {
                const v4i zero = {0, 0, 0, 0};
                d[s][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(v4i{f.a[s].x, f.a[s].y, f.a[s].z, f.a[s].w}, x.x[b], zero, 0, 0, 0);
            }
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const float wv[4] = {f.w[s].x, f.w[s].y, f.w[s].z, f.w[s].w};
#pragma unroll
            for (int b = 0; b < TB; b++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    int dot = d[s][b][r];
                    if constexpr (FMT == 0) dot = 2 * dot - ((1 << (4 + HP)) - 1) * x.su[b];
                    const float w = FMT == 2 && x.sx[b] == 0.0f ? 0.0f : wv[r];
                    acc[2 * k + s][b][r] = fmaf((float)dot * x.sx[b], w, acc[2 * k + s][b][r]);
                }
        }
    };
    auto run = [&](auto active) {  // active: this wave has a token block (the others only decode)
        constexpr bool kActive = decltype(active)::value;
        Wt wr[D];
        Bt br[D][W];
        // Stage i's products while the next stage is decoded into the other buffer.
        auto step = [&](Wt &wf, Bt(&bf)[W], int i, int live) {
            const int buf = i & 1;
            Ld ld[2];
            if constexpr (kActive) read(ld[0], buf, 0);
            __builtin_amdgcn_sched_barrier(0);
            decode(wf, buf ^ 1);
            fetch_w(wf, i + 1 + D);
            if constexpr (kActive) {
#pragma unroll
                for (int g = 0; g < W * NP; g++) {
                    const int q = g / NP;
                    if (q >= live) break;
                    if (g + 1 < W * NP) read(ld[(g + 1) & 1], buf, g + 1);
                    __builtin_amdgcn_sched_barrier(0);
                    mul(ld[g & 1], bf[q], g % NP);
                    __builtin_amdgcn_sched_barrier(0);
                    if (g % NP == NP - 1) fetch_b(bf[q], W * (i + D) + q);
                }
            }
            __syncthreads();
        };
        fetch_w(wr[0], 0);
#pragma unroll
        for (int d = 0; d < D; d++) {
            if (d > 0) fetch_w(wr[d], d);
            if constexpr (kActive)
#pragma unroll
                for (int q = 0; q < W; q++) fetch_b(br[d][q], W * d + q);
        }
        decode(wr[0], 0);
        fetch_w(wr[0], D);
        __syncthreads();
        const int full = nc / W;
        int i = 0;
        for (; i + D <= full; i += D)
#pragma unroll
            for (int d = 0; d < D; d++) step(wr[(d + 1) % D], br[d], i + d, W);
#pragma unroll
        for (int d = 0; d < D; d++)
            if (i + d < stages) step(wr[(d + 1) % D], br[d], i + d, nc - W * (i + d));
    };
    if (tb < A.nblk) run(std::true_type{});
    else run(std::false_type{});
    if constexpr (MODE != 0) {
        // the epilogues work on [token][row] in LDS
        constexpr int RP = 32 * NP + 4;
        float *ep = reinterpret_cast<float *>(tile_lds);
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int b = 0; b < TB; b++)
                *reinterpret_cast<float4 *>(ep + (16 * (TB * wave + b) + (int)li) * RP + 16 * s + 4 * (int)lg) =
                    make_float4(acc[s][b][0], acc[s][b][1], acc[s][b][2], acc[s][b][3]);
        __syncthreads();
        if constexpr (MODE == 1) mf_swiglu_epilogue<RP, W, TOK>(A, ep, tokb, wave, lane);
        else mf_qkv_epilogue<RP, W, TOK>(A, ep, tokb, wave, lane);
        return;
    }
#pragma unroll
    for (int b = 0; b < TB; b++) {
        const int t = (tb + b) * 16 + (int)li;
        if (t >= A.ntok) return;
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const int stripe = 2 * p0 + s, row0 = 16 * stripe + 4 * (int)lg;
            if (stripe >= A.stripes) break;
            float *o = A.out + (size_t)t * A.out_stride + row0;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                if (row0 + r >= A.rows) break;
                o[r] = A.accum ? o[r] + acc[s][b][r] : acc[s][b][r];
            }
        }
    }
}

// Tile-major copy of the activations: one 16-token x 64-column tile per 1 KB, in the
// order the MFMA's B operand is read (lane l = 16g + t holds token t's columns 16g ..
// 16g + 15), so each B load of a wave is 1 KB contiguous, with the chunk scales (and
// code sums, for bit planes) in 16-token groups.  Tokens past ntok repeat the last token.
// One thread per 16 bytes; blockIdx.y is the 16-token block.
__global__ __launch_bounds__(256) void mf_tile_kernel(const int8_t *xq, const float *xs, const int32_t *xsum, int K,
                                                      int nc, int ntok, int8_t *xt, float *st, int32_t *ut) {
    const int c = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6), tb = (int)blockIdx.y;
    if (c >= nc) return;
    const uint32_t lane = threadIdx.x & 63u, li = lane & 15u, lg = lane >> 4;
    const int tok = min(tb * 16 + (int)li, ntok - 1);
    const size_t tile = (size_t)tb * nc + c;
    *reinterpret_cast<int4 *>(xt + tile * 1024 + lane * 16) =
        *reinterpret_cast<const int4 *>(xq + (size_t)tok * K + (size_t)c * 64 + 16 * lg);
    if (lg == 0) st[tile * 16 + li] = xs[(size_t)tok * nc + c];
    if (lg == 1 && ut) ut[tile * 16 + li] = xsum[(size_t)tok * nc + c];
}

// ---------------------------------------------------------------- 2 .. 15 tokens, fast epilogue
// The GEMV's own work split (plan_gemv: a workgroup per stripe pair, or per stripe where
// pairs are fewer than CUs; its waves are K segments) with the chunk dots of up to 16 tokens
// from one MFMA per stripe-chunk.  The 4-token passes it replaces decode every weight once
// per 4 tokens and spend two v_dot4 per four codes and token; here the decode and the MFMA
// cost the same for 2 tokens as for 16, so what bounds it is the weight stream and, past
// about 8 tokens, the gather of the activation rows (16 lines per load).  Weights from the
// Infinity Cache, NF4 14336 x 4096, 4 / 8 / 15 tokens: 12.6 / 21.1 / 40.3 us as 4-token passes,
// 8.4 / 10.6 / 12.7 us here (one token 8.7); b6 4096 x 14336, 8 / 15 tokens: 27.7 / 54.8 us, 18.2 /
// 23.8 us here; from HBM, 4 / 8 tokens of the first 13.0 / 21.8 us and 10.1 / 12.1 us.
// gemv_four_token_passes says where the passes stay.
// Sums: the order of gemv_kernel's fast epilogue, so a batch gives each token the bits of
// the one-token GEMV.  A wave's chunks are dealt round-robin to G accumulators (the GEMV's
// lane groups: 4 in pair mode, 8 in stripe mode), which are added pairwise as the lane
// butterfly does, then the waves' sums in wave order.  (A chunk with scale 0 adds +-0.)
// Any number of tokens in groups of up to 16, a weight pass each.
// XL, groups of up to 4 tokens and K segments of up to 16 chunks: a wave first copies its segment's
// activation into LDS (4 KB, loads ahead of its first weights), so its ring holds weights alone and
// all G chunks are in flight where the planes' registers otherwise allow four, and a chunk's
// activation is one LDS read instead of three gathers.  b6 4096 x 14336, 4 tokens: 16.4 -> 11.3 us
// from HBM (4-token passes 15.5), 14.3 -> 10.6 us from the Infinity Cache (15.1).
struct GvArgs {
    const uint8_t *pair, *tail;
    size_t ptot;
    int rows, K, nc, np, sgc_log2, s0, s1, rb_lo, nseg, cps, ntok, accum;
    int tg;  // tokens per workgroup (blockIdx.y counts token groups)
    uint32_t t0, t1, u0, u1;
    int lane;
    const int8_t *xq;
    const float *xs;
    const int32_t *xsum;
    float *out;
    size_t out_stride;
    // Grouped form (sparse-MoE experts): blockIdx.y counts work items, each up to 16 (token,
    // slot) pairs of one expert; the matrix and its codebook are at the expert's record, pair
    // p reads activation row p / row_div and writes out + p * out_stride (gu_split: a [gate;
    // up] matrix's rows in [gate64, up64] blocks).
    GvGroup grp;
};

template <int FMT, int RS>
struct GvFrag {
    uint32_t d0[RS], d1[RS], hv[RS];
    uint2 sw[RS];
    v4i x;
    float sx;
    int32_t su;
};

constexpr int kXlTokens = 4, kXlChunks = 16;
constexpr int kXlBytes = kXlChunks * kXlTokens * (64 + 4 + 4);  // a wave's codes, scales, code sums

template <int FMT, int HP, bool SM, bool GRP = false, bool XL = false>
__global__ __launch_bounds__(1024) void gemv_mfma_kernel(GvArgs A) {
    constexpr int RS = SM ? 1 : 2, G = SM ? 8 : 4, RB = 16 * RS;
    constexpr int P = SM && FMT == 0 && HP > 0 && !XL ? 4 : G;  // chunks in flight (128 VGPRs at 16 waves)
    extern __shared__ __align__(16) float part[];  // [nseg][16 tokens][RB rows + 1], XL: then [nseg][kXlBytes]
    const uint32_t lane = threadIdx.x & 63u, li = lane & 15u, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    int rbi = (int)blockIdx.x;
    if (SM && (gridDim.x & 15u) == 0) {  // both stripes of a pair on one XCD, as in gemv_kernel
        const int a = rbi >> 4, s8 = (rbi >> 3) & 1, j = rbi & 7;
        rbi = 2 * (8 * a + j) + s8;
    }
    const int rb = A.rb_lo + rbi;  // pair index, or stripe index in stripe mode
    const bool is_tail = SM ? rb >= 2 * A.np : rb >= A.np;
    const int pidx = SM ? rb >> 1 : rb;
    const uint8_t *mbase = is_tail ? A.tail : A.pair + (size_t)pidx * A.ptot;
    int4 item = make_int4(0, 0, 0, 0);  // expert, first entry of the pair list, pairs
    if constexpr (GRP) {
        if ((int)blockIdx.y >= A.grp.n_items[0]) return;  // uniform: the grid covers the most items possible
        item = A.grp.items[blockIdx.y];
        const uint8_t *rec = A.grp.bank + (size_t)item.x * A.grp.bank_stride;
        mbase = rec + A.grp.mat_off + (size_t)pidx * A.ptot;
        const uint4 cb = *reinterpret_cast<const uint4 *>(rec + A.grp.cb_off);
        if constexpr (FMT == 1) nf4_xor_tables(cb.x, cb.y, cb.z, cb.w, A.t0, A.t1, A.u0, A.u1);
        else A.t0 = cb.x, A.t1 = cb.y;
    }
    MfLane L[RS];
#pragma unroll
    for (int s = 0; s < RS; s++)  // (pair mode on the tail stripe: side 1 repeats it, not stored)
        L[s] = mf_lane<FMT, HP>(lane, is_tail, is_tail ? 0u : SM ? (uint32_t)(rb & 1) : (uint32_t)s, A.lane);
    const int tok0 = GRP ? 0 : (int)blockIdx.y * A.tg, nt = GRP ? item.z : min(A.tg, A.ntok - tok0);
    uint32_t tok = min(li, (uint32_t)nt - 1u);  // columns past nt repeat the last token, not stored
    if constexpr (GRP) tok = (uint32_t)A.grp.list[item.y + (int)tok] / (uint32_t)A.grp.row_div;
    // (offsets count from the workgroup's first token, so they stay small for any batch)
    const size_t row0 = GRP ? 0 : (size_t)tok0;
    const uint32_t x_off = tok * (uint32_t)A.K + lg * 16u, sx_off = tok * (uint32_t)A.nc * 4u;
    const float *xs0 = A.xs + row0 * A.nc;
    const __amdgpu_buffer_rsrc_t rw = mf_rsrc(mbase), rx = mf_rsrc(A.xq + row0 * A.K), rs = mf_rsrc(xs0),
                                 ru = mf_rsrc(FMT == 0 ? (const void *)(A.xsum + row0 * A.nc) : xs0);
    const int cw0 = wave * A.cps, cw1 = min(A.nc, cw0 + A.cps), n = cw1 - cw0;
    auto fetch = [&](GvFrag<FMT, RS> &f, int c) {
        uint32_t rec, sgb;
        mf_record<FMT, HP>(A.sgc_log2, is_tail, c, rec, sgb);
#pragma unroll
        for (int s = 0; s < RS; s++) {
            f.d0[s] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rw, L[s].a_off, rec, 0);
            f.d1[s] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rw, L[s].b_off, rec, 0);
            if constexpr ((FMT == 0 && HP > 0) || FMT == 2)
                f.hv[s] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rw, L[s].h_off, rec, 0);
            const v2u sw = __builtin_amdgcn_raw_buffer_load_b64(rw, L[s].s_off, sgb, 0);
            f.sw[s] = make_uint2(sw[0], sw[1]);
        }
        if constexpr (!XL) {
            const v4u x = __builtin_amdgcn_raw_buffer_load_b128(rx, x_off, (uint32_t)c * 64u, 0);
            f.x = v4i{(int)x[0], (int)x[1], (int)x[2], (int)x[3]};
            f.sx = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, sx_off, (uint32_t)c * 4u, 0));
            if constexpr (FMT == 0) f.su = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(ru, sx_off, (uint32_t)c * 4u, 0);
        }
    };
    // XL: this wave's [chunk][token][64 codes], [chunk][token] scales and sums (chunks past the
    // segment and tokens past nt repeat the last ones)
    unsigned char *xl = nullptr;
    v4u xr[XL ? kXlChunks / 4 : 1];
    float sr = 0.0f;
    int32_t ur = 0;
    if constexpr (XL) {
        static_assert(kXlTokens == 4 && kXlChunks == 16, "the lane layout of the copies");
        xl = reinterpret_cast<unsigned char *>(part) + ((size_t)A.nseg * 16 * (RB + 1) * 4) + (size_t)wave * kXlBytes;
#pragma unroll
        for (int g = 0; g < kXlChunks / 4; g++) {
            const uint32_t c = (uint32_t)min(cw0 + 4 * g + (int)lg, cw1 - 1), t = (uint32_t)min((int)(li >> 2), nt - 1);
            xr[g] = __builtin_amdgcn_raw_buffer_load_b128(rx, t * (uint32_t)A.K + c * 64u + (li & 3u) * 16u, 0, 0);
        }
        const uint32_t c = (uint32_t)min(cw0 + (int)(lane >> 2), cw1 - 1), t = (uint32_t)min((int)(lane & 3u), nt - 1);
        const uint32_t at = (t * (uint32_t)A.nc + c) * 4u;
        sr = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, at, 0, 0));
        if constexpr (FMT == 0) ur = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(ru, at, 0, 0);
    }
    float acc[G][RS][4];
#pragma unroll
    for (int g = 0; g < G; g++)
#pragma unroll
        for (int s = 0; s < RS; s++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[g][s][r] = 0.0f;
    auto compute = [&](const GvFrag<FMT, RS> &w, int i, float (&o)[RS][4]) {  // i: chunk of the segment
        GvFrag<FMT, RS> f = w;
        if constexpr (XL) {
            const uint32_t t = li & 3u;
            f.x = *reinterpret_cast<const v4i *>(xl + i * 256 + t * 64u + lg * 16u);
            f.sx = *reinterpret_cast<const float *>(xl + kXlChunks * 256 + i * 16 + t * 4u);
            if constexpr (FMT == 0) f.su = *reinterpret_cast<const int32_t *>(xl + kXlChunks * 272 + i * 16 + t * 4u);
        }
#pragma unroll
        for (int s = 0; s < RS; s++) {
            const v4i a = mf_decode<FMT, HP>(f.d0[s], f.d1[s], f.hv[s], A.t0, A.t1, A.u0, A.u1, lane);
            const v4i zero = {0, 0, 0, 0};
            const v4i d = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, f.x, zero, 0, 0, 0);
            const uint2 sw = f.sx == 0.0f ? make_uint2(0u, 0u) : f.sw[s];  // (mf_step's note)
            const float ws[4] = {bf16_lo(sw.x), bf16_hi(sw.x), bf16_lo(sw.y), bf16_hi(sw.y)};
#pragma unroll
            for (int r = 0; r < 4; r++) {
                int dot = d[r];
                if constexpr (FMT == 0) dot = 2 * dot - ((1 << (4 + HP)) - 1) * f.su;
                o[s][r] = fmaf((float)dot * f.sx, ws[r], o[s][r]);
            }
        }
    };
    // One round = the G accumulators' next chunks; a chunk's registers take the load P chunks
    // on as soon as it is computed.  The last round issues only what it will use itself.
    GvFrag<FMT, RS> ring[P];
#pragma unroll
    for (int u = 0; u < P; u++) fetch(ring[u], min(cw0 + u, cw1 - 1));
    if constexpr (XL) {
        __builtin_amdgcn_sched_barrier(0);  // (the copies' loads and the first weights are under way)
#pragma unroll
        for (int g = 0; g < kXlChunks / 4; g++) *reinterpret_cast<v4i *>(xl + g * 1024 + lane * 16u) = v4i{(int)xr[g][0], (int)xr[g][1], (int)xr[g][2], (int)xr[g][3]};
        *reinterpret_cast<float *>(xl + kXlChunks * 256 + lane * 4u) = sr;
        if constexpr (FMT == 0) *reinterpret_cast<int32_t *>(xl + kXlChunks * 272 + lane * 4u) = ur;
    }
    int i0 = 0;
    for (; i0 + G < n; i0 += G) {
#pragma unroll
        for (int u = 0; u < G; u++) {
            compute(ring[u % P], i0 + u, acc[u]);
            __builtin_amdgcn_sched_barrier(0);
            fetch(ring[u % P], min(cw0 + i0 + P + u, cw1 - 1));
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int u = 0; u < G; u++) {
        if (i0 + u < n) compute(ring[u % P], i0 + u, acc[u]);
        if (u + P < G) fetch(ring[u % P], min(cw0 + i0 + P + u, cw1 - 1));
    }
    // the accumulators pairwise (neighbours, then pairs, ...), then into LDS
    constexpr int RP = RB + 1;
#pragma unroll
    for (int s = 0; s < RS; s++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            float v[G];
#pragma unroll
            for (int g = 0; g < G; g++) v[g] = acc[g][s][r];
#pragma unroll
            for (int w = G; w > 1; w >>= 1)
#pragma unroll
                for (int g = 0; g < w / 2; g++) v[g] = v[2 * g] + v[2 * g + 1];
            part[((size_t)wave * 16 + li) * RP + 16 * s + 4 * lg + r] = v[0];
        }
    __syncthreads();
    const int first = SM ? rb : is_tail ? 2 * A.np : 2 * rb;
    const int live = (!SM && is_tail) ? 16 : RB;
    for (int idx = (int)threadIdx.x; idx < nt * RB; idx += (int)blockDim.x) {
        const int t = idx / RB, rl = idx % RB, st = first + rl / 16, row = st * 16 + rl % 16;
        if (rl >= live || row >= A.rows || st < A.s0 || st >= A.s1) continue;
        float v = part[(size_t)t * RP + rl];
        for (int w = 1; w < A.nseg; w++) v += part[((size_t)w * 16 + t) * RP + rl];
        if constexpr (GRP) {
            int r = row;  // gate / up rows in blocks of 64
            if (A.grp.gu_split) {
                const int inter = A.rows >> 1, up = row >= inter ? 1 : 0, rr = row - up * inter;
                r = (rr >> 6) * 128 + up * 64 + (rr & 63);
            }
            A.out[(size_t)A.grp.list[item.y + t] * A.out_stride + r] = v;
            continue;
        }
        float *o = A.out + (size_t)(tok0 + t) * A.out_stride + row;
        *o = A.accum ? *o + v : v;
    }
}

// The grouped form where an expert's matrix is split by stripes and a wave's K segment is at most
// 8 chunks (one per accumulator of the GEMV's order: most experts): a workgroup takes one item
// and R stripes after each other, its activation in registers for all of them.  With a
// workgroup per stripe the gather of the activation rows and scales (16 lines a load) kept
// the address units busy 73% of the time; the weights alone are 3 or 2 loads per chunk.
// (Two thirds of a wave's time is still waiting for them.)
template <int FMT>
__global__ __launch_bounds__(1024) void gemv_mfma_items_kernel(GvArgs A, int R) {
    constexpr int G = 8;
    constexpr uint32_t CB = FMT == 2 ? 384u : 512u;  // bytes per stripe-chunk
    extern __shared__ float part[];                  // [2][nseg][16 tokens][17]
    const uint32_t lane = threadIdx.x & 63u, li = lane & 15u, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if ((int)blockIdx.y >= A.grp.n_items[0]) return;  // uniform: the grid covers the most items possible
    const int4 item = A.grp.items[blockIdx.y];        // expert, first entry of the pair list, pairs
    const uint8_t *rec0 = A.grp.bank + (size_t)item.x * A.grp.bank_stride;
    const MfLane L = mf_lane<FMT, 0>(lane, false, 0u, A.lane);
    const __amdgpu_buffer_rsrc_t rw = mf_rsrc(rec0 + A.grp.mat_off), rx = mf_rsrc(A.xq), rs = mf_rsrc(A.xs);
    const int cw0 = wave * A.cps, cw1 = min(A.nc, cw0 + A.cps), n = cw1 - cw0;
    struct Wt {
        uint32_t d0, d1, hv;
        uint2 sw;
    };
    const int s_first = (int)blockIdx.x * R, s_last = min(s_first + R, 2 * A.np) - 1;
    auto fetch = [&](Wt &f, int stripe, int u) {
        const int c = min(cw0 + u, cw1 - 1);
        uint32_t rec, sgb;
        mf_record<FMT, 0>(A.sgc_log2, false, c, rec, sgb);
        const uint32_t base = (uint32_t)(stripe >> 1) * (uint32_t)A.ptot, side = (uint32_t)(stripe & 1);
        const uint32_t code = base + rec + side * CB;
        f.d0 = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rw, L.a_off, code, 0);
        f.d1 = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rw, L.b_off, code, 0);
        if constexpr (FMT == 2) f.hv = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rw, L.h_off, code, 0);
        const v2u sw = __builtin_amdgcn_raw_buffer_load_b64(rw, L.s_off, base + sgb + side * 32u, 0);
        f.sw = make_uint2(sw[0], sw[1]);
    };
    Wt wt[G];
    v4i x[G];
    float sx[G];
#pragma unroll
    for (int u = 0; u < G; u++)
        if (u < n) fetch(wt[u], s_first, u);
    __builtin_amdgcn_sched_barrier(0);
    const int nt = item.z;
    const uint32_t pr = (uint32_t)A.grp.list[item.y + (int)min(li, (uint32_t)nt - 1u)], tok = pr / (uint32_t)A.grp.row_div;
    // (kept in LDS: a global load in the stripes' loop would wait for the weights in flight)
    __shared__ uint32_t pairs[16];
    if (threadIdx.x < 16) pairs[threadIdx.x] = pr;
    const uint32_t x_off = tok * (uint32_t)A.K + lg * 16u, sx_off = tok * (uint32_t)A.nc * 4u;
#pragma unroll
    for (int u = 0; u < G; u++) {
        if (u >= n) break;  // (uniform)
        const uint32_t c = (uint32_t)(cw0 + u);
        const v4u xv = __builtin_amdgcn_raw_buffer_load_b128(rx, x_off, c * 64u, 0);
        x[u] = v4i{(int)xv[0], (int)xv[1], (int)xv[2], (int)xv[3]};
        sx[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, sx_off, c * 4u, 0));
    }
    const uint4 cb = *reinterpret_cast<const uint4 *>(rec0 + A.grp.cb_off);
    if constexpr (FMT == 1) nf4_xor_tables(cb.x, cb.y, cb.z, cb.w, A.t0, A.t1, A.u0, A.u1);
    else A.t0 = cb.x, A.t1 = cb.y;
    for (int stripe = s_first; stripe <= s_last; stripe++) {
        float acc[G][4];
#pragma unroll
        for (int u = 0; u < G; u++) {
#pragma unroll
            for (int r = 0; r < 4; r++) acc[u][r] = 0.0f;
            if (u < n) {
                const v4i a = mf_decode<FMT, 0>(wt[u].d0, wt[u].d1, wt[u].hv, A.t0, A.t1, A.u0, A.u1, lane);
                const v4i zero = {0, 0, 0, 0};
                const v4i d = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, x[u], zero, 0, 0, 0);
                const uint2 sw = sx[u] == 0.0f ? make_uint2(0u, 0u) : wt[u].sw;  // (mf_step's note)
                const float ws[4] = {bf16_lo(sw.x), bf16_hi(sw.x), bf16_lo(sw.y), bf16_hi(sw.y)};
#pragma unroll
                for (int r = 0; r < 4; r++) acc[u][r] = fmaf((float)d[r] * sx[u], ws[r], 0.0f);
                __builtin_amdgcn_sched_barrier(0);
                fetch(wt[u], min(stripe + 1, s_last), u);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        float *pt = part + (size_t)(stripe & 1) * A.nseg * 16 * 17;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            float v[G];
#pragma unroll
            for (int g = 0; g < G; g++) v[g] = acc[g][r];
#pragma unroll
            for (int w = G; w > 1; w >>= 1)
#pragma unroll
                for (int g = 0; g < w / 2; g++) v[g] = v[2 * g] + v[2 * g + 1];
            pt[((size_t)wave * 16 + li) * 17 + 4 * lg + r] = v[0];
        }
        __syncthreads();
        for (int idx = (int)threadIdx.x; idx < nt * 16; idx += (int)blockDim.x) {
            const int t = idx >> 4, row = stripe * 16 + (idx & 15);
            float v = pt[(size_t)t * 17 + (idx & 15)];
            for (int w = 1; w < A.nseg; w++) v += pt[((size_t)w * 16 + t) * 17 + (idx & 15)];
            int r = row;  // gate / up rows in blocks of 64
            if (A.grp.gu_split) {
                const int inter = A.rows >> 1, up = row >= inter ? 1 : 0, rr = row - up * inter;
                r = (rr >> 6) * 128 + up * 64 + (rr & 63);
            }
            A.out[(size_t)pairs[t] * A.out_stride + r] = v;
        }
    }
}

}  // namespace

// Lookup words of an NF matrix: NF4's XOR tables, NF3's codebook (bit planes: none).
static void mf_tables(const k2t_mat *m, uint32_t &t0, uint32_t &t1, uint32_t &u0, uint32_t &u1) {
    if (m->fmt != K2T_FMT_NF) return;
    if (m->bits == 3) {
        t0 = m->cb[0];
        t1 = m->cb[1];
    } else {
        nf4_xor_tables(m->cb[0], m->cb[1], m->cb[2], m->cb[3], t0, t1, u0, u1);
    }
}

bool gemm_mfma_supported(const k2t_mat *m, int ntok) {
    if (ntok < kMfmaMinTokens || m->cols % 64 != 0) return false;
    // (the tiles are read at 32-bit offsets inside 2 GiB)
    if ((long)((ntok + 15) / 16) * m->nc * 1024 > 0x7FFFFFFFl) return false;
    if (m->fmt == K2T_FMT_NF) return (m->bits == 3 || m->bits == 4) && (m->sgc & (m->sgc - 1)) == 0;
    return m->fmt == K2T_FMT_NIBBLE4 && m->hp >= 0 && m->hp <= 2;
}

bool gemv_mfma_supported(const k2t_mat *m, int ntok) {
    return ntok >= 2 && ntok < kMfmaMinTokens && gemm_mfma_supported(m, kMfmaMinTokens);
}

// Where the 4-token passes stay the better form: their 16-byte loads stream weights better than this
// kernel's dwords, and what they pay is decode and dots per token.  NF3 with 2 or 3 tokens (weights
// from HBM, us in passes and here: 4096 x 14336 8.9 and 9.9, 9.7 and 10.0; 2048 x 8192 5.8 and 6.9, 6.5 and
// 6.9; 4 tokens 10.7 and 10.0, 7.2 and 6.9: not taken), and up to 4 tokens over K segments too long for
// the activation in LDS (b6 4096 x 14336 without it, 2 / 4 tokens 12.3 and 15.8, 15.5 and 16.4).
bool gemv_four_token_passes(const k2t_mat *m, const GemvPlan &plan, int ntok) {
    return (m->fmt == K2T_FMT_NF && m->bits == 3 && ntok <= 3) || (ntok <= 4 && plan.cps > kXlChunks);
}

template <int FMT, int HP>
static void launch_gemv_mfma_fmt(hipStream_t st, const GemvPlan &plan, dim3 grid, size_t lds, const GvArgs &A) {
    const dim3 block(64 * plan.nseg);
    // Activation in LDS for groups of up to four tokens, but over the shortest rows, which have little
    // to keep in flight (NF4 960 x 576, 4 tokens 3.4 us without and 3.7, 2048 x 2048 4.0 and 3.9; b5 3.4
    // and 3.4, 1536 x 1536 3.7 and 3.6).
    if (A.tg <= kXlTokens && plan.cps <= kXlChunks && A.nc > (FMT == 0 ? 16 : 24)) {
        const size_t l = lds + (size_t)plan.nseg * kXlBytes;
        if (plan.stripe_mode) hipLaunchKernelGGL((gemv_mfma_kernel<FMT, HP, true, false, true>), grid, block, l, st, A);
        else hipLaunchKernelGGL((gemv_mfma_kernel<FMT, HP, false, false, true>), grid, block, l, st, A);
        return;
    }
    if (plan.stripe_mode) hipLaunchKernelGGL((gemv_mfma_kernel<FMT, HP, true>), grid, block, lds, st, A);
    else hipLaunchKernelGGL((gemv_mfma_kernel<FMT, HP, false>), grid, block, lds, st, A);
}

// The arguments every launch over matrix m with this plan shares.
static GvArgs gemv_mfma_args(const k2t_mat *m, const GemvPlan &plan, const int8_t *xq, const float *xs,
                             const int32_t *xsum, float *out, size_t out_stride) {
    const bool planes = m->fmt == K2T_FMT_NIBBLE4;
    GvArgs A{};
    A.pair = m->pair;
    A.tail = m->tail;
    A.ptot = m->pairs ? m->pair_len / m->pairs : 0;
    A.rows = m->rows;
    A.K = m->cols;
    A.nc = m->nc;
    A.np = m->pairs;
    A.sgc_log2 = planes ? 0 : __builtin_ctz((unsigned)m->sgc);
    A.s1 = m->stripes;
    A.rb_lo = plan.rb_lo;
    A.nseg = plan.nseg;
    A.cps = plan.cps;
    A.lane = m->nf3_lane;
    mf_tables(m, A.t0, A.t1, A.u0, A.u1);
    A.xq = xq;
    A.xs = xs;
    A.xsum = xsum;
    A.out = out;
    A.out_stride = out_stride;
    return A;
}

static size_t gemv_mfma_lds(const GemvPlan &plan) {
    return (size_t)plan.nseg * 16 * ((plan.stripe_mode ? 16 : 32) + 1) * sizeof(float);
}

bool gemv_mfma_grouped_supported(const k2t_mat *geom) {
    return geom->fmt == K2T_FMT_NF && !geom->has_tail && gemm_mfma_supported(geom, kMfmaMinTokens);
}

void launch_gemv_mfma_grouped(k2t_ctx *ctx, const k2t_mat *geom, const GvGroup &g, int max_items, const int8_t *xq,
                              const float *xs, float *out, size_t out_stride) {
    if (!gemv_mfma_grouped_supported(geom) || max_items < 1 || max_items > 65535)
        throw Error(K2T_E_INTERNAL, "grouped mfma gemv: shape");
    const GemvPlan plan = plan_gemv(ctx, geom, 0, geom->stripes);
    GvArgs A = gemv_mfma_args(geom, plan, xq, xs, nullptr, out, out_stride);
    A.grp = g;
    const dim3 block(64 * plan.nseg);
    hipStream_t st = ctx->stream;
    // Items that are half full or more (the rows to gather are what the loop over stripes saves)
    // and two waves per SIMD with that: per layer, 300 tokens with 8 of 128 experts 396 -> 347 us
    // NF3; 96 tokens 212 -> 210 NF3, 208 -> 212 NF4; 32 tokens 147 -> 154.
    constexpr int R = 4;  // 2 / 8 stripes: 367 / 359 us
    const int groups = (geom->stripes + R - 1) / R;
    if (plan.stripe_mode && plan.cps <= 8 && g.pairs >= 8 * g.experts && (long)groups * max_items * plan.nseg >= 2048) {
        const dim3 grid(groups, max_items);
        const size_t lds = (size_t)2 * plan.nseg * 16 * 17 * sizeof(float);
        if (geom->bits == 3) hipLaunchKernelGGL((gemv_mfma_items_kernel<2>), grid, block, lds, st, A, R);
        else hipLaunchKernelGGL((gemv_mfma_items_kernel<1>), grid, block, lds, st, A, R);
        hip_check(hipGetLastError(), "grouped mfma gemv launch");
        return;
    }
    const dim3 grid(plan.rb_hi - plan.rb_lo, max_items);
    const size_t lds = gemv_mfma_lds(plan);
    if (geom->bits == 3 && plan.stripe_mode) hipLaunchKernelGGL((gemv_mfma_kernel<2, 0, true, true>), grid, block, lds, st, A);
    else if (geom->bits == 3) hipLaunchKernelGGL((gemv_mfma_kernel<2, 0, false, true>), grid, block, lds, st, A);
    else if (plan.stripe_mode) hipLaunchKernelGGL((gemv_mfma_kernel<1, 0, true, true>), grid, block, lds, st, A);
    else hipLaunchKernelGGL((gemv_mfma_kernel<1, 0, false, true>), grid, block, lds, st, A);
    hip_check(hipGetLastError(), "grouped mfma gemv launch");
}

void launch_gemv_mfma(k2t_ctx *ctx, const k2t_mat *m, const GemvPlan &plan, const int8_t *xq, const float *xs,
                      const int32_t *xsum, int ntok, int s0, int s1, float *out, size_t out_stride, bool accum) {
    GvArgs A = gemv_mfma_args(m, plan, xq, xs, xsum, out, out_stride);
    A.s0 = s0;
    A.s1 = s1;
    A.ntok = ntok;
    A.accum = accum ? 1 : 0;
    // A matrix with few row blocks leaves CUs idle: the tokens are then dealt to several
    // workgroups (four or more tokens each), which shortens each one's activation gather.
    // NF4 2048 x 8192, 8 / 15 tokens: 8.8 / 11.0 us in one group, 7.6 / 9.0 us.
    const int wgs = plan.rb_hi - plan.rb_lo;
    const int groups = std::max((ntok + 15) / 16, std::min(ctx->num_cus / wgs, (ntok + 3) / 4));
    A.tg = (ntok + groups - 1) / groups;
    const dim3 grid(wgs, (ntok + A.tg - 1) / A.tg);
    const size_t lds = gemv_mfma_lds(plan);
    hipStream_t st = ctx->stream;
    if (m->fmt == K2T_FMT_NF && m->bits == 3) launch_gemv_mfma_fmt<2, 0>(st, plan, grid, lds, A);
    else if (m->fmt == K2T_FMT_NF) launch_gemv_mfma_fmt<1, 0>(st, plan, grid, lds, A);
    else if (m->hp == 0) launch_gemv_mfma_fmt<0, 0>(st, plan, grid, lds, A);
    else if (m->hp == 1) launch_gemv_mfma_fmt<0, 1>(st, plan, grid, lds, A);
    else launch_gemv_mfma_fmt<0, 2>(st, plan, grid, lds, A);
    hip_check(hipGetLastError(), "mfma gemv launch");
}

// Where gemm_ks_kernel is considered for `blocks` 16-token blocks: few stripes, and no more (stripe,
// block) pairs than keep its exchange through LDS cheaper than a long chain per wave.  NF4
// 4096 x 14336 (256 stripes), 16 / 64 / 128 / 256 tokens: 16.5 / 28.9 / 41.5 / 76 us there,
// 40.5 / 46 / 47 / 58 us on the others; 2048 x 2048, 128: 8.6 and 10.8.  The bit planes' chains
// also subtract the code sums: b6 4096 x 14336, 64 / 128 tokens 33 / 63 us there, 40 / 49 us.
static bool ks_range(const k2t_mat *m, int blocks) {
    return m->stripes < 512 && (long)m->stripes * blocks <= (m->fmt == K2T_FMT_NIBBLE4 ? 1024 : 2048);
}

// And its workgroups (of four blocks from the third on, the last group padded) are one round: two per
// CU for NF, one for the bit planes.  A second round of a few workgroups costs as much as the
// first: NF4 5000 x 2112, 96 tokens (626 workgroups) 15.7 us there, 12.4 on a wave per stripe and
// block; b4, 48 tokens (313) 11.7 and 9.5.
static bool ks_fits(const k2t_ctx *ctx, const k2t_mat *m, int blocks) {
    return ks_range(m, blocks) &&
           (blocks <= 2 || m->stripes * ((blocks + 3) / 4) <= ctx->num_cus * (m->fmt == K2T_FMT_NIBBLE4 ? 1 : 2));
}

// Whether gemm_ks_kernel then reads a plain activation as its rows lie, rather than a tile-major
// copy made first: worth the copy's launch (2.5 us) only for short rows and few stripes (each
// gathers them again).  960 x 576, 16 tokens 7.3 -> 4.2 us, NF4 128 tokens 7.4 -> 6.6; NF4
// 2048 x 2048, 16 tokens 7.1 -> 6.0; not taken: 32 tokens of it 7.2 -> 8.1, 6144 x 2048, 16 tokens
// 7.6 -> 10.2, b6 960 x 576, 64 tokens 7.4 -> 8.0.
static bool ks_rows(const k2t_ctx *ctx, const k2t_mat *m, int blocks) {
    return ks_fits(ctx, m, blocks) && (long)m->stripes * m->nc * blocks <= 6000 &&
           m->nc * (blocks < 4 ? blocks : 4) <= (m->fmt == K2T_FMT_NIBBLE4 ? 20 : 40);
}

// The kernel of `blocks` blocks: gemm_ks_kernel unless its rounds of eight chunks are mostly padding
// (nine chunks: b4 3072 x 576, 64 tokens 7.0 us there, 6.3 on a wave per stripe and block; NF4 512
// tokens 8.6 and 7.7, but 64 tokens 6.8 and 6.6: from 900 pairs on); then a wave per stripe and
// block where those are at most 8 per CU and 64-token tiles would be more than one per CU (b4 5000 x
// 4096, 96 tokens, 314 tiles: 21.8 us and 19.2; 8192 x 4096, 64 tokens, 256 tiles: 17.5 and 18.1,
// not taken); else tiles.
enum class PlainForm { kKs, kWave, kTile };
static PlainForm plain_form(const k2t_ctx *ctx, const k2t_mat *m, int blocks) {
    const long pairs = (long)m->stripes * blocks;
    const bool full = (m->nc + 7) / 8 * 16 <= 3 * m->nc || (m->fmt == K2T_FMT_NF && pairs < 900);
    if (ks_fits(ctx, m, blocks) && (full || ks_rows(ctx, m, blocks))) return PlainForm::kKs;
    const int tiles = (m->stripes + 1) / 2 * ((blocks + 3) / 4);
    if (blocks <= 2 || (pairs <= 8 * ctx->num_cus && (ks_range(m, blocks) || tiles > ctx->num_cus))) return PlainForm::kWave;
    return PlainForm::kTile;
}

static bool stream_captured(k2t_ctx *ctx) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(ctx->stream, &cap) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return cap != hipStreamCaptureStatusNone;
}

bool gemm_mfma_nf3_passes(k2t_ctx *ctx, const k2t_mat *m, int ntok) {
    if (ntok <= 128 && (long)m->stripes * m->nc * ((ntok + 3) / 4) <= 36000) return true;
    return !ks_rows(ctx, m, (ntok + 15) / 16) && stream_captured(ctx);
}

// Arguments of one launch over all of m's stripes, and the tile-major activation (the
// producer's, else copied here into the context's scratch: 1 KB + 64 B of scales + 64 B
// of code sums per tile).
static void mfma_args(k2t_ctx *ctx, const k2t_mat *m, const int8_t *xq, const float *xs, const int32_t *xsum,
                     int ntok, ActTiles tiles, bool rows, MfArgs &A) {
    const bool planes = m->fmt == K2T_FMT_NIBBLE4;
    A = MfArgs{};
    A.pair = m->pair;
    A.tail = m->tail;
    A.ptot = m->pairs ? m->pair_len / m->pairs : 0;
    A.rows = m->rows;
    A.nc = m->nc;
    A.np = m->pairs;
    A.stripes = m->stripes;
    A.sgc_log2 = planes ? 0 : __builtin_ctz((unsigned)m->sgc);
    A.lane = m->nf3_lane;
    mf_tables(m, A.t0, A.t1, A.u0, A.u1);
    const int blocks = (ntok + 15) / 16;
    int8_t *xt = tiles.xt;
    float *stile = tiles.st;
    int32_t *utile = tiles.ut;
    A.tiled = 1;
    if ((!xt || (planes && !utile)) && rows) {
        xt = const_cast<int8_t *>(xq);
        stile = const_cast<float *>(xs);
        utile = const_cast<int32_t *>(xsum);
        A.tiled = 0;
    } else if (!xt || (planes && !utile)) {
        const size_t ntile = (size_t)blocks * m->nc;
        ensure_scratch(ctx, ntile * (1024 + 64 + 64) / sizeof(float));
        xt = reinterpret_cast<int8_t *>(ctx->scratch);
        stile = ctx->scratch + ntile * 256;
        utile = reinterpret_cast<int32_t *>(ctx->scratch + ntile * 272);
        hipLaunchKernelGGL(mf_tile_kernel, dim3((m->nc + 3) / 4, blocks), dim3(256), 0, ctx->stream, xq, xs, xsum,
                           m->cols, m->nc, ntok, xt, stile, planes ? utile : nullptr);
    }
    A.xt = xt;
    A.nblk = blocks;
    A.st = stile;
    A.ut = utile;
    A.K = m->cols;
    A.ntok = ntok;
}

template <int FMT, int HP, int NP, int TB, int D, int MODE>
static void launch_tile(hipStream_t st, const MfArgs &A) {
    const dim3 grid(((A.stripes + 1) / 2 + NP - 1) / NP, (A.nblk + 4 * TB - 1) / (4 * TB));
    const size_t lds = (size_t)2 * 4 * 2 * NP * (1024 + 64);
    hipLaunchKernelGGL((gemm_tile_kernel<FMT, HP, NP, TB, D, MODE>), grid, dim3(256), lds, st, A);
}

// f<FMT, HP>(...) for matrix m's format (NF4 or bit planes).
#define MF_FORMATS(m, f, ...)                             \
    do {                                                  \
        if ((m)->fmt == K2T_FMT_NF) f<1, 0>(__VA_ARGS__); \
        else if ((m)->hp == 0) f<0, 0>(__VA_ARGS__);      \
        else if ((m)->hp == 1) f<0, 1>(__VA_ARGS__);      \
        else f<0, 2>(__VA_ARGS__);                        \
    } while (0)

static bool is_nf3(const k2t_mat *m) { return m->fmt == K2T_FMT_NF && m->bits == 3; }

template <int FMT, int HP, bool ORD = false>
static void launch_ks(hipStream_t st, const MfArgs &A) {
    const dim3 blk(64 * kKsWaves);
    const int B = A.nblk, nb = B <= 1 ? 1 : B == 2 ? 2 : 4;
    const dim3 grid(A.stripes, (B + nb - 1) / nb);
    if (nb == 1) hipLaunchKernelGGL((gemm_ks_kernel<FMT, HP, 1, ORD>), grid, blk, 0, st, A);
    else if (nb == 2) hipLaunchKernelGGL((gemm_ks_kernel<FMT, HP, 2, ORD>), grid, blk, 0, st, A);
    else hipLaunchKernelGGL((gemm_ks_kernel<FMT, HP, 4, ORD>), grid, blk, 0, st, A);
}

template <int FMT, int HP>
static void launch_plain_fmt(hipStream_t st, PlainForm form, const MfArgs &A) {
    const int S = A.stripes, B = A.nblk;
    // Up to 32 tokens (and plain_form's cases): a wave per stripe (NF4 14336 x 4096, 16 tokens 16 us,
    // 18.6 in 64-token tiles).  Above, tiles of 32 rows x 64 tokens, or x 128 once those give 448
    // workgroups: NF4 14336 x 4096, 64 / 128 / 512 tokens 22 / 38 / 105 us in 64-token tiles,
    // 25 / 30 / 81 in 128-token ones (a wave per stripe and block, or 16 rows x 64 tokens per
    // wave: 31 / 41 / 94); 2048 x 8192, 512 tokens (256 workgroups of 128) 38 and 42.5.
    if (form == PlainForm::kKs) {
        launch_ks<FMT, HP>(st, A);
    } else if (form == PlainForm::kWave) {
        // two blocks per wave only where that leaves 8 waves per CU
        const int nb = B == 2 && S >= 2048 ? 2 : 1;
        const dim3 grid((S + 3) / 4, (B + nb - 1) / nb);
        if (nb == 1) hipLaunchKernelGGL((gemm_mfma_kernel<FMT, HP, 1, kMfmaDepth>), grid, dim3(256), 0, st, A);
        else hipLaunchKernelGGL((gemm_mfma_kernel<FMT, HP, 2, kMfmaDepth>), grid, dim3(256), 0, st, A);
    } else if (B >= 8 && (long)((S + 1) / 2) * ((B + 7) / 8) >= 448) {
        launch_tile<FMT, HP, 1, 2, 1, 0>(st, A);
    } else {
        launch_tile<FMT, HP, 1, 1, 3, 0>(st, A);
    }
}

template <int FMT, int HP>
static void launch_swiglu_fmt(hipStream_t st, const MfArgs &A) {
    if ((long)A.nci * ((A.nblk + 7) / 8) >= 384) launch_tile<FMT, HP, 4, 2, 1, 1>(st, A);
    else launch_tile<FMT, HP, 4, 1, 1, 1>(st, A);
}

template <int FMT, int HP>
static void launch_qkv_fmt(hipStream_t st, const MfArgs &A) {
    // A head and 16 tokens per workgroup while those are few: 48 heads, K 2048, 128 tokens (384
    // workgroups) 3.5 us a layer less than 64-token tiles, 512 tokens 14 us more.  The NF4 cache's
    // epilogue takes its tokens one by one, so tiles hold 16 of them in a row on each wave: 96
    // heads, 100 / 256 tokens 22.6 and 14.6 us a layer more than here, 400 tokens 3 more, 512 tokens 4 less.
    const dim3 grid(A.stripes / 4, A.nblk);
    if (grid.x * grid.y <= (A.qp.kr.bits == 8 ? 512u : 2560u)) hipLaunchKernelGGL((gemm_mfma_kernel<FMT, HP, 1, kMfmaDepth, true>), grid, dim3(256), 0, st, A);
    else launch_tile<FMT, HP, 2, 1, 2, 2>(st, A);
}

void launch_gemm_mfma(k2t_ctx *ctx, const k2t_mat *m, const int8_t *xq, const float *xs, const int32_t *xsum,
                      int ntok, float *out, size_t out_stride, bool accum, ActTiles tiles) {
    if (!gemm_mfma_supported(m, ntok)) throw Error(K2T_E_INTERNAL, "mfma gemm: unsupported matrix");
    MfArgs A;
    mfma_args(ctx, m, xq, xs, xsum, ntok, tiles, ks_rows(ctx, m, (ntok + 15) / 16), A);
    A.out = out;
    A.out_stride = out_stride;
    A.accum = accum ? 1 : 0;
    const PlainForm form = plain_form(ctx, m, A.nblk);
    if (is_nf3(m)) launch_plain_fmt<2, 0>(ctx->stream, form, A);
    else MF_FORMATS(m, launch_plain_fmt, ctx->stream, form, A);
    hip_check(hipGetLastError(), "mfma gemm launch");
}

// Whether `blocks` 16-token blocks of an ordered batch run on gemv_mfma_kernel, 16 tokens per weight
// pass, instead of gemm_ks_kernel: small products, whose copy into tiles costs more than it saves
// (NF3 5000 x 2112, 32 / 64 tokens 8.1 / 12.7 us there, 9.6 / 11.6 on gemm_ks_kernel; 2048 x 8192,
// 32 / 64 tokens 11.6 / 22.0 and 15.0 / 20.3); one block over many stripes (14336 x 4096, 13.4 and
// 16.3; 4096 x 14336, 18.2 and 16.1: not taken); rows of a round or two, which leave a K segment's
// exchange nothing to pay for it (8200 x 576, 512 tokens 26 and 43).
static bool ordered_gemv(const k2t_mat *m, int blocks) {
    return (long)m->stripes * m->nc * blocks <= 36000 || (blocks == 1 && m->stripes >= 512) || m->nc <= 12;
}

void launch_gemm_ordered(k2t_ctx *ctx, const k2t_mat *m, const GemvPlan &plan, const int8_t *xq, const float *xs,
                         int ntok, float *out, size_t out_stride, bool accum, ActTiles tiles) {
    if (!gemm_mfma_supported(m, ntok) || !is_nf3(m)) throw Error(K2T_E_INTERNAL, "ordered mfma gemm: unsupported matrix");
    // (a captured graph holds no scratch: gemm_mfma_nf3_passes' note; the bits are the same)
    if (ordered_gemv(m, (ntok + 15) / 16) || (!tiles.xt && stream_captured(ctx))) {
        launch_gemv_mfma(ctx, m, plan, xq, xs, nullptr, ntok, 0, m->stripes, out, out_stride, accum);
        return;
    }
    MfArgs A;
    mfma_args(ctx, m, xq, xs, nullptr, ntok, tiles, false, A);
    A.out = out;
    A.out_stride = out_stride;
    A.accum = accum ? 1 : 0;
    A.nseg = plan.nseg;
    A.cps = plan.cps;
    A.g_log2 = plan.stripe_mode ? 3 : 2;
    launch_ks<2, 0, true>(ctx->stream, A);
    hip_check(hipGetLastError(), "mfma gemm launch");
}

bool launch_gemm_mfma_qkv(k2t_ctx *ctx, const k2t_mat *qkv, ActTiles tiles, int ntok, float *out, size_t out_stride,
                          const QkvPostDev &qp) {
    if (!gemm_mfma_supported(qkv, ntok) || is_nf3(qkv) || !tiles.xt || qkv->rows % 64 != 0) return false;
    if (qkv->fmt == K2T_FMT_NIBBLE4 && !tiles.ut) return false;
    MfArgs A;
    mfma_args(ctx, qkv, nullptr, nullptr, nullptr, ntok, tiles, false, A);
    A.out = out;
    A.out_stride = out_stride;
    A.qp = qp;
    MF_FORMATS(qkv, launch_qkv_fmt, ctx->stream, A);
    hip_check(hipGetLastError(), "mfma qkv launch");
    return true;
}

bool launch_gemm_mfma_swiglu(k2t_ctx *ctx, const k2t_mat *gu, ActTiles tiles, int ntok, int8_t *q, float *s,
                             int32_t *sums, ActTiles out_tiles) {
    if (!gemm_mfma_supported(gu, ntok) || is_nf3(gu) || !tiles.xt || !out_tiles.xt || gu->rows % 128 != 0) return false;
    if (gu->fmt == K2T_FMT_NIBBLE4 && !tiles.ut) return false;
    // 512 or more workgroups of 128 rows x 64 tokens; with fewer the plain launch and the
    // activation's own spread better: 16384 x 2048 NF4, two layers, 512 / 256 tokens 403 / 282 us
    // apart and 375 / 275 fused; 128 / 64 tokens (256 / 128 workgroups) 219 / 202 and 228 / 222.
    if ((long)(gu->rows / 128) * ((ntok + 63) / 64) < 512) return false;
    MfArgs A;
    mfma_args(ctx, gu, nullptr, nullptr, nullptr, ntok, tiles, false, A);
    A.sq = q;
    A.ss = s;
    A.ssum = sums;
    A.stiles = out_tiles;
    A.nci = gu->rows / 128;
    MF_FORMATS(gu, launch_swiglu_fmt, ctx->stream, A);
    hip_check(hipGetLastError(), "mfma gate_up + swiglu launch");
    return true;
}

}  // namespace k2t
