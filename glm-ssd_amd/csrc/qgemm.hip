// gfx950 quantized GEMM for token batches (gs_gemm, gs_gemm_ex; Q8_0, Q4_K, Q5_K, Q6_K, IQ2_XXS,
// IQ3_XXS, rows of whole 256-element super-blocks):
//
//   Y[n][r] (+)= sum_k f16(deq(W[r][k])) * f16(X[n][k])     f32 accumulation
//
// on v_mfma_f32_16x16x32_f16, with the reference GEMM's operands (crates/cuda/kernels/
// gemm.cu:57-78): dequantized weights and activations rounded to f16. Workgroups of 8 waves in RG
// row groups x KG groups along K: wave (rg, kg) owns 16 NR weight rows and 16 NT tokens and takes
// 1/KG of every K step; the KG partial tiles are added through LDS at the end. So one workgroup
// decodes each of its weights once for up to 128 tokens, every decoded fragment feeds NT MFMAs,
// and every activation fragment read from LDS feeds NR.
//
// K runs in half super-blocks (128 elements): lane quarter q of a wave owns 32-element unit 4h + q
// of half h, MFMA g (0..3) takes elements 8g .. 8g+7 of the four quarters' units (the same
// permutation on both operands). Activations are staged per step as f16 in LDS, token rows of 256
// bytes per half, 16-byte chunk c of token t at c ^ (t & 15): 16 lanes reading one chunk column
// hit distinct banks. Weights are staged raw, RC super-blocks at a time (one slot of P bytes, an
// odd multiple of 16, per row and super-block, so 16 rows start in distinct banks), loaded a whole
// chunk of steps ahead of their use.
//
// Decode: a fragment's 8 values leave the packed bytes as f16 denormals (value q as the bits q,
// i.e. q * 2^-24, two per dword after one mask), one v_fma_mix_f32 per weight takes q * 2^-24 through
// (scale * 2^24) and the minimum in f32, and v_cvt_pk_f16_f32 rounds pairs: the reference's f32
// expression (its product is exact in f32 for every format here, so the fma rounds once where
// lib.rs's subtraction does), then the f16 rounding. About 7.5 issue cycles a weight for Q4_K
// against 9 through byte-to-float conversions.
//
// What bounds it: on gfx950 vector instructions hide behind an MFMA for only about a quarter of its 16
// cycles (a measured loop of 16x16x32 MFMAs and v_and: up to 2 per MFMA free, each further one adds its
// whole cost), so decode and matrix work add up, and the activations' LDS traffic with them. Hence
// many tokens per decoded weight (NT), the decode placed between MFMAs in program order, the B side of a
// step prepared during the step before, and loads straight to LDS (XH) spread over the MFMAs. A pass
// of 12288 x 4096 x 2048 tokens: 263 us (784 TFLOP/s); without MFMAs 205, without decode 217, without
// loads 220. Measured against the paths it replaced (Q4_K): 12288 x 4096 x 77 tokens 44 -> 24 us, x 256
// 65 -> 48, x 512 76 -> 64; 4096 x 12288 x 256 70 -> 48. host.cpp qg_pick has the rule.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "kargs.h"
#include "formats.h"
#include "lds_load.h"

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f8 __attribute__((ext_vector_type(8)));

#define QG_TH 512
#define QG_WV 8

// Sticky expiry flag of this code object's bounded LDS waits (host.cpp gs_wait_status).
__device__ uint32_t gs_wait_expired;

// fma(v, D, C) of an f16 denormal of a dword (hi: the upper one), in f32: one v_fma_mix_f32. The f16
// rounding follows in pairs (v_cvt_pk_f16_f32): 6 issue cycles a weight, where v_fma_mixlo/hi_f16,
// which round by themselves, take 8 each (half-register writes).
__device__ __forceinline__ float mix(uint32_t w, int hi, float D, float C) {
    const h2v p = __builtin_bit_cast(h2v, w);
    float r = __builtin_fmaf((float)(hi ? p[1] : p[0]), D, C);
    asm("" : "+v"(r));   // keeps the conversion apart
    return r;
}
__device__ __forceinline__ h8 to_h8(float a, float b, float c, float d, float e, float f, float g, float h) {
    return __builtin_convertvector((f8{a, b, c, d, e, f, g, h}), h8);
}
// eight weights from the dwords e0, o0 (elements 0,2 / 1,3) and e1, o1 (4,6 / 5,7)
__device__ __forceinline__ h8 mix8(uint32_t e0, uint32_t o0, uint32_t e1, uint32_t o1, float D, float C) {
    return to_h8(mix(e0, 0, D, C), mix(o0, 0, D, C), mix(e0, 1, D, C), mix(o0, 1, D, C),
                 mix(e1, 0, D, C), mix(o1, 0, D, C), mix(e1, 1, D, C), mix(o1, 1, D, C));
}
__device__ __forceinline__ uint32_t lw32(const uint8_t *p) { return *(const uint32_t *)p; }
__device__ __forceinline__ uint2 lw64(const uint8_t *p) { return *(const uint2 *)p; }

#define QG_2P24 16777216.0f
// 8 bytes at LDS offset p + sh (p dword-aligned, sh 0 or 2): three dwords shifted into place
struct W3 { uint32_t a, b, c; };
__device__ __forceinline__ W3 lw3(const uint8_t *p) { return W3{lw32(p), lw32(p + 4), lw32(p + 8)}; }
__device__ __forceinline__ uint2 sh8(const W3 &w, uint32_t sh) {
    return make_uint2(__builtin_amdgcn_alignbyte(w.b, w.a, sh), __builtin_amdgcn_alignbyte(w.c, w.b, sh));
}

// ---- formats: SB bytes per super-block in memory, P its LDS slot (an odd multiple of 16). A slot
// ---- holds the block from the dword boundary at or below its first byte; `lead` (0 or 2) is the
// ---- block's first byte in it, 0 for formats with LEAD = false (whole-dword blocks, aligned rows).
// ---- hdr(): the reads of unit u's scales; prep(): once per unit; fetch() + frag(): the 8 weights of
// ---- group g (0..3) of the unit
struct QgQ4K {   // lib.rs:204-218 with scale_min_k4 (lib.rs:87-93)
    static constexpr int TY = GS_Q4_K, SB = 144, P = 144, TAB = 0;
    static constexpr bool LEAD = false;
    using Hdr = uint4;
    struct Prep { const uint8_t *q; float D, C; uint32_t m; };
    __device__ static __forceinline__ void tables(uint8_t *, int) {}
    __device__ static __forceinline__ Hdr hdr(const uint8_t *s, uint32_t, int) { return *(const uint4 *)s; }
    __device__ static __forceinline__ void scales(const uint4 &h, int u, float &d, float &m) {
        const uint32_t sh = 8u * ((uint32_t)u & 3u);
        const uint32_t b1 = (h.y >> sh) & 0xffu, b2 = (h.z >> sh) & 0xffu, b3 = (h.w >> sh) & 0xffu;
        const uint32_t sc = u < 4 ? (b1 & 63u) : ((b3 & 0xfu) | ((b1 >> 6) << 4));
        const uint32_t mn = u < 4 ? (b2 & 63u) : ((b3 >> 4) | ((b2 >> 6) << 4));
        d = h2f(h.x & 0xffffu) * (float)sc;
        m = h2f(h.x >> 16) * (float)mn;
    }
    __device__ static __forceinline__ Prep prep(const Hdr &h, const uint8_t *s, uint32_t, int u) {
        float d, m;
        scales(h, u, d, m);
        // odd units are the high nibbles: 16 q under the mask, the 16 folded into the scale
        return Prep{s + 16 + 32 * (u >> 1), d * ((u & 1) ? QG_2P24 / 16 : QG_2P24), -m, (u & 1) ? 0x00f000f0u : 0x000f000fu};
    }
    using Raw = uint2;
    __device__ static __forceinline__ Raw fetch(const Prep &p, const uint8_t *, int g) { return lw64(p.q + 8 * g); }
    __device__ static __forceinline__ h8 frag(const Raw &w, const Prep &p, int) {
        return mix8(w.x & p.m, (w.x >> 8) & p.m, w.y & p.m, (w.y >> 8) & p.m, p.D, p.C);
    }
};
struct QgQ5K {   // lib.rs:221-240: Q4_K's nibbles and scales, bit u of qh[l] as the fifth bit
    static constexpr int TY = GS_Q5_K, SB = 176, P = 176, TAB = 0;
    static constexpr bool LEAD = false;
    using Hdr = uint4;
    struct Prep { const uint8_t *q, *h; float D, C; uint32_t m, u, s; };
    __device__ static __forceinline__ void tables(uint8_t *, int) {}
    __device__ static __forceinline__ Hdr hdr(const uint8_t *s, uint32_t, int) { return *(const uint4 *)s; }
    __device__ static __forceinline__ Prep prep(const Hdr &h, const uint8_t *s, uint32_t, int u) {
        float d, m;
        QgQ4K::scales(h, u, d, m);
        return Prep{s + 48 + 32 * (u >> 1), s + 16, d * ((u & 1) ? QG_2P24 / 16 : QG_2P24), -m,
                    (u & 1) ? 0x00f000f0u : 0x000f000fu, (uint32_t)u, (u & 1) ? 8u : 4u};
    }
    struct Raw { uint2 w, b; };
    __device__ static __forceinline__ Raw fetch(const Prep &p, const uint8_t *, int g) { return Raw{lw64(p.q + 8 * g), lw64(p.h + 8 * g)}; }
    __device__ static __forceinline__ h8 frag(const Raw &r, const Prep &p, int) {
        const uint2 w = r.w;
        const uint32_t b0 = r.b.x >> p.u, b1 = r.b.y >> p.u;
        return mix8((w.x & p.m) | ((b0 & 0x00010001u) << p.s), ((w.x >> 8) & p.m) | (((b0 >> 8) & 0x00010001u) << p.s),
                    (w.y & p.m) | ((b1 & 0x00010001u) << p.s), ((w.y >> 8) & p.m) | (((b1 >> 8) & 0x00010001u) << p.s),
                    p.D, p.C);
    }
};
struct QgQ6K {   // lib.rs:243-262; (q - 32) d sc: the product is exact in f32, so is the fma
    static constexpr int TY = GS_Q6_K, SB = 210, P = 240, TAB = 0;
    static constexpr bool LEAD = true;
    struct Hdr { uint32_t d, sc; };
    struct Prep { const uint8_t *l, *h; float D0, C0, D1, C1; uint32_t m, u, s, sh; };
    __device__ static __forceinline__ void tables(uint8_t *, int) {}
    __device__ static __forceinline__ Hdr hdr(const uint8_t *s, uint32_t lead, int u) {
        return Hdr{*(const uint16_t *)(s + lead + 208), *(const uint16_t *)(s + lead + 192 + 8 * (u >> 2) + 2 * (u & 3))};
    }
    __device__ static __forceinline__ Prep prep(const Hdr &h, const uint8_t *s, uint32_t lead, int u) {
        const int n = u >> 2, k = u & 3;   // quarter k of half n; scales of its two 16-element halves
        const float d = h2f(h.d);
        const float d0 = d * (float)(int)(int8_t)(h.sc & 0xffu), d1 = d * (float)(int)(int8_t)(h.sc >> 8);
        const float e = k >= 2 ? QG_2P24 / 16 : QG_2P24;   // high nibbles: 16 q under the mask
        return Prep{s + 64 * n + 32 * (k & 1), s + 128 + 32 * n, d0 * e, -32.f * d0, d1 * e, -32.f * d1,
                    k >= 2 ? 0x00f000f0u : 0x000f000fu, 2u * (uint32_t)k, k >= 2 ? 8u : 4u, lead};
    }
    struct Raw { W3 w, b; };
    __device__ static __forceinline__ Raw fetch(const Prep &p, const uint8_t *, int g) { return Raw{lw3(p.l + 8 * g), lw3(p.h + 8 * g)}; }
    __device__ static __forceinline__ h8 frag(const Raw &r, const Prep &p, int g) {
        const uint2 w = sh8(r.w, p.sh), b = sh8(r.b, p.sh);
        const uint32_t b0 = b.x >> p.u, b1 = b.y >> p.u;
        const float D = g < 2 ? p.D0 : p.D1, C = g < 2 ? p.C0 : p.C1;
        return mix8((w.x & p.m) | ((b0 & 0x00030003u) << p.s), ((w.x >> 8) & p.m) | (((b0 >> 8) & 0x00030003u) << p.s),
                    (w.y & p.m) | ((b1 & 0x00030003u) << p.s), ((w.y >> 8) & p.m) | (((b1 >> 8) & 0x00030003u) << p.s), D, C);
    }
};
struct QgQ8 {   // lib.rs:131-136; q + 128 as the denormal, -128 d in the fma (exact)
    static constexpr int TY = GS_Q8_0, SB = 272, P = 272, TAB = 0;
    static constexpr bool LEAD = false;
    using Hdr = uint32_t;
    struct Prep { const uint8_t *q; float D, C; uint32_t sh; };
    __device__ static __forceinline__ void tables(uint8_t *, int) {}
    __device__ static __forceinline__ Hdr hdr(const uint8_t *s, uint32_t, int u) { return *(const uint16_t *)(s + 34 * u); }
    __device__ static __forceinline__ Prep prep(const Hdr &h, const uint8_t *s, uint32_t, int u) {
        const float d = h2f(h);
        // the quants start at byte 34u + 2: 2 bytes past a dword for even u
        return Prep{s + ((34 * u + 2) & ~3), d * QG_2P24, -128.f * d, (u & 1) ? 0u : 2u};
    }
    using Raw = W3;
    __device__ static __forceinline__ Raw fetch(const Prep &p, const uint8_t *, int g) { return lw3(p.q + 8 * g); }
    __device__ static __forceinline__ h8 frag(const Raw &r, const Prep &p, int) {
        const uint2 w = sh8(r, p.sh);
        const uint32_t a = w.x ^ 0x80808080u, b = w.y ^ 0x80808080u;
        constexpr uint32_t M = 0x00ff00ffu;
        return mix8(a & M, (a >> 8) & M, b & M, (b >> 8) & M, p.D, p.C);
    }
};
// IQ tables in LDS: grid values as 16-bit pairs (an entry's elements in order), then the signs of
// the 128 seven-bit indices as two words P, Q (elements 0..3, 4..7): element 0 at bit 15, 1 at 31,
// 2 at 14, 3 at 30, so a mask and a one-bit shift give the sign bits of element pairs
__device__ __forceinline__ void qg_signs(uint8_t *tab, int tid) {
    if (tid < 128) {
        const uint32_t k = ksigns((uint32_t)tid);
        uint32_t w[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t b = k >> (4 * h);
            w[h] = ((b & 1u) << 15) | (((b >> 1) & 1u) << 31) | (((b >> 2) & 1u) << 14) | (((b >> 3) & 1u) << 30);
        }
        *(uint2 *)(tab + 8 * tid) = make_uint2(w[0], w[1]);
    }
}
__device__ __forceinline__ uint32_t qg_pair(uint32_t lo2) {   // bytes 0, 1 -> 16-bit halves
    return (lo2 & 0xffu) | ((lo2 & 0xff00u) << 8);
}
// d g sign (2s+1)/8 or /4: every product exact in f32, so one f16 rounding
__device__ __forceinline__ h8 iq_mix8(uint4 g, uint2 sm, float D) {
    constexpr uint32_t M = 0x80008000u;
    const uint32_t w[4] = {g.x ^ (sm.x & M), g.y ^ ((sm.x << 1) & M), g.z ^ (sm.y & M), g.w ^ ((sm.y << 1) & M)};
    return to_h8(mix(w[0], 0, D, -0.f), mix(w[0], 1, D, -0.f), mix(w[1], 0, D, -0.f), mix(w[1], 1, D, -0.f),
                 mix(w[2], 0, D, -0.f), mix(w[2], 1, D, -0.f), mix(w[3], 0, D, -0.f), mix(w[3], 1, D, -0.f));
}
struct QgIQ2 {   // lib.rs:274-288
    static constexpr int TY = GS_IQ2_XXS, SB = 66, P = 80, TAB = 1024 + 4096;
    static constexpr bool LEAD = true;
    struct Hdr { W3 w; uint32_t d; };
    struct Prep { uint32_t idx, aux; float D; };
    __device__ static __forceinline__ void tables(uint8_t *tab, int tid) {
        qg_signs(tab, tid);
        if (tid < 256) {
            const uint64_t g = iq2xxs_grid[tid];
            *(uint4 *)(tab + 1024 + 16 * tid) = make_uint4(qg_pair((uint32_t)g), qg_pair((uint32_t)g >> 16),
                                                           qg_pair((uint32_t)(g >> 32)), qg_pair((uint32_t)(g >> 48)));
        }
    }
    __device__ static __forceinline__ Hdr hdr(const uint8_t *s, uint32_t lead, int u) {
        return Hdr{lw3(s + ((lead + 2) & ~3u) + 8 * u), *(const uint16_t *)(s + lead)};
    }
    __device__ static __forceinline__ Prep prep(const Hdr &h, const uint8_t *, uint32_t lead, int) {
        const uint2 w = sh8(h.w, lead ^ 2u);
        return Prep{w.x, w.y, h2f(h.d) * (0.5f + (float)(w.y >> 28)) * 0.25f * QG_2P24};
    }
    struct Raw { uint4 v; uint2 sm; };
    __device__ static __forceinline__ Raw fetch(const Prep &p, const uint8_t *tab, int g) {
        return Raw{*(const uint4 *)(tab + 1024 + 16 * ((p.idx >> (8 * g)) & 0xffu)), *(const uint2 *)(tab + 8 * ((p.aux >> (7 * g)) & 127u))};
    }
    __device__ static __forceinline__ h8 frag(const Raw &r, const Prep &p, int) { return iq_mix8(r.v, r.sm, p.D); }
};
struct QgIQ3 {   // lib.rs:312-328
    static constexpr int TY = GS_IQ3_XXS, SB = 98, P = 112, TAB = 1024 + 2048;
    static constexpr bool LEAD = true;
    struct Hdr { W3 w; uint32_t x0, x1, d; };
    struct Prep { uint32_t i0, i1, aux; float D; };
    __device__ static __forceinline__ void tables(uint8_t *tab, int tid) {
        qg_signs(tab, tid);
        if (tid < 256) {
            const uint32_t g = iq3xxs_grid[tid];
            *(uint2 *)(tab + 1024 + 8 * tid) = make_uint2(qg_pair(g), qg_pair(g >> 16));
        }
    }
    __device__ static __forceinline__ Hdr hdr(const uint8_t *s, uint32_t lead, int u) {
        const uint8_t *b = s + ((lead + 2) & ~3u);
        return Hdr{lw3(b + 8 * u), lw32(b + 64 + 4 * u), lw32(b + 68 + 4 * u), *(const uint16_t *)(s + lead)};
    }
    __device__ static __forceinline__ Prep prep(const Hdr &h, const uint8_t *, uint32_t lead, int) {
        const uint2 w = sh8(h.w, lead ^ 2u);
        const uint32_t aux = __builtin_amdgcn_alignbyte(h.x1, h.x0, lead ^ 2u);
        return Prep{w.x, w.y, aux, h2f(h.d) * (0.5f + (float)(aux >> 28)) * 0.5f * QG_2P24};
    }
    struct Raw { uint2 a, b, sm; };
    __device__ static __forceinline__ Raw fetch(const Prep &p, const uint8_t *tab, int g) {
        const uint32_t iw = (g < 2 ? p.i0 : p.i1) >> (16 * (g & 1));
        return Raw{lw64(tab + 1024 + 8 * (iw & 0xffu)), lw64(tab + 1024 + 8 * ((iw >> 8) & 0xffu)),
                   *(const uint2 *)(tab + 8 * ((p.aux >> (7 * g)) & 127u))};
    }
    __device__ static __forceinline__ h8 frag(const Raw &r, const Prep &p, int) {
        return iq_mix8(make_uint4(r.a.x, r.a.y, r.b.x, r.b.y), r.sm, p.D);
    }
};

// XH: the activations come as f16 half-slabs from the workspace (gs_k_qgemm_x), else f32 rows.
template <class F, int NR, int NT, int RG, int KG, int RC, bool XH>
__device__ __forceinline__ void qgemm_body(const QGemmArgs &a) {
    static_assert(RG * KG == QG_WV && (KG == 2 || KG == 4 || KG == 8), "wave grid");
    constexpr int HS = KG == 8 ? 2 : 1;            // half super-blocks per step
    constexpr int SPC = 2 * RC / HS;               // steps per raw chunk
    constexpr int GPW = 4 * HS / KG;               // fragments per row block, wave and step
    constexpr int T = 16 * NT, RB = 16 * NR * RG;
    constexpr int XHB = T * 256, XB = XHB * HS;    // bytes of a half slab / of one step's activations
    constexpr int CPR = F::P / 16;                 // 16-byte pieces per slot
    constexpr int NPC = RB * RC * CPR;
    constexpr int NRAW = (NPC + QG_TH - 1) / QG_TH;
    constexpr int RAWB = (NPC + 63) / 64 * 1024;   // one raw chunk
    // activation buffers: three where they fit (XH: requested two steps ahead), else two
    constexpr int XR = XH && F::TAB + 3 * XB + 2 * RAWB + 64 <= 160 * 1024 ? 3 : 2;
    constexpr int NXP = XB / 16;                   // 16-byte f16 pieces of a step
    constexpr int NXA = (NXP + QG_TH - 1) / QG_TH;
    extern __shared__ __align__(16) uint8_t qg_lds[];
    __shared__ uint32_t qg_fill[XR + 1];   // activation buffers; raw chunks
    uint8_t *const tab = qg_lds, *const xbuf = qg_lds + F::TAB, *const rawbuf = xbuf + XR * XB;

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 15, q = lane >> 4;
    const int rg = wave / KG, kg = wave % KG;
    // workgroup -> (row block, token block): row block r on XCD r % 8, its token blocks in a row
    const int L = blockIdx.x, k8 = L >> 3;
    const int rblk = (L & 7) + 8 * (k8 / a.n_tb), tblk = k8 % a.n_tb;
    if (rblk >= a.n_rb) return;
    const int z = blockIdx.y, ks = blockIdx.z;
    const int kb0 = ks * a.ksb, kb1 = min(a.K / 256, kb0 + a.ksb), nst = (kb1 - kb0) * 2 / HS;   // steps of this slice
    const int r0 = rblk * RB, n0 = tblk * T;
    const int nrows = min(RB, a.rows - r0), ntok = min(T, a.N - n0);
    const float *X = a.X + (int64_t)z * a.x_bs;

    // raw pieces: piece zc = tid + 512 i -> (slot, 16-byte chunk c), slot = (super-block of the chunk,
    // row); read from the 4-byte boundary at or below the block, 20 bytes, shifted into place. One
    // buffer resource per tile, ending with the dword that holds the tile's last byte.
    const uint8_t *tile = uniform_ptr(a.W + (int64_t)z * a.w_bs + (int64_t)r0 * a.row_stride);
    const uint32_t d0 = (uint32_t)((uintptr_t)tile & 3u);
    const uint32_t row_bytes = (uint32_t)(a.K / 256) * F::SB, rs = (uint32_t)a.row_stride;
    // (the host checks that a tile spans less than 4 GiB)
    const uint32_t wbytes = __builtin_amdgcn_readfirstlane((d0 + (uint32_t)(nrows - 1) * rs + row_bytes + 3u) & ~3u);
    const BufferAt wt(tile - d0, 0, wbytes);
    // piece zc of a chunk -> (slot, 16-byte piece c), slot = (super-block of the chunk, row); read from
    // the dword boundary at or below the block. Pieces past the chunk (XH: the wave's own previous
    // piece, so every wave issues NRAW loads) are clamped to a valid one.
    uint32_t roff[NRAW];
    int rsb[NRAW], rdst[NRAW];
#pragma unroll
    for (int i = 0; i < NRAW; i++) {
        int zc = tid + QG_TH * i;
        if (XH && (zc & ~63) >= NPC) zc -= QG_TH;
        rdst[i] = 16 * zc;
        zc = min(zc, NPC - 1);
        const int slot = zc / CPR, c = zc % CPR, rr = slot % RB;
        rsb[i] = slot / RB;
        roff[i] = d0 + (uint32_t)min(rr, nrows - 1) * rs + 16u * c;
    }
    auto raw_off = [&](int i, int c) { return roff[i] + (uint32_t)F::SB * (uint32_t)min(kb0 + c * RC + rsb[i], kb1 - 1); };
    auto x_sb = [&](int s) { return (uint32_t)(s * XB); };
    const uint8_t *const x16 = uniform_ptr((const uint8_t *)a.X16 + ((int64_t)(z * a.n_tb + tblk) * (a.K / 128) + 2 * kb0) * XHB);
    const uint8_t *const xrow = uniform_ptr((const uint8_t *)(X + (int64_t)n0 * a.x_stride + 256 * kb0));

    // ---- XH = 0: through registers (raw pieces shifted to their dword, activations converted) ------
    uint4 rv[XH ? 1 : NRAW];
    uint32_t rx[XH ? 1 : NRAW];
    auto raw_load = [&](int c) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NRAW; i++) rv[i] = wt.u128(raw_off(i, c) & ~3u);
    };
    auto raw_store = [&](int c) __attribute__((always_inline)) {
        uint8_t *dst = rawbuf + (c & 1) * RAWB;
#pragma unroll
        for (int i = 0; i < NRAW; i++) {
            if (NPC % QG_TH != 0 && tid + QG_TH * i >= NPC) continue;
            *(uint4 *)(dst + rdst[i]) = rv[i];
        }
    };
    uint32_t xoff[XH ? 1 : NXA];   // byte offset of the piece in the token block's f32 rows (host: below 4 GiB)
    if constexpr (!XH) {
#pragma unroll
        for (int i = 0; i < NXA; i++) {
            const int y = min(tid + QG_TH * i, NXP - 1), h = y / (16 * T), t = (y >> 4) % T, c = y & 15;
            xoff[i] = 4u * ((uint32_t)min(t, ntok - 1) * (uint32_t)a.x_stride + 128u * h + 8u * c);
        }
    }
    f4 xv[XH ? 1 : NXA][2];
    auto x_load = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NXA; i++) {
            const GS_GLOBAL f4 *p = (const GS_GLOBAL f4 *)(const GS_GLOBAL uint8_t *)(xrow + (xoff[i] + 512u * (uint32_t)(s * HS)));
            xv[i][0] = p[0];
            xv[i][1] = p[1];
        }
    };
    auto x_store = [&](int s) __attribute__((always_inline)) {
        uint8_t *dst = xbuf + (s & 1) * XB;
#pragma unroll
        for (int i = 0; i < NXA; i++) {
            const int y = tid + QG_TH * i;
            if (NXP % QG_TH != 0 && y >= NXP) continue;
            const f8 v = {xv[i][0].x, xv[i][0].y, xv[i][0].z, xv[i][0].w, xv[i][1].x, xv[i][1].y, xv[i][1].z, xv[i][1].w};
            *(h8 *)(dst + (y & ~15) * 16 + (((y & 15) ^ ((y >> 4) & 15)) << 4)) = __builtin_convertvector(v, h8);
        }
    };

    // ---- XH = 1: straight to LDS (buffer loads with the LDS bit; 16 bytes per lane at M0 + 16 lane) --
    constexpr int NXD = XB / (1024 * QG_WV);       // activation loads per wave and step
    const u4 wrs = rsrc_words(tile - d0, wbytes), xrs = rsrc_words(x16, (uint32_t)(nst * XB));
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)qg_lds;
    const uint32_t xvo = 16u * (uint32_t)lane + 1024u * NXD * (uint32_t)wave;
    auto dma_x1 = [&](int s, int slot, int i) __attribute__((always_inline)) {
        dma16(lds0 + F::TAB + slot * XB + 1024 * (NXD * wave + i), xvo + 1024u * i, x_sb(s), xrs);
    };
    auto dma_raw1 = [&](int c, int i) __attribute__((always_inline)) {
        dma16(lds0 + F::TAB + XR * XB + (c & 1) * RAWB + __builtin_amdgcn_readfirstlane(rdst[i]), raw_off(i, c) & ~3u, 0u, wrs);
    };
    auto dma_x = [&](int s, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NXD; i++) dma_x1(s, slot, i);
    };
    auto dma_raw = [&](int c) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NRAW; i++) dma_raw1(c, i);
    };

    f4 acc[NR][NT];
#pragma unroll
    for (int n = 0; n < NR; n++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[n][t] = f4{0.f, 0.f, 0.f, 0.f};

    // Step s is read from its buffer once every wave has stored its share (fill count 8 (s / XR + 1)).
    // A wave counts step s + 1 at the end of step s, so a wave that reads step s knows that every wave
    // has finished step s - 1, the last reader of what is overwritten next. Counts are read relaxed
    // with an acquire fence on LDS after; bounded, and an expired wait is flagged (as in gemm.hip).
    auto wait_fill = [&](int slot, uint32_t want) __attribute__((always_inline)) {
        want += a.wait_force ? 0x40000000u : 0u;
        for (uint32_t spin = 0;; spin++) {
            if (__hip_atomic_load(&qg_fill[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) >= want) break;
            if (spin >= a.wait_limit) {
                if (lane == 0) __hip_atomic_fetch_or(&gs_wait_expired, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    auto count_fill = [&](int slot) __attribute__((always_inline)) {
        // XH: the data came by the loads just waited for and every read of the buffer it frees has been
        // used; else this wave's LDS stores come first
        if constexpr (XH) asm volatile("" ::: "memory");
        else __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        if (lane == 0) __hip_atomic_fetch_add(&qg_fill[slot], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    const uint8_t *const arow = xbuf + j * 256;
    uint32_t rlead[NR];   // first byte of the lane's rows, modulo 4
#pragma unroll
    for (int n = 0; n < NR; n++) rlead[n] = (d0 + (uint32_t)min(rg * 16 * NR + 16 * n + j, nrows - 1) * rs) & 3u;
    // The B side of a step: scales, raw bytes and first fragment, read and decoded during the step
    // before (between its last MFMAs), so a step starts with its MFMAs
    typename F::Prep p[NR];
    typename F::Raw raw[GPW][NR];
    h8 bf[2][NR];
    typename F::Hdr hd[NR];
    uint32_t lead[NR];
    const uint8_t *slots = nullptr;
    int bu = 0;
    auto b_hdr = [&](int c, int sbc, int h) __attribute__((always_inline)) {   // super-block sbc of raw chunk c, half h
        slots = rawbuf + (c & 1) * RAWB + (sbc * RB + rg * 16 * NR + j) * F::P;
        bu = 4 * h + q;
#pragma unroll
        for (int n = 0; n < NR; n++) {
            lead[n] = F::LEAD ? (rlead[n] + (uint32_t)F::SB * (uint32_t)(kb0 + c * RC + sbc)) & 2u : 0u;
            hd[n] = F::hdr(slots + 16 * n * F::P, lead[n], bu);
        }
    };
    auto b_prep = [&](int n) __attribute__((always_inline)) {
        p[n] = F::prep(hd[n], slots + 16 * n * F::P, lead[n], bu);
#pragma unroll
        for (int gi = 0; gi < GPW; gi++) raw[gi][n] = F::fetch(p[n], tab, (kg * GPW + gi) & 3);
    };
    // MFMAs of k-step gi on fragments av and bf[fb], with other work of this wave placed after each
    // token block by `mid` (a scheduling barrier keeps it there: it runs in the matrix core's shadow)
    h8 av[NT];
    auto mfmas = [&](int fb, auto mid) __attribute__((always_inline)) {
        __builtin_amdgcn_s_setprio(1);   // over waves that wait or decode: 262 -> 255 us at 12288 x 4096 x 2048 tokens
#pragma unroll
        for (int t = 0; t < NT; t++) {
#pragma unroll
            for (int n = 0; n < NR; n++) acc[n][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[t], bf[fb][n], acc[n][t], 0, 0, 0);
            mid(t);
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
    };
    // one step on the activations at xs; `next(stage)` (stage 0 .. 2 NR) prepares the next step's B side
    constexpr int NSTG = 2 * NR + 1;
    auto contract = [&](const uint8_t *xs, auto req, auto next) __attribute__((always_inline)) {
        auto a_ptr = [&](int gi) { return xs + (((4 * q + ((kg * GPW + gi) & 3)) ^ j) << 4); };
        {
            const uint8_t *xa = a_ptr(0);
#pragma unroll
            for (int t = 0; t < NT; t++) av[t] = *(const h8 *)(xa + t * 4096);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int gi = 0; gi + 1 < GPW; gi++) {
            const uint8_t *xa = a_ptr(gi + 1);
            mfmas(gi & 1, [&](int t) __attribute__((always_inline)) {
                if (gi == 0) req(t);
                av[t] = *(const h8 *)(xa + t * 4096);
#pragma unroll
                for (int n = 0; n < NR; n++)
                    if (t == n * NT / NR) bf[(gi + 1) & 1][n] = F::frag(raw[gi + 1][n], p[n], (kg * GPW + gi + 1) & 3);
            });
        }
        constexpr int LB = (GPW - 1) & 1;
        mfmas(LB, [&](int t) __attribute__((always_inline)) {
            if (GPW == 1) req(t);
#pragma unroll
            for (int st = 0; st < NSTG; st++)
                if (t == st * NT / NSTG) next(st);
        });
        // the next step's first fragments
        if (LB == 0) {
#pragma unroll
            for (int n = 0; n < NR; n++) bf[0][n] = bf[1][n];
        }
    };

    F::tables(tab, tid);
    if (tid < XR) qg_fill[tid] = tid == 0 ? QG_WV : 0u;
    if (tid == XR) qg_fill[XR] = 0u;   // raw chunks after the first, counted by every wave
    if constexpr (!XH) {
        raw_load(0);
        x_load(0);
        raw_store(0);
        x_store(0);
    } else {
        dma_raw(0);
        dma_x(0, 0);
        if (XR == 3) dma_x(min(1, nst - 1), 1);
        wait_vm<(XR - 2) * NXD>();   // chunk 0 and step 0 (this wave's share)
    }
    __syncthreads();
    constexpr int FB0 = GPW == 1 ? 1 : 0;
    b_hdr(0, 0, HS == 2 ? kg >> 2 : 0);
#pragma unroll
    for (int n = 0; n < NR; n++) {
        b_prep(n);
        bf[0][n] = F::frag(raw[0][n], p[n], (kg * GPW) & 3);
    }
    int slot = 0;
    uint32_t turn = QG_WV;
    for (int c = 0, s = 0; s < nst; c++) {
#pragma unroll
        for (int sc = 0; sc < SPC; sc++, s++) {
            if (sc > 0 && s >= nst) break;
            if constexpr (!XH) {
                // requested now, stored at the end of the step: the next step's activations, and behind
                // them (loads return in order) the next raw chunk. Past the end they re-read the last
                // step's data, so every wait on them is an exact count.
                x_load(min(s + 1, nst - 1));
                if (sc == 0) raw_load(c + 1);
            }
            if (s > 0) wait_fill(slot, turn);
            const int nslot = slot == XR - 1 ? 0 : slot + 1, pslot = slot == 0 ? XR - 1 : slot - 1;
            if constexpr (XH) {
                // every wave is past step s - 1: its activation buffer takes step s + 2, and at a chunk's
                // first step the other raw buffer the next chunk
                // the chunk requested at the first step (this wave's share), with what came after it
                if (sc == SPC / 2) wait_vm<XR == 3 ? (SPC / 2) * NXD : 0>();
            } else {
                if (sc == SPC / 2) raw_store(c + 1);
            }
            if (sc == SPC / 2) count_fill(XR);
            const bool last = sc == SPC - 1;
            const int h = HS == 2 ? kg >> 2 : sc & 1, s1 = last ? 0 : sc + 1;   // s1: the next step within its chunk
            // (requests go out one by one between the MFMAs: a burst of them stalls the wave at issue)
            auto req = [&](int t) __attribute__((always_inline)) {
                if constexpr (XH) {
                    // three buffers: the raw chunk, then step s + 2's activations; two: step s + 1's first,
                    // as they are waited for at the end of this step
                    constexpr int NQ = NRAW + NXD;
#pragma unroll
                    for (int i = 0; i < NQ; i++)
                        if (t == i * NT / NQ) {
                            if (XR == 3 && i >= NRAW) dma_x1(min(s + 2, nst - 1), pslot, i - NRAW);
                            else if (XR == 2 && i < NXD) dma_x1(min(s + 1, nst - 1), nslot, i);
                            else if (sc == 0) dma_raw1(c + 1, XR == 3 ? i : i - NXD);
                        }
                }
            };
            contract(arow + slot * XB + (HS == 2 ? h * XHB : 0), req, [&](int st) __attribute__((always_inline)) {
                if (st == 0) {
                    if (last) wait_fill(XR, (uint32_t)QG_WV * (uint32_t)(c + 1));
                    b_hdr(last ? c + 1 : c, HS == 2 ? s1 : s1 >> 1, HS == 2 ? kg >> 2 : s1 & 1);
                } else if (st <= NR) {
                    b_prep(st - 1);
                } else {
                    bf[FB0 ? 1 : 0][st - NR - 1] = F::frag(raw[0][st - NR - 1], p[st - NR - 1], (kg * GPW) & 3);
                }
            });
            if constexpr (XH) {
                // step s + 1's activations: only what was requested after them may be outstanding
                if (sc == 0) wait_vm<XR == 3 ? NXD + NRAW : NRAW>();
                else wait_vm<XR == 3 ? NXD : 0>();
            } else {
                if (s + 1 < nst) x_store(s + 1);
            }
            count_fill(nslot);
            if (nslot == 0) turn += QG_WV;
            slot = nslot;
        }
    }
    if constexpr (XH) wait_vm<0>();   // nothing may still land in LDS that the sums below reuse

    // The KG partial tiles are added in kg order through LDS and written; lane holds tokens 16t + 4q + i
    // (i < 4) of row 16n + j of its row group.
    // to Y (added to it with `accumulate`) or, for a K slice, to its partial, summed in slice order by
    // gs_k_gemm_reduce
    float *const obase = a.part ? a.part + ((int64_t)(ks * gridDim.y + z) * a.N + n0) * a.rows + r0
                                : a.Y + (int64_t)z * a.y_bs + (int64_t)n0 * a.y_stride + r0;
    const int64_t ostride = a.part ? a.rows : a.y_stride;
    const bool add = !a.part && a.accumulate;
    auto put = [&](int row, int tok, f4 v) __attribute__((always_inline)) {   // tokens tok .. tok + 3
        if (row >= nrows) return;
        float *dst = obase + (int64_t)tok * ostride + row;
        const int cnt = ntok - tok;
        if (add) {
            f4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (i < cnt) o[i] = dst[i * ostride];
            v += o;
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (i < cnt) dst[i * ostride] = v[i];
    };
    constexpr int WB = NR * NT * 1024;   // one wave's tile
    __syncthreads();
    if (KG == 2) {
        f4 *red = (f4 *)(qg_lds + rg * WB);
        if (kg == 1) {
#pragma unroll
            for (int n = 0; n < NR; n++)
#pragma unroll
                for (int t = 0; t < NT; t++) red[(n * NT + t) * 64 + lane] = acc[n][t];
        }
        __syncthreads();
        if (kg == 0) {
#pragma unroll
            for (int n = 0; n < NR; n++)
#pragma unroll
                for (int t = 0; t < NT; t++)
                    put(rg * 16 * NR + 16 * n + j, 16 * t + 4 * q, acc[n][t] + red[(n * NT + t) * 64 + lane]);
        }
    } else {
        {
            f4 *red = (f4 *)(qg_lds + wave * WB);
#pragma unroll
            for (int n = 0; n < NR; n++)
#pragma unroll
                for (int t = 0; t < NT; t++) red[(n * NT + t) * 64 + lane] = acc[n][t];
        }
        __syncthreads();
        // four outputs per thread and pass: the f4 that lane l of a wave's tile (n, t) holds
        for (int o = tid; o < RG * NR * NT * 64; o += QG_TH) {
            const int l = o & 63, nt = o >> 6, g = nt / (NR * NT), w = nt % (NR * NT), n = w / NT, t = w % NT;
            const f4 *src = (const f4 *)(qg_lds + g * KG * WB) + w * 64 + l;
            f4 v = src[0];
#pragma unroll
            for (int k = 1; k < KG; k++) v += src[k * (WB / 16)];
            put(g * 16 * NR + 16 * n + (l & 15), 16 * t + 4 * (l >> 4), v);
        }
    }
}

#define QG_K(NR, NT, RG, KG, RC, XH)                                                              \
    extern "C" __global__ void __launch_bounds__(QG_TH, 2)                                        \
        QG_NAME(NR, NT, RG, KG, XH)(QGemmArgs a) { qgemm_body<QG_F, NR, NT, RG, KG, RC, XH>(a); }
#define QG_CAT(T, A, B, C, D, E) gs_k_qgemm_##T##_##A##_##B##_##C##_##D##_##E
#define QG_CAT2(T, A, B, C, D, E) QG_CAT(T, A, B, C, D, E)
#define QG_NAME(A, B, C, D, E) QG_CAT2(QG_ID, A, B, C, D, E)

// raw super-blocks per chunk, so that the loads of about 190 slots are in flight: what fits in LDS
#define QG_RC48 (QG_F::P >= 176 ? 2 : 4)
#define QG_ROWS16(NT) QG_K(1, NT, 1, 8, 4, 0) QG_K(2, NT, 1, 8, QG_RC48, 0) QG_K(3, NT, 1, 8, QG_RC48, 0) QG_K(2, NT, 1, 8, QG_RC48, 1) QG_K(3, NT, 1, 8, QG_RC48, 1)
#if defined(QG_F)
QG_ROWS16(1) QG_ROWS16(2) QG_ROWS16(3) QG_ROWS16(4) QG_ROWS16(5) QG_ROWS16(6)
QG_K(2, 8, 4, 2, 1, 0) QG_K(2, 8, 4, 2, 1, 1)
#if QG_ID != 8
QG_K(3, 8, 4, 2, 1, 1)
#endif
#endif
