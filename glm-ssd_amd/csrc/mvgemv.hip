// gfx950 quantized GEMV of several vectors (gs_gemv with 2..8; Q8_0, Q4_K, Q5_K, Q6_K, rows of whole
// 256-element super-blocks): y[t][r] (+)= W[r] . q8_1(x[t]), crates/cuda/kernels/quants.cu:53-256,
// in one pass over the weights on v_mfma_i32_16x16x64_i8.
//
// Integer weights (Q8_0 int8, Q4_K nibbles, Q5_K 5-bit values, Q6_K 6-bit values - 32) against the
// vectors' q8_1 int8 values, exact int32 dots per unit (per 16-element half for Q6_K, whose halves have
// their own scales), taken into f32 with the unit's scales as the streaming kernels do:
//   Q8_0  d * d_x * dot;   Q4_K, Q5_K  (d*sc) * d_x * dot - (dmin*m) * s_x  (s_x = d_x * sum q_x);
//   Q6_K  (d*sc_h) * d_x * dot_h, per half h.
//
// One MFMA covers 64 elements per weight row (the B columns), 16 per lane quarter q. Its 16 A rows
// are block-diagonal: with up to 4 vectors, rows 4q .. 4q+3 hold the vectors' values of quarter q's
// elements and zeros elsewhere, so the lanes of quarter q (D rows 4q .. 4q+3) get the dots of just
// their own 16 elements and scale them by their own unit's (or half's) scale; with 5..8 vectors and
// whole-unit scales, rows 0..7 belong to the unit in quarters 0, 1 and rows 8..15 to the one in 2, 3
// (Q6_K runs the 4-vector form twice). The quarters are added at the end.
//
// Waves are independent between the sums: 8 waves as RG row tiles x KG along K; wave (rg, kg) takes
// super-blocks kg, kg + KG, .. of its tile's 16 rows, and its own ring of D items (16 rows x one
// super-block) in LDS is filled by loads straight to LDS that only it waits for (the vector-memory
// counter), D items ahead across tiles. The KG partial sums of TB tiles meet in LDS between two
// barriers. What bounds it: the weight stream, behind the quantization of the vectors that every
// workgroup does once per chunk of K.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "kargs.h"
#include "formats.h"
#include "lds_load.h"
#include "q8quant.h"

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

#define MV_TB 2   // tiles between two sums

__device__ __forceinline__ uint32_t lw32(const uint8_t *p) { return *(const uint32_t *)p; }
// 16 bytes at LDS offset p + sh (p dword-aligned, sh 0 or 2)
struct W5 { uint32_t w[5]; };
__device__ __forceinline__ W5 lw5(const uint8_t *p) { return W5{{lw32(p), lw32(p + 4), lw32(p + 8), lw32(p + 12), lw32(p + 16)}}; }
__device__ __forceinline__ W5 lw5a(const uint8_t *p) {   // p 16-byte aligned
    const uint4 v = *(const uint4 *)p;
    return W5{{v.x, v.y, v.z, v.w, lw32(p + 16)}};
}
__device__ __forceinline__ v4i sh16(const W5 &r, uint32_t sh) {
    v4i o;
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] = (int)__builtin_amdgcn_alignbyte(r.w[i + 1], r.w[i], sh);
    return o;
}

// ---- formats: SB bytes per super-block, P its LDS slot (odd multiple of 16, from the dword at or below
// ---- the block's first byte, `lead` bytes into it). load(): a lane's raw words of one item; pos(p): the
// ---- 16 int8 weights and the scales of position p (0..3): unit(p, q) of the super-block, half q & 1.
struct MvScaled { v4i w; float s, mn; };
struct MvQ4K {   // lib.rs:204-218 with scale_min_k4 (lib.rs:87-93)
    static constexpr int TY = GS_Q4_K, SB = 144, P = 144;
    static constexpr bool LEAD = false, MIN = true, HALVES = false;
    struct Raw { uint4 h, q[2]; };
    __device__ static __forceinline__ int unit(int p, int q) { return 4 * (p >> 1) + 2 * (q >> 1) + (p & 1); }
    __device__ static __forceinline__ void load(const uint8_t *s, uint32_t, int q, Raw &r) {
        r.h = *(const uint4 *)s;
#pragma unroll
        for (int i = 0; i < 2; i++) r.q[i] = *(const uint4 *)(s + 16 + 64 * i + 16 * q);
    }
    __device__ static __forceinline__ void scales(const uint4 &h, int p, int q, float &d, float &m) {
        // units 4i + 2(q >> 1) + nib: i = 0 the six-bit fields as they are, i = 1 the split ones
        const uint32_t sh = 8u * (uint32_t)((2 * (q >> 1) + (p & 1)));
        const uint32_t b1 = h.y >> sh, b2 = h.z >> sh, b3 = h.w >> sh;
        const uint32_t sc = p < 2 ? b1 & 63u : (b3 & 0xfu) | ((b1 >> 2) & 0x30u);
        const uint32_t mn = p < 2 ? b2 & 63u : ((b3 >> 4) & 0xfu) | ((b2 >> 2) & 0x30u);
        d = h2f(h.x & 0xffffu) * (float)sc;
        m = h2f(h.x >> 16) * (float)mn;
    }
    __device__ static __forceinline__ MvScaled pos(const Raw &r, int p, int q, uint32_t) {
        MvScaled o;
        const uint4 w = r.q[p >> 1];
        const uint32_t v[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int k = 0; k < 4; k++) o.w[k] = (int)((p & 1 ? v[k] >> 4 : v[k]) & 0x0f0f0f0fu);
        scales(r.h, p, q, o.s, o.mn);
        return o;
    }
};
struct MvQ5K {   // lib.rs:221-240: Q4_K's nibbles and scales, bit u of qh[l] as the fifth bit
    static constexpr int TY = GS_Q5_K, SB = 176, P = 176;
    static constexpr bool LEAD = false, MIN = true, HALVES = false;
    struct Raw { uint4 h, b, q[2]; };
    __device__ static __forceinline__ int unit(int p, int q) { return MvQ4K::unit(p, q); }
    __device__ static __forceinline__ void load(const uint8_t *s, uint32_t, int q, Raw &r) {
        r.h = *(const uint4 *)s;
        r.b = *(const uint4 *)(s + 16 + 16 * (q & 1));
#pragma unroll
        for (int i = 0; i < 2; i++) r.q[i] = *(const uint4 *)(s + 48 + 64 * i + 16 * q);
    }
    __device__ static __forceinline__ MvScaled pos(const Raw &r, int p, int q, uint32_t) {
        MvScaled o;
        const uint4 w = r.q[p >> 1];
        const uint32_t v[4] = {w.x, w.y, w.z, w.w}, b[4] = {r.b.x, r.b.y, r.b.z, r.b.w};
        const uint32_t u = (uint32_t)unit(p, q);
#pragma unroll
        for (int k = 0; k < 4; k++)
            o.w[k] = (int)(((p & 1 ? v[k] >> 4 : v[k]) & 0x0f0f0f0fu) | (((b[k] >> u) & 0x01010101u) << 4));
        MvQ4K::scales(r.h, p, q, o.s, o.mn);
        return o;
    }
};
struct MvQ6K {   // lib.rs:243-262: half n = q >> 1 of the super-block, quarter p of it
    static constexpr int TY = GS_Q6_K, SB = 210, P = 240;
    static constexpr bool LEAD = true, MIN = false, HALVES = true;
    struct Raw { W5 l[2], h; uint32_t sc0, sc1, d; };
    __device__ static __forceinline__ int unit(int p, int q) { return 4 * (q >> 1) + p; }
    __device__ static __forceinline__ void load(const uint8_t *s, uint32_t lead, int q, Raw &r) {
        const int n = q >> 1, e = 16 * (q & 1);
#pragma unroll
        for (int i = 0; i < 2; i++) r.l[i] = lw5a(s + 64 * n + 32 * i + e);
        r.h = lw5a(s + 128 + 32 * n + e);
        // the half's 8 scales, two per quarter (its two 16-element halves)
        const uint8_t *c = s + 192 + 8 * n;
        r.sc0 = __builtin_amdgcn_alignbyte(lw32(c + 4), lw32(c), lead);
        r.sc1 = __builtin_amdgcn_alignbyte(lw32(c + 8), lw32(c + 4), lead);
        r.d = *(const uint16_t *)(s + lead + 208);
    }
    __device__ static __forceinline__ MvScaled pos(const Raw &r, int p, int q, uint32_t lead) {
        MvScaled o;
        const v4i l = sh16(r.l[p & 1], lead), h = sh16(r.h, lead);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t lo = (p >= 2 ? (uint32_t)l[k] >> 4 : (uint32_t)l[k]) & 0x0f0f0f0fu;
            const uint32_t hi = p < 2 ? ((uint32_t)h[k] << (4 - 2 * p)) & 0x30303030u : ((uint32_t)h[k] >> (2 * p - 4)) & 0x30303030u;
            // bytewise v - 32 without borrows between bytes (v in 0..63)
            o.w[k] = (int)(((lo | hi | 0x80808080u) - 0x20202020u) ^ 0x80808080u);
        }
        const uint32_t sw = p < 2 ? r.sc0 : r.sc1;
        o.s = h2f(r.d) * (float)(int)(int8_t)(sw >> (16 * (p & 1) + 8 * (q & 1)));
        o.mn = 0.f;
        return o;
    }
};
struct MvQ8 {   // lib.rs:131-136
    static constexpr int TY = GS_Q8_0, SB = 272, P = 272;
    static constexpr bool LEAD = false, MIN = false, HALVES = false;
    struct Raw { W5 w[4]; uint32_t d[4]; };
    __device__ static __forceinline__ int unit(int p, int q) { return 2 * p + (q >> 1); }
    __device__ static __forceinline__ void load(const uint8_t *s, uint32_t, int q, Raw &r) {
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const int b = 34 * unit(p, q);
            r.d[p] = *(const uint16_t *)(s + b);
            r.w[p] = lw5(s + ((b + 2 + 16 * (q & 1)) & ~3));
        }
    }
    __device__ static __forceinline__ MvScaled pos(const Raw &r, int p, int q, uint32_t) {
        // block 34u: its quants start 2 bytes past a dword for even u = 2p + (q >> 1)
        return MvScaled{sh16(r.w[p], (q & 2) ? 0u : 2u), h2f(r.d[p]), 0.f};
    }
};

template <class F, int VG, int D>
__device__ __forceinline__ void mv_body(const MvArgs &a) {
    constexpr bool UD = VG == 2 && !F::HALVES;       // rows 0..7 / 8..15 for the quarter pairs
    constexpr int NM = VG == 2 && F::HALVES ? 2 : 1; // MFMAs per position
    constexpr int CPR = F::P / 16, ITEM = (16 * F::P + 1023) / 1024 * 1024, ND = ITEM / 1024;
    extern __shared__ __align__(16) uint8_t mv_lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 15, q = lane >> 4;
    const int KG = a.kg, RG = 8 / KG, rg = wave / KG, kg = wave % KG;
    const int nv = a.nv, ck = a.ck, nsb = ck / 256, U = ck / 32;   // units and super-blocks per chunk
    // LDS: zeros, quantized vectors [unit][nv][32], scales [unit][4 VG], sums [unit][4 VG] (MIN), partial
    // sums [MV_TB][8 waves][RL] f4, rings
    uint8_t *const xq = mv_lds + 64;
    float *const xd = (float *)(xq + 32 * (size_t)U * nv);
    float *const xs = xd + 4 * VG * U;
    f4 *const red = (f4 *)(xs + (F::MIN ? 4 * VG * U : 0));
    constexpr int RL = UD ? 32 : 16 * NM;   // f4 of a wave's partial tile: [vector group][row]
    const uint32_t ring0 = (uint32_t)(64 + 32 * U * nv + (F::MIN ? 2 : 1) * 16 * VG * U + MV_TB * 8 * RL * 16 + wave * D * ITEM);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)mv_lds;
    if (tid < 16) ((uint32_t *)mv_lds)[tid] = 0u;

    // ---- this wave's items: tiles t0, t0 + tstep, .. x super-blocks kg, kg + KG, .. ------------------
    const int ntile = (a.rows + 15) / 16, t0 = (int)blockIdx.x * RG + rg, tstep = (int)gridDim.x * RG;
    const int per = kg < nsb ? (nsb - 1 - kg) / KG + 1 : 0;                  // items per tile
    const int mytiles = t0 < ntile ? (ntile - 1 - t0) / tstep + 1 : 0, nitem = per * mytiles;
    const int maxtiles = (ntile - 1 - (int)blockIdx.x * RG) / tstep + 1;     // of any row group here
    const uint32_t rs = (uint32_t)a.row_stride, row_bytes = (uint32_t)(a.K / 256) * F::SB;
    // 16-byte pieces of an item: piece z -> row z / CPR, 16 (z % CPR) bytes into its slot
    uint32_t prow[ND], pcol[ND];
#pragma unroll
    for (int i = 0; i < ND; i++) {
        const int z = min(lane + 64 * i, 16 * CPR - 1);
        prow[i] = (uint32_t)(z / CPR);
        pcol[i] = 16u * (uint32_t)(z % CPR);
    }
    int dt = t0, ds = kg, di = 0;   // next item to request
    int chunk = 0;
    auto request = [&](int slot) __attribute__((always_inline)) {
        const uint32_t nr1 = (uint32_t)min(16, a.rows - 16 * dt) - 1u;
        const uint8_t *base = uniform_ptr(a.w + (int64_t)16 * dt * a.row_stride);
        const uint32_t d0 = (uint32_t)((uintptr_t)base & 3u), so = (uint32_t)(chunk * nsb + ds) * F::SB + d0;
        // ends with the dword that holds the tile's last byte: pieces past it read zeros
        const u4 r = rsrc_words(base - d0, __builtin_amdgcn_readfirstlane((d0 + nr1 * rs + row_bytes + 3u) & ~3u));
#pragma unroll
        for (int i = 0; i < ND; i++)
            dma16(lds0 + ring0 + slot * ITEM + 1024 * i, ((min(prow[i], nr1) * rs + so) & ~3u) + pcol[i], 0u, r);
        di++;
        ds += KG;
        if (ds >= nsb) {
            ds = kg;
            dt += tstep;
        }
    };

    // A operand: this lane's A row and quarter: active where the block diagonal has values
    const int vec = UD ? j & 7 : j & 3;
    const bool diag = UD ? (j >> 3) == (q >> 1) : (j >> 2) == q;
    uint32_t abase[NM], amask[NM];
#pragma unroll
    for (int m = 0; m < NM; m++) {
        const bool on = diag && vec + 4 * m < nv;
        amask[m] = on ? ~0u : 0u;
        abase[m] = on ? 64u + 32u * (uint32_t)(vec + 4 * m) + 16u * (q & 1) : 0u;
    }
    const int sel = UD ? q & 1 : 0;   // vector group of the lane's four D rows

    const int ntask = nv * U * 4;     // 8 floats per task, 4 tasks per unit
    const float rU = 1.0f / (float)U;
    for (chunk = 0; chunk < a.nchunk; chunk++) {
        // ---- the vectors' q8_1 units of this chunk (the streaming kernels' arithmetic) --------------
        constexpr int XC = 8;
        for (int b0 = 0; b0 < ntask; b0 += 512 * XC) {
            f4 f[XC][2];
#pragma unroll
            for (int i = 0; i < XC; i++) {
                const int t = min(b0 + 512 * i + tid, ntask - 1), sub = t & 3, vu = t >> 2, v = udiv_small(vu, rU), u = vu - v * U;
                const GS_GLOBAL f4 *src = (const GS_GLOBAL f4 *)(const GS_GLOBAL float *)(a.x + (int64_t)v * a.x_stride + chunk * ck + 32 * u + 8 * sub);
                f[i][0] = src[0];
                f[i][1] = src[1];
            }
            if (b0 + 512 * XC >= ntask) {   // the last batch is back: the rings' first items
#pragma unroll
                for (int i = 0; i < XC; i++) asm volatile("" : "+v"(f[i][0]), "+v"(f[i][1]));
                di = 0, dt = t0, ds = kg;
#pragma unroll
                for (int k = 0; k < D; k++)
                    if (di < nitem) request(k);
            }
#pragma unroll
            for (int i = 0; i < XC; i++) {
                if (b0 + 512 * i >= ntask) continue;   // uniform; quads are in or out together
                const int t = b0 + 512 * i + tid;
                const float e[8] = {f[i][0][0], f[i][0][1], f[i][0][2], f[i][0][3], f[i][1][0], f[i][1][1], f[i][1][2], f[i][1][3]};
                float amax = 0.f;
#pragma unroll
                for (int k = 0; k < 8; k++) amax = fmaxf(amax, fabsf(e[k]));
                uint32_t ab = __builtin_bit_cast(uint32_t, amax);
                ab = max(ab, __builtin_bit_cast(uint32_t, quad_swap<0xB1>(__builtin_bit_cast(float, ab))));
                ab = max(ab, __builtin_bit_cast(uint32_t, quad_swap<0x4E>(__builtin_bit_cast(float, ab))));
                amax = __builtin_bit_cast(float, ab);
                const float d = q8_div127(amax);
                float id = d != 0.f ? 1.0f / d : 0.f;
                id = id <= 3.40282347e38f ? id : 0.f;   // d < 2^-128: q = 0, as quant_unit
                uint32_t w[2];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    int qv[4];
#pragma unroll
                    for (int b = 0; b < 4; b++) qv[b] = q8_round_mul(e[4 * h + b], id);
                    w[h] = __builtin_amdgcn_perm((uint32_t)qv[1], (uint32_t)qv[0], 0x0c0c0400u) |
                           __builtin_amdgcn_perm((uint32_t)qv[3], (uint32_t)qv[2], 0x04000c0cu);
                }
                int sum = 0;
                if (F::MIN) {   // the unit's sum of q: this thread's 8, then the quad's
                    sum = __builtin_amdgcn_sdot4((int)w[1], 0x01010101, __builtin_amdgcn_sdot4((int)w[0], 0x01010101, 0, false), false);
                    sum += __builtin_bit_cast(int, quad_swap<0xB1>(__builtin_bit_cast(float, sum)));
                    sum += __builtin_bit_cast(int, quad_swap<0x4E>(__builtin_bit_cast(float, sum)));
                }
                if (t < ntask) {
                    const int sub = t & 3, vu = t >> 2, v = udiv_small(vu, rU), u = vu - v * U;
                    *(uint2 *)(xq + 32 * ((size_t)u * nv + v) + 8 * sub) = make_uint2(w[0], w[1]);
                    if (sub == 0) {
                        const float dh = h2f(f2h(d));
                        xd[4 * VG * u + v] = dh;
                        if (F::MIN) xs[4 * VG * u + v] = dh * (float)sum;
                    }
                }
            }
        }
        __syncthreads();

        f4 acc[NM] = {};
        int s = kg, slot = 0, done = 0;
        int tile = t0;
        for (int tb = 0; tb < maxtiles; tb += MV_TB) {
            for (int ti = 0; ti < MV_TB && tb + ti < maxtiles; ti++, tile += tstep) {
#pragma unroll
                for (int m = 0; m < NM; m++) acc[m] = f4{0.f, 0.f, 0.f, 0.f};
                if (tile < ntile) {
                    const uint32_t row0 = (uint32_t)(uintptr_t)(a.w + (int64_t)16 * tile * a.row_stride) + (uint32_t)min(j, a.rows - 16 * tile - 1) * rs;
                    for (s = kg; s < nsb; s += KG) {
                        // this item (they arrive in order): D - 1 younger ones may be in flight, fewer at the end
                        if (di - done >= D) wait_vm<(D - 1) * ND>();
                        else wait_vm<0>();
                        done++;
                        const uint32_t lead = F::LEAD ? (row0 + (uint32_t)F::SB * (uint32_t)(chunk * nsb + s)) & 2u : 0u;
                        typename F::Raw raw;
                        F::load(mv_lds + ring0 + slot * ITEM + j * F::P, lead, q, raw);
                        // the slot is free once the reads above are back
                        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                        __builtin_amdgcn_sched_barrier(0);
                        if (di < nitem) request(slot);
                        slot = slot == D - 1 ? 0 : slot + 1;
#pragma unroll
                        for (int p = 0; p < 4; p++) {
                            const int u = 8 * s + F::unit(p, q);
                            const MvScaled w = F::pos(raw, p, q, lead);
                            v4i dot[NM];
#pragma unroll
                            for (int m = 0; m < NM; m++) {
                                const v4i xa = *(const v4i *)(mv_lds + abase[m] + ((32u * (uint32_t)(u * nv)) & amask[m]));
                                dot[m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa, w.w, v4i{0, 0, 0, 0}, 0, 0, 0);
                            }
#pragma unroll
                            for (int m = 0; m < NM; m++) {
                                const f4 dx = *(const f4 *)(xd + 4 * (VG * u + sel + m));
#pragma unroll
                                for (int k = 0; k < 4; k++) acc[m][k] += (float)dot[m][k] * (w.s * dx[k]);
                                if (F::MIN) {
                                    // one quarter of each unit takes the minimum (UD: each vector group's)
                                    const f4 sx = *(const f4 *)(xs + 4 * (VG * u + sel + m));
                                    const float mn = UD || !(q & 1) ? w.mn : 0.f;
#pragma unroll
                                    for (int k = 0; k < 4; k++) acc[m][k] -= mn * sx[k];
                                }
                            }
                        }
                    }
                }
                // the quarters of the block diagonal: (0 + 1) + (2 + 3), or 0 + 2 and 1 + 3
#pragma unroll
                for (int m = 0; m < NM; m++) {
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        if (!UD) acc[m][k] += __shfl_xor(acc[m][k], 16);
                        acc[m][k] += __shfl_xor(acc[m][k], 32);
                    }
                    if (lane < (UD ? 32 : 16)) red[(ti * 8 + wave) * RL + 16 * m + lane] = acc[m];
                }
            }
            __syncthreads();
            // sums of the tiles' partials, in kg order
            for (int o = tid; o < MV_TB * RG * 16 * 8; o += 512) {
                const int jj = o & 15, v = (o >> 4) & 7, g = (o >> 7) % RG, ti = o / (128 * RG);
                const int tl = (int)blockIdx.x * RG + g + (tb + ti) * tstep, r = 16 * tl + jj;
                if (v < nv && tb + ti < maxtiles && r < a.rows) {
                    float pk[8], sum = 0.f;   // all read before the first is added
#pragma unroll
                    for (int k = 0; k < 8; k++) pk[k] = ((const float *)(red + (ti * 8 + g * KG + min(k, KG - 1)) * RL + 16 * (v >> 2) + jj))[v & 3];
#pragma unroll
                    for (int k = 0; k < 8; k++)
                        if (k < KG) sum += pk[k];
                    float *dst = a.y + (int64_t)v * a.y_stride + r;
                    *dst = a.accumulate || chunk > 0 ? *dst + sum : sum;
                }
            }
            __syncthreads();
        }
    }
}
#define MV_K(TY, F, VG, D)                                                                       \
    extern "C" __global__ void __launch_bounds__(512) gs_k_mv_##TY##_##VG##_##D(MvArgs a) { mv_body<F, VG, D>(a); }
MV_K(8, MvQ8, 1, 2) MV_K(8, MvQ8, 2, 2)
MV_K(12, MvQ4K, 1, 2) MV_K(12, MvQ4K, 2, 2) MV_K(12, MvQ4K, 1, 4) MV_K(12, MvQ4K, 2, 4)
MV_K(13, MvQ5K, 1, 2) MV_K(13, MvQ5K, 2, 2) MV_K(13, MvQ5K, 1, 4) MV_K(13, MvQ5K, 2, 4)
MV_K(14, MvQ6K, 1, 2) MV_K(14, MvQ6K, 2, 2)

// =============================================================================================
// The workgroup form: 16 rows per workgroup in chunks of 4096 elements that all 8 waves store to LDS
// (rows 16 bytes apart beyond their length so a fragment's 16 rows sit in different banks), the vectors'
// q8_1 units unit-major ([unit][vector][32 B]), the next chunk's loads issued before this chunk's
// contraction, the units split between the waves, one v_mfma_i32_16x16x32_i8 per 32-element unit with
// 8 bytes per lane. Q6_K: A rows 0..7 hold the vectors' first half of the unit (k < 16) and zeros, rows
// 8..15 the second, so lane quarters 0, 1 get the first half's dots and 2, 3 the second's, each scaled
// by its own.
// Better than the kernel above where that one's longer prologue and coarser items show: Q8_0, whose
// 34-byte blocks lie off 16-byte boundaries in LDS (there the lanes' dwords meet in a quarter of the
// banks), and Q6_K with 5..8 vectors on at most one tile per CU (there: two MFMAs per position).
// 4096 x 4096: Q8_0, 3/4/8 vectors 7.3/7.5/9.0 us against 8.5/8.9/9.9; Q6_K, 5/8
// vectors 9.5/10.5 against 10.4/11.7.
// =============================================================================================

// 8 bytes at a 2-byte aligned LDS offset: three aligned dwords, shifted into place
__device__ __forceinline__ uint64_t mvc_ld8(const uint8_t *r, uint32_t o) {
    const uint32_t oa = o & ~3u, sh = o & 3u;
    const uint32_t w0 = *(const uint32_t *)(r + oa), w1 = *(const uint32_t *)(r + oa + 4), w2 = *(const uint32_t *)(r + oa + 8);
    return (uint64_t)__builtin_amdgcn_alignbyte(w1, w0, sh) | ((uint64_t)__builtin_amdgcn_alignbyte(w2, w1, sh) << 32);
}
// unit u of a chunk row in LDS, lane quarter q: 8 weights, and the scale of the lane's D rows
struct MvcUnit { uint64_t b; float s; };
struct MvcQ8 {   // lib.rs:131-136
    static constexpr int QK = 32, BB = 34;
    static constexpr bool HALVES = false;
    __device__ static __forceinline__ void unit(const uint8_t *r, int u, int q, MvcUnit &m) {
        const uint32_t blk = 34u * (uint32_t)u;
        m.b = mvc_ld8(r, blk + 2u + 8u * (uint32_t)q);
        m.s = h2f(*(const uint16_t *)(r + blk));
    }
};
struct MvcQ6K {   // lib.rs:243-262
    static constexpr int QK = 256, BB = 210;
    static constexpr bool HALVES = true;
    __device__ static __forceinline__ void unit(const uint8_t *r, int u, int q, MvcUnit &m) {
        const uint32_t b = (uint32_t)u >> 3, uu = (uint32_t)u & 7u, n = uu >> 2, g = uu & 3u, blk = 210u * b;
        const uint64_t ql = mvc_ld8(r, blk + 64u * n + 32u * (g & 1u) + 8u * (uint32_t)q);
        const uint64_t qh = mvc_ld8(r, blk + 128u + 32u * n + 8u * (uint32_t)q);
        const uint64_t v = ((ql >> (4u * (g >> 1))) & 0x0f0f0f0f0f0f0f0full) | (((qh >> (2u * g)) & 0x0303030303030303ull) << 4);
        // v - 32 per byte without borrows between bytes (values 0..63)
        m.b = ((v | 0x8080808080808080ull) - 0x2020202020202020ull) ^ 0x8080808080808080ull;
        m.s = h2f(*(const uint16_t *)(r + blk + 208)) * (float)(int)(int8_t)r[blk + 192u + 8u * n + 2u * g + ((uint32_t)q >> 1)];
    }
};
template <class F, bool MULTI>
__device__ __forceinline__ void mvc_body(const MvArgs &a) {
    extern __shared__ __align__(16) uint8_t mvc_lds[];
    constexpr int CK = 4096;                                    // elements per chunk (at most)
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ck = a.K < CK ? a.K : CK, nch = a.K / ck;         // the host checks a.K % ck == 0
    const int U = ck / 32, nv = a.nv;                           // units per chunk
    const int rbytes = ck / F::QK * F::BB, RS = rbytes + 16;    // chunk row bytes (16-byte multiple), LDS pitch
    uint8_t *wl = mvc_lds;                                       // [16][RS] raw rows of the chunk
    uint8_t *xq = mvc_lds + 16 * (size_t)RS;                     // [U][8][32] int8
    float *xd = (float *)(xq + 256 * (size_t)U);                // [U][8] f16-rounded scales
    float *red = xd + 8 * (size_t)U;                            // [8 waves][64 lanes][4]
    const int r0 = blockIdx.x * 16;
    const int ntask = nv * U * 4;                               // 8 floats per task, 4 tasks per unit
    const int cpr = rbytes / 16, nchunk = 16 * cpr;             // 16-byte pieces per row, per tile
    constexpr int XC = 8, WC = 9;                               // per thread: tasks, pieces (<= 4352 B rows)

    float f[XC][8];
    u4 wc[WC];
    int wdst[WC];   // LDS byte offset of the piece (-1: none)
    // divisions by U and cpr through their reciprocals (exact below 2^21), and a scheduling
    // barrier after each load: the loads then go out as their addresses are ready, instead of
    // after every address of the step (which the compiler otherwise computes first: ~1 us later)
    const float rU = 1.0f / (float)U, rcpr = 1.0f / (float)cpr;
    auto issue_x = [&](int c) __attribute__((always_inline)) {
        const int k0 = c * ck;
#pragma unroll
        for (int i = 0; i < XC; i++) {
            // passes past the last task re-read a valid piece (uniform; no early exit, so the array
            // stays in registers)
            const int t = min(512 * i + tid, ntask - 1);
            const int sub = t & 3, vu = t >> 2, v = udiv_small(vu, rU), u = vu - v * U;
            const float4 *src = (const float4 *)(a.x + (int64_t)v * a.x_stride + k0 + 32 * u + 8 * sub);
            const float4 p0 = src[0], p1 = src[1];
            f[i][0] = p0.x; f[i][1] = p0.y; f[i][2] = p0.z; f[i][3] = p0.w;
            f[i][4] = p1.x; f[i][5] = p1.y; f[i][6] = p1.z; f[i][7] = p1.w;
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto issue_w = [&](int tile, int c) __attribute__((always_inline)) {
        const int64_t wk0 = (int64_t)(c * ck / F::QK) * F::BB;
#pragma unroll
        for (int i = 0; i < WC; i++) {
            const int z = min(512 * i + tid, nchunk - 1), rr = udiv_small(z, rcpr), cc = z - rr * cpr;
            const uint8_t *row = a.w + (int64_t)min(16 * tile + rr, a.rows - 1) * a.row_stride + wk0;   // tail rows: clamped, dropped
            wc[i] = *(const u4 *)(row + 16 * cc);
            wdst[i] = 512 * i + tid < nchunk ? rr * RS + 16 * cc : -1;
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto stage_x = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < XC; i++) {
            if (512 * i >= ntask) continue;                      // uniform; quads are in or out together
            const int t = 512 * i + tid;
            float amax = 0.f;
#pragma unroll
            for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(f[i][e]));
            uint32_t ab = __builtin_bit_cast(uint32_t, amax);
            ab = max(ab, __builtin_bit_cast(uint32_t, quad_swap<0xB1>(__builtin_bit_cast(float, ab))));
            ab = max(ab, __builtin_bit_cast(uint32_t, quad_swap<0x4E>(__builtin_bit_cast(float, ab))));
            amax = __builtin_bit_cast(float, ab);
            const float d = q8_div127(amax);
            float id = d != 0.f ? 1.0f / d : 0.f;
            id = id <= 3.40282347e38f ? id : 0.f;   // d < 2^-128: q = 0, as quant_unit
            uint32_t w[2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                int qv[4];
#pragma unroll
                for (int b = 0; b < 4; b++) qv[b] = q8_round_mul(f[i][4 * h + b], id);
                w[h] = __builtin_amdgcn_perm((uint32_t)qv[1], (uint32_t)qv[0], 0x0c0c0400u) |
                       __builtin_amdgcn_perm((uint32_t)qv[3], (uint32_t)qv[2], 0x04000c0cu);
            }
            if (t < ntask) {
                const int sub = t & 3, vu = t >> 2, v = udiv_small(vu, rU), u = vu - v * U;
                *(uint2 *)(xq + 256 * (size_t)u + 32 * v + 8 * sub) = make_uint2(w[0], w[1]);
                if (sub == 0) xd[8 * u + v] = h2f(f2h(d));
            }
        }
    };

    const int j = lane & 15, q = lane >> 4;
    const int ta = j & 7;                 // the lane's A row's vector
    const int tq = 4 * (q & 1);           // first vector of the lane's four D rows
    // rows 8..15: the vectors' second halves (HALVES), else repeats of 0..7 whose dots are dropped
    const uint64_t amask = F::HALVES && (j >> 3) != (q >> 1) ? 0ull : ~0ull;
    const uint8_t *wrow = wl + (size_t)j * RS;
    const int upw = (U + 7) / 8, u0 = wave * upw, u1 = min(U, u0 + upw);
    // the workgroup's (chunk, tile) steps, chunk-major over its tiles blockIdx.x, blockIdx.x +
    // gridDim.x, ...: the activations of a chunk are staged once for all the workgroup's tiles, and
    // with several tiles each step adds its chunk's partial sums into y (chunk 0 stores them), in
    // chunk order; a single tile keeps them in registers until its last chunk
    // (MULTI = false: the host launched one step per workgroup, so no load is issued during a
    // contraction and the load registers are free there)
    const int ntile = (a.rows + 15) / 16;
    const int ntw = MULTI ? (ntile - 1 - (int)blockIdx.x) / (int)gridDim.x + 1 : 1;   // tiles of this workgroup
    const int nstep = MULTI ? ntw * nch : 1;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    issue_x(0);
    issue_w(blockIdx.x, 0);
    for (int k = 0; k < nstep; k++) {
        const int c = k / ntw, ti = k - c * ntw, tile = blockIdx.x + ti * gridDim.x;
        __builtin_amdgcn_sched_barrier(0);
        if (ti == 0) stage_x();
#pragma unroll
        for (int i = 0; i < WC; i++)
            if (wdst[i] >= 0) *(u4 *)(wl + wdst[i]) = wc[i];
        __syncthreads();
        if (MULTI && k + 1 < nstep) {   // in flight during this step's contraction
            const int k1 = k + 1, c1 = k1 / ntw, t1 = k1 - c1 * ntw;
            if (t1 == 0) issue_x(c1);
            issue_w(blockIdx.x + t1 * gridDim.x, c1);
        }
        // four units per step: their LDS reads and MFMAs overlap
        constexpr int US = 4;
        for (int ub = u0; ub < u1; ub += US) {
            MvcUnit m[US];
            uint64_t xa[US];
            f4 dx[US];
#pragma unroll
            for (int i = 0; i < US; i++) {
                const int u = min(ub + i, u1 - 1);   // past the wave's last unit: re-read it, dropped below
                F::unit(wrow, u, q, m[i]);
                xa[i] = *(const uint64_t *)(xq + 256 * (size_t)u + 32 * ta + 8 * q) & amask;
                dx[i] = *(const f4 *)(xd + 8 * u + tq);
            }
            v4i dot[US];
#pragma unroll
            for (int i = 0; i < US; i++) dot[i] = __builtin_amdgcn_mfma_i32_16x16x32_i8((long)xa[i], (long)m[i].b, v4i{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < US; i++) {
                if (ub + i >= u1) continue;   // uniform
#pragma unroll
                for (int k = 0; k < 4; k++) acc[k] += (float)dot[i][k] * (m[i].s * dx[i][k]);
            }
        }
        if (ntw > 1 || c == nch - 1) {   // the waves' partial sums, in wave order
            *(float4 *)(red + 4 * (64 * wave + lane)) = make_float4(acc[0], acc[1], acc[2], acc[3]);
            acc[0] = acc[1] = acc[2] = acc[3] = 0.f;
            __syncthreads();
            if (tid < 16 * 8) {
                const int t = tid >> 4, jj = tid & 15, r = 16 * tile + jj;
                const int src = 16 * (t >> 2) + jj, i = t & 3;   // the lane that holds D[t][jj]
                float sum = 0.f;
#pragma unroll
                for (int w = 0; w < 8; w++) {
                    sum += red[4 * (64 * w + src) + i];
                    if (F::HALVES) sum += red[4 * (64 * w + src + 32) + i];
                }
                if (t < nv && r < a.rows) {
                    float *dst = a.y + (int64_t)t * a.y_stride + r;
                    *dst = a.accumulate || (ntw > 1 && c > 0) ? *dst + sum : sum;
                }
            }
        }
        __syncthreads();   // every wave is done with this step's LDS before the next is stored
    }
}
// _0: one (chunk, tile) step per workgroup; _1: a walk over several (chunk-major over its tiles)
extern "C" __global__ void __launch_bounds__(512) gs_k_mvc_8_0(MvArgs a) { mvc_body<MvcQ8, false>(a); }
extern "C" __global__ void __launch_bounds__(512) gs_k_mvc_8_1(MvArgs a) { mvc_body<MvcQ8, true>(a); }
extern "C" __global__ void __launch_bounds__(512) gs_k_mvc_14_0(MvArgs a) { mvc_body<MvcQ6K, false>(a); }
