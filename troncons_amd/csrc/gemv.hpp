// gemv.hpp — y = W x + b over a decoded slot's MXFP4 matrix (gfx950), shared by the reference-API
// kernels (noyaux.hip) and the fused path's long-tile layers (fusion.hip).
#pragma once

#include "commun.hpp"
#include "fusion_corps.hpp"

// ============================================================================ GEMVs, reference order
//
// Operation-order contract (the bits of the reference's gemv_mxfp4 / gemv_f32, gemv.cuh:61-126,
// passe.cuh:104-130), for row r of y = W x + b:
//   MXFP4: P(b) = fma chain from 0 over bytes i = 0..15 of block b's 16 code bytes, each byte's low
//          nibble times x[32b + i] then its high nibble times x[32b + 16 + i], with the doubled E2M1
//          values (exact: 2 * {0, .5, 1, 1.5, 2, 3, 4, 6}, code 8 = -0);
//          A(l) = fma chain from 0 over blocks b = l, l + 32, l + 64, ... < B of 2^(e_b - 128) * P(b);
//   f32:   A(l) = fma chain from 0 over quads c = l, l + 32, ... < C/4 of w[4c + k] * x[4c + k], k = 0..3;
//   y[r] = S + b[r] (f32 add; no bias term when b is absent), S the pairwise tree over l = 0..31:
//          pairs at lane distance 16, then 8, 4, 2, 1 (every lane of the tree ends with the same S).
// Mapping here: a 32-lane half-wavefront owns a row (l = its lane), two rows per half for MXFP4
// (the x loads of a block serve both); E2M1 pairs are expanded by v_cvt_scalef32_pk_f32_fp4 (scale
// 2: the doubled values); the tree runs on DPP exchanges (somme_demi_f32); the loads of a
// lane's next block are issued before the current block's arithmetic.
namespace trc {

constexpr uint32_t GEMV_LIGNES_PAR_DEMI = 2;

// Bytes 4t .. 4t + 3 of a block (code word t) continuing the chain s: byte 4t + k pairs with
// x[4t + k] (low nibble) and x[16 + 4t + k] (high nibble), i.e. xa[k] and xb[k].
__device__ __forceinline__ float chaine_mot(uint32_t mot, const f32x4 xa, const f32x4 xb, float s) {
    const f32x2 w0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(mot, 2.0f, 0);
    const f32x2 w1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(mot, 2.0f, 1);
    const f32x2 w2 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(mot, 2.0f, 2);
    const f32x2 w3 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(mot, 2.0f, 3);
    s = fmaf(w0.x, xa.x, s);
    s = fmaf(w0.y, xb.x, s);
    s = fmaf(w1.x, xa.y, s);
    s = fmaf(w1.y, xb.y, s);
    s = fmaf(w2.x, xa.z, s);
    s = fmaf(w2.y, xb.z, s);
    s = fmaf(w3.x, xa.w, s);
    s = fmaf(w3.y, xb.w, s);
    return s;
}

// P(b) for one block: q its 16 code bytes, xs its 32 x values as 8 float4.
__device__ __forceinline__ float chaine_bloc(const u32x4 q, const f32x4 (&xs)[8]) {
    float s = chaine_mot(q.x, xs[0], xs[4], 0.0f);
    s = chaine_mot(q.y, xs[1], xs[5], s);
    s = chaine_mot(q.z, xs[2], xs[6], s);
    return chaine_mot(q.w, xs[3], xs[7], s);
}

struct BlocGemv {
    u32x4 q[GEMV_LIGNES_PAR_DEMI];
    uint32_t e[GEMV_LIGNES_PAR_DEMI];
    f32x4 xs[8];
};

// Rows r0, r0 + 1 of an MXFP4 matrix in its slot (rows past R are read as row R - 1 and not written).
__device__ __forceinline__ void gemv_mxfp4_demi(const uint8_t* __restrict__ mat, const float* __restrict__ x,
                                                float* __restrict__ y, uint32_t R, uint32_t C, uint32_t r0,
                                                uint32_t l) {
    const uint32_t B = C / 32u;
    const trc_disposition d = disposition_matrice(R, C);
    const gptr<u32x4> codes = glob<u32x4>(mat);
    const gptr<uint8_t> ech = glob<uint8_t>(mat + d.echelles);
    const gptr<f32x4> x4 = glob<f32x4>(x);
    uint64_t base[GEMV_LIGNES_PAR_DEMI];
#pragma unroll
    for (uint32_t i = 0; i < GEMV_LIGNES_PAR_DEMI; ++i) base[i] = uint64_t(min(r0 + i, R - 1u)) * B;
    auto charger = [&](uint32_t b, BlocGemv& c) {
#pragma unroll
        for (uint32_t i = 0; i < GEMV_LIGNES_PAR_DEMI; ++i) {
            c.q[i] = codes[base[i] + b];
            c.e[i] = ech[base[i] + b];
        }
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) c.xs[k] = x4[8u * b + k];
    };
    float acc[GEMV_LIGNES_PAR_DEMI] = {};
    BlocGemv cur;
    if (l < B) charger(l, cur);
    for (uint32_t b = l; b < B; b += 32u) {
        BlocGemv suiv;
        charger(min(b + 32u, B - 1u), suiv);  // unconditional (the last one reloads a block): no wait of
                                              // the current block's arithmetic covers these loads
#pragma unroll
        for (uint32_t i = 0; i < GEMV_LIGNES_PAR_DEMI; ++i)
            acc[i] = fmaf(echelle_e8m0(cur.e[i]), chaine_bloc(cur.q[i], cur.xs), acc[i]);
        cur = suiv;
    }
    const gptr<float> biais = glob<float>(mat + d.biais);
#pragma unroll
    for (uint32_t i = 0; i < GEMV_LIGNES_PAR_DEMI; ++i) {
        const float s = somme_demi_f32(acc[i]);
        if (l == 0u && r0 + i < R) y[r0 + i] = s + biais[r0 + i];
    }
}

// The same rows for matrices of at most GEMV_X_COLONNES columns, x staged in LDS once per block of
// FILS threads (FILS / 32 halves of PD rows each), every code and scale load of a lane issued
// before the block's barrier. A lane's blocks are l, l + 32, l + 64 (B <= 96); the arithmetic of
// each row is gemv_mxfp4_demi's, so the bits are the same whatever the block shape. x lies in LDS
// as 144 bytes per block (32 f32 and 16 bytes of padding): lane l's reads of its block start 4
// banks past lane l - 1's, so each group of 8 lanes covers the 32 banks once. The scales of a
// half's rows, contiguous in the slot, come in as 4-byte words (the vector memory unit takes as
// long over a byte load as over a 16-byte one) and are read back from LDS byte by byte.
constexpr uint32_t GEMV_X_BLOCS = 3;                            // blocks per lane at most
constexpr uint32_t GEMV_X_COLONNES = 32u * 32u * GEMV_X_BLOCS;  // 3072
constexpr uint32_t GEMV_X_PAS = 144;                            // LDS bytes per block of x

template <uint32_t FILS, uint32_t PD>  // threads per block, rows per half-wavefront
struct FormeGemvX {
    static constexpr uint32_t DEMIS = FILS / 32u;
    static constexpr uint32_t LIGNES = DEMIS * PD;                              // rows per block
    static constexpr uint32_t MOTS_ECH = PD * 32u * GEMV_X_BLOCS / 4u + 1u;     // scale words per half
    static constexpr uint32_t ECH_DEMI = 4u * MOTS_ECH;
    static constexpr uint32_t NE = (MOTS_ECH + 31u) / 32u;                     // scale words per lane
    static constexpr uint32_t NX = (GEMV_X_COLONNES / 4u + FILS - 1u) / FILS;  // float4 of x per thread
    static constexpr uint32_t LDS = (GEMV_X_COLONNES / 32u) * GEMV_X_PAS + DEMIS * ECH_DEMI;
};

// lire_x(g): values 4g .. 4g + 3 of x.
template <uint32_t FILS, uint32_t PD, uint32_t NB, class LireX>  // NB: blocks per lane, ceil(B / 32)
__device__ __forceinline__ void gemv_mxfp4_x_lds_n(const uint8_t* __restrict__ mat, LireX lire_x,
                                                   float* __restrict__ y, uint32_t R, uint32_t C, uint32_t r_bloc,
                                                   uint8_t* __restrict__ xl) {
    using F = FormeGemvX<FILS, PD>;
    const uint32_t B = C / 32u;
    const uint32_t l = threadIdx.x & 31u;
    const uint32_t r0 = r_bloc + (threadIdx.x >> 5) * PD;
    const trc_disposition d = disposition_matrice(R, C);
    const gptr<u32x4> codes = glob<u32x4>(mat);
    const gptr<uint32_t> ech32 = glob<uint32_t>(mat + d.echelles);  // 256-aligned region of R * B bytes
    // x first, then the scale words: the waits before their LDS stores leave the code loads, issued
    // after them, in flight
    f32x4 xv[F::NX];
#pragma unroll
    for (uint32_t k = 0; k < F::NX; ++k) xv[k] = lire_x(min(threadIdx.x + k * FILS, C / 4u - 1u));
    // the half's scale bytes [r0 B, (r0 + PD) B) as the words from the one holding byte r0 B
    const uint32_t o0 = r0 * B, a0 = o0 >> 2, dernier_mot = (R * B + 3u) / 4u - 1u;
    uint32_t ev[F::NE];
#pragma unroll
    for (uint32_t k = 0; k < F::NE; ++k) ev[k] = ech32[min(a0 + l + 32u * k, dernier_mot)];
    u32x4 q[PD][NB];
    // block by block, so that the arithmetic of a lane's first block waits for its loads only
    // (vector memory completes in order)
#pragma unroll
    for (uint32_t j = 0; j < NB; ++j) {
        const uint32_t b = min(l + 32u * j, B - 1u);  // past B: a block reloaded, never used
#pragma unroll
        for (uint32_t i = 0; i < PD; ++i) q[i][j] = codes[uint64_t(min(r0 + i, R - 1u)) * B + b];
    }
#pragma unroll
    for (uint32_t k = 0; k < F::NX; ++k) {
        const uint32_t g = threadIdx.x + k * FILS;  // float4 g: block g / 8, quarter g % 8
        if (g < C / 4u) *reinterpret_cast<f32x4*>(xl + (g >> 3) * GEMV_X_PAS + 16u * (g & 7u)) = xv[k];
    }
    uint8_t* el = xl + (GEMV_X_COLONNES / 32u) * GEMV_X_PAS + (threadIdx.x >> 5) * F::ECH_DEMI;
#pragma unroll
    for (uint32_t k = 0; k < F::NE; ++k)
        if (4u * (l + 32u * k) < F::ECH_DEMI) *reinterpret_cast<uint32_t*>(el + 4u * (l + 32u * k)) = ev[k];
    __syncthreads();
    // scale of row i, block b: byte (o0 & 3) + i B + b of the half's words (rows past R: unused)
    const uint8_t* el_r = el + (o0 & 3u);
    float acc[PD] = {};
#pragma unroll
    for (uint32_t j = 0; j < NB; ++j) {
        const uint32_t b = l + 32u * j;
        if (b < B) {
            // word by word (x values 4t .. 4t + 3 and 16 + 4t ..): each row's chain keeps
            // chaine_bloc's order, and only two float4 of x are live at a time
            float p[PD] = {};
#pragma unroll
            for (uint32_t t = 0; t < 4; ++t) {
                const f32x4 xa = *reinterpret_cast<const f32x4*>(xl + b * GEMV_X_PAS + 16u * t);
                const f32x4 xb = *reinterpret_cast<const f32x4*>(xl + b * GEMV_X_PAS + 64u + 16u * t);
#pragma unroll
                for (uint32_t i = 0; i < PD; ++i) p[i] = chaine_mot(q[i][j][t], xa, xb, p[i]);
            }
#pragma unroll
            for (uint32_t i = 0; i < PD; ++i) acc[i] = fmaf(echelle_e8m0(el_r[i * B + b]), p[i], acc[i]);
        }
    }
    const gptr<float> biais = glob<float>(mat + d.biais);
#pragma unroll
    for (uint32_t i = 0; i < PD; ++i) {
        const float s = somme_demi_f32(acc[i]);
        if (l == 0u && r0 + i < R) y[r0 + i] = s + biais[r0 + i];
    }
}

// gemv_mxfp4_x_lds_n for the matrix's blocks per lane (uniform over the block), so that only the
// loads a lane can use are held in registers.
template <uint32_t FILS, uint32_t PD, class LireX>
__device__ __forceinline__ void gemv_mxfp4_x_lds(const uint8_t* __restrict__ mat, LireX x, float* __restrict__ y, uint32_t R, uint32_t C, uint32_t r_bloc,
                                                 uint8_t* __restrict__ xl) {
    const uint32_t nb = (C / 32u + 31u) / 32u;
    if (nb <= 1u)
        gemv_mxfp4_x_lds_n<FILS, PD, 1>(mat, x, y, R, C, r_bloc, xl);
    else if (nb == 2u)
        gemv_mxfp4_x_lds_n<FILS, PD, 2>(mat, x, y, R, C, r_bloc, xl);
    else
        gemv_mxfp4_x_lds_n<FILS, PD, 3>(mat, x, y, R, C, r_bloc, xl);
}

// x read from device memory.
struct XCarte {
    gptr<f32x4> x4;
    __device__ __forceinline__ f32x4 operator()(uint32_t g) const { return x4[g]; }
};

}  // namespace trc
