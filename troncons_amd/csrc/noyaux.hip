// noyaux.hip — the reference kernel API of the expert hot path (Noyaux, moteur/crates/trc-noyaux/
// src/lib.rs), written for gfx950.
//
// Same kernel names, arguments and results as the reference's (decodeur.cuh, gemv.cuh, passe.cuh),
// so that the engine's launch layer maps one to one. The slot decoders run the fused path's rANS
// engine (two tiles per wavefront, LDS word rings, 8-byte LUT entries) with a consumer that stores
// into the slot; the GEMVs produce the reference's bits under the operation-order contract stated
// above them, on a wave64 mapping of their own.
//
// Determinism: no floating-point atomics; the only atomics are integer control counters.
#include <hip/hip_runtime.h>

#include "commun.hpp"
#include "emplacement.hpp"
#include "entiers.hpp"
#include "erreurs.hpp"
#include "fusion_corps.hpp"
#include "gemv.hpp"
#include "selection.hpp"

namespace trc {

struct DescDecodage {
    uint64_t partie, emplacement, luts, controle;
};
struct DescGemv {
    uint64_t matrice, x, y;
    uint32_t lignes, colonnes;
};

}  // namespace trc

extern "C" __global__ void __launch_bounds__(trc::FILS_ECHELLES)
decoder_echelles(const uint8_t* __restrict__ partie, uint8_t* __restrict__ emplacement,
                 const uint32_t* __restrict__ luts, trc_dims_expert dims, uint32_t* __restrict__ controle) {
    __shared__ trc::LdsEchelles<trc::FILS_ECHELLES> s;
    trc::decoder_echelles_corps(partie, emplacement, luts, dims, controle, s);
}

extern "C" __global__ void __launch_bounds__(trc::FILS_CODES_SLOT)
decoder_codes(const uint8_t* __restrict__ partie, uint8_t* __restrict__ emplacement, const uint32_t* __restrict__ luts,
              trc_dims_expert dims, uint32_t* __restrict__ controle) {
    __shared__ trc::LdsCodes s;
    trc::decoder_codes_corps(partie, emplacement, luts, dims, controle, s);
}

extern "C" __global__ void __launch_bounds__(trc::FILS_ECHELLES)
decoder_echelles_lot(const trc::DescDecodage* __restrict__ descs, trc_dims_expert dims) {
    __shared__ trc::LdsEchelles<trc::FILS_ECHELLES> s;
    const trc::DescDecodage d = descs[blockIdx.z];
    trc::decoder_echelles_corps(reinterpret_cast<const uint8_t*>(d.partie), reinterpret_cast<uint8_t*>(d.emplacement),
                                reinterpret_cast<const uint32_t*>(d.luts), dims,
                                reinterpret_cast<uint32_t*>(d.controle), s);
}

extern "C" __global__ void __launch_bounds__(trc::FILS_CODES_SLOT)
decoder_codes_lot(const trc::DescDecodage* __restrict__ descs, trc_dims_expert dims) {
    __shared__ trc::LdsCodes s;
    const trc::DescDecodage d = descs[blockIdx.z];
    trc::decoder_codes_corps(reinterpret_cast<const uint8_t*>(d.partie), reinterpret_cast<uint8_t*>(d.emplacement),
                             reinterpret_cast<const uint32_t*>(d.luts), dims, reinterpret_cast<uint32_t*>(d.controle),
                             s);
}

// Raw-file path (flag bit 2): the slot's three regions — codes (16 bytes per block), scales (one
// byte per block), biases (4 bytes per row) — copied from the CODES_BRUTS, ECHELLES_BRUTES and
// BIAIS streams as one list of 16-byte units over the grid. Sources are 16-byte aligned (streams
// are, in a 16-byte aligned part), destinations 256-byte aligned; a region's last unit, when its
// length is not a multiple of 16, is copied byte by byte, so no byte outside a region is written.
namespace trc {
__device__ __forceinline__ void copier_unite(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, uint32_t u,
                                             uint32_t octets) {
    const uint32_t o = 16u * u;
    if (o + 16u <= octets) {
        ecrire_global<u32x4>(dst + o, *glob<u32x4>(src + o));
    } else {
        for (uint32_t k = o; k < octets; ++k) dst[k] = glob<uint8_t>(src)[k];
    }
}
}  // namespace trc

extern "C" __global__ void __launch_bounds__(trc::FILS_BRUT)
copier_brut(const uint8_t* __restrict__ partie, uint8_t* __restrict__ emplacement, trc_dims_expert dims,
            uint32_t* __restrict__ controle) {
    using namespace trc;
    const uint32_t j = blockIdx.y;
    const uint32_t R = choisir(dims.lignes, j), C = choisir(dims.colonnes, j);
    const uint32_t B = C / 32u, nblocs = R * B;
    constexpr uint8_t sortes[4] = {SORTE_CODES_BRUTS, SORTE_ECHELLES_BRUTES, SORTE_BIAIS, 0};
    DescFlux f[4];
    const bool bon = C % 32u == 0 && B > 0 && R > 0 && trouver_flux_n(partie, sortes, 3, j, f) &&
                     f[0].produits == 16u * nblocs && f[0].longueur >= 16u * nblocs && f[1].produits == nblocs &&
                     f[1].longueur >= nblocs && f[2].produits == 4u * R && f[2].longueur >= 4u * R;
    if (!bon) {
        if (threadIdx.x == 0) atomicAdd(&controle[CTL_FORMAT], 1u);
        return;
    }
    const trc_disposition disp = disposition(dims, j);
    uint8_t* mat = emplacement + disp.base;
    const uint32_t n_codes = nblocs, n_ech = (nblocs + 15u) / 16u, n_biais = (4u * R + 15u) / 16u;
    const uint32_t total = n_codes + n_ech + n_biais;
    for (uint32_t u = blockIdx.x * blockDim.x + threadIdx.x; u < total; u += gridDim.x * blockDim.x) {
        if (u < n_codes)
            copier_unite(f[0].p, mat, u, 16u * nblocs);
        else if (u < n_codes + n_ech)
            copier_unite(f[1].p, mat + disp.echelles, u - n_codes, nblocs);
        else
            copier_unite(f[2].p, mat + disp.biais, u - n_codes - n_ech, 4u * R);
    }
}

// ============================================================================ GEMVs (gemv.hpp)
// y = W x + b, x in LDS (C <= GEMV_X_COLONNES): FormeGemvX<FILS, PD>::LIGNES rows per block.
template <uint32_t FILS, uint32_t PD>
__global__ void __launch_bounds__(FILS)
gemv_mxfp4_x(const uint8_t* __restrict__ matrice, const float* __restrict__ x, float* __restrict__ y, uint32_t R,
             uint32_t C) {
    __shared__ __attribute__((aligned(16))) uint8_t xl[trc::FormeGemvX<FILS, PD>::LDS];
    trc::gemv_mxfp4_x_lds<FILS, PD>(matrice, trc::XCarte{trc::glob<trc::f32x4>(x)}, y, R, C, blockIdx.x * trc::FormeGemvX<FILS, PD>::LIGNES, xl);
}

// The batch form: grid y = product; a product wider than GEMV_X_COLONNES takes gemv_mxfp4_demi for
// the same rows (each half-wavefront two at a time). Both branches are uniform over the block (its
// rows belong to one product), so the barrier of the LDS form is reached by all.
template <uint32_t FILS, uint32_t PD>
__global__ void __launch_bounds__(FILS) gemv_mxfp4_lot_x(const trc::DescGemv* __restrict__ descs) {
    using F = trc::FormeGemvX<FILS, PD>;
    __shared__ __attribute__((aligned(16))) uint8_t xl[F::LDS];
    const trc::DescGemv dsc = descs[blockIdx.y];
    const uint32_t r_bloc = blockIdx.x * F::LIGNES;
    if (r_bloc >= dsc.lignes || dsc.colonnes % 32u != 0) return;
    if (dsc.colonnes > trc::GEMV_X_COLONNES) {
        for (uint32_t r0 = r_bloc + (threadIdx.x >> 5) * trc::GEMV_LIGNES_PAR_DEMI;
             r0 < min(r_bloc + F::LIGNES, dsc.lignes); r0 += F::DEMIS * trc::GEMV_LIGNES_PAR_DEMI)
            trc::gemv_mxfp4_demi(reinterpret_cast<const uint8_t*>(dsc.matrice), reinterpret_cast<const float*>(dsc.x),
                                 reinterpret_cast<float*>(dsc.y), dsc.lignes, dsc.colonnes, r0, threadIdx.x & 31u);
        return;
    }
    trc::gemv_mxfp4_x_lds<FILS, PD>(reinterpret_cast<const uint8_t*>(dsc.matrice),
                                    trc::XCarte{trc::glob<trc::f32x4>(reinterpret_cast<const void*>(dsc.x))},
                                    reinterpret_cast<float*>(dsc.y), dsc.lignes, dsc.colonnes, r_bloc, xl);
}

// y = W x + b for one slot matrix: 8 halves x 2 rows per block of 256 threads.
extern "C" __global__ void __launch_bounds__(trc::GEMV_FILS)
gemv_mxfp4(const uint8_t* __restrict__ matrice, const float* __restrict__ x, float* __restrict__ y, uint32_t R,
           uint32_t C) {
    const uint32_t r0 = (blockIdx.x * (trc::GEMV_FILS / 32u) + (threadIdx.x >> 5)) * trc::GEMV_LIGNES_PAR_DEMI;
    if (r0 >= R || C % 32u != 0) return;
    trc::gemv_mxfp4_demi(matrice, x, y, R, C, r0, threadIdx.x & 31u);
}

// Independent products (e.g. the 12 matrices of a layer's 4 experts) in one launch: grid y = product.
extern "C" __global__ void __launch_bounds__(trc::GEMV_FILS) gemv_mxfp4_lot(const trc::DescGemv* __restrict__ descs) {
    const trc::DescGemv dsc = descs[blockIdx.y];
    const uint32_t r0 = (blockIdx.x * (trc::GEMV_FILS / 32u) + (threadIdx.x >> 5)) * trc::GEMV_LIGNES_PAR_DEMI;
    if (r0 >= dsc.lignes || dsc.colonnes % 32u != 0) return;
    trc::gemv_mxfp4_demi(reinterpret_cast<const uint8_t*>(dsc.matrice), reinterpret_cast<const float*>(dsc.x),
                         reinterpret_cast<float*>(dsc.y), dsc.lignes, dsc.colonnes, r0, threadIdx.x & 31u);
}

// y = W x (+ b), W f32 row-major: one row per half-wavefront, four quads per lane in flight.
extern "C" __global__ void __launch_bounds__(trc::GEMV_FILS)
gemv_f32(const float* __restrict__ W, const float* __restrict__ x, const float* __restrict__ biais,
         float* __restrict__ y, uint32_t R, uint32_t C) {
    using namespace trc;
    const uint32_t r = blockIdx.x * (GEMV_FILS / 32u) + (threadIdx.x >> 5);
    const uint32_t l = threadIdx.x & 31u;
    if (r >= R || C % 4u != 0) return;
    const uint32_t C4 = C / 4u;
    const gptr<f32x4> w4 = glob<f32x4>(W + uint64_t(r) * C);
    const gptr<f32x4> x4 = glob<f32x4>(x);
    constexpr uint32_t LOT = 4;
    float acc = 0.0f;
    uint32_t c = l;
    for (; c + 32u * (LOT - 1u) < C4; c += 32u * LOT) {  // whole batches: every load goes out first
        f32x4 w[LOT], xv[LOT];
#pragma unroll
        for (uint32_t u = 0; u < LOT; ++u) {
            w[u] = w4[c + 32u * u];
            xv[u] = x4[c + 32u * u];
        }
#pragma unroll
        for (uint32_t u = 0; u < LOT; ++u) {
            acc = fmaf(w[u].x, xv[u].x, acc);
            acc = fmaf(w[u].y, xv[u].y, acc);
            acc = fmaf(w[u].z, xv[u].z, acc);
            acc = fmaf(w[u].w, xv[u].w, acc);
        }
    }
    for (; c < C4; c += 32u) {
        const f32x4 w = w4[c], xv = x4[c];
        acc = fmaf(w.x, xv.x, acc);
        acc = fmaf(w.y, xv.y, acc);
        acc = fmaf(w.z, xv.z, acc);
        acc = fmaf(w.w, xv.w, acc);
    }
    const float s = somme_demi_f32(acc);
    if (l == 0u) y[r] = biais != nullptr ? s + biais[r] : s;
}

// =========================================================================== router, SwiGLU, combine

// Top-k of E logits by (value desc, index asc); weights = softmax of the k in f64 (m = first,
// exp, ordered sum, division), rounded to f32. One wavefront: 64 lanes x 4 values (E <= 256).
extern "C" __global__ void __launch_bounds__(64)
routeur_topk(const float* __restrict__ logits, uint32_t E, uint32_t k, uint32_t* __restrict__ indices,
             float* __restrict__ poids, uint32_t* boite, uint32_t sequence) {
    using namespace trc;
    if (E == 0 || E > EXPERTS_MAX || k == 0 || k > TOPK_MAX || k > E) return;
    uint32_t choisi[TOPK_MAX];
    float w[TOPK_MAX];
    topk_vague(logits, E, k, choisi, w);
    if (threadIdx.x != 0) return;
#pragma unroll
    for (uint32_t r = 0; r < TOPK_MAX; ++r) {
        if (r < k) {
            indices[r] = choisi[r];
            poids[r] = w[r];
            if (boite != nullptr) {
                reinterpret_cast<volatile uint32_t*>(boite)[1 + r] = choisi[r];
                reinterpret_cast<volatile uint32_t*>(boite)[1 + k + r] = __float_as_uint(w[r]);
            }
        }
    }
    if (boite != nullptr) {
        __threadfence_system();
        reinterpret_cast<volatile uint32_t*>(boite)[0] = sequence;
    }
}

// The cache-biased router (passe.cuh:516-580): the k are chosen on the f32 score logit + biais
// (biais[e] = beta for an expert already in a VRAM slot, 0 else; score desc, index asc), then
// returned by unbiased logit desc, index asc, with the f64 softmax of the unbiased logits as
// weights. With a zero bias: routeur_topk's indices and weights, bit for bit. Same outputs and
// mailbox protocol as routeur_topk. A slot left unchosen (NaN scores) keeps index 0xFFFFFFFF and
// sorts last with weight 0.
extern "C" __global__ void __launch_bounds__(64)
routeur_topk_biais(const float* __restrict__ logits, const float* __restrict__ biais, uint32_t E, uint32_t k,
                   uint32_t* __restrict__ indices, float* __restrict__ poids, uint32_t* boite, uint32_t sequence) {
    using namespace trc;
    if (E == 0 || E > EXPERTS_MAX || k == 0 || k > TOPK_MAX || k > E) return;
    __shared__ float score[EXPERTS_MAX];
    for (uint32_t e = threadIdx.x; e < E; e += blockDim.x) score[e] = logits[e] + biais[e];
    __syncthreads();
    uint32_t choisi[TOPK_MAX];
    float w_score[TOPK_MAX];  // softmax of the scores: not used
    topk_vague(score, E, k, choisi, w_score);
    if (threadIdx.x != 0) return;
    float u[TOPK_MAX];
#pragma unroll
    for (uint32_t r = 0; r < TOPK_MAX; ++r) u[r] = r < k && choisi[r] < E ? logits[choisi[r]] : -INFINITY;
    for (uint32_t r = 1; r < k; ++r)
        for (uint32_t j = r; j > 0 && meilleur(u[j], choisi[j], u[j - 1], choisi[j - 1]); --j) {
            const float tv = u[j];
            u[j] = u[j - 1];
            u[j - 1] = tv;
            const uint32_t ti = choisi[j];
            choisi[j] = choisi[j - 1];
            choisi[j - 1] = ti;
        }
    double ex[TOPK_MAX];
    const double m = u[0];
    double z = 0.0;
    for (uint32_t r = 0; r < k; ++r) {
        ex[r] = exp(double(u[r]) - m);
        z += ex[r];
    }
    for (uint32_t r = 0; r < k; ++r) {
        const float w = float(ex[r] / z);
        indices[r] = choisi[r];
        poids[r] = w;
        if (boite != nullptr) {
            reinterpret_cast<volatile uint32_t*>(boite)[1 + r] = choisi[r];
            reinterpret_cast<volatile uint32_t*>(boite)[1 + k + r] = __float_as_uint(w);
        }
    }
    if (boite != nullptr) {
        __threadfence_system();
        reinterpret_cast<volatile uint32_t*>(boite)[0] = sequence;
    }
}

// gpt-oss clamped SwiGLU in f64, rounded once: g <- min(g,7); u <- clamp(u,-7,7);
// y = g / (1 + exp(-1.702 g)) * (u + 1).
extern "C" __global__ void __launch_bounds__(256)
swiglu_oai(const float* __restrict__ g, const float* __restrict__ u, float* __restrict__ y, uint32_t n) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    const double gv = fmin(double(g[i]), 7.0);
    const double uv = fmin(fmax(double(u[i]), -7.0), 7.0);
    y[i] = float(gv / (1.0 + exp(-1.702 * gv)) * (uv + 1.0));
}

// residu[i] += ((w0 s0[i] + w1 s1[i]) + w2 s2[i]) + ..., each product and sum rounded on its own.
extern "C" __global__ void __launch_bounds__(256)
combiner(float* __restrict__ residu, const float* __restrict__ sorties, uint32_t pas, const float* __restrict__ poids,
         uint32_t n, uint32_t d) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= d || n == 0) return;
    float s = poids != nullptr ? poids[0] * sorties[i] : sorties[i];
    for (uint32_t j = 1; j < n; ++j) {
        const float sj = sorties[uint64_t(j) * pas + i];
        const float p = poids != nullptr ? poids[j] * sj : sj;
        s = s + p;
    }
    residu[i] = residu[i] + s;
}

// ============================================================================ C-ABI launch layer
namespace {

using trc::usage;

inline hipStream_t flux_de(void* f) { return reinterpret_cast<hipStream_t>(f); }

int verifier_dims(const trc_dims_expert* dims) {
    if (dims == nullptr) return usage("dims absent");
    return trc_dims_verifier(dims);
}

}  // namespace

extern "C" int trc_decoder_expert(trc_vue partie, trc_vue emplacement, trc_vue luts, const trc_dims_expert* dims,
                                  trc_vue controle, void* flux) {
    int r = verifier_dims(dims);
    if (r != TRC_OK) return r;
    uint32_t g1[3], g2[3];
    trc_grilles_decodeur(dims, g1, g2);
    return trc_decoder_expert_grilles(partie, emplacement, luts, dims, controle, g1, g2, flux);
}

extern "C" int trc_decoder_expert_grilles(trc_vue partie, trc_vue emplacement, trc_vue luts,
                                          const trc_dims_expert* dims, trc_vue controle, const uint32_t g1[3],
                                          const uint32_t g2[3], void* flux) {
    int r = verifier_dims(dims);
    if (r != TRC_OK) return r;
    const uint64_t te = trc_taille_emplacement(dims);
    TRC_VERIFIER(partie.adresse != 0 && partie.octets >= 64, "partie de %llu o (en-tete de 64 o au moins)",
                 (unsigned long long)partie.octets);
    TRC_VERIFIER(partie.adresse % 16 == 0, "partie non alignee sur 16");
    TRC_VERIFIER(emplacement.octets >= te, "emplacement de %llu o, %llu o demandes",
                 (unsigned long long)emplacement.octets, (unsigned long long)te);
    TRC_VERIFIER(emplacement.adresse != 0 && emplacement.adresse % 256 == 0, "emplacement non aligne sur 256");
    TRC_VERIFIER(luts.adresse != 0 && luts.octets >= uint64_t(trc::LUTS_PAR_COUCHE) * 4, "LUT de %llu o",
                 (unsigned long long)luts.octets);
    TRC_VERIFIER(controle.adresse != 0 && controle.octets >= 16, "controle de moins de 16 o");
    TRC_VERIFIER(g1 != nullptr && g2 != nullptr && g1[1] == 3 && g2[1] == 3 && g1[0] > 0 && g2[0] > 0,
                 "grilles fausses");
    const hipStream_t f = flux_de(flux);
    auto p = reinterpret_cast<const uint8_t*>(partie.adresse);
    auto e = reinterpret_cast<uint8_t*>(emplacement.adresse);
    auto l = reinterpret_cast<const uint32_t*>(luts.adresse);
    auto c = reinterpret_cast<uint32_t*>(controle.adresse);
    hipLaunchKernelGGL(decoder_echelles, dim3(g1[0], 3, 1), dim3(trc::FILS_ECHELLES), 0, f, p, e, l, *dims, c);
    if ((r = trc::apres_lancement("decoder_echelles")) != TRC_OK) return r;
    hipLaunchKernelGGL(decoder_codes, dim3(g2[0], 3, 1), dim3(trc::FILS_CODES_SLOT), 0, f, p, e, l, *dims, c);
    return trc::apres_lancement("decoder_codes");
}

extern "C" int trc_decoder_lot(trc_vue descs, uint32_t n, const trc_dims_expert* dims, void* flux) {
    int r = verifier_dims(dims);
    if (r != TRC_OK) return r;
    TRC_VERIFIER(n > 0 && n <= 65535, "lot de %u experts", n);
    TRC_VERIFIER(descs.adresse != 0 && descs.octets >= uint64_t(n) * sizeof(trc_desc_decodage),
                 "descripteurs trop courts");
    uint32_t g1[3], g2[3];
    trc_grilles_decodeur(dims, g1, g2);
    const hipStream_t f = flux_de(flux);
    auto d = reinterpret_cast<const trc::DescDecodage*>(descs.adresse);
    hipLaunchKernelGGL(decoder_echelles_lot, dim3(g1[0], 3, n), dim3(trc::FILS_ECHELLES), 0, f, d, *dims);
    if ((r = trc::apres_lancement("decoder_echelles_lot")) != TRC_OK) return r;
    hipLaunchKernelGGL(decoder_codes_lot, dim3(g2[0], 3, n), dim3(trc::FILS_CODES_SLOT), 0, f, d, *dims);
    return trc::apres_lancement("decoder_codes_lot");
}

extern "C" int trc_copier_brut(trc_vue partie, trc_vue emplacement, const trc_dims_expert* dims, trc_vue controle,
                               void* flux) {
    int r = verifier_dims(dims);
    if (r != TRC_OK) return r;
    TRC_VERIFIER(partie.adresse != 0 && partie.octets >= 64, "partie trop courte");
    TRC_VERIFIER(partie.adresse % 16 == 0, "partie non alignee sur 16");
    TRC_VERIFIER(emplacement.adresse != 0 && emplacement.octets >= trc_taille_emplacement(dims),
                 "emplacement trop court");
    TRC_VERIFIER(emplacement.adresse % 256 == 0, "emplacement non aligne sur 256");
    TRC_VERIFIER(controle.adresse != 0 && controle.octets >= 16, "controle de moins de 16 o");
    uint32_t g[3];
    trc_grille_brut(dims, g);
    hipLaunchKernelGGL(copier_brut, dim3(g[0], 3, 1), dim3(trc::FILS_BRUT), 0, flux_de(flux),
                       reinterpret_cast<const uint8_t*>(partie.adresse), reinterpret_cast<uint8_t*>(emplacement.adresse),
                       *dims, reinterpret_cast<uint32_t*>(controle.adresse));
    return trc::apres_lancement("copier_brut");
}

namespace {

template <uint32_t FILS, uint32_t PD>
int lancer_gemv_lot_x_forme(const trc::DescGemv* descs, uint32_t n, uint32_t lignes_max, hipStream_t f) {
    constexpr uint32_t L = trc::FormeGemvX<FILS, PD>::LIGNES;
    hipLaunchKernelGGL((gemv_mxfp4_lot_x<FILS, PD>), dim3((lignes_max + L - 1) / L, n), dim3(FILS), 0, f, descs);
    return trc::apres_lancement("gemv_mxfp4_lot_x");
}

// The block shape of a batch of n products of at most lignes_max rows: one row per
// half-wavefront (32 VGPRs, so that a CU holds many wavefronts whose loads and arithmetic overlap),
// 16 halves per block, or 8 when that leaves fewer than 512 blocks. Measured on MI355X over 4, 8
// and 12 gpt-oss matrices against 2 and 4 rows per half and 4 to 32 halves per block.
int lancer_gemv_lot_x(const trc::DescGemv* descs, uint32_t n, uint32_t lignes_max, hipStream_t f) {
    if (uint64_t(n) * ((lignes_max + 15u) / 16u) < 512u) return lancer_gemv_lot_x_forme<256, 1>(descs, n, lignes_max, f);
    return lancer_gemv_lot_x_forme<512, 1>(descs, n, lignes_max, f);
}

}  // namespace

extern "C" int trc_gemv(trc_vue matrice, trc_vue x, trc_vue y, uint32_t lignes, uint32_t colonnes, void* flux) {
    TRC_VERIFIER(lignes > 0 && colonnes > 0 && colonnes % 32 == 0, "forme %u x %u", lignes, colonnes);
    const uint64_t pas = trc::disposition_matrice(lignes, colonnes).pas;
    TRC_VERIFIER(matrice.adresse != 0 && matrice.octets >= pas, "matrice de %llu o, %llu o demandes",
                 (unsigned long long)matrice.octets, (unsigned long long)pas);
    TRC_VERIFIER(matrice.adresse % 256 == 0, "matrice non alignee sur 256");
    TRC_VERIFIER(x.adresse != 0 && x.octets >= 4ull * colonnes && x.adresse % 16 == 0,
                 "x trop court ou non aligne sur 16");
    TRC_VERIFIER(y.adresse != 0 && y.octets >= 4ull * lignes, "y trop court");
    if (colonnes <= trc::GEMV_X_COLONNES) {
        constexpr uint32_t L = trc::FormeGemvX<256, 1>::LIGNES;  // a single product: 8 rows per block
        hipLaunchKernelGGL((gemv_mxfp4_x<256, 1>), dim3((lignes + L - 1) / L), dim3(256), 0, flux_de(flux),
                           reinterpret_cast<const uint8_t*>(matrice.adresse), reinterpret_cast<const float*>(x.adresse),
                           reinterpret_cast<float*>(y.adresse), lignes, colonnes);
        return trc::apres_lancement("gemv_mxfp4_x");
    }
    hipLaunchKernelGGL(gemv_mxfp4, dim3((lignes + trc::GEMV_LIGNES_PAR_BLOC - 1) / trc::GEMV_LIGNES_PAR_BLOC),
                       dim3(trc::GEMV_FILS), 0, flux_de(flux), reinterpret_cast<const uint8_t*>(matrice.adresse),
                       reinterpret_cast<const float*>(x.adresse), reinterpret_cast<float*>(y.adresse), lignes,
                       colonnes);
    return trc::apres_lancement("gemv_mxfp4");
}

extern "C" int trc_gemv_lot(trc_vue descs, uint32_t n, uint32_t lignes_max, void* flux) {
    TRC_VERIFIER(n > 0 && n <= 65535, "lot de %u produits", n);
    TRC_VERIFIER(descs.adresse != 0 && descs.octets >= uint64_t(n) * sizeof(trc_desc_gemv), "descripteurs trop courts");
    TRC_VERIFIER(lignes_max > 0, "lignes_max nul");
    return lancer_gemv_lot_x(reinterpret_cast<const trc::DescGemv*>(descs.adresse), n, lignes_max, flux_de(flux));
}

extern "C" int trc_gemv_f32(trc_vue w, trc_vue x, trc_vue biais, trc_vue y, uint32_t lignes, uint32_t colonnes,
                            void* flux) {
    TRC_VERIFIER(lignes > 0 && colonnes > 0 && colonnes % 4 == 0, "forme %u x %u", lignes, colonnes);
    TRC_VERIFIER(w.adresse != 0 && w.octets >= 4ull * lignes * colonnes && w.adresse % 16 == 0,
                 "matrice f32 trop courte ou non alignee sur 16");
    TRC_VERIFIER(x.adresse != 0 && x.octets >= 4ull * colonnes && x.adresse % 16 == 0,
                 "x trop court ou non aligne sur 16");
    TRC_VERIFIER(y.adresse != 0 && y.octets >= 4ull * lignes, "y trop court");
    TRC_VERIFIER(biais.adresse == 0 || biais.octets >= 4ull * lignes, "biais trop court");
    constexpr uint32_t lignes_bloc = trc::GEMV_FILS / 32u;  // one row per half-wavefront
    hipLaunchKernelGGL(gemv_f32, dim3((lignes + lignes_bloc - 1) / lignes_bloc),
                       dim3(trc::GEMV_FILS), 0, flux_de(flux), reinterpret_cast<const float*>(w.adresse),
                       reinterpret_cast<const float*>(x.adresse), reinterpret_cast<const float*>(biais.adresse),
                       reinterpret_cast<float*>(y.adresse), lignes, colonnes);
    return trc::apres_lancement("gemv_f32");
}

extern "C" int trc_routeur_topk(trc_vue logits, uint32_t experts, uint32_t k, trc_vue indices, trc_vue poids,
                                uint64_t boite, uint32_t sequence, void* flux) {
    TRC_VERIFIER(experts > 0 && experts <= 256 && k > 0 && k <= 8 && k <= experts, "top-%u sur %u", k, experts);
    TRC_VERIFIER(logits.adresse != 0 && logits.octets >= 4ull * experts && indices.adresse != 0 &&
                     indices.octets >= 4ull * k && poids.adresse != 0 && poids.octets >= 4ull * k,
                 "routeur : vues trop courtes");
    hipLaunchKernelGGL(routeur_topk, dim3(1), dim3(64), 0, flux_de(flux), reinterpret_cast<const float*>(logits.adresse),
                       experts, k, reinterpret_cast<uint32_t*>(indices.adresse), reinterpret_cast<float*>(poids.adresse),
                       reinterpret_cast<uint32_t*>(boite), sequence);
    return trc::apres_lancement("routeur_topk");
}

extern "C" int trc_routeur_topk_biais(trc_vue logits, trc_vue biais, uint32_t experts, uint32_t k, trc_vue indices,
                                      trc_vue poids, uint64_t boite, uint32_t sequence, void* flux) {
    TRC_VERIFIER(experts > 0 && experts <= 256 && k > 0 && k <= 8 && k <= experts, "top-%u sur %u", k, experts);
    TRC_VERIFIER(logits.adresse != 0 && logits.octets >= 4ull * experts && biais.adresse != 0 &&
                     biais.octets >= 4ull * experts && indices.adresse != 0 && indices.octets >= 4ull * k &&
                     poids.adresse != 0 && poids.octets >= 4ull * k,
                 "routeur biaise : vues trop courtes");
    hipLaunchKernelGGL(routeur_topk_biais, dim3(1), dim3(64), 0, flux_de(flux),
                       reinterpret_cast<const float*>(logits.adresse), reinterpret_cast<const float*>(biais.adresse),
                       experts, k, reinterpret_cast<uint32_t*>(indices.adresse), reinterpret_cast<float*>(poids.adresse),
                       reinterpret_cast<uint32_t*>(boite), sequence);
    return trc::apres_lancement("routeur_topk_biais");
}

extern "C" int trc_swiglu_oai(trc_vue g, trc_vue u, trc_vue y, uint32_t n, void* flux) {
    const uint64_t o = 4ull * n;
    TRC_VERIFIER(n > 0 && g.adresse && u.adresse && y.adresse && g.octets >= o && u.octets >= o && y.octets >= o,
                 "swiglu : vues trop courtes");
    hipLaunchKernelGGL(swiglu_oai, dim3((n + 255) / 256), dim3(256), 0, flux_de(flux),
                       reinterpret_cast<const float*>(g.adresse), reinterpret_cast<const float*>(u.adresse),
                       reinterpret_cast<float*>(y.adresse), n);
    return trc::apres_lancement("swiglu_oai");
}

extern "C" int trc_combiner(trc_vue residu, trc_vue sorties, uint32_t pas, trc_vue poids, uint32_t n, uint32_t d,
                            void* flux) {
    TRC_VERIFIER(n > 0 && d > 0 && (n == 1 || pas >= d), "combiner %u sorties de %u (pas %u)", n, d, pas);
    TRC_VERIFIER(residu.adresse && sorties.adresse && residu.octets >= 4ull * d &&
                     sorties.octets >= 4ull * ((uint64_t(n) - 1) * pas + d),
                 "combiner : vues trop courtes");
    TRC_VERIFIER(poids.adresse == 0 || poids.octets >= 4ull * n, "poids trop courts");
    hipLaunchKernelGGL(combiner, dim3((d + 255) / 256), dim3(256), 0, flux_de(flux),
                       reinterpret_cast<float*>(residu.adresse), reinterpret_cast<const float*>(sorties.adresse), pas,
                       reinterpret_cast<const float*>(poids.adresse), n, d);
    return trc::apres_lancement("combiner");
}
