// chaines.hpp — decoding of long DELTA tiles (gfx950): one tile per wavefront, one LDS round trip per
// decode step.
//
// A tile of 256 macro-steps is a chain of 1024 dependent steps, and a 2880 x 2880 matrix has 8 DELTA
// tiles: a launch over a layer's 12 matrices has 96 chains for 1024 SIMDs, and its time is the chain's
// latency. Decoded the way of short tiles (anneau.hpp), a step waits for two LDS reads, one after the
// other: the renormalisation word, then the LUT entry that this word selects. Here a lane that
// renormalises reads one record holding both. As the tile's words are consumed strictly in order, they
// are turned into records ahead of the decode: word w becomes the LUT entry of slot w mod 4096 with the
// word's upper bits folded in,
//     entry {f | s << 24, b}  ->  record {f | s << 24, f * (w >> 12) + b},
// since the next state's update f * (x >> 12) + b with x = y << 16 | w is f * (y << 4) plus the
// record's second word. A lane that does not renormalise reads its LUT entry (x = y), so every lane
// makes one 8-byte read per step, from the records or from the LUT, and multiplies by y << 4 or
// y >> 12: y' = f * m + b'. The word itself is only needed after the last step (the end check).
//
// One tile per wavefront: lanes 0-31 decode, and as the half's ballot is the low word of the
// wavefront's, the word pointer is a scalar and a lane's rank one v_mbcnt_lo. Lanes 32-63 run the same
// instructions on a state of their own that is equal in all of them (they read one common address
// and store nothing); all 64 lanes translate words, 64 at a time, and load them (256 words per load,
// requested 256 words before they are needed).
//
// Measured: 1024 steps in 90 us (88 ns a step, about 140 cycles of them the LDS read) against 192 us
// with two reads, over the 96 tiles of four gpt-oss experts. The same form for CODES_CTX was measured
// and left out: a word's record is needed for three contexts, and their LUT reads and stores took back
// what the steps gained (four experts: 138 us against 137 us).
#pragma once

#include "anneau.hpp"
#include "commun.hpp"
#include "entiers.hpp"
#include "fusion_corps.hpp"

namespace trc {

constexpr uint32_t CHAINE_N_MIN = 64;   // macro-steps per tile from which tiles are decoded as chains
constexpr uint32_t CHAINE_MOTS = 512;    // words of the raw ring (two halves of 256)
constexpr uint32_t CHAINE_FICHES = 256;  // records per context
constexpr uint32_t CHAINE_MIROIR = 32;   // the ring's first records again past its end: no lane's index wraps
constexpr uint32_t CHAINE_AVANCE = 128;  // records a macro-step can use: 4 steps of 32 lanes
constexpr uint32_t CHAINE_LOT = 64;      // words translated at a time
static_assert(CHAINE_AVANCE + CHAINE_LOT <= CHAINE_FICHES, "a batch fits beside a macro-step's records");
// LDS of one wavefront's chain (raw ring, then records), 16-byte aligned.
constexpr uint32_t CHAINE_OCTETS = 2u * CHAINE_MOTS + 8u * (CHAINE_FICHES + CHAINE_MIROIR);

// The tile being decoded. Words are counted from g0, the 16-byte aligned origin of the tile's words;
// translation starts there, so that batches of 64 never straddle the rings' ends.
struct Chaine {
    const uint8_t* flux;
    uint32_t g0, dernier;        // byte offsets in the stream: origin of the words, its last 8 bytes
    uint32_t a_brut, a_fiches;   // LDS: raw ring, records
    uint32_t a_lut;              // LDS: 4096 8-byte entries
    uint32_t lane;
    uint32_t p, tr, charge;      // next word to consume, next to translate, words requested into the ring
    u32x2 vol;                   // this lane's 4 of the words charge .. charge + 255, not yet in LDS
    // the lane's state before a step: LUT entry (or record) and multiplier
    u32x2 e;
    uint32_t m;
    // after a step: the lane's state before renormalisation, the lanes that renormalise, their first word
    uint32_t y, vote, p_vote;

    __device__ __forceinline__ u32x2 lire(uint32_t mot) const {
        const uint32_t o = g0 + 2u * mot + 8u * lane;
        u32x2 d = {0u, 0u};
        if (o <= dernier) d = *glob<u32x2>(flux + o);
        return d;
    }

    // Tile whose words start at word `debut`, lane states x (lanes 0-31).
    __device__ __forceinline__ void ouvrir(const EnteteRans& h, const DescFlux& f, uint32_t debut, uint32_t x,
                                           uint32_t lut, uint32_t zone) {
        lane = __lane_id();
        const uint32_t mot0 = uint32_t(reinterpret_cast<const uint8_t*>(h.mots) - f.p) + 2u * debut;
        flux = f.p;
        g0 = mot0 & ~15u;
        dernier = dernier_depart(8u, f.longueur);  // (its header, checked, is 16 bytes long)
        a_brut = zone;
        a_fiches = zone + 2u * CHAINE_MOTS;
        a_lut = lut;
        p = (mot0 - g0) / 2u;
        tr = 0u;
        const u32x2 d0 = lire(0u), d1 = lire(256u);
        vol = lire(512u);
        charge = CHAINE_MOTS;
        e = lire_lds<u32x2>(a_lut + ((x & (M - 1u)) << 3));
        m = x >> PROBA_BITS;
        if (lane >= VOIES) {  // one common state
            e = u32x2{0u, 0u};
            m = 0u;
        }
        ecrire_lds<u32x2>(a_brut + 8u * lane, d0);
        ecrire_lds<u32x2>(a_brut + 512u + 8u * lane, d1);
        y = L;
        vote = p_vote = 0;
        traduire();  // tr is past p from here on
    }

    // A batch's translation in three stages, each one LDS round trip, so that a macro-step runs them
    // in the shadow of its steps.
    struct Lot {
        uint32_t w;
        u32x2 f;
    };
    __device__ __forceinline__ void lot_mots(Lot& l) const {
        l.w = lire_lds<uint16_t>(a_brut + 2u * (tr & (CHAINE_MOTS - 1u)) + 2u * lane);
    }
    __device__ __forceinline__ void lot_entrees(Lot& l) const {
        l.f = lire_lds<u32x2>(a_lut + ((l.w & (M - 1u)) << 3));
    }
    __device__ __forceinline__ void lot_fiches(const Lot& l) {
        const uint32_t o = tr & (CHAINE_FICHES - 1u), a = a_fiches + 8u * o + 8u * lane;
        const u32x2 r = {l.f.x, __umul24(l.f.x, l.w >> PROBA_BITS) + l.f.y};
        ecrire_lds<u32x2>(a, r);
        if (o == 0u && lane < CHAINE_MIROIR) ecrire_lds<u32x2>(a + 8u * CHAINE_FICHES, r);
        tr += CHAINE_LOT;
        if (tr + 256u >= charge) {  // the older half of the ring is translated: the next 256 words over it
            ecrire_lds<u32x2>(a_brut + 2u * (charge & (CHAINE_MOTS - 1u)) + 8u * lane, vol);
            charge += 256u;
            vol = lire(charge);
        }
    }
    __device__ __forceinline__ void traduire() {
        Lot l;
        lot_mots(l);
        lot_entrees(l);
        lot_fiches(l);
    }

    // One step. Returns the entry used (its top byte is the decoded symbol).
    __device__ __forceinline__ uint32_t pas() {
        const uint32_t s = e.x;
        uint32_t ici = (a_fiches >> 3) + (p & (CHAINE_FICHES - 1u));  // the first record's address / 8
        asm("" : "+v"(ici));  // added up before the vote, which v_mbcnt counts on from it
        y = __umul24(e.x, m) + e.y;
        const bool besoin = y < L;
        vote = uint32_t(__builtin_amdgcn_ballot_w64(besoin));
        p_vote = p;
        uint32_t a_fiche = __builtin_amdgcn_mbcnt_lo(vote, ici) << 3, a_entree = ((y & (M - 1u)) << 3) + a_lut;
        // both addresses whole before the selection (the compiler would select before the shifts, a
        // longer chain from the vote to the read)
        asm("" : "+v"(a_fiche), "+v"(a_entree));
        m = besoin ? y << 4 : y >> PROBA_BITS;
        p += __popc(vote);
        e = lire_lds<u32x2>(besoin ? a_fiche : a_entree);
        return s;
    }

    // A macro-step: the four decoded bytes, step k in byte k. `entre` runs in the shadow of the first
    // step's read. Enough records are ahead when it starts.
    template <class Entre>
    __device__ __forceinline__ uint32_t macro(Entre entre) {
        while (tr - p < CHAINE_AVANCE) traduire();  // words used faster than 64 a macro-step: rare
        // the batch's reads are unconditional (with no branch around them the waits for the steps' reads
        // stay exact); its records are stored when there is room for them
        const bool lot = tr - p <= CHAINE_FICHES - CHAINE_LOT;
        Lot l;
        lot_mots(l);
        const uint32_t s0 = pas();
        entre();
        lot_entrees(l);
        const uint32_t s1 = pas();
        if (lot) lot_fiches(l);
        const uint32_t s2 = pas(), s3 = pas();
        return __builtin_amdgcn_perm(s1, s0, 0x0c0c0703u) | __builtin_amdgcn_perm(s3, s2, 0x07030c0cu);
    }

    // After the last macro-step: lanes that do not end on L, and whether the words end at `attendu`
    // (counted like `debut`). A lane that renormalised last reads its word back from the stream.
    __device__ __forceinline__ void verifier(const EnteteRans& h, uint32_t debut, uint32_t attendu, uint32_t& hors_l,
                                             uint32_t& pointeur) const {
        if (lane >= VOIES) return;
        uint32_t x = y;
        if (y < L) {
            const uint32_t o = g0 + 2u * __builtin_amdgcn_mbcnt_lo(vote, p_vote);
            x = (y << 16) | (o <= dernier + 6u ? uint32_t(*glob<uint16_t>(flux + o)) : 0u);
        }
        hors_l += x != L ? 1u : 0u;
        const uint32_t mot0 = uint32_t(reinterpret_cast<const uint8_t*>(h.mots) - flux) + 2u * debut;
        pointeur += (lane == 0u && debut + p - (mot0 - g0) / 2u != attendu) ? 1u : 0u;
    }
};

// Byte-wise (med + delta - 128) mod 256.
__device__ __forceinline__ uint32_t echelles_de_deltas(uint32_t med, uint32_t delta) {
    return ((med & 0x7F7F7F7Fu) + (delta & 0x7F7F7F7Fu)) ^ ((med ^ delta) & 0x80808080u) ^ 0x80808080u;
}

// DELTA tiles -> E8M0 scales of blocks of a slot: e(block) = (med[row] + delta - 128) mod 256 (as
// echelles_vers_emplacement). The block's wavefronts (`vagues` of them) take tiles in turn, `zone` the
// calling wavefront's LDS; lut is staged in LDS by the caller, its barrier passed. MED_LDS: the medians
// are too, at med; otherwise (more than MED_LDS_MAX rows) they are read from the stream, med_g.
template <bool MED_LDS>
__device__ __forceinline__ void chaine_echelles(const DescFlux& fd, const EnteteRans& h, uint32_t R, uint32_t B,
                                                uint8_t* ech, const uint2* lut, uint8_t* zone, const uint8_t* med,
                                                const uint8_t* med_g, uint32_t vagues, uint32_t* __restrict__ controle) {
    const uint32_t nblocs = R * B, nmacro = h.P / 128u;
    const uint32_t lane = __lane_id(), v = lane & 31u;
    const bool bas = lane < VOIES;
    const uint32_t a_lut = adresse_lds(lut), a_med = adresse_lds(med);
    const gptr<uint8_t> g_med = glob<uint8_t>(med_g);
    auto mediane = [&](uint32_t r) -> uint32_t {
        const uint32_t i = min(r, R - 1u);
        return MED_LDS ? uint32_t(lire_lds<uint8_t>(a_med + i)) : uint32_t(g_med[i]);
    };
    const uint32_t q128 = 128u / B, r128 = 128u - q128 * B;  // a macro-step's 128 blocks
    uint32_t hors_l = 0, pointeur = 0;
    for (uint32_t t = uniforme32(blockIdx.x * vagues + (threadIdx.x >> 6)); t < h.T; t += gridDim.x * vagues) {
        const uint32_t nb = min(h.N, nmacro - t * h.N);
        const uint32_t debut = uniforme32(h.debut[t]), attendu = uniforme32(t + 1u < h.T ? h.debut[t + 1u] : h.W);
        const uint32_t x = glob<uint32_t>(h.etats)[t * VOIES + v];
        Chaine c;
        c.ouvrir(h, fd, debut, x, a_lut, adresse_lds(zone));
        // the lane's blocks b0 .. b0 + 3, whose first is block `reste` of row `ligne`, and the medians of
        // that row and the next one, read a macro-step before their use; the scales of a macro-step
        // are stored during the next one
        uint32_t b0 = 4u * (t * h.N * VOIES + v), ligne = b0 / B, reste = b0 - ligne * B;
        uint32_t m0 = mediane(ligne), m1 = mediane(ligne + 1u);
        uint32_t deltas = 0;
        auto poser = [&]() {
            uint32_t e4;
            if (B >= 4u) {  // uniform: the four blocks lie in at most two rows
                const uint32_t k = B - reste;
                const uint32_t apres = k >= 4u ? 0u : 0xFFFFFFFFu << (8u * k);  // bytes of the next row
                e4 = echelles_de_deltas(__builtin_amdgcn_perm(m1, m0, apres & 0x04040404u), deltas);
            } else {
                uint32_t meds = 0;
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) meds |= mediane((b0 + k) / B) << (8u * k);
                e4 = echelles_de_deltas(meds, deltas);
            }
            if (bas && b0 + 4u <= nblocs) {
                ecrire_global<uint32_t>(ech + b0, e4);  // b0 % 4 == 0 and the scales are 256-aligned
            } else if (bas) {
                for (uint32_t k = 0; b0 + k < nblocs; ++k) ecrire_global<uint8_t>(ech + b0 + k, uint8_t(e4 >> (8u * k)));
            }
            b0 += 128u;
            ligne += q128;
            reste += r128;
            if (reste >= B) {
                reste -= B;
                ++ligne;
            }
            m0 = mediane(ligne);
            m1 = mediane(ligne + 1u);
        };
        deltas = c.macro([]() {});
        for (uint32_t mm = 1; mm < nb; ++mm) deltas = c.macro(poser);
        poser();
        c.verifier(h, debut, attendu, hors_l, pointeur);
    }
    verser_controle(controle, hors_l, pointeur);
}

}  // namespace trc
