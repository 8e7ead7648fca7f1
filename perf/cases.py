"""The work that a user of this framework has it do, as cases that can be timed and checked.

Every case is one call (or one decode step) through the public entry points of `troncons_amd`:
the rANS-coded MoE layer at batch 1, the batched prefill, one expert, the slot decoder, the MXFP4
and Q8_0 GEMVs, the decode attention, and a whole decode step. Shapes are gpt-oss ones (hidden and
expert width 2880, 64 query heads and 8 KV heads of 64, 201088 vocabulary rows) and smaller or
ragged ones; weights are drawn as a trained layer's are (normal values, quantised to MXFP4 blocks
or Q8_0 blocks) and coded by the framework's encoder.

Tile lengths are written "delta/codes" in macro-steps: "256/256" is what the reference encoder
writes into every file, "mixte" is the encoding of the benchmark (gate and up at 2/32, down at
1/16), the others are lengths that the tests use.
"""
from __future__ import annotations

import math
import os
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

CARTE = "cuda:0"
E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)
JETONS = 8  # activations that the decode cases take in turn, so that the routing moves between passes


# ------------------------------------------------------------------------------------- the cases

def listed():
    return [
        # A token through one MoE layer, batch 1: the call that a decode step makes once per layer.
        {"name": "couche", "sorte": "couche", "E": 32, "k": 4, "d": 2880, "r": 2880, "tuiles": "mixte"},
        # The same over a file of the reference encoder, whose tiles are 256 macro-steps long.
        {"name": "couche_256", "sorte": "couche", "E": 32, "k": 4, "d": 2880, "r": 2880, "tuiles": "256/256"},
        # A prompt's positions through one layer: the benchmark's 512, activations in bf16.
        {"name": "prefill_512", "sorte": "prefill", "E": 32, "k": 4, "d": 2880, "r": 2880, "tuiles": "1/16", "T": 512,
         "x": "bf16"},
        # A short prompt over a reference file, with the f32 activations that a norm leaves.
        {"name": "prefill_37", "sorte": "prefill", "E": 32, "k": 4, "d": 2880, "r": 2880, "tuiles": "256/256", "T": 37,
         "x": "f32"},
        # One expert's MLP from its coded part (the streamed layer runs one per arriving part).
        {"name": "expert", "sorte": "expert", "d": 2880, "r": 2880, "tuiles": "1/16"},
        # The scheduler's decode of a layer's four missing experts into their slots.
        {"name": "decoder_4", "sorte": "decoder", "n": 4, "d": 2880, "r": 2880, "tuiles": "256/256"},
        # The scheduler's MLP matrices over decoded slots: three of each of four experts.
        {"name": "gemv_lot_12", "sorte": "gemv", "n": 12, "lignes": 2880, "colonnes": 2880},
        # The output head, the largest matrix of a decode step.
        {"name": "tete_q8", "sorte": "q8", "lignes": 201088, "colonnes": 2880, "biais": False},
        # The attention output projection.
        {"name": "projection_q8", "sorte": "q8", "lignes": 2880, "colonnes": 4096, "biais": True},
        # Decode attention of a full-context layer at the longest context, and of a windowed layer
        # (128 positions on a ring: the smallest call of a step).
        {"name": "attention_8192", "sorte": "attention", "tetes": 64, "kv": 8, "n": 8192, "anneau": 0, "cache": "f16"},
        {"name": "attention_128", "sorte": "attention", "tetes": 64, "kv": 8, "n": 128, "anneau": 128, "cache": "f16"},
        # A whole decode step (embedding, a windowed and a full-context layer, head, greedy token).
        {"name": "pas", "sorte": "pas", "E": 8, "k": 4, "d": 2880, "vocab": 65536, "position": 4500, "contexte": 8192},
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    sorte = rng.choice(["couche", "couche", "prefill", "expert", "decoder", "gemv", "q8", "attention", "attention"])
    tuiles = rng.choice(["mixte", "1/16", "2/16", "2/32", "256/256", "256/256", "16/64", "4/8"])
    d, r = 32 * _log(rng, 8, 90), 32 * _log(rng, 8, 90)
    if sorte == "couche":
        E = rng.randint(4, 32)
        return {"sorte": sorte, "E": E, "k": min(E, rng.choice([1, 2, 4, 4, 6, 8])), "d": d, "r": r, "tuiles": tuiles}
    if sorte == "prefill":
        E = rng.randint(4, 32)
        return {"sorte": sorte, "E": E, "k": min(E, rng.choice([1, 2, 4])), "d": d, "r": r,
                "tuiles": rng.choice(["1/16", "2/32", "256/256", "4/8"]), "T": _log(rng, 1, 512),
                "x": rng.choice(["bf16", "f32"])}
    if sorte == "expert":
        return {"sorte": sorte, "d": d, "r": r, "tuiles": tuiles}
    if sorte == "decoder":
        return {"sorte": sorte, "n": rng.randint(1, 4), "d": d, "r": r, "tuiles": tuiles}
    if sorte == "gemv":
        return {"sorte": sorte, "n": rng.randint(1, 12), "lignes": _log(rng, 64, 2880), "colonnes": d}
    if sorte == "q8":
        return {"sorte": sorte, "lignes": _log(rng, 64, 201088), "colonnes": 32 * _log(rng, 8, 90),
                "biais": rng.random() < 0.5}
    kv = rng.choice([1, 2, 4, 8])
    n = _log(rng, 1, 8192)
    return {"sorte": sorte, "tetes": kv * rng.choice([1, 4, 8]), "kv": kv, "n": n,
            "anneau": 0 if rng.random() < 0.6 else n + rng.randint(0, 64), "cache": rng.choice(["f16", "f16", "f32"])}


# ------------------------------------------------------------------- seeded weights and their values

def _gen(seed, *cles):
    g = torch.Generator(device=CARTE)
    s = seed & 0xFFFFFFFF
    for c in cles:
        s = (s * 1000003 + c + 1) & 0x7FFFFFFFFFFF
    return g.manual_seed(s)


def _normale(g, *forme, sigma=1.0):
    return torch.randn(*forme, generator=g, device=CARTE) * sigma


def _bf16(t):
    return t.to(torch.bfloat16).to(torch.float32)


def _mxfp4(g, lignes, colonnes):
    """Normal weights of variance 1/colonnes as MXFP4 blocks: codes u8[R][B][16] (byte i of a block:
    weight i in the low nibble, weight 16 + i in the high one) and E8M0 exponents u8[R][B]."""
    w = _normale(g, lignes, colonnes // 32, 32, sigma=colonnes ** -0.5)
    e = torch.floor(torch.log2(w.abs().amax(-1).clamp_min(1e-30))).to(torch.int32) - 2 + 127
    m = w.abs() * torch.exp2((127 - e).to(torch.float32))[..., None]
    bornes = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=CARTE)
    q = torch.bucketize(m, bornes).to(torch.uint8)
    q = torch.where((w < 0) & (q > 0), q | 8, q)  # no negative zero: the coded form folds it
    return q[..., :16] | (q[..., 16:] << 4), e.to(torch.uint8)


def _valeurs64(codes, e):
    """The weights of MXFP4 blocks in 64 bits, [R][C]."""
    table = torch.tensor(E2M1 + tuple(-v for v in E2M1), dtype=torch.float64, device=CARTE)
    w = torch.cat([table[(codes & 15).long()], table[(codes >> 4).long()]], -1)
    return (w * torch.exp2(e.to(torch.float64) - 127.0)[..., None]).reshape(codes.shape[0], -1)


def _formes(c):
    """(rows, columns) of gate, up and down."""
    return [(c["r"], c["d"]), (c["r"], c["d"]), (c["d"], c["r"])]


def _experts(c, seed, n):
    """[expert][matrix] -> (codes, exponents, biases) on the GPU."""
    out = []
    for x in range(n):
        g = _gen(seed, 1, x)
        out.append([(*_mxfp4(g, R, C), _normale(g, R, sigma=0.02)) for R, C in _formes(c)])
    return out


def _tuiles(t):
    """Per matrix (delta, codes) tile lengths, and the two that the calls take (down's)."""
    if t == "mixte":
        return (2, 2, 1), (32, 32, 16), 1, 16
    nd, nc = (int(v) for v in t.split("/"))
    return nd, nc, nd, nc


def _fils(f, n):
    with ThreadPoolExecutor(min(n, 16, os.cpu_count() or 1)) as ex:
        return list(ex.map(f, range(n)))


def _coder(c, experts):
    """The experts' coded parts (bytes) and the layer's LUTs, from the framework's encoder."""
    from troncons_amd import codeur
    from troncons_amd import noyaux as K
    formes = _formes(c)
    dims = K.DimsExpert.de([f[0] for f in formes], [f[1] for f in formes])
    nd, nc, _, _ = _tuiles(c["tuiles"])
    hote = []
    for mats in experts:
        bl = [torch.cat([e[..., None], q], -1).reshape(-1).cpu().numpy() for q, e, _ in mats]
        hote.append((bl, [b.cpu().numpy() for _, _, b in mats]))
    freqs = _fils(lambda j: codeur.tables([h[0][j] for h in hote], formes[j][0], formes[j][1] // 32), 3)
    parts = _fils(lambda x: codeur.partie(hote[x][0], hote[x][1], freqs, dims, expert=x, N_delta=nd, N_codes=nc)[0],
                  len(hote))
    luts = K.luts_couche([[freqs[j][t] for t in range(4)] for j in range(3)])
    return dims, parts, torch.from_numpy(luts.view(np.int32).copy()).to(CARTE), freqs


def _sur_carte(parts):
    """The parts in one allocation (256-aligned each): the tensor and the address of each part."""
    pas = [(len(p) + 255) // 256 * 256 for p in parts]
    bloc = torch.zeros(sum(pas), dtype=torch.uint8, device=CARTE)
    adresses, o = [], 0
    for p, n in zip(parts, pas):
        bloc[o:o + len(p)].copy_(torch.from_numpy(np.frombuffer(p, np.uint8).copy()))
        adresses.append(bloc.data_ptr() + o)
        o += n
    return bloc, adresses


def _travail(octets):
    from troncons_amd.noyaux import VueCarte
    t = torch.zeros(octets + 256, dtype=torch.uint8, device=CARTE)
    return t, VueCarte.de(t, (-t.data_ptr()) % 256, octets)


def _controle():
    return torch.zeros(4, dtype=torch.int32, device=CARTE)


def _routeur(seed, E, d):
    """A router of bf16 rows (the values, and their bits as the calls take them)."""
    w = _normale(_gen(seed, 2), E, d, sigma=d ** -0.5).to(torch.bfloat16)
    return w


def _routage(seed, T, E, k):
    """Top-k choices of T positions, skewed over the experts as real routing is, and softmax weights."""
    g = torch.Generator().manual_seed((seed * 7919 + 13) & 0x7FFFFFFF)
    p = 1.0 / torch.arange(1, E + 1, dtype=torch.float64)
    idx = torch.multinomial(p.expand(T, E), k, generator=g)
    lg = torch.randn(T, k, generator=g, dtype=torch.float64).sort(-1, descending=True).values
    return idx.to(torch.int32), torch.softmax(lg, -1).to(torch.float32)


def _q8(g, lignes, colonnes):
    """Normal weights of variance 1/colonnes as Q8_0 blocks u8[R][B][34] (f16 d, 32 codes of 8 bits)."""
    sortie = torch.empty(lignes, colonnes // 32, 34, dtype=torch.uint8, device=CARTE)
    for r in range(0, lignes, 16384):
        w = _normale(g, min(16384, lignes - r), colonnes // 32, 32, sigma=colonnes ** -0.5)
        s = (w.abs().amax(-1) / 127.0).to(torch.float16)
        q = torch.round(w / s.to(torch.float32).clamp_min(1e-12)[..., None]).clamp(-127, 127).to(torch.int8)
        sortie[r:r + w.shape[0], :, :2] = s[..., None].view(torch.uint8)
        sortie[r:r + w.shape[0], :, 2:] = q.view(torch.uint8)
    return sortie


def _q8_64(blocs):
    s = blocs[..., :2].contiguous().view(torch.float16).to(torch.float64)
    return (blocs[..., 2:].view(torch.int8).to(torch.float64) * s).reshape(blocs.shape[0], -1)


# ------------------------------------------------------------------------------- prepare and run

def prepare(case, seed):
    return globals()["_prepare_" + case["sorte"]](case, seed)


def run(state):
    return globals()["_run_" + state["sorte"]](state)


def _jetons(c, seed):
    return _bf16(_normale(_gen(seed, 3), JETONS, c["d"]))


def _prepare_couche(c, seed):
    from troncons_amd import fusion
    from troncons_amd.noyaux import VueCarte
    V = VueCarte.de
    dims, parts, luts, _ = _coder(c, _experts(c, seed, c["E"]))
    bloc, adresses = _sur_carte(parts)
    fz = fusion.Fusion()
    table = torch.tensor(adresses, dtype=torch.int64, device=CARTE)
    rep = torch.zeros(fusion.taille_repertoire(c["E"]), dtype=torch.uint8, device=CARTE)
    ctl = _controle()
    fz.monter_couche(V(table), c["E"], dims, V(rep), V(ctl))
    _, _, nd, nc = _tuiles(c["tuiles"])
    garde, travail = _travail(fusion.taille_travail_couche(dims, c["E"], c["k"], nc))
    routeur = _routeur(seed, c["E"], c["d"])
    x = _jetons(c, seed)
    residu = _normale(_gen(seed, 4), c["d"])
    idx = torch.zeros(c["k"], dtype=torch.int32, device=CARTE)
    poids = torch.zeros(c["k"], dtype=torch.float32, device=CARTE)
    return {"sorte": "couche", "c": c, "fz": fz, "dims": dims, "rep": V(rep), "luts": V(luts), "routeur": V(routeur),
            "x": [V(x[i]) for i in range(JETONS)], "i": 0, "residu": residu, "idx": idx, "poids": poids, "ctl": ctl,
            "travail": travail, "nd": nd, "nc": nc, "garde": (garde, bloc, table, x)}


def _run_couche(s):
    c = s["c"]
    x = s["x"][s["i"] % JETONS]
    s["i"] += 1
    s["fz"].couche_moe(s["rep"], c["E"], s["luts"], s["dims"], s["routeur"], None, x, c["k"], s["residu"], s["idx"],
                       s["poids"], s["ctl"], s["travail"], s["nd"], s["nc"])
    return {"residu": s["residu"], "indices": s["idx"], "poids": s["poids"], "controle": s["ctl"]}


def _x_prefill(c, seed):
    x = _normale(_gen(seed, 3), c["T"], c["d"])
    return _bf16(x) if c["x"] == "bf16" else x


def _prepare_prefill(c, seed):
    from troncons_amd import fusion
    from troncons_amd.noyaux import VueCarte
    V = VueCarte.de
    dims, parts, luts, _ = _coder(c, _experts(c, seed, c["E"]))
    bloc, adresses = _sur_carte(parts)
    fz = fusion.Fusion()
    table = torch.tensor(adresses, dtype=torch.int64, device=CARTE)
    rep = torch.zeros(fusion.taille_repertoire(c["E"]), dtype=torch.uint8, device=CARTE)
    ctl = _controle()
    fz.monter_couche(V(table), c["E"], dims, V(rep), V(ctl))
    _, _, nd, nc = _tuiles(c["tuiles"])
    garde, travail = _travail(fusion.taille_travail_prefill(dims, c["E"], c["T"], c["k"], nc))
    idx, poids = (t.to(CARTE) for t in _routage(seed, c["T"], c["E"], c["k"]))
    residus = _normale(_gen(seed, 4), c["T"], c["d"])
    return {"sorte": "prefill", "c": c, "fz": fz, "dims": dims, "rep": V(rep), "luts": V(luts),
            "x": V(_x_prefill(c, seed)), "idx": V(idx), "poids": V(poids), "residus": residus, "ctl": ctl,
            "travail": travail, "nd": nd, "nc": nc, "garde": (garde, bloc, table)}


def _run_prefill(s):
    c = s["c"]
    s["fz"].prefill_moe(s["rep"], c["E"], s["luts"], s["dims"], s["x"], c["T"], s["idx"], s["poids"], c["k"],
                        s["residus"], s["ctl"], s["travail"], s["nd"], s["nc"])
    return {"residus": s["residus"], "controle": s["ctl"]}


def _prepare_expert(c, seed):
    from troncons_amd import fusion
    from troncons_amd.noyaux import VueCarte
    dims, parts, luts, _ = _coder(c, _experts(c, seed, 1))
    bloc, _ = _sur_carte(parts)
    _, _, nd, nc = _tuiles(c["tuiles"])
    garde, travail = _travail(fusion.taille_travail_expert(dims, nc))
    return {"sorte": "expert", "fz": fusion.Fusion(), "dims": dims, "partie": VueCarte.de(bloc),
            "luts": VueCarte.de(luts), "x": VueCarte.de(_jetons(c, seed)[0].contiguous()),
            "sortie": torch.zeros(c["d"], device=CARTE), "ctl": _controle(), "travail": travail, "nd": nd, "nc": nc,
            "garde": garde}


def _run_expert(s):
    s["fz"].expert_fusionne(s["partie"], s["luts"], s["dims"], s["x"], s["sortie"], s["ctl"], s["travail"], s["nd"],
                            s["nc"])
    return {"sortie": s["sortie"], "controle": s["ctl"]}


def _prepare_decoder(c, seed):
    from troncons_amd import noyaux as K
    dims, parts, luts, _ = _coder(c, _experts(c, seed, c["n"]))
    bloc, adresses = _sur_carte(parts)
    taille = K.taille_emplacement(dims)
    slots = torch.zeros(c["n"], taille, dtype=torch.uint8, device=CARTE)
    ctl = torch.zeros(c["n"], 4, dtype=torch.int32, device=CARTE)
    descs = b"".join(K.DescDecodage(adresses[i], slots[i].data_ptr(), luts.data_ptr(), ctl[i].data_ptr()).octets()
                     for i in range(c["n"]))
    d = torch.from_numpy(np.frombuffer(descs, np.uint8).copy()).to(CARTE)
    return {"sorte": "decoder", "n": c["n"], "noyaux": K.Noyaux.charger(), "dims": dims, "descs": K.VueCarte.de(d),
            "slots": slots, "ctl": ctl, "garde": (bloc, luts)}


def _run_decoder(s):
    s["noyaux"].decoder_lot(s["descs"], s["n"], s["dims"])
    return {"emplacements": s["slots"], "controle": s["ctl"]}


def _matrices(c, seed):
    """The slot matrices of a GEMV batch, (codes, exponents, biases) each, and an x for each."""
    out = []
    for i in range(c["n"]):
        g = _gen(seed, 5, i)
        out.append((*_mxfp4(g, c["lignes"], c["colonnes"]), _normale(g, c["lignes"], sigma=0.02),
                    _normale(g, c["colonnes"])))
    return out


def _prepare_gemv(c, seed):
    from troncons_amd import noyaux as K
    R, C = c["lignes"], c["colonnes"]
    d = K.disposition_matrice(R, C)
    garde, descs = [], b""
    y = torch.zeros(c["n"], R, device=CARTE)
    for i, (codes, e, b, x) in enumerate(_matrices(c, seed)):
        m = torch.zeros(d.pas, dtype=torch.uint8, device=CARTE)
        m[:codes.numel()] = codes.reshape(-1)
        m[d.echelles:d.echelles + e.numel()] = e.reshape(-1)
        m[d.biais:d.biais + 4 * R] = b.view(torch.uint8)
        garde += [m, x]
        descs += bytes(K.DescGemv(m.data_ptr(), x.data_ptr(), y[i].data_ptr(), R, C))
    t = torch.from_numpy(np.frombuffer(descs, np.uint8).copy()).to(CARTE)
    return {"sorte": "gemv", "n": c["n"], "lignes": R, "noyaux": K.Noyaux.charger(), "descs": K.VueCarte.de(t), "y": y,
            "garde": garde}


def _run_gemv(s):
    s["noyaux"].gemv_lot(s["descs"], s["n"], s["lignes"])
    return s["y"]


def _entrees_q8(c, seed):
    g = _gen(seed, 6)
    w = _q8(g, c["lignes"], c["colonnes"])
    return w, _normale(g, c["colonnes"]), _normale(g, c["lignes"], sigma=0.1) if c["biais"] else None


def _prepare_q8(c, seed):
    from troncons_amd import noyaux as K
    V = K.VueCarte.de
    w, x, b = _entrees_q8(c, seed)
    return {"sorte": "q8", "c": c, "noyaux": K.Noyaux.charger(), "w": V(w), "x": V(x),
            "biais": V(b) if b is not None else None, "y": torch.zeros(c["lignes"], device=CARTE)}


def _run_q8(s):
    c = s["c"]
    s["noyaux"].gemv_q8_0(s["w"], s["x"], s["biais"], s["y"], c["lignes"], c["colonnes"])
    return s["y"]


def _bornes(c):
    """[debut, fin) and the cache's slots: a windowed layer is some positions past its first wrap."""
    if c["anneau"]:
        fin = c["n"] + c["anneau"] // 2 + 3
        return fin - c["n"], fin, c["anneau"]
    return 0, c["n"], c["n"]


def _entrees_attention(c, seed):
    g = _gen(seed, 7)
    _, _, cases = _bornes(c)
    t = torch.float16 if c["cache"] == "f16" else torch.float32
    k, v = (_normale(g, cases, c["kv"], 64).to(t) for _ in range(2))
    return _normale(g, c["tetes"], 64), k, v, _normale(g, c["tetes"])


def _prepare_attention(c, seed):
    from troncons_amd import noyaux as K
    V = K.VueCarte.de
    q, k, v, puits = _entrees_attention(c, seed)
    debut, fin, _ = _bornes(c)
    n = K.Noyaux.charger()
    return {"sorte": "attention", "appel": n.attention if c["cache"] == "f16" else n.attention_kvf32, "q": V(q),
            "k": V(k), "v": V(v), "puits": V(puits), "sortie": torch.zeros(c["tetes"], 64, device=CARTE),
            "p": K.ParamsAttention(c["tetes"], c["kv"], 64, debut, fin, c["anneau"], 0.125, 0)}


def _run_attention(s):
    s["appel"](s["q"], s["k"], s["v"], s["puits"], s["sortie"], s["p"])
    return s["sortie"]


PAS = {"tetes": 64, "kv": 8, "couches": 2, "fenetre": 128, "eps": 1e-5}
JETON = 1234


def _modele_poids(c, seed):
    """The weights of the decode step's model as tensors: layers, embedding, output norm, head."""
    d, dq, dkv = c["d"], PAS["tetes"] * 64, PAS["kv"] * 64
    couches = []
    for l in range(PAS["couches"]):
        g = _gen(seed, 8, l)
        cases = PAS["fenetre"] if l % 2 == 0 else c["contexte"]
        couches.append({
            "attn_norm": 1.0 + _normale(g, d, sigma=0.1), "post_norm": 1.0 + _normale(g, d, sigma=0.1),
            "wq": _q8(g, dq, d), "bq": _normale(g, dq, sigma=0.1), "wk": _q8(g, dkv, d),
            "bk": _normale(g, dkv, sigma=0.1), "wv": _q8(g, dkv, d), "bv": _normale(g, dkv, sigma=0.1),
            "wo": _q8(g, d, dq), "bo": _normale(g, d, sigma=0.1), "puits": _normale(g, PAS["tetes"]),
            "routeur": _routeur(seed + 1000 + l, c["E"], d), "routeur_biais": _normale(g, c["E"], sigma=0.1),
            "experts": _experts({"d": d, "r": d}, seed + 2000 + l, c["E"]),
            "ck": _normale(g, cases, dkv).to(torch.float16), "cv": _normale(g, cases, dkv).to(torch.float16)})
    g = _gen(seed, 9)
    return couches, _q8(g, c["vocab"], d), 1.0 + _normale(g, d, sigma=0.1), _q8(g, c["vocab"], d)


def _prepare_pas(c, seed):
    from troncons_amd import modele as M
    from troncons_amd import noyaux as K
    couches, emb, norme, tete = _modele_poids(c, seed)
    d = c["d"]
    h = M.Hyper(couches=PAS["couches"], d=d, tetes=PAS["tetes"], tetes_kv=PAS["kv"], experts=c["E"], actifs=c["k"],
                vocab=c["vocab"], eps=PAS["eps"], rope=K.ParamsRope.gpt_oss(), fenetre=PAS["fenetre"],
                contexte=c["contexte"], dims=K.DimsExpert.de([d] * 3, [d] * 3), n_delta=1, n_codes=16)
    poids = []
    for w in couches:
        _, parts, _, freqs = _coder({"d": d, "r": d, "tuiles": "mixte"}, w["experts"])
        plat = {n: w[n].reshape(-1).cpu().numpy() for n in ("attn_norm", "post_norm", "wq", "bq", "wk", "bk", "wv",
                                                          "bv", "wo", "bo", "puits", "routeur_biais")}
        poids.append(M.PoidsCouche(routeur=w["routeur"].view(torch.int16).cpu().numpy().view(np.uint16),
                                   parties=[np.frombuffer(p, np.uint8) for p in parts],
                                   freqs=[[f for f in fj] for fj in freqs], **plat))
    m = M.Modele(h, poids, emb.reshape(-1).cpu().numpy(), norme.cpu().numpy(), tete.reshape(-1).cpu().numpy())
    for l, w in enumerate(couches):  # the positions before this step
        m.c[l]["ck"].copy_(w["ck"].reshape(-1).view(torch.uint8))
        m.c[l]["cv"].copy_(w["cv"].reshape(-1).view(torch.uint8))
    m.natif()
    return {"sorte": "pas", "m": m, "position": c["position"]}


def _run_pas(s):
    m = s["m"]
    m.pas_natif(JETON, s["position"])
    return {"logits": m.logits_natif(), "cle": [c["ck"] for c in m.c], "valeur": [c["cv"] for c in m.c]}


# ------------------------------------------------------------------------------------ work of a pass

def _octets_codes(c):
    """Bytes of one expert's coded streams: about 3.73 bits per weight, and the biases."""
    return sum(R * C * 3.73 / 8 + 4 * R for R, C in _formes(c))


def work(case):
    c, s = case, case["sorte"]
    if s in ("couche", "prefill", "expert"):
        poids3 = 3 * c["d"] * c["r"]
        if s == "expert":
            return {"bytes": _octets_codes(c) + 8 * c["d"], "flops": 2 * poids3}
        if s == "couche":
            return {"bytes": c["k"] * _octets_codes(c) + 2 * c["E"] * c["d"] + 12 * c["d"],
                    "flops": 2 * poids3 * c["k"] + 2 * c["E"] * c["d"]}
        n = min(c["E"], c["T"] * c["k"])
        return {"bytes": n * _octets_codes(c) + 12 * c["T"] * c["d"], "flops": 2 * poids3 * c["T"] * c["k"]}
    if s == "decoder":
        slot = sum(R * C * 17 / 32 + 4 * R for R, C in _formes(c))
        return {"bytes": c["n"] * (_octets_codes(c) + slot), "flops": 0}
    if s == "gemv":
        R, C = c["lignes"], c["colonnes"]
        return {"bytes": c["n"] * (R * C * 17 / 32 + 8 * R + 4 * C), "flops": 2 * c["n"] * R * C}
    if s == "q8":
        R, C = c["lignes"], c["colonnes"]
        return {"bytes": R * C * 34 / 32 + 8 * R + 4 * C, "flops": 2 * R * C}
    if s == "attention":
        o = 2 if c["cache"] == "f16" else 4
        return {"bytes": 2 * o * c["n"] * c["kv"] * 64 + 8 * c["tetes"] * 64, "flops": 4 * c["n"] * c["tetes"] * 64}
    d, dq, dkv = c["d"], PAS["tetes"] * 64, PAS["kv"] * 64
    att = (d * (dq + 2 * dkv) + dq * d) * 34 / 32
    kv = 4 * dkv * (PAS["fenetre"] + c["position"] + 1)
    mlp = c["k"] * _octets_codes({"d": d, "r": d})
    poids = PAS["couches"] * (2 * d * dq + 2 * d * dkv + 3 * c["k"] * d * d) + c["vocab"] * d
    return {"bytes": PAS["couches"] * (att + mlp) + kv + c["vocab"] * d * 34 / 32 + 4 * c["vocab"], "flops": 2 * poids}


# ------------------------------------------------------------------------------ tolerance and oracle

def tolerance(case):
    """Against 64 bits the calls measure 7e-8 to 2.4e-7 (relative 2-norm; two correct orders of the
    same f32 sums may be twice that apart), the decode step's logits 6e-7."""
    s = case["sorte"]
    if s == "decoder":
        return "exact"  # bytes
    if s == "pas":
        # a rounding of one layer's key or residual moves everything after it; the caches are f16 bits
        return {"rel": 4e-6, "max": 4e-5, "differ": 1e-4}
    return {"rel": 2e-6, "max": 2e-5}


def _swiglu64(g, u):
    g = g.clamp(max=7.0)
    return g * torch.sigmoid(1.702 * g) * (u.clamp(-7.0, 7.0) + 1.0)


def _mlp64(mats, x):
    """One expert over rows x [n][d] in 64 bits."""
    g, u = (x @ _valeurs64(q, e).T + b.double() for q, e, b in mats[:2])
    q, e, b = mats[2]
    return _swiglu64(g, u) @ _valeurs64(q, e).T + b.double()


def _topk64(lg, k):
    v, i = torch.sort(lg, descending=True, stable=True)
    return i[:k], torch.softmax(v[:k], -1)


def exact(case, seed):
    c, s = case, case["sorte"]
    if s == "couche":
        x = _jetons(c, seed)[0].double()
        idx, w = _topk64(_routeur(seed, c["E"], c["d"]).double() @ x, c["k"])
        mats = _experts(c, seed, c["E"])
        r = _normale(_gen(seed, 4), c["d"]).double()
        for e, p in zip(idx.tolist(), w):
            r = r + p * _mlp64(mats[e], x[None])[0]
        return {"residu": r, "indices": None, "poids": w, "controle": None}
    if s == "prefill":
        x = _x_prefill(c, seed).double()
        idx, w = (t.to(CARTE) for t in _routage(seed, c["T"], c["E"], c["k"]))
        r = _normale(_gen(seed, 4), c["T"], c["d"]).double()
        mats = _experts(c, seed, c["E"])
        for e in range(c["E"]):
            pos, place = (idx == e).nonzero(as_tuple=True)
            if len(pos):
                r.index_add_(0, pos, w[pos, place].double()[:, None] * _mlp64(mats[e], x[pos]))
        return {"residus": r, "controle": None}
    if s == "expert":
        x = _jetons(c, seed)[0].double()
        return {"sortie": _mlp64(_experts(c, seed, 1)[0], x[None])[0], "controle": None}
    if s == "gemv":
        return torch.stack([_valeurs64(q, e) @ x.double() + b.double() for q, e, b, x in _matrices(c, seed)])
    if s == "q8":
        w, x, b = _entrees_q8(c, seed)
        y = torch.cat([_q8_64(w[r:r + 16384]) @ x.double() for r in range(0, c["lignes"], 16384)])
        return y + b.double() if b is not None else y
    if s == "attention":
        q, k, v, puits = _entrees_attention(c, seed)
        debut, fin, cases = _bornes(c)
        pos = torch.arange(debut, fin, device=CARTE) % cases
        return _attention64(q.double(), k[pos].double(), v[pos].double(), puits.double())
    if s == "pas":
        return _pas64(c, seed)
    return None


def _attention64(q, k, v, puits):
    """q [tetes][64], k and v [n][kv][64] -> [tetes][64], the sink in the denominator."""
    groupe = q.shape[0] // k.shape[1]
    k, v = (t.repeat_interleave(groupe, 1) for t in (k, v))
    sc = (q[None] * k).sum(-1) * 0.125
    m = torch.maximum(sc.max(0).values, puits)
    e = torch.exp(sc - m)
    return (e[..., None] * v).sum(0) / (e.sum(0) + torch.exp(puits - m))[:, None]


def _rope64(x, position):
    """YaRN rotation of heads x [n][64], gpt-oss's parameters."""
    base, facteur, ctx, d = 150000.0, 32.0, 4096.0, 64
    i = torch.arange(d // 2, dtype=torch.float64, device=CARTE)
    theta = base ** (-2.0 * i / d)
    lo, hi = (0.5 * d * math.log(ctx / (2.0 * math.pi * b)) / math.log(base) for b in (32.0, 1.0))
    g = ((i - lo) / (hi - lo)).clamp(0.0, 1.0)
    angle = position * theta * ((1.0 - g) + g / facteur)
    m = 1.0 + 0.1 * math.log(facteur)
    co, si = torch.cos(angle) * m, torch.sin(angle) * m
    a, b = x[:, :d // 2], x[:, d // 2:]
    return torch.cat([a * co - b * si, b * co + a * si], -1)


def _norme64(x, w):
    return x / torch.sqrt((x * x).mean() + PAS["eps"]) * w.double()


def _pas64(c, seed):
    couches, emb, norme, tete = _modele_poids(c, seed)
    x = _q8_64(emb[JETON:JETON + 1])[0]
    cles, valeurs = [], []
    for l, w in enumerate(couches):
        h = _norme64(x, w["attn_norm"])
        q, k, v = (_q8_64(w["w" + n]) @ h + w["b" + n].double() for n in "qkv")
        q, k = _rope64(q.view(-1, 64), c["position"]), _rope64(k.view(-1, 64), c["position"])
        cases = w["ck"].shape[0]
        ck, cv = w["ck"].clone(), w["cv"].clone()
        ck[c["position"] % cases] = k.reshape(-1).to(torch.float16)
        cv[c["position"] % cases] = v.to(torch.float16)
        debut = max(c["position"] + 1 - PAS["fenetre"], 0) if l % 2 == 0 else 0
        pos = torch.arange(debut, c["position"] + 1, device=CARTE) % cases
        a = _attention64(q, ck[pos].double().view(len(pos), -1, 64), cv[pos].double().view(len(pos), -1, 64),
                         w["puits"].double())
        x = x + _q8_64(w["wo"]) @ a.reshape(-1) + w["bo"].double()
        h = _norme64(x, w["post_norm"])
        idx, p = _topk64(w["routeur"].double() @ h + w["routeur_biais"].double(), c["k"])
        for e, pe in zip(idx.tolist(), p):
            x = x + pe * _mlp64(w["experts"][e], h[None])[0]
        cles.append(None)
        valeurs.append(None)
    h = _norme64(x, norme)
    z = torch.cat([_q8_64(tete[r:r + 16384]) @ h for r in range(0, c["vocab"], 16384)])
    return {"logits": z, "cle": cles, "valeur": valeurs}
