"""Timed workloads over the library's public entry points: attention steps of a serving engine with cached keys.

A case names an entry point (`op`) and its sizes.  `listed()` holds one case per kind of call that an engine makes,
from the first tokens of a chat to the largest batch a card serves in one call; `draw(rng)` picks further sizes from
the same ranges.  Calls are eager, one call per pass, as a program issues them; outputs are the entry points' own.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "verified-metal-kernels_amd"))
import vmk                                                            # noqa: E402
from vmk.ops import dsa, dsa_project as proj, prefix, spec            # noqa: E402

HKV, D = 8, 128
MAX_BYTES = 540e6          # a drawn case reads no more than the largest listed one
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # one chat, its first thousand tokens: the smallest call, two launches and the host's own time
        dict(name="decode_chat", op="decode", B=1, L=1000, L_min=0, Hq=32, dtype="fp16"),
        # a long document decoded by one user: the whole card on one request (configuration D1)
        dict(name="decode_long", op="decode", B=1, L=65536, L_min=0, Hq=32, dtype="fp16"),
        # continuous batching: eight requests at different positions of caches of 8192 rows
        dict(name="decode_batch", op="decode", B=8, L=8192, L_min=500, Hq=32, dtype="bf16"),
        # the same over a page pool in the token-major layout (configuration D2n with requests of unequal length)
        dict(name="decode_pages", op="decode_paged", B=4, L=16384, L_min=1000, Hq=32, ps=64, layout="NHD",
             dtype="bf16"),
        # eight drafts of one request checked in one pass (the first benchmark shape of the verification op)
        dict(name="verify_chain", op="spec", B=1, L=8192, k=8, tree=False, dtype="fp16"),
        # trees of 64 drafts over long caches: the largest call (configuration C4)
        dict(name="verify_tree", op="spec", B=2, L=65536, k=64, tree=True, dtype="fp16"),
        # a system prompt shared by eight chats (configuration C1)
        dict(name="prefix_small", op="prefix", N=8, P=2048, S=256, S_min=0, Hq=32, dtype="fp16", outlier=False),
        # a long document shared by 64 requests, with answers of unequal length (configuration C2)
        dict(name="prefix_large", op="prefix", N=64, P=16384, S=2048, S_min=128, Hq=32, dtype="fp16", outlier=True),
        # a shared prefix in a page pool, a middling batch whose last pages are partly filled
        dict(name="prefix_pages", op="prefix_paged", N=24, P=8192, S=1000, S_min=100, Hq=32, ps=64, layout="HND",
             dtype="bf16", outlier=False),
        # sparse decode of one request at the shortest benchmark length
        dict(name="dsa_single", op="dsa", B=1, L=8192, L_min=0, dtype="bf16"),
        # sparse decode of four long requests (configuration C5)
        dict(name="dsa_batch", op="dsa", B=4, L=65536, L_min=0, dtype="fp16"),
        # the projections of four new tokens (configuration DP): every weight read once
        dict(name="dsa_project", op="dsa_project", B=4, L=4096, dtype="fp16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ones' ranges.  Sizes over their logarithm, odd ones as they fall; page-sized where a
    page table asks for it."""
    op = rng.choice(("decode", "decode", "decode_paged", "spec", "spec", "prefix", "prefix_paged", "dsa", "dsa",
                     "dsa_project"))
    dtype = rng.choice(("fp16", "bf16"))
    paged = dict(ps=rng.choice((32, 64, 128)), layout=rng.choice(("HND", "NHD")))
    while True:
        if op in ("decode", "decode_paged"):
            c = dict(op=op, B=_log(rng, 1, 32), L=_log(rng, 500, 65536), Hq=rng.choice((32, 32, 64)), dtype=dtype)
            c["L_min"] = rng.choice((0, max(1, c["L"] // 16)))
        elif op == "spec":
            c = dict(op=op, B=_log(rng, 1, 8), L=_log(rng, 1000, 65536), k=_log(rng, 2, 64), dtype=dtype)
            c["tree"] = c["k"] > 16 or rng.random() < 0.5
        elif op in ("prefix", "prefix_paged"):
            c = dict(op=op, N=_log(rng, 2, 64), P=_log(rng, 1000, 32768), S=_log(rng, 32, 2048),
                     Hq=rng.choice((32, 32, 64)), dtype=dtype, outlier=rng.random() < 0.3)
            c["S_min"] = rng.choice((0, max(1, c["S"] // 16)))
        elif op == "dsa":
            c = dict(op=op, B=_log(rng, 1, 8), L=_log(rng, 1000, 65536), dtype=dtype)
            c["L_min"] = rng.choice((0, max(1, c["L"] // 4)))
        else:
            c = dict(op=op, B=_log(rng, 1, 32), L=4096, dtype=dtype)
        if op.endswith("_paged"):
            c.update(paged)
            if op == "prefix_paged":
                c["P"] = -(-c["P"] // c["ps"]) * c["ps"]
        if _full_bytes(c) <= MAX_BYTES:
            return c


def _full_bytes(c):
    """Bytes of the keys and values that a case's caches hold (every length at its largest)."""
    if c["op"] in ("decode", "decode_paged", "spec"):
        return c["B"] * c["L"] * HKV * D * 4
    if c["op"] in ("prefix", "prefix_paged"):
        return (c["P"] + c["N"] * c["S"]) * HKV * D * 4
    return c["B"] * c["L"] * (dsa.DK + dsa.DI) * 2


def _lengths(case, seed):
    """Rows in use of each request: all of them, or uniform between the case's smallest and largest."""
    n, hi = (case["N"], case["S"]) if "N" in case else (case["B"], case["L"])
    lo = case.get("S_min", 0) or case.get("L_min", 0)
    if not lo:
        return None
    return np.random.default_rng([seed, 7]).integers(lo, hi + 1, n).astype(np.int32)


class _Draw:
    """Seeded normal values made on the card."""

    def __init__(self, case, seed):
        self.dt = DTYPES[case["dtype"]]
        self.g = torch.Generator(device="cuda").manual_seed(int(seed) * 2 + 1)

    def __call__(self, *shape, scale=1.0, dtype=None):
        x = torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32)
        return (x * scale if scale != 1.0 else x).to(dtype or self.dt)

    def outliers(self, k):
        """One value in a hundred twenty times larger, as key channels of trained models have them."""
        return torch.where(torch.rand(k.shape, generator=self.g, device="cuda") < 0.01, k * 20.0, k)


def _pool(rows, ps, layout, ids, num_pages):
    """Caches (n, Hkv, S, D) cut into pages of ps rows at the places `ids` (n, pages) of a pool."""
    n, h, s, d = rows.shape
    npg = ids.shape[1]
    full = torch.zeros(n, h, npg * ps, d, dtype=rows.dtype, device=rows.device)
    full[:, :, :s] = rows
    pages = full.view(n, h, npg, ps, d).transpose(1, 2).reshape(n * npg, h, ps, d)
    if layout == "NHD":
        pages = pages.transpose(1, 2)
    pool = torch.zeros((num_pages,) + tuple(pages.shape[1:]), dtype=rows.dtype, device=rows.device)
    pool[ids.reshape(-1).long()] = pages
    return pool


def _page_ids(seed, count):
    return torch.from_numpy(np.random.default_rng([seed, 9]).permutation(count).astype(np.int32)).cuda()


def _logical(case, seed):
    """A case's inputs with the caches in one piece: (q, the caches and masks by name, lengths or None)."""
    r, op = _Draw(case, seed), case["op"]
    n = _lengths(case, seed) if "B" not in case or op in ("decode", "decode_paged", "dsa") else None
    if op in ("decode", "decode_paged"):
        B, L = case["B"], case["L"]
        return dict(q=r(B, case["Hq"], D), k=r(B, HKV, L, D), v=r(B, HKV, L, D)), n
    if op == "spec":
        B, L, kd = case["B"], case["L"], case["k"]
        rng = np.random.default_rng([seed, 5])
        w = np.stack([spec.tree_bits_bounded(kd, rng) if case["tree"] else spec.chain_bits(kd) for _ in range(B)])
        return dict(q=r(B, kd, 32, D), k=r(B, HKV, L, D), v=r(B, HKV, L, D),
                    words=torch.from_numpy(w.view(np.int32)).cuda()), n
    if op in ("prefix", "prefix_paged"):
        N, P, S = case["N"], case["P"], case["S"]
        t = dict(q=r(N, case["Hq"], D), kp=r(HKV, P, D), vp=r(HKV, P, D), ks=r(N, HKV, S, D), vs=r(N, HKV, S, D))
        if case["outlier"]:
            t.update(kp=r.outliers(t["kp"]), ks=r.outliers(t["ks"]))
        return t, n
    if op == "dsa":
        B, L = case["B"], case["L"]
        return dict(q=r(B, dsa.H, dsa.DK), kv=r(B, L, dsa.DK), iq=r(B, dsa.HI, dsa.DI), ik=r(B, L, dsa.DI),
                    w=r(B, dsa.HI, scale=dsa.HI ** -0.5 * dsa.DI ** -0.5, dtype=torch.float32)), n
    B, L = case["B"], case["L"]
    weights = {}
    for name, shape in proj.WEIGHT_SHAPES.items():
        if name in proj.NORMS:
            weights[name] = (0.0 if name == "ik_norm_b" else 1.0) + r(*shape, scale=0.1, dtype=torch.float32)
        else:
            weights[name] = r(*shape, scale=shape[-1] ** -0.5)
    cos, sin = proj.rope_tables(L)
    pos = torch.from_numpy(np.random.default_rng([seed, 3]).integers(0, L, B).astype(np.int32)).cuda()
    return dict(x=r(B, proj.DIM), pos=pos, rope_cos=cos.cuda(), rope_sin=sin.cuda(), weights=weights,
                kv=r(B, L, proj.DC + proj.DR), ik=r(B, L, proj.DI)), None


def prepare(case, seed):
    t, n = _logical(case, seed)
    op, lens = case["op"], None if n is None else torch.from_numpy(n).cuda()
    if op == "decode_paged":
        ps, B = case["ps"], case["B"]
        mp = -(-case["L"] // ps)
        ids = _page_ids(seed, B * mp).view(B, mp)
        if lens is None:                       # caches that end inside their last page
            lens = torch.full((B,), case["L"], dtype=torch.int32, device="cuda")
        t = dict(q=t["q"], k_pages=_pool(t["k"], ps, case["layout"], ids, B * mp),
                 v_pages=_pool(t["v"], ps, case["layout"], ids, B * mp), page_table=ids, layout=case["layout"])
    elif op == "prefix_paged":
        ps, N = case["ps"], case["N"]
        npp, nsp = case["P"] // ps, -(-case["S"] // ps)
        total = npp + N * nsp
        ids = _page_ids(seed, total)
        if lens is None:
            lens = torch.full((N,), case["S"], dtype=torch.int32, device="cuda")
        pp, sp = ids[:npp].contiguous(), ids[npp:].view(N, nsp).contiguous()
        kp, vp = (_pool(t[a][None], ps, case["layout"], pp[None], total) for a in ("kp", "vp"))
        t = dict(q=t["q"], k_pages=kp + _pool(t["ks"], ps, case["layout"], sp, total),
                 v_pages=vp + _pool(t["vs"], ps, case["layout"], sp, total), prefix_pages=pp, suffix_pages=sp,
                 layout=case["layout"])
    if op in ("prefix", "prefix_paged"):
        t["slens"] = lens
    elif op in ("decode", "decode_paged", "dsa"):
        t["lens"] = lens
    return dict(op=op, args=t)


_CALLS = dict(decode=vmk.decode, decode_paged=vmk.decode_paged, spec=vmk.spec_verify, prefix=vmk.prefix_decode,
              prefix_paged=vmk.prefix_decode_paged, dsa=vmk.dsa_decode, dsa_project=vmk.dsa_project)


def run(state):
    op, t = state["op"], state["args"]
    out = _CALLS[op](**t)
    if op == "dsa_project":                     # the new rows of the caches are outputs too
        q, iq, w = out
        return dict(q=q, iq=iq, w=w, kv=t["kv"], ik=t["ik"])
    return out


def work(case):
    op = case["op"]
    # the lengths are drawn per seed; their mean stands for them
    mean = lambda lo, hi: (lo + hi) / 2 if lo else hi                 # noqa: E731
    if op in ("decode", "decode_paged"):
        n = case["B"] * mean(case["L_min"], case["L"])
        table = n / case["ps"] * 4 if op == "decode_paged" else 0
        return dict(bytes=n * HKV * D * 4 + 2 * case["B"] * case["Hq"] * D * 2 + table, flops=4 * n * case["Hq"] * D)
    if op == "spec":
        return dict(bytes=spec.algorithmic_bytes(case), flops=spec.flops(case))
    if op in ("prefix", "prefix_paged"):
        n = case["N"] * mean(case["S_min"], case["S"])
        rows = case["P"] + n
        table = rows / case["ps"] * 4 if op == "prefix_paged" else 0
        return dict(bytes=rows * HKV * D * 4 + 2 * case["N"] * case["Hq"] * D * 2 + table,
                    flops=4 * case["Hq"] * D * (case["N"] * case["P"] + n))
    if op == "dsa":
        n = [mean(case["L_min"], case["L"])] * case["B"]
        return dict(bytes=dsa.algorithmic_bytes(case, n), flops=dsa.flops(case, n))
    return dict(bytes=proj.algorithmic_bytes(case), flops=proj.flops(case))


def tolerance(case):
    # 16-bit probabilities, partial rows and results of 32-bit sums.  Measured over the listed cases and fourteen drawn
    # ones, the distance from the float64 result is at most 3.6e-4 in fp16 and 2.33e-3 in bf16 (largest difference
    # 1.9e-3 and 9.8e-3); the tolerance is four times that.
    return {"rel": 1.5e-3, "max": 8e-3} if case["dtype"] == "fp16" else {"rel": 9.5e-3, "max": 4e-2}


# ---------------------------------------------------------------------------------------- results in 64 bits
def _attend(q, k, v, mask=None, scale=D ** -0.5):
    """softmax(q k^T scale) v in float64; q (R, D), k/v (n, D), mask (R, n) or None.  Plain 2D products."""
    s = torch.mm(q.double(), k.double().t().contiguous()) * scale
    if mask is not None:
        s = s.masked_fill(~mask, float("-inf"))
    return torch.mm(torch.softmax(s, -1), v.double())


def exact(case, seed):
    t, n = _logical(case, seed)
    op = case["op"]
    if op in ("decode", "decode_paged", "spec"):
        q = t["q"] if op == "spec" else t["q"][:, None]                # (B, kd, Hq, D)
        B, kd, Hq, _ = q.shape
        L, G = case["L"], Hq // HKV
        out = torch.empty(B, kd, Hq, D, dtype=torch.float64, device="cuda")
        m = spec.draft_mask(t["words"], L, kd) if op == "spec" else None
        for b in range(B):
            u = L if n is None else int(n[b])
            mb = None if m is None else m[b][:, None].expand(kd, G, L).reshape(kd * G, L)
            for h in range(HKV):
                rows = q[b, :, h * G:(h + 1) * G].reshape(kd * G, D)
                out[b, :, h * G:(h + 1) * G] = _attend(rows, t["k"][b, h, :u], t["v"][b, h, :u], mb).view(kd, G, D)
        return out if op == "spec" else out[:, 0]
    if op in ("prefix", "prefix_paged"):
        N, Hq, G = case["N"], case["Hq"], case["Hq"] // HKV
        out = torch.empty(N, Hq, D, dtype=torch.float64, device="cuda")
        for h in range(HKV):
            kp, vp = t["kp"][h].double(), t["vp"][h].double()
            for i in range(N):
                u = case["S"] if n is None else int(n[i])
                k, v = torch.cat([kp, t["ks"][i, h, :u].double()]), torch.cat([vp, t["vs"][i, h, :u].double()])
                out[i, h * G:(h + 1) * G] = _attend(t["q"][i, h * G:(h + 1) * G], k, v)
        return out
    if op == "dsa":
        out = torch.empty(case["B"], dsa.H, dsa.DC, dtype=torch.float64, device="cuda")
        for b in range(case["B"]):
            u = case["L"] if n is None else int(n[b])
            s = torch.relu(torch.mm(t["ik"][b, :u].double(), t["iq"][b].double().t().contiguous()))
            s = torch.mv(s, t["w"][b].double())
            kv = t["kv"][b, torch.topk(s, min(u, dsa.TOPK)).indices].double()
            out[b] = _attend(t["q"][b], kv, kv[:, :dsa.DC].contiguous(), scale=dsa.SCALE)
        return out
    return _exact_project(t, DTYPES[case["dtype"]])


def _exact_project(t, dt):
    """The projections' definition (include/vmk.h) in float64, with its two roundings to the 16-bit type."""
    W = {k: v.double() for k, v in t["weights"].items()}
    x, p = t["x"].double(), t["pos"].long()
    c, s = t["rope_cos"].double()[p], t["rope_sin"].double()[p]

    def rms(a, w):
        return a / torch.sqrt(a.pow(2).mean(-1, keepdim=True) + proj.EPS) * w

    def rope(a, c, s):
        a0, a1 = a[..., 0::2], a[..., 1::2]
        return torch.stack([a0 * c - a1 * s, a0 * s + a1 * c], -1).flatten(-2)

    def rope_half(a, c, s):
        a0, a1 = a[..., :proj.DR // 2], a[..., proj.DR // 2:]
        return torch.cat([a0 * c - a1 * s, a0 * s + a1 * c], -1)

    lin = lambda a, w: torch.mm(a, w.t().contiguous())                # noqa: E731
    cq = rms(lin(x, W["wq_a"]), W["q_norm"]).to(dt).double()
    yq = lin(cq, W["wq_b"]).view(-1, proj.H, proj.DN + proj.DR)
    nope = yq[..., :proj.DN].to(dt).double()
    lat = torch.stack([lin(nope[:, h], W["w_uk"][h]) for h in range(proj.H)], 1)
    q = torch.cat([lat, rope(yq[..., proj.DN:], c[:, None], s[:, None])], -1)
    yi = lin(cq, W["iwq_b"]).view(-1, proj.HI, proj.DI)
    iq = torch.cat([rope_half(yi[..., :proj.DR], c[:, None], s[:, None]), yi[..., proj.DR:]], -1)
    w = lin(x, W["iw"]) * (proj.HI ** -0.5 * proj.DI ** -0.5)
    kvx, ikx = lin(x, W["wkv_a"]), lin(x, W["iwk"])
    ikx = torch.nn.functional.layer_norm(ikx, (proj.DI,), W["ik_norm_w"], W["ik_norm_b"], proj.EPS)
    kv, ik, b = t["kv"].double(), t["ik"].double(), torch.arange(len(p), device=p.device)
    kv[b, p] = torch.cat([rms(kvx[:, :proj.DC], W["kv_norm"]), rope(kvx[:, proj.DC:], c, s)], -1)
    ik[b, p] = torch.cat([rope_half(ikx[:, :proj.DR], c, s), ikx[:, proj.DR:]], -1)
    return dict(q=q, iq=iq, w=w, kv=kv, ik=ik)
