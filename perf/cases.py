"""Performance cases of the bit-plane key scan: what a user's program has this framework do.

A serving program packs a layer's keys once (`build`, `pack`), then for every generated token plans, scans, selects and
attends (`decode`: one call with the index and the rows in HBM; `klt`: the rotated store of models without QK-norm;
`select`: the separate calls, for selections too long for one workgroup; `host`: index and rows in pinned host memory).
`scores` and `chan4` are the drop-in forms that return score rows, the second over the 4-bit baseline store.

Keys follow the benchmark's distribution: lognormal channel scales with outlier channels, normal tokens, and planted keys
near the queries.  Shapes are the benchmark's five configurations, the ragged and small shapes of its tests, and the
ranges between them."""
import math
import weakref

import torch

from fathom_amd import bitplane as bp
from fathom_amd import klt
from fathom_amd import offload as off

BLK, D = 64, 128
SINK, LOCAL = 4, 32
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def listed():
    return [
        # The smallest call: one short conversation, one KV head, one query head. Launches and latency.
        {"name": "decode_short", "kind": "decode", "BH": 1, "G": 1, "n": 1000, "k": 128, "budget": 48.0, "sub": 16},
        # One of 36 layers of a decode step, batch 4 x 8 KV heads, at 32k tokens.
        {"name": "decode_32k_batch4", "kind": "decode", "BH": 32, "G": 4, "n": 32768, "k": 512, "budget": 64.0, "sub": 16},
        # One layer of a single 128k conversation.
        {"name": "decode_128k", "kind": "decode", "BH": 8, "G": 4, "n": 131072, "k": 512, "budget": 48.0, "sub": 16},
        # The headline layer: 1M tokens, the store in the whole-sequence layout.
        {"name": "decode_1m", "kind": "decode", "BH": 8, "G": 4, "n": 1048576, "k": 512, "budget": 48.0, "sub": 0},
        # Batch 2 x 4 KV heads with 7 query heads each, 2048 tokens selected, on the rotated store.
        {"name": "klt_128k_g7", "kind": "klt", "BH": 8, "G": 7, "n": 131072, "k": 2048, "budget": 48.0, "sub": 16},
        # A selection longer than one workgroup ranks, over a ragged length.
        {"name": "select_300k_k4096", "kind": "select", "BH": 8, "G": 4, "n": 300007, "k": 4096, "budget": 56.0, "sub": 16},
        # The drop-in chain that returns score rows, one budget per row, deep plans, a ragged length.
        {"name": "scores_50k", "kind": "scores", "BH": 8, "G": 4, "n": 50021, "k": 512, "budget": 92.0, "sub": 16},
        # The store of a 128k prefill of one layer.
        {"name": "build_128k", "kind": "build", "BH": 8, "n": 131072, "dtype": "bf16", "sub": 16, "keep_code": True,
         "klt": False},
        # The rotated store of a ragged 20k prefill; only the store is kept.
        {"name": "build_klt_20k", "kind": "build", "BH": 8, "n": 20011, "dtype": "f16", "sub": 16, "keep_code": False,
         "klt": True},
        # The drop-in packers one by one, for a caller that keeps the logical planes: one head of float32 keys.
        {"name": "pack_16k_f32", "kind": "pack", "BH": 1, "n": 16384, "dtype": "f32", "sub": 16},
        # Index and rows in pinned host memory, read over PCIe, with tokens newer than the index on the device.
        {"name": "host_128k", "kind": "host", "BH": 8, "G": 4, "n": 131072, "k": 512, "budget": 48.0, "recent": 17,
         "copy": False},
        # The 4-bit baseline store with a quarter of the channels listed.
        {"name": "chan4_128k", "kind": "chan4", "BH": 8, "G": 4, "n": 131072, "nact": 32, "sub": 16},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "klt", "select", "scores", "build", "build", "pack", "host", "chan4"])
    BH = rng.choice([1, 2, 4, 8, 8, 16, 32])
    G = rng.choice([1, 2, 4, 4, 5, 7, 8, 12])
    budget = float(rng.randint(40, 92))
    sub = rng.choice([16, 16, 64, 0])
    dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
    if kind == "decode":
        n = _log(rng, 400, min(1048576, 8388608 // BH))
        G = min(G, 4) if BH * n > 1 << 21 else G
        return {"kind": kind, "BH": BH, "G": G, "n": n, "k": min(_log(rng, 64, 2048), n // 2), "budget": budget,
                "sub": sub}
    if kind == "klt":
        n = _log(rng, 4000, min(262144, 2097152 // BH))
        return {"kind": kind, "BH": BH, "G": G, "n": n, "k": min(_log(rng, 128, 2048), n // 2), "budget": budget,
                "sub": sub}
    if kind == "select":
        n = _log(rng, 20000, min(1048576, 2097152 // BH))
        return {"kind": kind, "BH": BH, "G": min(G, 8), "n": n, "k": min(_log(rng, 1000, 8192), n // 2),
                "budget": budget, "sub": sub}
    if kind == "scores":
        n = _log(rng, 1000, min(262144, 2097152 // BH))
        return {"kind": kind, "BH": BH, "G": G, "n": n, "k": min(_log(rng, 64, 2048), n // 2), "budget": budget,
                "sub": sub}
    if kind == "build":
        return {"kind": kind, "BH": BH, "n": _log(rng, 1000, min(262144, 1048576 // BH)), "dtype": dtype, "sub": sub,
                "keep_code": rng.random() < 0.5, "klt": rng.random() < 0.25}
    if kind == "pack":
        return {"kind": kind, "BH": BH, "n": _log(rng, 1000, min(131072, 262144 // BH)), "dtype": dtype, "sub": sub}
    if kind == "host":
        return {"kind": kind, "BH": min(BH, 8), "G": min(G, 8), "n": _log(rng, 20000, 1048576 // max(8, BH)),
                "k": _log(rng, 128, 1024), "budget": budget, "recent": rng.randint(1, 31), "copy": rng.random() < 0.3}
    return {"kind": kind, "BH": BH, "G": G, "n": _log(rng, 1000, min(262144, 1048576 // BH)),
            "nact": rng.choice([8, 16, 24, 32, 48, 77]), "sub": sub}


# --------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _keys(case, seed):
    """Keys [BH, n, D], queries [BH, G, D] and the calibration variance [BH, D] of one layer."""
    gen = _gen(seed)
    BH, n, G = case["BH"], case["n"], case.get("G", 4)
    dtype = DTYPES[case.get("dtype", "bf16")]
    sigma = torch.exp(torch.randn(BH, D, generator=gen, device="cuda"))
    outliers = torch.rand(BH, D, generator=gen, device="cuda").topk(4, 1).indices
    sigma.scatter_(1, outliers, sigma.gather(1, outliers) * 10.0)
    q = torch.randn(BH, G, D, generator=gen, device="cuda")
    K = torch.empty(BH, n, D, dtype=dtype, device="cuda")
    planted, stride = torch.arange(32, device="cuda"), (n - SINK - 64) // 32
    heads = planted % G
    for b in range(BH):
        x = torch.randn(n, D, generator=gen, device="cuda") * sigma[b]
        at = SINK + planted * stride + torch.randint(stride, (32,), generator=gen, device="cuda")
        x[at] = 0.8 * q[b, heads] + 0.05 * sigma[b] * torch.randn(32, D, generator=gen, device="cuda")
        K[b] = x
    var = torch.stack([K[b, 16:].float().var(0) for b in range(BH)])
    return K, q, var


def _rows(case, seed):
    gen = _gen(seed + 7)
    V = torch.empty(case["BH"], case["n"], D, dtype=torch.bfloat16, device="cuda")
    for b in range(case["BH"]):
        V[b] = torch.randn(case["n"], D, generator=gen, device="cuda")
    return V


def _recent(case, seed):
    gen = _gen(seed + 8)
    return torch.randn(2, case["BH"], case["recent"], D, generator=gen, device="cuda").bfloat16()


def _basis(K, q):
    """The rotated store's calibration from the first tokens, as the user's calibration run leaves it: mean, basis
    (columns), variances, in the order of the components' share of the score variance."""
    Kc = K[:, 16:4112].double().cpu()
    mu = Kc.mean(1)
    Kc = Kc - mu[:, None]
    lam, V = torch.linalg.eigh(Kc.transpose(1, 2) @ Kc / Kc.shape[1])
    lam = lam.clamp_min(0)
    w = (q.double().cpu() @ V).square().mean(1) * lam
    order = w.argsort(-1, descending=True)
    V = V.gather(2, order[:, None].expand_as(V))
    return {"mu": mu.float().cuda(), "Vt": V.float().contiguous().cuda(), "lam": lam.gather(1, order).float().cuda(),
            "w": w.gather(1, order).float().cuda()}


def _budgets(case):
    """One budget per row, up to the case's."""
    return torch.linspace(max(40.0, case["budget"] - 16), case["budget"], case["BH"]).round()


def _active(case, q, var):
    """The listed channels of the baseline store: the largest gains of each row."""
    gain = (q.square() * var[:, None]).sum(1)
    return torch.zeros(case["BH"], D, dtype=torch.bool, device="cuda").scatter_(1, gain.topk(case["nact"], 1).indices,
                                                                               True)


def _with_sub(sub, n, make):
    """A store built with superblocks of `sub` blocks (0: one superblock per row)."""
    keep = bp.SUB
    bp.SUB = sub or math.ceil(n / BLK)
    try:
        return make()
    finally:
        bp.SUB = keep


class _Pinned:
    """Host copies that are given back when the state goes."""

    def __init__(self):
        self.held = []
        weakref.finalize(self, _Pinned._free, self.held)

    @staticmethod
    def _free(held):
        torch.cuda.synchronize()
        for p in held:
            off.free_host(p)

    def put(self, t):
        _, dev, p = off.host_mapped(t)
        self.held.append(p)
        return dev


def prepare(case, seed):
    kind, n = case["kind"], case["n"]
    K, q, var = _keys(case, seed)
    sub = case.get("sub", 16)
    s = {"case": case, "kind": kind, "q": q}
    if kind == "build":
        s.update(K=K, params=_basis(K, q) if case["klt"] else None)
        return s
    if kind == "pack":
        s.update(K=K)
        return s
    if kind == "chan4":
        s.update(store=_with_sub(sub, n, lambda: bp.Chan4Store(K, keep_code=False)), active=_active(case, q, var))
        return s
    if kind == "host":
        pin = _Pinned()
        rec = _recent(case, seed)
        store = _with_sub(0 if case["copy"] else 64, n, lambda: bp.PlaneStore(K, keep_code=False))
        if case["copy"]:
            s["staging"] = off.staging_store(store)
            store, held = off.host_store(store)
            pin.held.extend(held)
        else:
            store.planes32, store.scales_k = pin.put(store.planes_k), pin.put(store.scales_k)
            del store.planes_k
        s.update(pin=pin, store=store, K=pin.put(K), V=pin.put(_rows(case, seed)), Krec=rec[0], Vrec=rec[1], var=var)
        return s
    if kind == "klt":
        params = _basis(K, q)
        s.update(store=_with_sub(sub, n, lambda: klt.KLTPlaneStore(K, params, keep_code=False)))
    else:
        s.update(store=_with_sub(sub, n, lambda: bp.PlaneStore(K, keep_code=False)),
                 g=(q.square() * var[:, None]).sum(1))
    if kind == "scores":
        s["budgets"] = _budgets(case)
    else:
        s.update(K=K, V=_rows(case, seed))
    return s


def run(s):
    c, kind, q = s["case"], s["kind"], s["q"]
    n, k = c["n"], c.get("k")
    if kind == "decode":
        idx, out = s["store"].plan_scan_topk_attention(q, s["g"], c["budget"], k, s["K"], s["V"], SINK, LOCAL)
        return {"idx": idx, "out": out}
    if kind == "klt":
        plan = s["store"].plan(q, c["budget"])
        idx = s["store"].scan_topk(q, plan, k, SINK, LOCAL)
        out, _ = off.gather_attention(q, idx, n, s["K"], s["V"], n)
        return {"t": plan["t"], "idx": idx, "out": out}
    if kind == "select":
        plan = bp.make_plan(s["g"], c["budget"])
        idx = s["store"].scan_topk(q, plan, k, SINK, LOCAL)
        return {"t": plan["t"], "idx": idx, "out": off.gather_attn(q, s["K"], s["V"], idx)}
    if kind == "scores":
        plan = bp.make_plan(s["g"], s["budgets"])
        scores = s["store"].scan(q, plan)
        return {"t": plan["t"], "scores": scores, "idx": bp.sink_local_topk(scores, k, SINK, LOCAL)}
    if kind == "host":
        m = n + c["recent"]
        if c["copy"]:
            plan = bp.make_plan((q.square() * s["var"][:, None]).sum(1), c["budget"])
            off.copy_index(s["store"], s["staging"], plan)
            idx = s["staging"].scan_topk(q, plan, k, SINK, LOCAL, m=m)
            out, seen = off.gather_attention(q, idx, n, s["K"], s["V"], n, s["Krec"], s["Vrec"])
            return {"t": plan["t"], "idx": idx, "out": out, "seen": seen}
        r = off.select_and_gather(s["store"], q, s["var"], c["budget"], k, s["K"], s["V"], SINK, LOCAL, m, s["Krec"],
                                  s["Vrec"])
        return {"t": r["plan"]["t"], "idx": r["idx"], "K": r["K"], "V": r["V"], "seen": r["n_unique"]}
    if kind == "chan4":
        act, nact = bp.channel_list(s["active"])
        return {"act": act, "nact": nact, "scores": s["store"].scan(q, act, nact)}
    if kind == "build":
        K = s["K"]
        if c["klt"]:
            st = _with_sub(c["sub"], n, lambda: klt.KLTPlaneStore(K, s["params"], keep_code=c["keep_code"]))
        else:
            st = _with_sub(c["sub"], n, lambda: bp.PlaneStore(K, keep_code=c["keep_code"]))
        return {"planes": st.planes_k, "scales": st.scales_k, "scales_blk": st.scales_blk, "code": st.code}
    code, scales = bp.quantise_u4(s["K"])
    planes = bp.pack_planes(code)
    planes_k, scales_k = _with_sub(c["sub"], n, lambda: bp.to_superblocks(planes, scales))
    return {"code": code, "scales": scales, "planes": planes, "planes_k": planes_k, "scales_k": scales_k}


# --------------------------------------------------------------------------- the least that a pass moves and computes
def work(case):
    kind, BH, n = case["kind"], case["BH"], case["n"]
    G, k = case.get("G", 0), case.get("k", 0)
    nblk = math.ceil(n / BLK)
    if kind in ("build", "pack"):
        size = {"bf16": 2, "f16": 2, "f32": 4}[case["dtype"]]
        blocks = math.ceil(nblk / case["sub"]) * case["sub"] if case["sub"] else nblk
        store = BH * blocks * D * 34  # four planes of 8 bytes and the scale of each block and channel
        by = BH * n * D * size + store + BH * nblk * D * 2
        fl = 4.0 * BH * n * D  # absmax, divide, floor, pack
        if kind == "pack":  # codes and logical planes are results too, and each call reads the one before it
            by += 2 * BH * n * D + 2 * BH * nblk * D * 32 + BH * nblk * D * 2
        else:
            by += BH * n * D if case["keep_code"] else 0
            if case["klt"]:
                fl += 2.0 * BH * n * D * D
        return {"bytes": by, "flops": fl}
    if kind == "chan4":
        return {"bytes": BH * nblk * case["nact"] * 34 + BH * G * n * 4, "flops": 2.0 * BH * G * n * case["nact"]}
    bits = float(_budgets(case).mean()) if kind == "scores" else case["budget"]
    # planes read, and the scales of the listed channels: about 0.62 channels for each plane at these distributions
    index = BH * nblk * bits * (8 + 2 * 0.62)
    by = index + BH * G * k * 8
    fl = 2.0 * BH * G * n * bits
    if kind == "scores":
        by += BH * G * n * 4
    else:
        rows = BH * min(n, G * k)  # the heads of a row share few of their selected tokens
        by += rows * 2 * D * 2
        fl += 4.0 * BH * G * k * D
        if kind == "host":
            by += index if case["copy"] else 0  # staged in HBM, then scanned there
            by += BH * G * k * 2 * D * 2
        else:
            by += BH * G * D * 4
    return {"bytes": by, "flops": fl}


def tolerance(case):
    kind = case["kind"]
    if kind == "pack" or (kind == "build" and not case["klt"]):
        return "exact"
    if kind == "host" and not case["copy"]:
        return "exact"  # the rows are copies, in the order of the selection
    if kind == "build":
        # float32 rotations in another order move a value over a code's edge, or a scale by its last bit, now and then
        return {"rel": 4e-5, "differ": 1e-3}
    if kind in ("scores", "chan4"):
        return {"rel": 2.5e-6, "differ": 2e-3}  # 1e-7 to 6e-7 off the sums in 64 bits
    # 1e-6 off the sums in 64 bits where the same tokens are selected, 1e-4 where a score's last bits decide which of
    # two nearly equal tokens is the last one
    return {"rel": 4e-4, "differ": 2e-3}


# --------------------------------------------------------------------------- the same in 64 bits
def _plan64(g, budgets):
    lg = torch.log2(g.double().clamp_min(1e-30))
    lo, hi = torch.full_like(lg[:, :1], -60.0), torch.full_like(lg[:, :1], 60.0)
    B = torch.as_tensor(budgets, dtype=torch.float64).to(g.device).expand(g.shape[0])[:, None]
    for _ in range(30):
        mid = (lo + hi) / 2
        over = ((lg - mid) / 2).round().clamp(0, 4).sum(1, keepdim=True) > B
        lo, hi = torch.where(over, mid, lo), torch.where(over, hi, mid)
    return ((lg - hi) / 2).round().clamp(0, 4)


def _dequant64(x, t):
    """The t-bit values of one row's keys x [n, D], each block of 64 with its absmax in half precision."""
    n = x.shape[0]
    x = torch.nn.functional.pad(x.double(), (0, 0, 0, -n % BLK)).view(-1, BLK, D)
    a = x.abs().amax(1, keepdim=True).clamp_min(1e-8).half().double()
    code = (x / (a / 8)).floor_().clamp_(-8, 7).add_(8)
    half = torch.exp2(t - 1)
    val = ((code / torch.exp2(4 - t)).floor_() + 0.5 - half) * (a / half)
    return torch.where(t > 0, val, torch.zeros((), dtype=torch.float64, device=x.device)).view(-1, D)[:n]


def _topk64(s, k, m):
    n = s.shape[-1]
    s = s.clone()
    s[:, :SINK] = -math.inf
    s[:, m - LOCAL:] = -math.inf
    top = s.topk(k - SINK - LOCAL, -1).indices
    fixed = torch.cat([torch.arange(SINK), torch.arange(m - LOCAL, m)]).to(s.device)
    return torch.cat([top, fixed.expand(s.shape[0], -1)], 1)


def _attend64(q, K, V, idx):
    Ks, Vs = K[idx].double(), V[idx].double()
    p = ((Ks * q.double()[:, None]).sum(-1) * D ** -0.5).softmax(-1)
    return (p[..., None] * Vs).sum(1)


def exact(case, seed):
    kind, n, k = case["kind"], case["n"], case.get("k")
    K, q, var = _keys(case, seed)
    if kind in ("build", "pack"):
        x = K
        if kind == "build" and case["klt"]:
            P = _basis(K, q)
            x = torch.stack([(K[b].double() - P["mu"][b].double()) @ P["Vt"][b].double() for b in range(case["BH"])])
        a = torch.stack([torch.nn.functional.pad(x[b].double(), (0, 0, 0, -n % BLK)).view(-1, BLK, D).abs().amax(1)
                         for b in range(case["BH"])]).clamp_min(1e-8)
        sub = case["sub"] or a.shape[1]
        a_sb = torch.nn.functional.pad(a, (0, 0, 0, -a.shape[1] % sub)).view(case["BH"], -1, sub, D).transpose(2, 3)
        if kind == "pack":
            return {"code": None, "scales": a, "planes": None, "planes_k": None, "scales_k": a_sb.contiguous()}
        return {"planes": None, "scales": a_sb.contiguous(), "scales_blk": a, "code": None}
    if kind == "chan4":
        full = torch.full((D,), 4.0, dtype=torch.float64, device="cuda")
        active = _active(case, q, var)
        return {"act": None, "nact": None, "scores": torch.stack(
            [(q[b].double() * active[b]) @ _dequant64(K[b], full).T for b in range(case["BH"])])}
    if kind == "host" and not case["copy"]:
        return None
    basis = _basis(K, q) if kind == "klt" else None
    if basis:
        qr = torch.bmm(q.double(), basis["Vt"].double())
        gain = (qr.square() * basis["lam"].double()[:, None]).sum(1)
    else:
        qr, gain = q.double(), (q.square() * var[:, None]).sum(1)
    t = _plan64(gain, _budgets(case) if kind == "scores" else case["budget"])
    if kind != "scores":
        V = _rows(case, seed)
        rec = _recent(case, seed) if kind == "host" else None
    m = n + case.get("recent", 0)
    scores, outs = [], []
    for b in range(case["BH"]):
        x = (K[b].double() - basis["mu"][b].double()) @ basis["Vt"][b].double() if basis else K[b]
        s = qr[b] @ _dequant64(x, t[b]).T
        if kind == "scores":
            scores.append(s)
            continue
        Kb, Vb = (K[b], V[b]) if rec is None else (torch.cat([K[b], rec[0, b]]), torch.cat([V[b], rec[1, b]]))
        outs.append(_attend64(q[b], Kb, Vb, _topk64(s, k, m)))
    if kind == "scores":
        return {"t": None, "scores": torch.stack(scores), "idx": None}
    out = {"idx": None, "out": torch.stack(outs)}
    if kind != "decode":
        out["t"] = None
    if kind == "host":
        out["seen"] = None
    return out
