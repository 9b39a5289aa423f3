"""Selection over 16-token group maxima, rows of up to 131072 tokens, at the edges of its shapes: equal to the top-k of the
scan's scores (itself checked against the oracle), whatever the order of the scores, the layout of the store and the
route a length takes on either side of the limits."""
import math

import numpy as np
import pytest
import torch

from fathom_amd import bitplane as bp
from fathom_amd import offload as off
from fathom_amd import workloads as W
from oracle import fathom_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def _oracle_topk(scores, k, sink, local, m):
    s = scores.cpu().numpy()
    return torch.from_numpy(O.sink_local_topk(s, k, sink, local, m=m))


@pytest.mark.parametrize("BH,G,n,k,sub,extra", [(2, 4, 32769, 512, 16, 0), (1, 4, 131072, 2084, 0, 9), (2, 3, 131071, 100, 64, 0),
                                                (1, 7, 131072, 512, 16, 0), (2, 5, 32833, 2084, 64, 31),
                                                (1, 8, 100001, 300, 0, 5), (3, 1, 65600, 512, 64, 0),
                                                (1, 4, 131073, 512, 16, 0), (2, 7, 140000, 600, 64, 0), (24, 4, 33333, 512, 16, 0)])
def test_fused_selection_at_its_limits(BH, G, n, k, sub, extra, monkeypatch):
    print(f"[group-select] {BH}x{G} n={n} k={k} sub={sub}", flush=True)
    monkeypatch.setattr(bp, "SUB", sub or -(-n // 64))
    x = W.synth_layer(BH, n, G, seed=n % 97, device=DEV, kdtype=torch.bfloat16)
    g = ((x["q"] ** 2) * x["var"][:, None, :]).sum(1)
    st = bp.PlaneStore(x["K"])
    for budget in (48.0, 110.0):  # plans held in registers, and in register groups
        plan = bp.make_plan(g, budget)
        scores = st.scan(x["q"], plan)
        want = _oracle_topk(scores, k, 4, 32, n + extra)
        got = st.scan_topk(x["q"], plan, k, 4, 32, m=n + extra)
        idx, t = st.plan_scan_topk(x["q"], g, budget, k, 4, 32, m=n + extra, return_t=True)
        assert torch.equal(got.cpu(), want) and torch.equal(idx, got) and torch.equal(t, plan["t"])
        if extra == 0:
            i2, out = st.plan_scan_topk_attention(x["q"], g, budget, k, x["K"], x["K"], 4, 32)
            ref, _ = off.gather_attention(x["q"], got, n, x["K"], x["K"], n)
            assert torch.equal(i2, got) and torch.equal(out, ref)


def test_planned_call_with_nothing_to_select():
    """k = sink + local: the fixed positions, and the plan's depths where asked for, on short and long rows."""
    print("[group-select] k = sink + local", flush=True)
    for n in (5000, 140000):
        x = W.synth_layer(2, n, 4, seed=1, device=DEV, kdtype=torch.bfloat16)
        g = ((x["q"] ** 2) * x["var"][:, None, :]).sum(1)
        st = bp.PlaneStore(x["K"], keep_code=False)
        idx, t = st.plan_scan_topk(x["q"], g, 48.0, 36, 4, 32, return_t=True)
        assert torch.equal(t, bp.make_plan(g, 48.0)["t"])
        want = torch.cat([torch.arange(4), torch.arange(n - 32, n)]).expand(2, 4, 36)
        assert torch.equal(idx.cpu(), want) and torch.equal(st.plan_scan_topk(x["q"], g, 48.0, 36, 4, 32).cpu(), want)


@pytest.mark.parametrize("n", [65536, 131072, 140001])
@pytest.mark.parametrize("G", [4, 7])
def test_ties_and_masks(n, G):
    """Every score equal, and scores that fall or rise along the row (every group of one end reaches the threshold; past
    the limit the sample misleads the chain and its rows are rescanned)."""
    print(f"[group-select ties] n={n} G={G}", flush=True)
    for kind in ("equal", "falling", "rising"):
        K = torch.zeros(1, n, 128, device=DEV)
        if kind != "equal":
            K[0, :, 0] = torch.linspace(3, -3, n, device=DEV) * (1 if kind == "falling" else -1)
            K[0, :, 1] = torch.randn(n, device=DEV, generator=torch.Generator(DEV).manual_seed(2)) * 0.01
        st = bp.PlaneStore(K, keep_code=False)
        q = torch.zeros(1, G, 128, device=DEV)
        q[..., 0], q[:, 1::2, 1] = 1.0, 1.0
        gain = torch.ones(1, 128, device=DEV)
        gain[0, 0], gain[0, 1] = 1000.0, 10.0
        plan = bp.make_plan(gain, 6.0)
        scores = st.scan(q, plan)
        got = st.scan_topk(q, plan, 2000, 4, 32)
        assert torch.equal(got.cpu(), _oracle_topk(scores, 2000, 4, 32, n)), kind
        idx, t = st.plan_scan_topk(q, gain, 6.0, 2000, 4, 32, return_t=True)
        assert torch.equal(idx, got) and torch.equal(t, plan["t"]), kind


@pytest.mark.parametrize("n,G", [(40000, 4), (131072, 6), (200000, 4)])
def test_host_resident_staged_scan_equals_hbm(n, G, monkeypatch):
    """Superblocks of 64 blocks in mapped host memory: the staged passes give the same indices, whatever the plan."""
    print(f"[group-select host] n={n} G={G}", flush=True)
    monkeypatch.setattr(bp, "SUB", 64)
    x = W.synth_layer(2, n, G, seed=3, device=DEV, kdtype=torch.bfloat16)
    g = ((x["q"] ** 2) * x["var"][:, None, :]).sum(1)
    st = bp.PlaneStore(x["K"], keep_code=False)
    plans = [bp.make_plan(g, b) for b in (20.0, 48.0, 64.0, 100.0)]
    want = [st.scan_topk(x["q"], p, 512, 4, 32) for p in plans]
    ref = [bp.sink_local_topk(st.scan(x["q"], p), 512, 4, 32) for p in plans]
    _, pl, h1 = off.host_mapped(st.planes_k)
    _, sc, h2 = off.host_mapped(st.scales_k)
    try:
        st.planes32, st.scales_k = pl, sc
        got = [st.scan_topk(x["q"], p, 512, 4, 32) for p in plans]
        torch.cuda.synchronize()
    finally:
        off.free_host(h1)
        off.free_host(h2)
    for a, b, c in zip(got, want, ref):
        assert torch.equal(a, b) and torch.equal(a, c)


@pytest.mark.parametrize("n,G", [(40000, 4), (40000, 6), (200000, 4)])
def test_staged_scan_of_plans_without_units(n, G, monkeypatch):
    """Superblocks of 64 blocks (staged tiles): rows whose plan lists no channel -- budget 0, and a zero query row among
    others -- give the indices of the direct scan over superblocks of 16."""
    print(f"[group-select empty plan] n={n} G={G}", flush=True)
    x = W.synth_layer(2, n, G, seed=4, device=DEV, kdtype=torch.bfloat16)
    q = x["q"].clone()
    q[1] = 0.0                              # a padded batch slot: every gain at the floor
    g = ((q ** 2) * x["var"][:, None, :]).sum(1)
    got = {}
    for sub in (16, 64):
        monkeypatch.setattr(bp, "SUB", sub)
        st = bp.PlaneStore(x["K"], keep_code=False)
        for budget in (0.0, 48.0, torch.tensor([0.5, 48.0])):
            plan = bp.make_plan(g, budget)
            idx, t = st.plan_scan_topk(q, g, budget, 512, 4, 32, return_t=True)
            assert torch.equal(st.scan_topk(q, plan, 512, 4, 32), idx) and torch.equal(t, plan["t"])
            got.setdefault(sub, []).append(idx)
    assert all(torch.equal(a, b) for a, b in zip(got[16], got[64]))
    first = torch.cat([torch.arange(4, 480), torch.arange(4), torch.arange(n - 32, n)])  # every score equal
    assert torch.equal(got[64][0].cpu(), first.expand(2, G, 512))


@pytest.mark.parametrize("n,G,k", [(160000, 4, 512), (160000, 7, 512), (300011, 4, 2084)])
@pytest.mark.parametrize("sub", [16, 64])
def test_rescan_of_a_misled_first_pass(n, G, k, sub, monkeypatch):
    """The sampled tiles hold one high score per 16-token group, the others none: fewer than kk keys reach the first
    pass's threshold (checked on the scores), and the row is rescanned with the lower one -- after a direct first pass
    (superblocks of 16) and a staged one (of 64), with the plan given and made in the sample pass."""
    print(f"[rescan] n={n} G={G} k={k} sub={sub}", flush=True)
    monkeypatch.setattr(bp, "SUB", sub)
    kk, tile = k - 36, 1024
    ntiles = -(-n // tile)
    want = max(32, -(-2 * k // 64), -(-32 * n // (5 * k * tile)))
    S = -(-ntiles // min(want, 64))                       # every S-th tile is sampled
    gen = torch.Generator().manual_seed(n)
    tok = torch.arange(0, ntiles, S)[:, None] * tile + torch.arange(64) * 16
    tok = (tok + torch.randint(0, 16, tok.shape, generator=gen)).flatten()
    tok = tok[(tok >= 4) & (tok < n - 32)]
    K = torch.randn(2, n, 128, generator=gen) * 0.01
    sampled = sum(min(tile, n - t * S * tile) for t in range(-(-ntiles // S)))
    r_hi = min(max(1, (5 * kk * sampled + 2 * n - 1) // (2 * n)), kk)
    high = (r_hi + kk) // 2                               # high scores: the threshold's rank and more, fewer than kk
    K[:, tok[torch.randperm(len(tok), generator=gen)[:high]], 0] = 3.0 + torch.rand(2, high, generator=gen)
    K = K.to(DEV)
    q = torch.zeros(2, G, 128, device=DEV)
    q[..., 0], q[:, 1::2, 1] = 1.0, 0.5
    gain = torch.ones(2, 128, device=DEV)
    gain[:, 0], gain[:, 1] = 1000.0, 10.0
    st = bp.PlaneStore(K, keep_code=False)
    plan = bp.make_plan(gain, 6.0)
    scores = st.scan(q, plan)
    sc = scores.clone()
    sc[..., :4], sc[..., n - 32:] = -math.inf, -math.inf
    grp = torch.nn.functional.pad(sc, (0, ntiles * tile - n), value=-math.inf).view(2, G, ntiles, 64, 16)[:, :, ::S].amax(-1)
    t_hi = grp.flatten(2).topk(r_hi, -1).values[..., -1:]
    assert bool(((sc >= t_hi).sum(-1) < kk).any()) and r_hi < high < kk
    want_idx = _oracle_topk(scores, k, 4, 32, n)
    assert torch.equal(st.scan_topk(q, plan, k, 4, 32).cpu(), want_idx)
    idx, t = st.plan_scan_topk(q, gain, 6.0, k, 4, 32, return_t=True)
    assert torch.equal(idx.cpu(), want_idx) and torch.equal(t, plan["t"])
    i2, out = st.plan_scan_topk_attention(q, gain, 6.0, k, K.bfloat16(), K.bfloat16(), 4, 32)
    ref, _ = off.gather_attention(q, idx, n, K.bfloat16(), K.bfloat16(), n)
    assert torch.equal(i2, idx) and torch.equal(out, ref)


def _score_rows(kind, rows, n, seed):
    rng = np.random.default_rng(seed)
    s = rng.standard_normal((rows, n)).astype(np.float32)
    if kind == "equal":
        s[:] = -1.5
    elif kind == "specials":
        for v in (np.nan, np.inf, -np.inf, 0.0, -0.0, 3e38, -3e38, 1e-45):
            s[:, rng.integers(0, n, max(1, n // 20))] = v
    elif kind == "outliers":
        s[:, rng.integers(0, n, 3)] = 1e30
        s[0] = np.abs(s[0])
    elif kind == "lowest":  # more -inf than finite scores
        s[:, rng.random(n) < 0.8] = -np.inf
    elif kind == "steps":
        s = np.round(s * 2) / 2
    return s


@pytest.mark.parametrize("n,k,sink,local,extra", [
    (64, 60, 4, 32, 0), (50, 50, 0, 0, 0), (1000, 1000, 4, 32, 0), (1024, 128, 4, 32, 3), (1025, 700, 0, 1, 0),
    (4096, 2084, 4, 32, 0), (4097, 257, 1, 0, 0), (4097, 300, 4, 32, 40), (8192, 548, 4, 32, 0), (8193, 549, 4, 32, 0),
    (8193, 512, 4, 32, 0), (16384, 1060, 4, 32, 0), (32192, 2048, 4, 32, 0), (32768, 2084, 4, 32, 0), (32768, 2048, 0, 0, 0),
    (32769, 512, 4, 32, 0), (40003, 2084, 4, 32, 31), (131072, 512, 4, 32, 0), (131071, 2084, 4, 32, 0),
    (131073, 512, 4, 32, 0)])
def test_score_rows_at_every_route(n, k, sink, local, extra):
    print(f"[row-select] n={n} k={k} sink={sink} local={local}", flush=True)
    for i, kind in enumerate(("normal", "equal", "specials", "outliers", "lowest", "steps")):
        s = _score_rows(kind, 3, n, n + i)
        got = bp.sink_local_topk(torch.from_numpy(s).to(DEV), k, sink, local, m=n + extra).cpu().numpy()
        np.testing.assert_array_equal(got, O.sink_local_topk(s, k, sink, local, m=n + extra), err_msg=kind)


@pytest.mark.parametrize("n,k", [(700, 128), (3000, 512), (6000, 512), (8192, 600), (20000, 1500), (30001, 2048)])
def test_fused_selection_of_short_rows(n, k):
    print(f"[row-select fused] n={n} k={k}", flush=True)
    for BH, G in ((1, 1), (2, 5), (24, 4)):
        x = W.synth_layer(BH, n, G, seed=n, device=DEV, kdtype=torch.bfloat16)
        g = ((x["q"] ** 2) * x["var"][:, None, :]).sum(1)
        st = bp.PlaneStore(x["K"], keep_code=False)
        plan = bp.make_plan(g, 48.0)
        want = _oracle_topk(st.scan(x["q"], plan), k, 4, 32, n)
        assert torch.equal(st.scan_topk(x["q"], plan, k, 4, 32).cpu(), want)
        idx, out = st.plan_scan_topk_attention(x["q"], g, 48.0, k, x["K"], x["K"], 4, 32)
        ref, _ = off.gather_attention(x["q"], idx, n, x["K"], x["K"], n)
        assert torch.equal(idx.cpu(), want) and torch.equal(out, ref)


@pytest.mark.parametrize("n,k,extra", [(2100, 2085, 0), (4097, 4097, 0), (8192, 4096, 0), (8193, 8228, 40), (30000, 4096, 0),
                                       (32768, 8000, 0), (32769, 8228, 0), (131072, 4000, 0), (131073, 2085, 0),
                                       (200001, 8228, 7), (524289, 3000, 0), (1048576, 2100, 0), (1048577, 2100, 0)])
def test_wide_selection_at_every_route(n, k, extra):
    print(f"[wide-select] n={n} k={k}", flush=True)
    rows = 2 if n < 300000 else 1
    for i, kind in enumerate(("normal", "equal", "specials", "outliers", "lowest", "steps")):
        s = _score_rows(kind, rows, n, n + i)
        got = bp.sink_local_topk(torch.from_numpy(s).to(DEV), k, 4, 32, m=n + extra).cpu().numpy()
        np.testing.assert_array_equal(got, O.sink_local_topk(s, k, 4, 32, m=n + extra), err_msg=kind)


@pytest.mark.parametrize("n,k", [(900, 400), (4096, 512), (8192, 600), (30000, 2048), (32768, 512), (32769, 2084), (131072, 1000),
                                 (131071, 2084), (8193, 4096), (32768, 8228), (131072, 4000), (131073, 2085), (300007, 4096),
                                 (524288, 6136)])
def test_more_candidates_than_one_sort_takes(n, k):
    """Rows whose first bound leaves more scores than one sort (or the LDS list) takes: neighbouring tokens alike, two and
    three levels of equal scores with the cut inside one, a ramp, and levels whose lowest group of tokens is the row's last."""
    print(f"[narrowed] n={n} k={k}", flush=True)
    rng = np.random.default_rng(n + k)
    t = np.arange(n)
    knots = -(-n // 256) + 2
    smooth = np.stack([np.interp(t, np.arange(knots) * 256, rng.standard_normal(knots)) for _ in range(2)])
    kk = k - 36
    two = np.where(rng.random((2, n)) < 1.5 * kk / n, 2.0, 1.0)
    three = np.where(rng.random((2, n)) < 0.3 * kk / n, 5.0, np.where(rng.random((2, n)) < 0.9, 1.0, -3.0))
    tail = np.where(t >= n - n // 3, 1.0 + t % 7 * 1e-6, -1.0)[None].repeat(2, 0)
    for s in (smooth + rng.standard_normal((2, n)) * 1e-4, two, three, t[None] * 1e-3 - 5.0, tail):
        s = np.ascontiguousarray(s, dtype=np.float32)
        got = bp.sink_local_topk(torch.from_numpy(s).to(DEV), k, 4, 32).cpu().numpy()
        np.testing.assert_array_equal(got, O.sink_local_topk(s, k, 4, 32))


@pytest.mark.parametrize("BH,G,n,k", [(2, 4, 4000, 512), (2, 4, 20000, 512), (2, 3, 131072, 512), (2, 7, 131071, 512),
                                      (1, 7, 131072, 2048), (1, 4, 300007, 4096)])
def test_fused_selection_of_clustered_and_equal_rows(BH, G, n, k):
    """The same in the fused scan's score orders, and the attention over such rows."""
    print(f"[narrowed fused] {BH}x{G} n={n} k={k}", flush=True)
    gen = torch.Generator(DEV).manual_seed(n)
    knots = -(-n // 300) + 1
    K = torch.randn(BH, knots, 128, device=DEV, generator=gen).repeat_interleave(300, 1)[:, :n]
    K = (K + 0.05 * torch.randn(BH, n, 128, device=DEV, generator=gen)).to(torch.bfloat16).contiguous()
    q = torch.randn(BH, G, 128, device=DEV, generator=gen)
    g = (q ** 2).sum(1)
    q[-1, -1] = 0.0                               # every score of this head equal
    st = bp.PlaneStore(K, keep_code=False)
    plan = bp.make_plan(g, 48.0)
    want = _oracle_topk(st.scan(q, plan), k, 4, 32, n)
    assert torch.equal(st.scan_topk(q, plan, k, 4, 32).cpu(), want)
    idx, out = st.plan_scan_topk_attention(q, g, 48.0, k, K, K, 4, 32)
    ref, _ = off.gather_attention(q, idx, n, K, K, n)
    assert torch.equal(idx.cpu(), want) and torch.equal(out, ref)


@pytest.mark.parametrize("BH,G,n,k", [(2, 5, 200001, 4096), (1, 4, 40000, 3000), (1, 8, 9000, 8228), (1, 4, 600000, 5000)])
def test_wide_fused_selection(BH, G, n, k):
    print(f"[wide-select fused] {BH}x{G} n={n} k={k}", flush=True)
    x = W.synth_layer(BH, n, G, seed=n % 31, device=DEV, kdtype=torch.bfloat16)
    g = ((x["q"] ** 2) * x["var"][:, None, :]).sum(1)
    st = bp.PlaneStore(x["K"], keep_code=False)
    plan = bp.make_plan(g, 56.0)
    want = _oracle_topk(st.scan(x["q"], plan), k, 4, 32, n)
    assert torch.equal(st.scan_topk(x["q"], plan, k, 4, 32).cpu(), want)
    assert torch.equal(st.plan_scan_topk(x["q"], g, 56.0, k, 4, 32).cpu(), want)


@pytest.mark.parametrize("BH,G,k", [(1, 1, 1), (1, 3, 33), (2, 4, 128), (2, 4, 129), (1, 5, 500), (8, 4, 512), (3, 2, 513),
                                    (1, 7, 1024), (2, 4, 1030), (14, 7, 2048), (1, 2, 4200), (40, 3, 1500)])
def test_attention_splits(BH, G, k):
    """Splits of 128 and 512 positions, merged over up to 4, 8 and more of them, against softmax attention in float64 on
    the CPU: float32 products and sums over k terms stay within 1e-5 of the largest value."""
    print(f"[attention] {BH}x{G} k={k}", flush=True)
    n = 5000
    gen = torch.Generator().manual_seed(k)
    K, V = (torch.randn(BH, n, 128, generator=gen).bfloat16() for _ in range(2))
    q = torch.randn(BH, G, 128, generator=gen)
    idx = torch.randint(0, n, (BH, G, k), generator=gen)
    idx[0, 0, :1] = -1                           # a zero row
    out, _ = off.gather_attention(q.to(DEV), idx.to(DEV), n, K.to(DEV), V.to(DEV), n)
    for b in range(BH):
        for h in range(G):
            rows = idx[b, h]
            Ks, Vs = K[b, rows.clamp_min(0)].double(), V[b, rows.clamp_min(0)].double()
            Ks[rows < 0], Vs[rows < 0] = 0.0, 0.0
            ref = torch.softmax(Ks @ q[b, h].double() * 128 ** -0.5, 0) @ Vs
            assert (out[b, h].cpu().double() - ref).abs().max() <= 1e-5 * ref.abs().max().clamp_min(1.0)


def test_single_split_rounds_no_more_than_merged_ones():
    """512 positions in one split of 16 waves: mean relative error against float64 over 384 fixed heads.  Four merged splits
    of four waves give 2.49e-7 on them, sixteen partial sums added in a row 2.58e-7; the limit lies between."""
    print("[attention] single-split error", flush=True)
    err = []
    for seed in range(6):
        for mult in (1.0, 3.0):
            gen = torch.Generator().manual_seed(seed * 1000 + 512)
            K, V = (torch.randn(8, 6000, 128, generator=gen).bfloat16() for _ in range(2))
            q = torch.randn(8, 4, 128, generator=gen) * mult
            idx = torch.randint(0, 6000, (8, 4, 512), generator=gen)
            out, _ = off.gather_attention(q.to(DEV), idx.to(DEV), 6000, K.to(DEV), V.to(DEV), 6000)
            bh = torch.arange(8)[:, None, None]
            w = torch.softmax((K[bh, idx].double() * q.double()[:, :, None]).sum(-1) * 128 ** -0.5, -1)
            ref = (w[..., None] * V[bh, idx].double()).sum(2)
            err.append(((out.cpu().double() - ref).norm(dim=-1) / ref.norm(dim=-1)).mean())
    assert torch.stack(err).mean() < 2.53e-7


@pytest.mark.parametrize("BH", [1, 3, 64, 65, 200, 257])
def test_host_budgets_equal_device_budgets(BH):
    """Per-row budgets from the host, of any dtype and shape that expands, reused at once by the caller."""
    print(f"[budgets] BH={BH}", flush=True)
    g = torch.rand(BH, 128, generator=torch.Generator().manual_seed(BH)).to(DEV) * 100
    for host in (torch.linspace(40, 92, BH), torch.arange(BH) % 50 + 40, torch.tensor([48.5], dtype=torch.float64)):
        want = bp.make_plan(g, host.to(DEV))["t"]
        mine = host.clone()
        got = bp.make_plan(g, mine)
        mine.zero_()
        assert torch.equal(got["t"], want)
    with pytest.raises(RuntimeError):
        bp.make_plan(g, torch.ones(BH + 1 if BH > 1 else 2))
