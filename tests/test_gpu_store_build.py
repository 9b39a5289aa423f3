"""Store builders of D = 128 rows at the edges of their tiles: codes, scales and plane words equal the oracle's bit for
bit, whichever of the workgroup shapes the size picks."""
import math

import numpy as np
import pytest
import torch

from fathom_amd import bitplane as bp
from oracle import fathom_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
SDT = {"f16": torch.float16, "f32": torch.float32, "bf16": torch.bfloat16}


def _edge_keys(BH, n, dtype, sdt, seed):
    """Random keys, and per channel the quotient's edges: multiples of the block's scale step and the representable
    values next to them, both signs; next to zero the smallest normal of 32-bit keys, whose denormals (a block that
    holds one divides) come in the second block."""
    g = torch.Generator().manual_seed(seed)
    K = torch.randn(BH, n, 128, generator=g) * torch.exp(2 * torch.randn(BH, 1, 128, generator=g))
    K = K.to(dtype)
    a = K.float().abs().reshape(BH, n, 128)[:, :64].amax(1)          # the first block's absmax,
    K[:, 0] = a.to(dtype)                                            # kept past the rows below
    step = a.to(SDT[sdt]).float() / 8
    m = torch.arange(-8, 9, dtype=torch.float32)
    at = (m[None, :, None] * step[:, None, :]).to(dtype)
    near = [at, torch.nextafter(at, torch.full_like(at, math.inf)), torch.nextafter(at, torch.full_like(at, -math.inf))]
    rows = torch.cat(near, 1)                                        # [BH, 51, 128]
    rows = torch.where(rows.float().abs() <= a[:, None], rows, torch.zeros((), dtype=dtype))
    if n >= 128:
        K[:, 64] = a.to(dtype)
        K[:, 69:120] = rows                      # with 32-bit denormals
    if dtype == torch.float32:
        rows = torch.where((rows != 0) & (rows.abs() < 2.0 ** -126), 2.0 ** -126 * rows.sign(), rows)
    K[:, 5:56] = rows[:, :min(51, n - 5)]
    return K


@pytest.mark.parametrize("sdt", ["f16", "bf16"])
def test_edge_keys_reach_the_division_free_path(sdt):
    """The first block of 32-bit edge keys has neither denormals nor scales that divide, and its quotients touch every
    integer from both sides; the second has denormals."""
    K = _edge_keys(1, 256, torch.float32, sdt, 3)
    tiny = (K != 0) & (K.abs() < 2.0 ** -126)
    assert not tiny[:, :64].any() and tiny[:, 64:128].any()
    s = K[:, :64].abs().amax(1).to(SDT[sdt]).float() / 8
    assert (8 * s >= 2.0 ** -14).all() and (8 * s <= 65504).all()
    x, m = K[0, 5:56].double() / s[0].double(), torch.arange(-8.0, 9.0, dtype=torch.float64)
    inside = (m[:, None] * s[0].double()).abs() < K[0, :64].abs().amax(0).double() * (1 - 2.0 ** -20)
    for i in range(17):
        at, up, down = x[i], x[17 + i], x[34 + i]
        assert ((up > m[i]) | ~inside[i]).all() and ((down < m[i]) | ~inside[i]).all()
        assert ((at - m[i]).abs()[inside[i]] <= 2.0 ** -22 * 8).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("sdt", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("BH,n,sub", [(1, 64, 16), (2, 1000, 3), (3, 65536 + 33, 16), (9, 7777, 64), (1, 1049000, 0),
                                      (2, 530000, 5)])
def test_build_equals_oracle_at_tile_edges(BH, n, sub, sdt, dtype, monkeypatch):
    print(f"[build] {BH}x{n} sub={sub} {sdt} {dtype}", flush=True)
    nb = -(-n // 64)
    monkeypatch.setattr(bp, "SUB", sub or nb)
    K = _edge_keys(BH, n, dtype, sdt, n)
    if n > 500000:                          # the large shapes' rows repeat their head: the oracle is slow
        K[:, 8192:] = K[:, :8192].repeat(1, -(-n // 8192), 1)[:, 8192:n]
    st = bp.PlaneStore(K.to(DEV), scale_dtype=SDT[sdt])
    lean = bp.PlaneStore(K.to(DEV), scale_dtype=SDT[sdt], keep_code=False)
    torch.cuda.synchronize()
    assert torch.equal(st.planes_k, lean.planes_k) and torch.equal(st.scales_k, lean.scales_k)
    assert torch.equal(bp.unpack_planes(bp.pack_planes(st.code), n), st.code)
    pl, sc = bp.to_superblocks(bp.pack_planes(st.code), st.scales_blk)
    assert torch.equal(pl, st.planes_k)
    if sdt == "f16":
        assert torch.equal(sc, st.scales_k)
    keep = min(n, 8192 if n > 500000 else n)
    head = K[:, :keep].float().numpy()
    code_r, sc_r = O.quantise_u4(head, sdt)
    np.testing.assert_array_equal(st.code[:, :keep].cpu().numpy(), code_r)
    np.testing.assert_array_equal(st.scales_blk[:, :-(-keep // 64)].float().cpu().numpy(), sc_r)
    tail = (n - 1) // 64 * 64               # the last, ragged block
    code_t, sc_t = O.quantise_u4(K[:, tail:].float().numpy(), sdt)
    np.testing.assert_array_equal(st.code[:, tail:].cpu().numpy(), code_t)
    np.testing.assert_array_equal(st.scales_blk[:, -1:].float().cpu().numpy(), sc_t)
    planes = bp.pack_planes(st.code[:, tail:].contiguous())
    np.testing.assert_array_equal(planes.cpu().numpy().view(np.uint64), O.pack_planes(code_t))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("BH,n,cut", [(1, 1, 0), (3, 257, 0), (2, 1000, 1)])
def test_klt_centering_equals_torch(BH, n, cut, dtype):
    """One rounding per element, as the conversion and the subtraction: equal bit for bit, whatever the alignment."""
    from fathom_amd.klt import _centered
    print(f"[klt center] {BH}x{n} {dtype}", flush=True)
    flat = torch.randn(BH * n * 128 + cut, generator=torch.Generator().manual_seed(n)).to(dtype).to(DEV)
    K = flat[cut:].view(BH, n, 128)             # cut = 1: rows off the vector loads' alignment
    mu = torch.randn(BH, 128, generator=torch.Generator().manual_seed(1)).to(DEV)
    assert torch.equal(_centered(K, mu), K.float() - mu[:, None, :])
    assert torch.equal(_centered(K.transpose(0, 1).contiguous().transpose(0, 1), mu), K.float() - mu[:, None, :])


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,D", [(33, 1), (1001, 12), (180000, 100), (700001, 24), (560000, 128)])
def test_klt_centering_of_other_widths(n, D, dtype):
    """Widths that the vector forms take for some key types only, and rows longer than one step of the grid."""
    from fathom_amd.klt import _centered
    print(f"[klt center] n={n} D={D} {dtype}", flush=True)
    g = torch.Generator(DEV).manual_seed(D)
    K = torch.randn(2, n, D, device=DEV, generator=g).to(dtype)
    mu = torch.randn(2, D, device=DEV, generator=g)
    assert torch.equal(_centered(K, mu), K.float() - mu[:, None, :])
