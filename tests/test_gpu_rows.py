"""Kind 8 (more than 64 batch rows) against the oracle, at the edges of its tiles, its ring and its
row groups."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import assert_close, case, to_dev
from oracle import bsg_oracle as orc

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import bsa_mi355x as bsa  # noqa: E402
from bsa_mi355x import tuning  # noqa: E402
from bsa_mi355x.select import select_gemm_packed  # noqa: E402


@pytest.mark.parametrize("cols", [32, 48, 64, 96])
@pytest.mark.parametrize("bt,k,n", [
    (65, 64, 16),       # one subtile, one block, the last row group all but empty
    (128, 1000, 523),   # ragged last block and subtile, odd output width
    (129, 712, 1040),   # a second row group of one row
    (300, 4096, 1610),  # three row groups
])
def test_rows_kernel(dev, cols, bt, k, n):
    nblk = orc.nblk_of(k)
    x, w_nk, _ = case(cols + bt, bt, k, n, 1, "normal")
    # rows past bt and columns past K lie in NaN
    xw = torch.full((bt + 130, k + 64), float("nan"), dtype=torch.float16, device=dev)
    xt = xw[:bt, :k]
    xt.copy_(to_dev(x, dev))
    packed = bsa.pack_weight(to_dev(w_nk, dev))
    p = bsa.Plan(1, cols, 8, 4, 128, 8)
    rng = np.random.default_rng(bt)
    for na in sorted({a for a in (1, 2, 3, 4, 5, 7, 8, 9, nblk) if a <= nblk}):
        idx = rng.permutation(nblk)[:na].astype(np.int32)
        print(f"rows kernel cols={cols} bt={bt} K={k} N={n} na={na}", flush=True)
        out = torch.full((bt, n), float("nan"), dtype=torch.float16, device=dev)
        used = bsa.gemm_packed(xt, packed, n, to_dev(idx, dev), out, plan=p, sort_list=True)
        assert used.as_tuple() == p.as_tuple()
        assert_close(out.float().cpu().numpy(), orc.gemm_ref64(x, w_nk, np.sort(idx)), f"kind 8 {cols} na={na}")
    # skipped entries (no such block) among the active ones, a device count, a bitmap, every block
    ref = orc.gemm_ref64(x, w_nk, np.arange(nblk))
    ids = np.repeat(np.arange(nblk), 2).astype(np.int32)
    ids[1::2] = np.where(np.arange(nblk) % 2, -1, nblk)
    # (every output starts as NaN: memory reused from the loop above may hold the right answer)
    out = torch.full_like(out, float("nan"))
    cnt = torch.tensor([2 * nblk], dtype=torch.int32, device=dev)
    bsa.gemm_packed(xt, packed, n, to_dev(np.r_[ids, ids], dev), out, plan=p, num_active_dev=cnt)
    bit = torch.ones(nblk, dtype=torch.uint8, device=dev)
    out_b, out_d = torch.full_like(out, float("nan")), torch.full_like(out, float("nan"))
    bsa.gemm_packed(xt, packed, n, None, out_b, bitmap=bit, plan=p)
    bsa.gemm_packed(xt, packed, n, None, out_d, plan=p)
    for o in (out, out_b, out_d):
        assert_close(o.float().cpu().numpy(), ref, f"kind 8 {cols} every block")
    assert torch.equal(out_b.view(torch.int16), out_d.view(torch.int16))


def test_rows_kernel_bf16_and_stale_slots(dev):
    """bf16, and: a launch that leaves Inf in every ring stage does not show in the next one's slots
    past the list (they load zeros)."""
    bt, k, n = 200, 640, 4096
    x, w_nk, idx = case(9, bt, k, n, 5, "normal")
    p = bsa.Plan(1, 96, 8, 4, 128, 8)
    xb, wb = torch.from_numpy(x).to(torch.bfloat16), torch.from_numpy(w_nk).to(torch.bfloat16)
    packed = bsa.pack_weight(wb.to(dev))
    every = torch.arange(orc.nblk_of(k), dtype=torch.int32, device=dev)
    out = torch.full((bt, n), float("nan"), dtype=torch.bfloat16, device=dev)
    bsa.gemm_packed(torch.full((bt, k), float("inf"), dtype=torch.bfloat16, device=dev), packed, n, every, out, plan=p)
    out.fill_(float("nan"))
    bsa.gemm_packed(xb.to(dev), packed, n, to_dev(idx, dev), out, plan=p)
    ref = orc.gemm_ref64(xb.float().numpy(), wb.float().numpy(), idx)
    got = out.float().cpu().numpy()
    # the output's own rounding: half a unit in the last place of 8 bits, 2^-9 of the value
    assert np.linalg.norm(got - ref) <= 2.0 ** -9 * np.linalg.norm(ref) * 1.05


@pytest.mark.parametrize("bt,k,n,na", [(65, 4096, 11008, 31), (256, 4096, 4096, 31), (130, 11008, 4096, 40),
                                       (192, 4096, 4096, 20), (100, 512, 2048, 8)])
def test_many_rows_through_the_public_calls(dev, bt, k, n, na):
    """The plans that tuning.many_rows_plan gives, through the drop-in, the selection and the 2-D
    entry (which keeps its own tiles)."""
    x, w_nk, idx = case(bt, bt, k, n, na, "normal")
    xt, wt = to_dev(x, dev).view(bt, 1, k), to_dev(w_nk, dev)
    out = torch.full((bt, 1, n), float("nan"), dtype=torch.float16, device=dev)
    bsa._prepacked_block_sparse_gemm_from_active_blocks(xt, wt, to_dev(idx[::-1].copy(), dev), out, cache_prefix="rows")
    assert_close(out.view(bt, n).float().cpu().numpy(), orc.gemm_ref64(x, w_nk, idx), "drop-in")
    want = tuning.many_rows_plan(bt, n)
    assert bsa.resolve_plan(bt, n, orc.nblk_of(k), na, dev).as_tuple() == want.as_tuple()
    out.fill_(float("nan"))
    sel, _ = bsa.select_sparse_gemm(xt, wt, out, na, cache_prefix="rows")
    kept = sel.cpu().numpy()
    assert np.array_equal(kept, orc.select_topk_l1(x, na))
    assert_close(out.view(bt, n).float().cpu().numpy(), orc.gemm_ref64(x, w_nk, kept), "selection")
    nb = np.arange(0, n // 64, 3, dtype=np.int32)
    out.fill_(0)
    bsa._prepacked_block_sparse_gemm_2d_from_active_blocks(xt, wt, to_dev(idx, dev), to_dev(nb, dev), out,
                                                           cache_prefix="rows")
    cols = (nb[:, None] * 64 + np.arange(64)).reshape(-1)
    got = out.view(bt, n).float().cpu().numpy()
    assert_close(got[:, cols], orc.gemm_ref64(x, w_nk, idx)[:, cols], "2-D")
    assert not np.delete(got, cols, axis=1).any()


@pytest.mark.parametrize("bt,k,n,na,select_kind", [
    (160, 4096, 4096, 64, 4),    # kind 4 over a long list: split two ways, three row groups
    (320, 4160, 2050, 50, 4),    # split three ways, five row groups, odd width of the last subtile
    (72, 1024, 11016, 12, 7),    # a GEMM on kind 8, a selection on kind 7
    (128, 4096, 6912, 31, 7),    # four subtiles per unit on kind 7
    (320, 1024, 8200, 9, 8),     # kind 8 over two rounds of 64 columns
])
def test_many_rows_plans_by_list_length_and_selection(dev, bt, k, n, na, select_kind):
    """The automatic plans past 64 rows that depend on the list's length or on a selection."""
    nblk = orc.nblk_of(k)
    x, w_nk, idx = case(bt, bt, k, n, na, "normal")
    xt, packed = to_dev(x, dev), bsa.pack_weight(to_dev(w_nk, dev))
    pl = tuning.many_rows_plan(bt, n, na)
    out = torch.full((bt, n), float("nan"), dtype=torch.float16, device=dev)
    print(f"many rows bt={bt} K={k} N={n} na={na} plan={pl.as_tuple()}", flush=True)
    bsa.gemm_packed(xt, packed, n, to_dev(idx, dev), out, plan=pl)
    assert_close(out.float().cpu().numpy(), orc.gemm_ref64(x, w_nk, idx), "list")
    assert bsa.resolve_plan(bt, n, nblk, na, dev, select=True).kind == select_kind
    out.fill_(float("nan"))
    sel, _ = select_gemm_packed(xt, packed, n, na, out)
    kept = sel.cpu().numpy()
    assert np.array_equal(kept, orc.select_topk_l1(x, na))
    assert_close(out.float().cpu().numpy(), orc.gemm_ref64(x, w_nk, kept), "selection")
