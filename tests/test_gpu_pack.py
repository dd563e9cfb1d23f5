"""Weight packing: each source layout's kernel against the oracle's permutation, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import bsg_oracle as orc

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import bsa_mi355x as bsa  # noqa: E402


@pytest.mark.parametrize("layout", ["nk", "kn"])
@pytest.mark.parametrize("n,k,lead,skip", [
    (16, 64, 0, 0),      # one tile
    (1, 8, 0, 0),        # smallest
    (17, 72, 0, 0),      # a ragged second tile and block
    (250, 60, 4, 0),     # column count below 256, channels not a multiple of 8
    (259, 127, 9, 0),    # tails in both, padded rows
    (272, 320, 8, 16),   # rows of a wider matrix, aligned start
    (255, 192, 8, 1),    # rows of a wider matrix, unaligned start: the gather
    (520, 200, 3, 4),    # 8-byte start
])
def test_pack_sources_bit_exact(dev, layout, n, k, lead, skip):
    rng = np.random.default_rng(n * 1000 + k)
    w_nk = rng.normal(0, 0.02, size=(n, k)).astype(np.float16)
    want = orc.tile_permute(orc.pack_kmajor(w_nk)).view(np.uint16)
    src = torch.from_numpy(w_nk if layout == "nk" else np.ascontiguousarray(w_nk.T)).to(dev)
    # NaN around the matrix: anything read from there shows
    wide = torch.full((src.shape[0], skip + src.shape[1] + lead), float("nan"), dtype=torch.float16, device=dev)
    view = wide[:, skip:skip + src.shape[1]]
    view.copy_(src)
    for w in (src, view, view.view(torch.bfloat16)):
        # the packed tensor is likely to take the memory of this one, not the previous answer's
        del_me = torch.full(want.shape, float("nan"), dtype=torch.float16, device=dev)
        del del_me
        got = bsa.pack_weight(w, layout=layout).view(torch.float16).cpu().numpy()
        assert np.array_equal(got.view(np.uint16), want), (layout, n, k, tuple(w.stride()))
