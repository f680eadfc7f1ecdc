"""The expansion of a whole tile per LDS read (csrc/rank_whole.hpp): the quantised operators with up to eight weight rows.

Every weight row picks a single channel (keys) or token (values), so that a result is one dequantised element and nothing
else: it must be the oracle's number, whichever of the 64 positions of whichever tile it is.  Tiles are full, empty, hold one
element at every position, only their first or only their second half, and everything in between at random."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu
D = 128


def rows(rng, tokens):
    keep = rng.random((1, tokens, D)) < rng.random((1, 1, D))
    t = np.arange(tokens)
    for c in range(64):                       # key tiles of one element; value tiles too where tokens allow
        keep[0, :, c] = t % 64 == c
    keep[0, :, 64], keep[0, :, 65] = True, False
    keep[0, :, 66], keep[0, :, 67] = t % 64 < 32, t % 64 >= 32
    last = tokens - 5
    keep[0, last], keep[0, last + 1] = True, False
    keep[0, last + 2], keep[0, last + 3] = np.arange(D) % 64 < 32, np.arange(D) % 64 >= 32
    return np.where(keep, rng.standard_normal((1, tokens, D)), 0).astype(np.float16)


@pytest.mark.parametrize("groups,n_rows", [(1, 1), (4, 1), (5, 1), (1, 8)])
@pytest.mark.parametrize("bit", [2, 4, 8])
def test_every_element(groups, n_rows, bit):
    from mustafar_amd import compression_quant as cq
    from mustafar_amd._lib import check, lib
    rng = np.random.default_rng(10 * groups + n_rows + bit)
    tokens, rpk = 128, groups * n_rows
    x = rows(rng, tokens)
    g = torch.from_numpy(x).cuda()
    L, st = lib(), torch.cuda.current_stream().cuda_stream
    tail = (groups, groups, n_rows, bit, 32 // bit, 0, 64)
    for value in (False, True):
        c = cq.convert_value_batched_quant(g, bit) if value else cq.convert_key_batched_quant(g, True, bit)
        h = [t.cpu().numpy() for t in c]
        want = orc.decode_quant(h[0], h[2], h[1], h[5], h[6], 0, tokens, D, int(value), bit, 0)  # [tokens, D]
        ptrs = [c[i].data_ptr() for i in (0, 2, 1, 5, 6)]
        n = tokens if value else D                                                              # channels or tokens to pick
        ws = torch.empty(max(16, L.mstf_value_spmv_quant_workspace_bytes(D, tokens, groups, groups, n_rows)), dtype=torch.uint8,
                         device="cuda")
        for first in range(0, n, rpk):
            picks = (first + np.arange(rpk)) % n
            w = torch.zeros((groups, n_rows, n), dtype=torch.float16, device="cuda")
            w.view(rpk, n)[torch.arange(rpk), torch.from_numpy(picks)] = 1
            out = torch.empty((groups, n_rows, D if value else tokens), dtype=torch.float16, device="cuda")
            if value:
                check(L.mstf_value_spmv_quant_grouped(st, *ptrs, w.data_ptr(), out.data_ptr(), D, tokens, *tail, ws.data_ptr(),
                                                      ws.numel()), "value")
            else:
                check(L.mstf_key_spmv_quant_grouped(st, *ptrs, w.data_ptr(), out.data_ptr(), tokens, D, *tail), "key")
            ref = np.stack([want[p] if value else want[:, p] for p in picks])
            assert np.array_equal(out.view(rpk, -1).float().cpu().numpy(), ref.astype(np.float32)), (value, first)
