"""Quantised value products over more than 8192 blocks, whose tiles are read whole (csrc/quant_spmv.hip, value_whole): every
weight row picks a single token, so that a result is one dequantised element, the same number as calls over fewer blocks give,
which read half of two tiles (tests/test_gpu_rank_whole.py holds those against the oracle)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
D = 128


@pytest.mark.parametrize("groups", [1, 4, 5, 8])
@pytest.mark.parametrize("bit,group_size", [(2, 64), (4, 32), (8, 64)])
def test_whole_tiles_equal_halves(bit, group_size, groups):
    from mustafar_amd import compression_quant as cq
    from mustafar_amd._lib import check, lib
    heads, tokens = 8200, 64
    g = torch.Generator(device="cuda").manual_seed(bit + groups)
    x = torch.randn((heads, tokens, D), generator=g, device="cuda", dtype=torch.float16)
    x[torch.rand(x.shape, generator=g, device="cuda") < torch.rand((heads, 1, 1), generator=g, device="cuda")] = 0
    x[7], x[4100, :, 64:] = 0, 0
    x[8, :, :64], x[9] = 1, torch.arange(tokens, device="cuda").view(-1, 1) + 1
    c = cq.convert_value_batched_quant(x, bit, group_size)
    p = torch.zeros((heads * groups, tokens), device="cuda", dtype=torch.float16)
    p.scatter_(1, torch.randint(0, tokens, (heads * groups, 1), generator=g, device="cuda"), 1.0)
    L = lib()

    def product(first, last):
        out = torch.full(((last - first) * groups, D), float("nan"), device="cuda", dtype=torch.float16)
        n = (last - first) * groups
        ws = torch.empty(max(256, L.mstf_value_spmv_quant_workspace_bytes(D, tokens, n, groups, 1)), dtype=torch.uint8, device="cuda")
        arrays = [c[i][first:last].contiguous() for i in (0, 1, 5, 6)]
        check(L.mstf_value_spmv_quant_grouped(torch.cuda.current_stream().cuda_stream, arrays[0].data_ptr(), c[2].data_ptr(),
                                              arrays[1].data_ptr(), arrays[2].data_ptr(), arrays[3].data_ptr(),
                                              p[first * groups:last * groups].data_ptr(), out.data_ptr(), D, tokens, n, groups, 1, bit,
                                              32 // bit, 0, group_size, ws.data_ptr(), ws.numel()), "value")
        return out

    whole = product(0, heads)
    halves = torch.cat([product(0, 4100), product(4100, heads)])
    # (8-bit codes of nearly constant groups, as in head 8 and in tiles of few elements, have infinite zero-points: NaN at the
    # same places)
    assert torch.equal(whole.isnan(), halves.isnan()) and torch.equal(whole.nan_to_num(), halves.nan_to_num())
    plain = torch.isfinite(c[6]).reshape(heads, -1).all(1)
    assert int(plain.sum()) > heads // 2 and bool(torch.isfinite(whole.view(heads, groups, D)[plain]).all())
