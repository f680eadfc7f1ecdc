"""An infinite weight times a kept element is infinite, with its sign, in the products of eight, sixteen and 32 rows: the
element multiplies its own weight only (an absent one, or a code that stands for zero, is 0 x inf and gives NaN, and so do
the neighbours of its group of four tiles in the products of one to four rows).  The column that an infinite weight meets
comes from a product with a one in its place, which is exact."""
import pytest
import torch

pytestmark = pytest.mark.gpu
D, TOKENS, HEADS = 128, 192, 2


@pytest.mark.parametrize("groups,n_rows", [(8, 1), (2, 8), (4, 8)])
@pytest.mark.parametrize("bit", [0, 2, 4])
@pytest.mark.parametrize("value", [False, True])
def test_infinite_weights(groups, n_rows, bit, value):
    from mustafar_amd import compression_quant as cq, ops
    from mustafar_amd._lib import check, lib
    gen = torch.Generator(device="cuda")
    gen.manual_seed(groups + bit)
    x = torch.randn((HEADS, TOKENS, D), generator=gen, device="cuda", dtype=torch.float16)
    rows, n = HEADS * groups * n_rows, TOKENS if value else D    # n: weights of a row
    L = lib()
    if bit:
        c = cq.convert_value_batched_quant(x, bit, kth=39) if value else cq.convert_key_batched_quant(x, True, bit, kth=39)
        need = L.mstf_value_spmv_quant_workspace_bytes(D, TOKENS, HEADS * groups, groups, n_rows)
        ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")

        def product(w):
            out = torch.empty((rows, D if value else TOKENS), dtype=torch.float16, device="cuda")
            args = [None] + [c[i].data_ptr() for i in (0, 2, 1, 5, 6)] + [w.data_ptr(), out.data_ptr()]
            shape = [D, TOKENS] if value else [TOKENS, D]
            tail = [HEADS * groups, groups, n_rows, bit, 32 // bit, 0, 64] + ([ws.data_ptr(), ws.numel()] if value else [])
            check((L.mstf_value_spmv_quant_grouped if value else L.mstf_key_spmv_quant_grouped)(*args, *shape, *tail), "spmv")
            return out
    else:
        c = ops.compress(x, value, kth=39)
        call = ops.value_spmv if value else ops.key_spmv

        def product(w):
            return call(c, w.view(HEADS * groups, n_rows, n), groups, n_rows).view(rows, -1)

    at = torch.randint(0, n, (rows,), generator=gen, device="cuda")
    at[:8] = torch.arange(8, device="cuda") * 9       # every place in a group of eight tiles
    one = torch.zeros((rows, n), dtype=torch.float16, device="cuda")
    one[torch.arange(rows), at] = 1.0
    column = product(one).float()
    w = torch.rand((rows, n), generator=gen, device="cuda").half() / n
    w[torch.arange(rows), at] = float("inf")
    got = product(w)
    kept = column != 0
    assert 0.3 < float(kept.float().mean()) < 0.95    # both kinds are there
    want = torch.where(kept, torch.copysign(torch.full_like(column, float("inf")), column), float("nan"))
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(got[kept].float(), want[kept])
