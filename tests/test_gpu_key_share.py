"""Key products with more than eight rows where the four wavefronts of a workgroup share a token block, a channel stage each (few
blocks; kKeyShare in csrc/spmv.hip, kKeyShareQuant in csrc/quant_spmv.hip), against the form with a block per wavefront, which
the same rows take in a call with many heads.  Only the order of the 32-bit sums differs: of 128 products, by at most
128 x 2^-24 of the sum of their magnitudes, and then one rounding to fp16."""
import pytest
import torch

pytestmark = pytest.mark.gpu
D = 128


def product(K, q, groups, n_rows, bit, group_size):
    from mustafar_amd import compression_quant as cq, ops
    from mustafar_amd._lib import check, lib
    heads, tokens = K.shape[:2]
    if bit == 0:
        return ops.key_spmv(ops.compress(K, False), q, groups, n_rows)
    c = cq.convert_key_batched_quant(K, True, bit, group_size=group_size)
    s = torch.empty((heads * groups, n_rows, tokens), dtype=torch.float16, device="cuda")
    check(lib().mstf_key_spmv_quant_grouped(torch.cuda.current_stream().cuda_stream, *[c[i].data_ptr() for i in (0, 2, 1, 5, 6)],
                                            q.data_ptr(), s.data_ptr(), tokens, D, heads * groups, groups, n_rows, bit, 32 // bit,
                                            0, group_size), "key")
    return s


@pytest.mark.parametrize("bit,group_size", [(0, 64), (2, 64), (2, 32), (4, 64), (4, 32), (8, 64), (8, 32)])
@pytest.mark.parametrize("groups,n_rows,heads,blocks", [(4, 8, 1, 1), (2, 8, 3, 5), (6, 8, 2, 7), (4, 8, 32, 24), (4, 8, 32, 25),
                                                        (2, 8, 40, 32), (2, 8, 61, 21)])
def test_shared_blocks(bit, group_size, groups, n_rows, heads, blocks):
    many = (1281 + blocks - 1) // blocks
    g = torch.Generator(device="cuda").manual_seed(heads + blocks)
    K = torch.randn((max(heads, many), blocks * 64, D), generator=g, device="cuda", dtype=torch.float16)
    K *= torch.rand(K.shape, generator=g, device="cuda") < torch.rand((*K.shape[:2], 1), generator=g, device="cuda")
    q = torch.randn((K.shape[0] * groups, n_rows, D), generator=g, device="cuda", dtype=torch.float16)
    few = product(K[:heads].contiguous(), q[: heads * groups].contiguous(), groups, n_rows, bit, group_size).double()
    want = product(K, q, groups, n_rows, bit, group_size)[: heads * groups].double()
    terms = (q[: heads * groups].view(heads, -1, D).abs().float() @ K[:heads].abs().float().transpose(1, 2)).view_as(want).double()
    # (the dequantised magnitudes are within a step of the tile's codes, at most its range, of K's: twice the largest covers them)
    if bit:
        terms = q[: heads * groups].abs().sum(-1, keepdim=True).double() * 2 * K.abs().max().double()
    limit = 2.0 ** -10 * want.abs() + 2.0 ** -24 + D * 2.0 ** -23 * terms
    assert ((few - want).abs() <= limit).all(), float(((few - want).abs() / limit).max())
