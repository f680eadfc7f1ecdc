"""Operands that start between two sixteen-byte boundaries - the entry points accept weights at any multiple of four bytes and
results at any multiple of two: the products of more than eight rows go to passes of eight then (their wide accesses want
the alignment), query rows come four bytes a lane.  Against the same call on aligned copies: one rounding of the result
to fp16 (2^-11) and another order of the 32-bit sums."""
import pytest
import torch

pytestmark = pytest.mark.gpu
D, HEADS = 128, 3


def at_offset(t, elements):
    """A copy of t that starts `elements` behind a 256-byte boundary."""
    room = torch.full((t.numel() + elements + 8,), float("nan"), dtype=t.dtype, device=t.device)
    out = room[elements:elements + t.numel()].view(t.shape)
    out.copy_(t)
    return out


@pytest.mark.parametrize("groups,n_rows,tokens", [(2, 8, 64), (4, 8, 1024), (7, 8, 2112), (4, 1, 640)])
@pytest.mark.parametrize("bit", [0, 2])
def test_offset_operands(groups, n_rows, tokens, bit):
    from mustafar_amd import compression_quant as cq, ops
    from mustafar_amd._lib import check, lib
    gen = torch.Generator(device="cuda")
    gen.manual_seed(tokens + bit)
    K, V = (torch.randn((HEADS, tokens, D), generator=gen, device="cuda", dtype=torch.float16) for _ in range(2))
    rows, Bq = HEADS * groups * n_rows, HEADS * groups
    q = torch.randn((rows, D), generator=gen, device="cuda", dtype=torch.float16)
    p = torch.softmax(torch.randn((rows, tokens), generator=gen, device="cuda"), -1).half()
    L = lib()
    need = (L.mstf_value_spmv_quant_workspace_bytes if bit else L.mstf_value_spmv_workspace_bytes)(D, tokens, Bq, groups, n_rows)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    if bit:
        ck, cv = ([c[i] for i in (0, 2, 1, 5, 6)] for c in (cq.convert_key_batched_quant(K, True, bit, kth=89),
                                                            cq.convert_value_batched_quant(V, bit, kth=89)))
        fk, fv, tail = L.mstf_key_spmv_quant_grouped, L.mstf_value_spmv_quant_grouped, [bit, 32 // bit, 0, 64]
    else:
        ck, cv = ((c.bmp, c.nz, c.idx, c.nz_off) for c in (ops.compress(K, False, 89), ops.compress(V, True, 89)))
        fk, fv, tail = L.mstf_key_spmv_f16, L.mstf_value_spmv_f16, []

    def keys(w, out):
        check(fk(None, *[t.data_ptr() for t in ck], w.data_ptr(), out.data_ptr(), tokens, D, Bq, groups, n_rows, *tail), "keys")
        return out.clone()

    def values(w, out):
        check(fv(None, *[t.data_ptr() for t in cv], w.data_ptr(), out.data_ptr(), D, tokens, Bq, groups, n_rows, *tail,
                 ws.data_ptr() if need else None, need), "values")
        return out.clone()

    s, o = torch.zeros((rows, tokens), dtype=torch.float16, device="cuda"), torch.zeros((rows, D), dtype=torch.float16, device="cuda")
    for call, w, out in ((keys, q, s), (values, p, o)):
        want = call(w, out).float()
        for wo, oo in ((2, 0), (6, 1), (0, 3), (8, 4)):
            got = call(at_offset(w, wo), at_offset(torch.zeros_like(out), oo)).float()
            err = (got - want).abs()
            assert bool((err <= 2.0 ** -10 * want.abs() + 2.0 ** -18 * want.abs().max()).all()), (call.__name__, wo, oo)
