"""Value products whose wavefronts walk several token blocks, a ragged last one among them, and both products at head_dim 64 (a
key walk of two stages, weight rows of 128 bytes, one half of channels), each for weight rows of the narrow and of the wide
form.  Reference: the products in 64 bits; a result is a 32-bit sum of at most n products, rounded once to fp16:
|error| <= 2^-11 |x| + n 2^-24 sum |terms|."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def close(got, weights, rows):
    """got: weights @ rows; [heads, rows per head, n] @ [heads, n, m]"""
    w, x = weights.double(), rows.double()
    want, bound = torch.matmul(w, x), torch.matmul(w.abs(), x.abs())
    limit = 2.0 ** -11 * want.abs() + 2.0 ** -24 + w.shape[-1] * 2.0 ** -24 * bound
    assert bool(((got.double().view_as(want) - want).abs() <= limit).all())


def tiles_of(x, value):
    """The 64-element tiles [heads, T, 64] of rows x [heads, tokens, D]."""
    heads, tokens, D = x.shape
    blocks = x.view(heads, tokens // 64, 64, D)
    if not value:
        return blocks.transpose(2, 3).reshape(heads, -1, 64)
    return blocks.view(heads, tokens // 64, 64, D // 64, 64).transpose(2, 3).reshape(heads, -1, 64)


def bitmaps(keep):
    return (keep.long() << (63 - torch.arange(64, device=keep.device))).sum(-1)      # (wraps to the sign bit: element 0)


def packed_fp16(x, value):
    """bmp, nz, idx, nz_off of rows x (zeros absent): values of a tile padded to eight, offsets in four-byte units."""
    t = tiles_of(x, value)
    keep = t != 0
    count = keep.sum(-1)
    room = (count + 7) // 8 * 8
    idx = torch.zeros((t.shape[0], t.shape[1] + 1), dtype=torch.int32, device=t.device)
    idx[:, 1:] = room.cumsum(1) // 2
    head = torch.zeros(t.shape[0], dtype=torch.int64, device=t.device)
    head[1:] = room.sum(1).cumsum(0)[:-1]
    nz = torch.zeros(int(room.sum()) + 64, dtype=torch.float16, device=t.device)
    at = head[:, None, None] + 2 * idx[:, :-1, None].long() + keep.long().cumsum(-1) - 1
    nz[at[keep]] = t[keep]
    return bitmaps(keep), nz, idx, (head // 8).int()


def packed_quant(x, value, bit):
    """bmp, packed, tile_off, scales, zeros and the rows they stand for."""
    t = tiles_of(x, value)
    heads, T, _ = t.shape
    keep, cap = t != 0, 32 // bit
    inf = torch.tensor(float("inf"), device=t.device)
    lo, hi = torch.where(keep, t.float(), inf).amin(-1), torch.where(keep, t.float(), -inf).amax(-1)
    none = ~keep.any(-1)
    scale = torch.where(none | (hi == lo), 1.0, (hi - lo) / (2 ** bit - 1)).half()
    zero = torch.where(none, 0.0, torch.floor(-lo / scale.float() + 0.5)).half()
    code = (torch.floor(t.float() / scale.float()[..., None] + 0.5) + zero.float()[..., None]).clamp(0, 2 ** bit - 1)
    rows = torch.where(keep, ((code - zero.float()[..., None]) * scale.float()[..., None]).half(), torch.zeros_like(t))
    words = (keep.sum(-1) + cap - 1) // cap
    off = (words.flatten().cumsum(0) - words.flatten()).view(heads, T)
    rank = keep.long().cumsum(-1) - 1
    packed = torch.zeros(int(words.sum()) + 64, dtype=torch.int64, device=t.device)
    packed.index_add_(0, (off[..., None] + rank // cap)[keep], (code.long() << (bit * (rank % cap)))[keep])
    packed = torch.where(packed >= 2 ** 31, packed - 2 ** 32, packed).int()
    D = x.shape[2]
    if value:
        rows = rows.view(heads, -1, D // 64, 64, 64).transpose(2, 3).reshape(x.shape)
    else:
        rows = rows.view(heads, -1, D, 64).transpose(2, 3).reshape(x.shape)
    return (bitmaps(keep), packed, off.int(), scale, zero), rows


def pruned(gen, heads, tokens, D):
    x = torch.randn((heads, tokens, D), generator=gen, device="cuda", dtype=torch.float16)
    keep = torch.rand((heads, tokens, D), generator=gen, device="cuda") < torch.rand((heads, tokens, 1), generator=gen, device="cuda")
    keep[:, 0], keep[:, 1] = True, False
    return torch.where(keep, x, torch.zeros_like(x))


def product(x, w, value, bit, groups, n_rows):
    from mustafar_amd._lib import check, lib
    L = lib()
    heads, tokens, D = x.shape
    Bq = heads * groups
    out = torch.empty((heads, groups * n_rows, D if value else tokens), dtype=torch.float16, device="cuda")
    c, rows = packed_quant(x, value, bit) if bit else (packed_fp16(x, value), x)
    args = [None] + [t.data_ptr() for t in c] + [w.data_ptr(), out.data_ptr()]
    args += [D, tokens] if value else [tokens, D]
    args += [Bq, groups, n_rows] + ([bit, 32 // bit, 0, 64] if bit else [])
    if value:
        ask = L.mstf_value_spmv_quant_workspace_bytes if bit else L.mstf_value_spmv_workspace_bytes
        ws = torch.empty(max(ask(D, tokens, Bq, groups, n_rows), 16), dtype=torch.uint8, device="cuda")
        args += [ws.data_ptr(), ws.numel()]
    name = "mstf_%s_spmv_%s" % ("value" if value else "key", "quant_grouped" if bit else "f16")
    check(getattr(L, name)(*args), name)
    torch.cuda.synchronize()
    return out, rows


@pytest.mark.parametrize("heads,blocks", [(130, 67), (257, 33)])      # five blocks a wavefront, two splits; five, one
@pytest.mark.parametrize("groups,n_rows", [(4, 1), (2, 8), (4, 8)])
@pytest.mark.parametrize("bit", [0, 2, 4])
def test_walk(heads, blocks, groups, n_rows, bit):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(blocks + bit)
    V = pruned(gen, heads, blocks * 64, 128)
    p = torch.rand((heads, groups * n_rows, blocks * 64), generator=gen, device="cuda").half()
    out, rows = product(V, p, True, bit, groups, n_rows)
    for h in range(0, heads, 8):
        close(out[h:h + 8], p[h:h + 8], rows[h:h + 8])


@pytest.mark.parametrize("tokens", [64, 320, 1088])
@pytest.mark.parametrize("groups,n_rows", [(1, 1), (4, 1), (8, 1), (2, 8), (4, 8)])
@pytest.mark.parametrize("bit", [0, 2, 8])
def test_head_dim_64(tokens, groups, n_rows, bit):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(tokens + bit)
    heads, rows = 3, groups * n_rows
    K, V = pruned(gen, heads, tokens, 64), pruned(gen, heads, tokens, 64)
    q = torch.randn((heads, rows, 64), generator=gen, device="cuda", dtype=torch.float16)
    p = torch.rand((heads, rows, tokens), generator=gen, device="cuda").half()
    s, k = product(K, q, False, bit, groups, n_rows)
    close(s, q, k.transpose(1, 2).contiguous())
    o, v = product(V, p, True, bit, groups, n_rows)
    close(o, p, v)
