"""Four wavefronts per block in the fused attention over codes (SHARE, csrc/fused_quant.hip): on both sides of the sizes where the
launch takes that form (1024 blocks of all heads, 768 with more than four query heads, 128 of a head), one block a head, with and
without (max, sum), and with a workspace that has no room for a slot per block, where the call goes without.  The forms add
the same products up in the same order: they give the same numbers, bit for bit, wherever the call is one that may share.  Reference:
the three operators over the same codes; the bound is the one of scores rounded to fp16 in front of the softmax."""
import pytest
import torch

pytestmark = pytest.mark.gpu
D = 128


@pytest.mark.parametrize("bit,group_size", [(2, 64), (2, 32), (4, 64), (4, 32), (8, 64), (8, 32)])
@pytest.mark.parametrize("heads,groups,blocks", [(1, 1, 1), (3, 4, 1), (2, 8, 3), (1, 4, 128), (1, 4, 129), (8, 3, 9)])
def test_against_the_operators(bit, group_size, heads, groups, blocks):
    check(bit, group_size, heads, groups, blocks)


@pytest.mark.parametrize("heads,groups,blocks", [(256, 4, 4), (205, 4, 5), (8, 4, 128), (96, 5, 8), (97, 5, 8), (257, 8, 3)])
def test_around_the_most_blocks(heads, groups, blocks):
    check(2, 64, heads, groups, blocks)


def check(bit, group_size, heads, groups, blocks):
    from mustafar_amd import compression_quant as cq, mustafar_package_quant as mq, ops
    g = torch.Generator(device="cuda").manual_seed(heads * blocks + bit)
    tokens, rows = blocks * 64, heads * groups
    K, V = (torch.randn((heads, tokens, D), generator=g, device="cuda", dtype=torch.float16) for _ in range(2))
    K[:, :, 7] *= 10
    q = 0.25 * torch.randn((rows, D), generator=g, device="cuda", dtype=torch.float16)
    kth = 89 if bit < 8 else 40     # (8 bits: a few values that lie together have an infinite zero-point)
    k = cq.convert_key_batched_quant(K, True, bit, group_size, kth=kth)
    v = cq.convert_value_batched_quant(V, bit, group_size, kth=kth)
    assert k[6].isfinite().all() and v[6].isfinite().all()
    lse = torch.empty((rows, 2), device="cuda")
    got = mq.decode_attention_quant(k, v, q, groups, bit)
    with_lse = mq.decode_attention_quant(k, v, q, groups, bit, lse=lse)
    least = torch.empty(ops.attention_workspace_least(tokens, 0, rows), dtype=torch.uint8, device="cuda")
    alone = mq.decode_attention_quant(k, v, q, groups, bit, ws=least)
    dense = [dequantised(side, tokens, is_value, bit).float() for side, is_value in ((k, False), (v, True))]
    q32 = q.float().view(heads, groups, D)
    s = (q32 @ dense[0].transpose(1, 2).contiguous()).half()
    w = torch.softmax((s / D ** 0.5).float(), -1)
    want = (w @ dense[1]).view(rows, D)
    for o in (got, with_lse, alone):
        err = (o.float() - want).abs().amax(-1) / want.abs().amax(-1)
        assert float(err.max()) < 2e-3
    assert torch.equal(got, with_lse)
    if blocks <= 128 and heads * blocks <= (1024 if groups <= 4 else 768):
        assert torch.equal(got, alone)
    assert torch.allclose(lse[:, 0], (s / D ** 0.5).float().amax(-1).view(-1), atol=2e-2)


def dequantised(side, tokens, is_value, bit):
    """Dense rows [heads, tokens, D] of a side, (code - zero) * scale rounded to fp16, in torch."""
    bmp, off, packed, _, _, sc, zp = side
    H, T = bmp.shape
    place = torch.arange(63, -1, -1, device="cuda")
    bits = (bmp.unsqueeze(-1) >> place) & 1                                            # element order
    rank = bits.cumsum(-1) - bits
    cap = 32 // bit
    word = packed.long()[(off.long().unsqueeze(-1) + rank // cap).clamp(max=packed.numel() - 1)]
    code = (word >> ((rank % cap) * bit)) & ((1 << bit) - 1)
    if sc.dim() == 3:
        sc, zp = (t.repeat_interleave(32, -1) for t in (sc, zp))
    else:
        sc, zp = (t.unsqueeze(-1) for t in (sc, zp))
    x = torch.where(bits > 0, ((code.float() - zp.float()) * sc.float()).half(), 0).view(H, tokens // 64, -1, 64)
    if not is_value:
        return x.transpose(2, 3).reshape(H, tokens, D)
    return x.view(H, tokens // 64, 2, 64, 64).transpose(2, 3).reshape(H, tokens, D)


@pytest.mark.parametrize("bit", [2, 4, 8])
@pytest.mark.parametrize("heads,groups,tokens,window", [(4, 4, 768, 60), (2, 8, 256, 100), (64, 4, 1024, 1), (61, 4, 1024, 130)])
def test_step_and_windows_without_room(bit, heads, groups, tokens, window):
    """A step over pools, with room for a slot per block and without: the same numbers, and those of append and attention apart.
    64 heads of 16 blocks and a window block each are one workgroup too many for the shared form, 61 too few heads for that."""
    from mustafar_amd import mustafar_package_quant as mq, ops
    from mustafar_amd.cache import QuantSparseKVCache
    g = torch.Generator(device="cuda").manual_seed(tokens + bit)
    rand = lambda *shape: torch.randn(shape, generator=g, device="cuda", dtype=torch.float16)  # noqa: E731
    K, V = rand(1, heads, tokens + window, D), rand(1, heads, tokens + window, D)
    cache = QuantSparseKVCache(groups, D, 0.7, 0.7, window, bit=bit, window_kernel=True, max_tokens=tokens + 256)
    cache.prefill(K, V)
    q, k, v = rand(1, heads * groups * D), rand(1, heads * D), rand(1, heads * D)
    rows, win = heads * groups, cache._kbuf.shape[1]
    length = torch.tensor([window + 1], dtype=torch.int32, device="cuda")
    outs = []
    for room in (ops.attention_workspace_least(tokens + 256, win, rows), 16 << 20):
        kw, vw = cache._kbuf.clone(), cache._vbuf.clone()
        for step in (True, False):
            ws = torch.empty(room, dtype=torch.uint8, device="cuda")
            if step:
                outs.append(mq.decode_step_quant_pool(cache.k_pool, cache.v_pool, q, k, v, kw, vw, win, win_len_dev=length, ws=ws))
            else:
                outs.append(mq.decode_attention_window_quant_pool(cache.k_pool, cache.v_pool, q.view(rows, D), kw, vw, win, groups,
                                                                  win_len_dev=length, ws=ws))
    assert all(torch.equal(o, outs[0]) for o in outs[1:])
    assert outs[0].isfinite().all()


@pytest.mark.parametrize("bit", [2, 4, 8])
@pytest.mark.parametrize("heads,groups,blocks,window", [(3, 4, 1, 1), (8, 4, 9, 300), (2, 8, 16, 65), (96, 8, 2, 512), (5, 1, 0, 70)])
def test_window_calls_without_room(bit, heads, groups, blocks, window):
    """decode_attention_window_quant, with room for a slot per block and with the least workspace: the same numbers."""
    from mustafar_amd import compression_quant as cq, mustafar_package_quant as mq, ops
    g = torch.Generator(device="cuda").manual_seed(heads * blocks + bit)
    tokens, rows = blocks * 64, heads * groups
    k = v = None
    if blocks:
        K, V = (torch.randn((heads, tokens, D), generator=g, device="cuda", dtype=torch.float16) for _ in range(2))
        k = cq.convert_key_batched_quant(K, True, bit, kth=89 if bit < 8 else 40)
        v = cq.convert_value_batched_quant(V, bit, kth=89 if bit < 8 else 40)
    q = 0.25 * torch.randn((rows, D), generator=g, device="cuda", dtype=torch.float16)
    kw, vw = (torch.randn((heads, window, D), generator=g, device="cuda", dtype=torch.float16) for _ in range(2))
    outs, lses = [], []
    for room in (ops.attention_workspace_least(tokens, window, rows), 64 << 20):
        lses.append(torch.empty((rows, 2), device="cuda"))
        ws = torch.empty(room, dtype=torch.uint8, device="cuda")
        outs.append(mq.decode_attention_window_quant(k, v, q, kw, vw, window, groups, bit, lse=lses[-1], ws=ws))
    assert torch.equal(*outs) and torch.equal(*lses) and outs[0].isfinite().all()
