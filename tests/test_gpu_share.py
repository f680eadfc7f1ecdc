"""Few token blocks: the four wavefronts of a workgroup share a block (fused_shares_blocks, csrc/fused_common.hpp), and the
merge takes one split per block.  Every stage is summed up on its own with one wavefront per block too, so the result must
be the same numbers, bit for bit, as from the two-phase entry points, which never share: (max, sum) and output.  Sizes: one
block, a ragged last group of eight, more splits than one run of the merge, more than its groups, and both sides of the
limit; the pooled step likewise against the calls it fuses, with and without sharing."""
import pytest
import torch

pytestmark = pytest.mark.gpu
D = 128


def kv(gen, heads, tokens):
    K = torch.randn((heads, tokens, D), generator=gen, device="cuda", dtype=torch.float16)
    K[:, :, 7] *= 10
    return K, torch.randn((heads, tokens, D), generator=gen, device="cuda", dtype=torch.float16)


@pytest.mark.parametrize("heads,groups,tokens", [(1, 4, 64), (3, 1, 128), (2, 8, 576), (1, 5, 1600), (2, 2, 4608), (1, 4, 8192), (1, 4, 33344),
                                                 (16, 4, 4096), (17, 4, 4096), (12, 8, 4096), (13, 8, 4096)])
def test_shared_blocks_give_the_same_numbers(heads, groups, tokens):
    from mustafar_amd import ops
    gen = torch.Generator(device="cuda")
    gen.manual_seed(tokens + groups)
    K, V = kv(gen, heads, tokens)
    ck, cv = ops.compress(K, False, kth=89), ops.compress(V, True, kth=89)
    q = torch.randn((heads * groups, D), generator=gen, device="cuda", dtype=torch.float16)
    lse, lse2 = (torch.empty((heads * groups, 2), device="cuda") for _ in range(2))
    o = ops.decode_attention(ck, cv, q, groups, lse=lse)
    ws = ops.decode_attention_partial(ck, cv, q, groups, ws=ops.Workspace("cuda", 64 << 20))
    o2 = ops.decode_attention_merge(ws, tokens, D, heads * groups, groups, lse=lse2)
    assert torch.equal(lse, lse2)
    assert torch.equal(o.view(torch.int16), o2.view(torch.int16))
    assert torch.equal(ops.decode_attention_static(ck, cv, q, groups).view(torch.int16), o.view(torch.int16))


@pytest.mark.parametrize("bs,n_kv,groups,tokens", [(1, 1, 4, 256), (2, 8, 4, 1024), (9, 8, 2, 1024), (7, 8, 8, 1024)])
@pytest.mark.parametrize("bit", [0, 2])
def test_pooled_step_equals_the_calls_it_fuses(bs, n_kv, groups, tokens, bit):
    from mustafar_amd import mustafar_package_quant as mpq, ops
    from mustafar_amd.cache import QuantSparseKVCache, SparseKVCache
    gen = torch.Generator(device="cuda")
    gen.manual_seed(bs * tokens + groups)
    K, V = kv(gen, bs * n_kv, tokens + 300)     # `tokens` compressed, 300 in the window
    make = (lambda: QuantSparseKVCache(groups, D, bit=bit, window_kernel=True, max_tokens=tokens + 256)) if bit else \
           (lambda: SparseKVCache(groups, D, window_kernel=True, max_tokens=tokens + 256))
    a = make()
    a.prefill(K.view(bs, n_kv, -1, D), V.view(bs, n_kv, -1, D))
    kb, vb = a._kbuf.clone(), a._vbuf.clone()
    n_q = n_kv * groups
    proj = torch.randn((bs, (n_q + 2 * n_kv) * D), generator=gen, device="cuda", dtype=torch.float16)
    q, k, v = proj[:, :n_q * D], proj[:, n_q * D:(n_q + n_kv) * D], proj[:, (n_q + n_kv) * D:]
    ang = torch.rand(D, generator=gen, device="cuda") * 6
    cos, sin = ang.cos().half(), ang.sin().half()
    wlen = torch.tensor([a._wlen + 1], dtype=torch.int32, device="cuda")
    one, two = (torch.empty((bs * n_q, 2), device="cuda") for _ in range(2))
    step = mpq.decode_step_quant_pool if bit else ops.decode_step_pool
    got = step(a.k_pool, a.v_pool, q, k, v, kb, vb, kb.shape[1], cos, sin, win_len_dev=wlen, lse=one)
    rows = ops.window_append(k, v, a._kbuf, a._vbuf, a._wlen + 1, q_in=q, cos=cos, sin=sin, win_len_dev=wlen)
    if bit:
        want = mpq.decode_attention_window_quant_pool(a.k_pool, a.v_pool, rows, a._kbuf, a._vbuf, kb.shape[1], groups,
                                                      win_len_dev=wlen, lse=two)
    else:
        want = ops.decode_attention_window_pool(a.k_pool, a.v_pool, rows, a._kbuf, a._vbuf, kb.shape[1], groups, wlen, lse=two)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16)) and torch.equal(one, two)
    n = int(wlen)
    assert torch.equal(kb[:, :n], a._kbuf[:, :n]) and torch.equal(vb[:, :n], a._vbuf[:, :n])


@pytest.mark.parametrize("heads,groups,tokens", [(8, 4, 512), (8, 4, 4096), (2, 8, 4096), (17, 4, 3840)])
def test_a_workspace_without_room_for_sharing_serves_the_call(heads, groups, tokens):
    """The least a call demands - a slot per 512 tokens and row, what a workspace made for a longer context or more rows
    may come to - gives the same numbers as the size the query answers."""
    from mustafar_amd import compression_quant as cq, mustafar_package_quant as mpq, ops
    gen = torch.Generator(device="cuda")
    gen.manual_seed(tokens + groups)
    K, V = kv(gen, heads, tokens)
    ck, cv = ops.compress(K, False, kth=89), ops.compress(V, True, kth=89)
    rows, n = heads * groups, -(-tokens // 512)
    q = torch.randn((rows, D), generator=gen, device="cuda", dtype=torch.float16)

    def least(slots):
        return torch.empty(-(-rows * slots * 520 // 256) * 256, dtype=torch.uint8, device="cuda")
    lse, lse2 = (torch.empty((rows, 2), device="cuda") for _ in range(2))
    assert torch.equal(ops.decode_attention(ck, cv, q, groups, lse=lse, ws=least(n)),
                       ops.decode_attention(ck, cv, q, groups, lse=lse2)) and torch.equal(lse, lse2)
    ws = ops.decode_attention_partial(ck, cv, q, groups, ws=least(n))
    assert torch.equal(ops.decode_attention_merge(ws, tokens, D, rows, groups), ops.decode_attention(ck, cv, q, groups))
    kw, vw = kv(gen, heads, 320)
    assert torch.equal(ops.decode_attention_window(ck, cv, q, kw, vw, 300, groups, ws=least(n + 5)),
                       ops.decode_attention_window(ck, cv, q, kw, vw, 300, groups))
    k, v = cq.convert_key_batched_quant(K, True, 2, kth=89), cq.convert_value_batched_quant(V, 2, kth=89)
    assert torch.equal(mpq.decode_attention_quant(k, v, q, groups, 2, ws=least(n)),
                       mpq.decode_attention_quant(k, v, q, groups, 2))
    with pytest.raises(RuntimeError):
        ops.decode_attention(ck, cv, q, groups, ws=least(n)[:-256])


def test_a_workspace_reserved_for_the_longest_context_holds_in_a_capture():
    """`Workspace` sized before the capture for 8256 tokens of 8 heads, which do not share; the shorter calls, which would
    like more room than that, are captured with it."""
    from mustafar_amd import ops
    from mustafar_amd._lib import lib
    heads, groups = 8, 4
    gen = torch.Generator(device="cuda")
    gen.manual_seed(9)
    ws = ops.Workspace("cuda", lib().mstf_decode_attention_workspace_bytes(8256, D, heads * groups, groups))
    assert ws.tensor.numel() < lib().mstf_decode_attention_workspace_bytes(8192, D, heads * groups, groups)
    q = torch.randn((heads * groups, D), generator=gen, device="cuda", dtype=torch.float16)
    sides = []
    for tokens in (1024, 8192):
        K, V = kv(gen, heads, tokens)
        sides.append((ops.compress(K, False, kth=89), ops.compress(V, True, kth=89)))
    want = [ops.decode_attention(k, v, q, groups) for k, v in sides]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = [ops.decode_attention(k, v, q, groups, ws=ws) for k, v in sides]
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))


# window rows: splits of 512 tokens and window blocks on both sides of the 64 that the merge keeps in LDS, and far beyond
@pytest.mark.parametrize("heads,groups,tokens,window", [(1, 4, 512, 63 * 64), (1, 4, 512, 63 * 64 + 1), (3, 2, 8192, 48 * 64 + 5),
                                                        (1, 8, 64, 6000), (2, 4, 512, 20480)])
def test_a_long_window_behind_shared_blocks(heads, groups, tokens, window):
    from mustafar_amd import ops
    from mustafar_amd.cache import CompressedPool, append_pair
    gen = torch.Generator(device="cuda")
    gen.manual_seed(window + groups)
    K, V = kv(gen, heads, tokens)
    kw, vw = kv(gen, heads, window)
    rows = heads * groups
    proj = torch.randn((1, (rows + 2 * heads) * D), generator=gen, device="cuda", dtype=torch.float16)
    q, k_in, v_in = proj[:, :rows * D], proj[:, rows * D:(rows + heads) * D], proj[:, (rows + heads) * D:]
    kw[:, -1], vw[:, -1] = k_in.view(heads, D), v_in.view(heads, D)
    q = q.contiguous().view(rows, D)
    ck, cv = ops.compress(K, False, kth=89), ops.compress(V, True, kth=89)
    one, two, three = (torch.empty((rows, 2), device="cuda") for _ in range(3))
    got = ops.decode_attention_window(ck, cv, q, kw, vw, window, groups, lse=one)
    least = torch.empty(ops.attention_workspace_least(tokens, window, rows), dtype=torch.uint8, device="cuda")
    assert torch.equal(got, ops.decode_attention_window(ck, cv, q, kw, vw, window, groups, lse=two, ws=least))
    assert torch.equal(one, two)
    # the step over pools of the same tokens, which appends the last row of the window itself
    kp, vp = CompressedPool(heads, D, tokens, False, "cuda"), CompressedPool(heads, D, tokens, True, "cuda")
    append_pair(kp, vp, K, V, 89, 89)
    kb, vb = kw.clone(), vw.clone()
    kb[:, -1], vb[:, -1] = 0, 0
    step = ops.decode_step_pool(kp, vp, q.view(1, -1), k_in, v_in, kb, vb, window, lse=three)
    assert torch.equal(step.view(rows, D), got) and torch.equal(one, three)
    assert torch.equal(kb, kw) and torch.equal(vb, vw)
    keys = torch.cat([ops.prune_rows(K, 89), kw], 1).float().repeat_interleave(groups, 0)
    values = torch.cat([ops.prune_rows(V, 89), vw], 1).float().repeat_interleave(groups, 0)
    s = torch.matmul(keys, q.float().view(rows, D, 1))[..., 0].half()
    want = torch.matmul(torch.softmax((s / D ** 0.5).float(), -1).view(rows, 1, -1), values)[:, 0]
    # weights and outputs rounded to fp16, a score rounded to the neighbouring fp16 value now and then (test_gpu_deal.py)
    assert float((got.float() - want).norm(dim=-1).div(want.norm(dim=-1)).max()) < 5e-3
