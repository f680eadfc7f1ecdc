"""Totals that the producers' kernels store to pinned host memory themselves (mstf_compress_kv_landing_f16, ..._sized): the
same numbers as the device totals, at every number of wavefronts per workgroup and from one workgroup to many; what becomes
of the words when results are dropped early, when none is free, when the call is recorded and when a workgroup gives up."""
import pytest
import torch

pytestmark = pytest.mark.gpu
D, KTH = 128, 89


def kv(heads, tokens, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn((heads, tokens, D), generator=g, device="cuda", dtype=torch.float16) for _ in range(2)]


def same(c):
    idx = c.idx.cpu()
    assert c.packed().numel() == int(c.total_halfs) == int(2 * idx[:, -1].to(torch.int64).sum())


@pytest.mark.parametrize("heads,tokens", [(1, 64), (1, 128), (3, 192), (2, 256), (5, 1344), (130, 1024), (300, 2048)])
def test_totals_land(heads, tokens):
    from mustafar_amd import compression_quant as cq, ops
    k, v = kv(heads, tokens)
    for c in ops.compress_kv(k, v, KTH, 20):
        same(c)
    for x, is_value in ((k, False), (v, True)):
        rows = x.view(1, heads, tokens, D).transpose(1, 2)
        c, _ = ops.compress_proj(rows, is_value, KTH, tokens)
        assert c.total_halfs == c.nz.numel() == int(2 * c.idx[:, -1].to(torch.int64).sum())
        for bit, gs in ((2, 64), (4, 32), (8, 64)):
            out = (cq.convert_value_batched_quant(x, bit, gs, kth=KTH) if is_value
                   else cq.convert_key_batched_quant(x, True, bit, gs, kth=KTH))
            ref = cq._produce(x, is_value, bit, KTH, gs)
            assert out[2].numel() == int(out[4].to(torch.int64).sum()) == int(ref[-1])
            assert torch.equal(out[2], ref[2][:out[2].numel()])


def test_pairs_are_bounded_and_come_back():
    from mustafar_amd import ops
    from mustafar_amd._lib import lib
    held, L = [], lib()
    while True:
        p = L.mstf_landing_take()
        if not p:
            break
        held.append(p)
    assert len(held) <= 1024
    k, v = kv(4, 256)
    c = ops.compress_kv(k, v, KTH, KTH)        # none free: by way of the device totals
    assert c[0]._landing is None
    same(c[0]), same(c[1])
    for p in held:
        L.mstf_landing_give(p)
    for i in range(3000):                       # dropped while their kernels are still to run
        ops.compress_kv(k, v, KTH, KTH)
    for i in range(64):
        c = ops.compress_kv(k, v, KTH - i, 1 + i)
        same(c[0]), same(c[1])


def test_recorded_calls_do_not_land():
    from mustafar_amd import ops
    k, v = kv(4, 512)
    ws = ops.Workspace("cuda")
    ops.compress_kv(k, v, KTH, KTH, ws=ws)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        c = ops.compress_kv(k, v, KTH, KTH, ws=ws)
    for seed in range(1, 4):
        for dst, src in zip((k, v), kv(4, 512, seed)):
            dst.copy_(src)
        graph.replay()
        assert not any(bool(s.any()) for s in ws._status)
        same(c[0]), same(c[1])
        ref = ops.compress_kv(k, v, KTH, KTH)
        assert torch.equal(c[0].packed(), ref[0].packed()) and torch.equal(c[1].packed(), ref[1].packed())


def test_a_wait_that_ran_out_lands_as_such():
    """With no polls at all a call raises or is exactly right."""
    from mustafar_amd import compression_quant as cq, ops
    from mustafar_amd._lib import lib
    k, v = kv(16, 1024)
    rows = v.view(1, 16, 1024, D).transpose(1, 2)
    want_kv = [c.packed().clone() for c in ops.compress_kv(k, v, KTH, KTH)]
    want_q = cq.convert_value_batched_quant(v, 2, kth=KTH)[2]
    lib().mstf_test_set_spin_limit(0)
    try:
        for _ in range(4):
            for c, want in zip(ops.compress_kv(k, v, KTH, KTH), want_kv):
                try:
                    assert torch.equal(c.packed(), want)
                except RuntimeError as e:
                    assert "gave up" in str(e)
            try:
                assert torch.equal(cq.convert_value_batched_quant(v, 2, kth=KTH)[2], want_q)
            except RuntimeError as e:
                assert "gave up" in str(e)
            try:
                c, _ = ops.compress_proj(rows, True, KTH, 1024)
                assert torch.equal(c.nz, want_kv[1])
            except RuntimeError as e:
                assert "gave up" in str(e)
    finally:
        lib().mstf_test_set_spin_limit(-1)
    for c, want in zip(ops.compress_kv(k, v, KTH, KTH), want_kv):      # behind calls whose totals nobody read, too
        try:
            assert torch.equal(c.packed(), want)
        except RuntimeError as e:
            assert "gave up" in str(e)
    for c, want in zip(ops.compress_kv(k, v, KTH, KTH), want_kv):      # (a total that was read has brought cleared words)
        assert torch.equal(c.packed(), want)


@pytest.mark.parametrize("heads,tokens", [(1, 64), (3, 192), (40, 1024), (130, 2048), (33, 3264)])
def test_status_words_are_left_as_they_were(heads, tokens):
    """Calls of several sizes over the same kept words, one behind the other and without a wait between them; a launch that
    clears words in the workspace gives the same arrays."""
    from mustafar_amd import compression_quant as cq, ops
    k, v = kv(heads, tokens, 3)
    ws, bare = ops.Workspace("cuda"), torch.empty(1 << 22, dtype=torch.uint8, device="cuda")
    got = [ops.compress_kv(k, v, KTH, 10 + i, ws=ws) for i in range(6)]
    rows = k.view(1, heads, tokens, D).transpose(1, 2)
    part = max(64, tokens // 128 * 64)
    for i, pair in enumerate(got):
        ref = ops.compress_kv(k, v, KTH, 10 + i, ws=bare)
        for a, b in zip(pair, ref):
            assert int(a.total_halfs) == int(b.total_halfs)
            assert all(torch.equal(x, y) for x, y in ((a.bmp, b.bmp), (a.idx, b.idx), (a.nz_off, b.nz_off), (a.packed(), b.packed())))
        c, _ = ops.compress_proj(rows, False, KTH, part, ws=ws)
        r, _ = ops.compress_proj(rows, False, KTH, part, ws=bare)
        assert torch.equal(c.idx, r.idx) and torch.equal(c.nz, r.nz)
        x, y = (cq.convert_value_batched_quant(v, 2, ws=w, kth=KTH) for w in (ws, bare))
        assert all(torch.equal(p, q) for p, q in zip(x, y))
    assert len(ws._status) >= 1 and not any(bool(s.any()) for s in ws._status)
