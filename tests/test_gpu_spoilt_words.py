"""Kept status words of the producers behind a call whose bounded wait ran out (csrc/compress_common.hpp, Handover): until its
caller has brought cleared words, calls of any size over the same words raise or are exactly right."""
import pytest
import torch

pytestmark = pytest.mark.gpu
D, KTH = 128, 89


def kv(heads, tokens, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn((heads, tokens, D), generator=g, device="cuda", dtype=torch.float16) for _ in range(2)]


def spoil(ws, heads, tokens):
    """A call without polls over the words of ws, its totals unread.  Skips where every wait ended at once."""
    from mustafar_amd import ops
    from mustafar_amd._lib import lib
    k, v = kv(heads, tokens)
    for _ in range(4):
        lib().mstf_test_set_spin_limit(0)
        try:
            c = ops.compress_kv(k, v, KTH, KTH, ws=ws)
            torch.cuda.synchronize()
        finally:
            lib().mstf_test_set_spin_limit(-1)
        if any(int(t.total_halfs) == -1 for t in c):
            return
    pytest.skip("no wait ran out")


def exact(got, want):
    """Whether the arrays are `want`'s; False where reading them raises."""
    try:
        packed = got.packed()
    except RuntimeError as e:
        assert "gave up" in str(e)
        return False
    assert all(torch.equal(a, b) for a, b in ((got.bmp, want.bmp), (got.idx, want.idx), (got.nz_off, want.nz_off), (packed, want.packed())))
    return True


# workgroups of a side: 4500 of one wavefront, 2048 of four; behind them 1, 3, 48, 1040 and 4800
@pytest.mark.parametrize("spoiling", [(60, 4800), (128, 4096)])
def test_calls_of_other_sizes_behind_a_give_up(spoiling):
    from mustafar_amd import compression_quant as cq, ops
    bare = torch.empty(1 << 22, dtype=torch.uint8, device="cuda")
    sizes = [(1, 256), (1, 192), (12, 1024), (130, 2048), (64, 4800)]
    inputs = [kv(h, t, 3 + i) for i, (h, t) in enumerate(sizes)]
    wants = [ops.compress_kv(k, v, KTH, 10, ws=bare) for k, v in inputs]
    for order in (1, -1):
        ws = ops.Workspace("cuda")
        ws.status(ops.status_words(64 * 75, 2))
        spoil(ws, *spoiling)
        gots = [ops.compress_kv(k, v, KTH, 10, ws=ws) for k, v in inputs[::order]]     # none of their totals read yet
        torch.cuda.synchronize()
        for got, want in zip(gots, wants[::order]):
            for g, w in zip(got, want):
                exact(g, w)
        for (k, v), want in zip(inputs, wants):                  # the reads have brought cleared words
            assert all([exact(g, w) for g, w in zip(ops.compress_kv(k, v, KTH, 10, ws=ws), want)])
        spoil(ws, *spoiling)
        rows = inputs[2][0].view(1, 12, 1024, D).transpose(1, 2)
        for _ in range(2):
            try:
                assert torch.equal(ops.compress_proj(rows, False, KTH, 1024, ws=ws)[0].nz, wants[2][0].packed())
            except RuntimeError as e:
                assert "gave up" in str(e)
        assert torch.equal(ops.compress_proj(rows, False, KTH, 1024, ws=ws)[0].nz, wants[2][0].packed())
        spoil(ws, *spoiling)
        for _ in range(2):
            try:
                out = cq.convert_value_batched_quant(inputs[3][1], 2, ws=ws, kth=KTH)
            except RuntimeError as e:
                assert "gave up" in str(e)
        want = cq.convert_value_batched_quant(inputs[3][1], 2, ws=bare, kth=KTH)
        assert all(torch.equal(a, b) for a, b in zip(out, want))


@pytest.mark.parametrize("heads,tokens", [(1, 192), (12, 1024), (64, 4800)])
def test_a_recorded_call_clears_its_own_words(heads, tokens):
    """Behind a call that gave up over the words of the same Workspace a graph's replays are exact, every one."""
    from mustafar_amd import ops
    k, v = kv(heads, tokens, 5)
    ws = ops.Workspace("cuda", 1 << 22)
    want = ops.compress_kv(k, v, KTH, 10, ws=ws)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        c = ops.compress_kv(k, v, KTH, 10, ws=ws)
    for _ in range(3):
        spoil(ws, 60, 4800)
        for t in c[0].bmp, c[0].idx, c[0].nz, c[1].bmp, c[1].idx, c[1].nz:
            t.zero_()
        graph.replay()
        assert all([exact(g, w) for g, w in zip(c, want)])


def test_cleared_words_come_on_the_stream_that_uses_them():
    """The read that finds a give-up may be made on another, busy stream: the next call does not wait for that one."""
    from mustafar_amd import ops
    k, v = kv(12, 1024, 6)
    ws = ops.Workspace("cuda", 1 << 22)
    want = ops.compress_kv(k, v, KTH, 10, ws=torch.empty(1 << 22, dtype=torch.uint8, device="cuda"))
    spoil(ws, 60, 4800)
    c = ops.compress_kv(k, v, KTH, 10, ws=ws)
    torch.cuda.synchronize()
    other = torch.cuda.Stream()
    with torch.cuda.stream(other):
        # what such words hold in front of their clearing: the ready mark and a total
        used = [torch.full((4096,), -(1 << 63) + 64, dtype=torch.int64, device="cuda") for _ in range(8)]
        torch.cuda.synchronize()
        del used
        torch.cuda._sleep(int(2e8))
        with pytest.raises(RuntimeError, match="gave up"):
            c[0].packed()
    got = ops.compress_kv(k, v, KTH, 10, ws=ws)
    assert all([exact(g, w) for g, w in zip(got, want)])
    torch.cuda.synchronize()
