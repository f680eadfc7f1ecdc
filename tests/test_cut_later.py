"""Results whose values are cut to size when somebody asks for them (ops.CompressedKV.cut, ops.compress_proj): the same arrays and
numbers as of a call that waits, also as a copy, and an error where a wait on the GPU ran out."""
import copy
import ctypes
import pickle

import pytest
import torch

D, KTH = 128, 89


def uncut(total):
    from mustafar_amd import ops
    pair = (ctypes.c_int64 * 2)(7, total)
    landing = ops._LandingPair(ctypes.addressof(pair), 0, None, None)
    c = ops.CompressedKV.cut(torch.arange(2).view(1, 2), torch.tensor([[0, 1, 2]], dtype=torch.int32),
                             torch.arange(16, dtype=torch.float16), torch.zeros(1, dtype=torch.int32), 64, D, True,
                             torch.tensor([max(total, -1)]), landing)
    given = []
    landing._give = given.append
    return c, pair, given


@pytest.mark.parametrize("ask", [lambda c: c.nz, lambda c: c.total_halfs, lambda c: c.packed(), lambda c: c.used_halfs(),
                                 lambda c: c.nbytes(), copy.copy, copy.deepcopy, pickle.dumps])
def test_asked_for_in_any_way(ask):
    c, pair, given = uncut(8)
    ask(c)
    assert given == [ctypes.addressof(pair)] and c._uncut is None
    pair[1] = 5                                     # another call's by now
    other = pickle.loads(pickle.dumps(copy.deepcopy(c)))
    for r in (c, other):
        assert r.nz.numel() == r.total_halfs == r.used_halfs() == r.packed().numel() == 8
        assert r.nbytes() == 16 + 12 + 16 and torch.equal(r.nz, torch.arange(8, dtype=torch.float16))


def test_an_error_each_time_and_no_other_attribute():
    c, pair, given = uncut(-1)
    for _ in range(2):
        for name in ("nz", "total_halfs"):
            with pytest.raises(RuntimeError, match="gave up"):
                getattr(c, name)
    assert not hasattr(c, "values") and given == [] and pair[1] == -1


@pytest.mark.gpu
@pytest.mark.parametrize("heads,tokens,whole", [(1, 64, 64), (3, 200, 192), (64, 2048, 1984)])
def test_the_same_as_of_a_call_that_waits(heads, tokens, whole):
    from mustafar_amd import ops
    from mustafar_amd._lib import lib
    g = torch.Generator(device="cuda").manual_seed(heads)
    x = torch.randn((1, tokens, heads, D), generator=g, device="cuda", dtype=torch.float16)
    cos, sin = (torch.randn((tokens, D), generator=g, device="cuda").clamp(-1, 1).half() for _ in range(2))
    ws, rot = ops.Workspace("cuda", 1 << 20), [torch.empty_like(x) for _ in range(2)]

    def both(r):
        return [ops.compress_proj(x, False, KTH, whole, cos, sin, r, ws=ws)[0], ops.compress_proj(x, True, KTH, whole, ws=ws)[0]]

    got, held = both(rot[0]), []
    assert all(c._uncut is not None for c in got)
    while True:                                     # no words left: the calls wait
        p = lib().mstf_landing_take()
        if not p:
            break
        held.append(p)
    want = both(rot[1])
    for p in held:
        lib().mstf_landing_give(p)
    assert all(c._uncut is None for c in want)
    for a, b in zip(got, want):
        assert a.total_halfs == b.total_halfs == a.nz.numel() == int(2 * a.idx[:, -1].to(torch.int64).sum())
        assert all(torch.equal(p, q) for p, q in ((a.nz, b.nz), (a.bmp, b.bmp), (a.idx, b.idx), (a.nz_off, b.nz_off)))
    assert torch.equal(rot[0], rot[1])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with pytest.raises(RuntimeError):               # as before: a size cannot be waited for in a graph
        with torch.cuda.graph(graph):
            ops.compress_proj(x, True, KTH, whole, ws=ws)
