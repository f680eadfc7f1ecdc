"""Sizes of the prefill producer (ops.compress_proj, compress_proj_both): known, or an error, when the call returns; keys and values
whose sizes are waited for together are the arrays of two calls; and a result that several threads ask for its size."""
import ctypes

import pytest
import torch

D, KTH = 128, 89


@pytest.mark.parametrize("access", range(1, 8))
def test_a_total_that_two_threads_ask_for(access):
    """The other thread's whole call in front of any access to the result's attributes: the total comes from its landing, never from
    the device word (5 here), which the asking thread's stream may not be ordered behind."""
    from mustafar_amd import ops
    pair = (ctypes.c_int64 * 2)(7, 8)
    left = [-1]

    class Result(ops.CompressedKV):
        def __getattribute__(self, name):
            if name in ("_landing", "_used"):
                left[0] -= 1
                if left[0] == 0:
                    assert self.used_halfs() == 8
            return super().__getattribute__(name)

        def __setattr__(self, name, value):
            super().__setattr__(name, value)
            if name in ("_landing", "_used"):
                left[0] -= 1
                if left[0] == 0:
                    assert self.used_halfs() == 8

    landing = ops._LandingPair(ctypes.addressof(pair), 0, None, None)
    landing._give = lambda p: None
    c = Result(None, None, torch.ones(16), None, 64, D, True, torch.tensor([5]), landing)
    left[0] = access
    assert c.used_halfs() == 8 and c.packed().numel() == 8


def rows(heads, tokens):
    g = torch.Generator(device="cuda").manual_seed(heads)
    x = torch.randn((1, tokens, heads, D), generator=g, device="cuda", dtype=torch.float16)
    return (x, *(torch.randn((tokens, D), generator=g, device="cuda").clamp(-1, 1).half() for _ in range(2)))


@pytest.mark.gpu
def test_known_or_an_error_when_the_call_returns():
    from mustafar_amd import ops
    from mustafar_amd._lib import lib
    x, cos, sin = rows(64, 4096)
    want = ops.compress_proj(x, True, KTH, 4096)[0]
    for _ in range(4):
        lib().mstf_test_set_spin_limit(0)
        try:
            c = ops.compress_proj(x, True, KTH, 4096)[0]
        except RuntimeError as e:
            assert "gave up" in str(e)
            continue
        finally:
            lib().mstf_test_set_spin_limit(-1)
        held = vars(c)
        assert held["total_halfs"] == held["nz"].numel() == want.total_halfs and torch.equal(held["nz"], want.nz)


@pytest.mark.gpu
@pytest.mark.parametrize("heads,tokens,whole", [(1, 64, 64), (3, 200, 192), (64, 2048, 1984)])
def test_both_sides_are_those_of_two_calls(heads, tokens, whole):
    from mustafar_amd import ops
    from mustafar_amd._lib import lib
    x, cos, sin = rows(heads, tokens)
    ws = ops.Workspace("cuda", 1 << 20)
    rot = torch.empty_like(x)
    want = [ops.compress_proj(x, False, KTH, whole, cos, sin, rot, ws=ws)[0], ops.compress_proj(x, True, 40, whole, ws=ws)[0]]

    def same():
        k = x.clone()
        settle = ops.compress_proj_both(k, x, KTH, 40, whole, cos, sin, ws=ws)
        got = settle()
        assert torch.equal(k, rot)
        for a, b in zip(got, want):
            assert a.total_halfs == b.total_halfs == a.nz.numel() == int(2 * a.idx[:, -1].to(torch.int64).sum())
            assert all(torch.equal(p, q) for p, q in ((a.nz, b.nz), (a.bmp, b.bmp), (a.idx, b.idx), (a.nz_off, b.nz_off)))
            assert (a.tokens, a.head_dim, a.is_value) == (whole, D, b.is_value)
    same()
    held = []
    while True:                                     # no words left: the two calls wait
        p = lib().mstf_landing_take()
        if not p:
            break
        held.append(p)
    try:
        same()
    finally:
        for p in held:
            lib().mstf_landing_give(p)
    torch.cuda.synchronize()
    for call in (lambda: ops.compress_proj(x, True, KTH, whole, ws=ws),
                 lambda: ops.compress_proj_both(rot, x, KTH, KTH, whole, cos, sin, ws=ws)):
        graph = torch.cuda.CUDAGraph()
        with pytest.raises(RuntimeError):           # a size cannot be waited for in a graph
            with torch.cuda.graph(graph):
                call()
    same()
