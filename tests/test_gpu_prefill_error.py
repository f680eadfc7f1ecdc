"""A prompt whose compressor gave up (SparseKVCache.prefill_proj): the call raises and the cache is as it was in front of it, so that
the caller can try again."""
import pytest
import torch

pytestmark = pytest.mark.gpu
D = 128


@pytest.mark.parametrize("window_kernel", [False, True])
def test_a_prompt_that_gave_up_leaves_the_cache_empty(monkeypatch, window_kernel):
    from mustafar_amd import ops
    from mustafar_amd.cache import SparseKVCache
    g = torch.Generator(device="cuda").manual_seed(3)
    kx, vx = (torch.randn((2, 700, 3, D), generator=g, device="cuda", dtype=torch.float16) for _ in range(2))
    one = torch.ones((700, D), device="cuda", dtype=torch.float16)      # (no rotation, so that the rows can be taken again)
    cache, want = (SparseKVCache(2, D, 0.7, 0.7, 128, window_kernel=window_kernel) for _ in range(2))

    def state():
        return cache.k, cache.v, cache.compressed_length, cache.kv_len, cache._wlen, cache._kbuf, cache.k_win, cache.v_win
    before = state()
    with monkeypatch.context() as m:
        m.setattr(ops._LandingPair, "read", lambda self, side: -1)
        with pytest.raises(RuntimeError, match="gave up"):
            cache.prefill_proj(kx, vx, one, one * 0)
    assert state() == before and cache.kv_len == 0
    cache.prefill_proj(kx, vx, one, one * 0)
    want.prefill(kx.transpose(1, 2), vx.transpose(1, 2))
    assert cache.kv_len == want.kv_len == 700 and cache.compressed_length == want.compressed_length == 512
    for a, b in ((cache.k, want.k), (cache.v, want.v)):
        assert torch.equal(a.bmp, b.bmp) and torch.equal(a.idx, b.idx) and torch.equal(a.packed(), b.packed())
    assert torch.equal(cache.k_win, want.k_win) and torch.equal(cache.v_win, want.v_win)
