"""The first step of a new cache: the scratch memory made with its first append is large enough for the step, so that no
layer allocates in front of its first attention call."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["fp16", "2 bits"])
@pytest.mark.parametrize("max_tokens", [0, 1280])
@pytest.mark.parametrize("heads,groups,tokens", [(20, 8, 1309), (64, 4, 1100), (24, 8, 200)])
@pytest.mark.parametrize("from_projection", [False, True])
def test_the_first_step_finds_its_workspace(kind, max_tokens, heads, groups, tokens, from_projection):
    from mustafar_amd.cache import QuantSparseKVCache, SparseKVCache
    cls = SparseKVCache if kind == "fp16" else QuantSparseKVCache
    bs, n_kv, D = heads // 4, 4, 128
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)
    rand = lambda *shape: torch.randn(shape, generator=gen, device="cuda", dtype=torch.float16)  # noqa: E731
    cache = cls(groups, D, 0.7, 0.7, 256, window_kernel=True, max_tokens=max_tokens)
    K, V = rand(bs, tokens, n_kv, D), rand(bs, tokens, n_kv, D)
    one = torch.ones((tokens, D), device="cuda", dtype=torch.float16)
    if from_projection:
        cache.prefill_proj(K, V, one, one * 0)
    else:
        cache.prefill(K.transpose(1, 2).contiguous(), V.transpose(1, 2).contiguous())
    made = cache.ws.tensor
    out = cache.decode_device_proj(rand(bs, groups * n_kv * D), rand(bs, n_kv * D), rand(bs, n_kv * D), one[0], one[0] * 0)
    assert torch.isfinite(out).all()
    assert cache.ws.tensor is made and len(cache.ws._bufs) == 1
