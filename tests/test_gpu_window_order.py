"""The dense window's blocks behind compressed blocks that divide evenly over a split's wavefronts, that do not, and behind splits
without any (fused_window_order): the step in one launch against append and attention calls on a twin cache, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
D = 128


# (128 heads: with the capacities below neither format shares blocks; none to 16 compressed blocks per head; one split of four
# blocks, whose idle wavefronts are fewer than the window's blocks)
@pytest.mark.parametrize("bit", [0, 2, 8])
@pytest.mark.parametrize("tokens,groups,max_tokens",
                         [(t, g, m) for t in (256, 600, 767, 800, 1100, 1500) for g, m in ((2, 1536), (8, 2560))] +
                         [(t, 4, 512) for t in (256, 512, 543, 544, 600, 767, 800)])
def test_step_equals_the_calls(bit, tokens, groups, max_tokens):
    from mustafar_amd.cache import QuantSparseKVCache, SparseKVCache
    bs, n_kv = 16, 8
    gen = torch.Generator(device="cuda")
    gen.manual_seed(tokens)
    K = torch.randn((bs, n_kv, tokens, D), generator=gen, device="cuda", dtype=torch.float16)
    V = torch.randn((bs, n_kv, tokens, D), generator=gen, device="cuda", dtype=torch.float16)
    proj = torch.randn((bs, (groups + 2) * n_kv * D), generator=gen, device="cuda", dtype=torch.float16)
    angle = torch.rand(D // 2, generator=gen, device="cuda").repeat(2) * 6
    nq, nk = groups * n_kv * D, n_kv * D
    outs = []
    for step_launch in (True, False):
        extra = {"bit": bit} if bit else {}
        c = (QuantSparseKVCache if bit else SparseKVCache)(groups, D, 0.7, 0.7, 256, window_kernel=True, max_tokens=max_tokens,
                                                           **extra)
        c.step_launch = step_launch
        c.prefill(K, V)
        o = c.decode_device_proj(proj[:, :nq], proj[:, nq:nq + nk], proj[:, nq + nk:], angle.cos().half(), angle.sin().half())
        outs.append([o, c._kbuf[:, :c._wlen + 1].clone(), c._vbuf[:, :c._wlen + 1].clone()])
    for a, b in zip(*outs):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
