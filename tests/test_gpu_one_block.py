"""The quantised fused attention in its form for one token block per wavefront and in the one for several: both sides of the
block count at which one gives way to the other (which depends on the LDS of width and group size), and a cache whose
capacity lies on either side of it."""
import pytest
import torch

from test_gpu_deal import D, _kv, _rel

pytestmark = pytest.mark.gpu


# 24 heads: 512 workgroups of eight blocks fit the chip (168 blocks a head), 256 of 8-bit codes (80)
@pytest.mark.parametrize("bit,group_size,blocks", [(2, 32, 168), (2, 32, 169), (4, 64, 168), (4, 64, 169), (4, 32, 80),
                                                   (4, 32, 169), (8, 64, 80), (8, 64, 81), (8, 32, 5), (8, 32, 81)])
def test_both_forms(bit, group_size, blocks):
    """Against the three operators; the bound is derived in test_gpu_deal."""
    from mustafar_amd import compression_quant, mustafar_package_quant as mpq, ops
    bkv, groups, n = 24, 4, blocks * 64
    kth = ops.kth_from_sparsity(0.7, D)
    K, V, g = _kv(bkv, blocks)
    k = compression_quant.convert_key_batched_quant(K, True, bit, group_size, kth=kth)
    v = compression_quant.convert_value_batched_quant(V, bit, group_size, kth=kth)
    Bq = bkv * groups
    q = torch.randn((Bq, D), generator=g, device="cuda", dtype=torch.float16)
    padded = torch.nn.functional.pad(q.view(Bq, 1, D), (0, 0, 0, 7))
    s = mpq.mustafar_key_formulation_quant_meta(k[0], k[2], k[1], k[3], k[4], k[5], k[6], padded, n, D, Bq, groups, bit,
                                                32 // bit)
    p = ops.scale_softmax(s[:, 0].contiguous(), D)
    ref = mpq.mustafar_value_formulation_quant_decode_n1(v[0], v[2], v[1], v[3], v[4], v[5], v[6], p, None, D, n, Bq, groups,
                                                         bit, 32 // bit)
    o = mpq.decode_attention_quant(k, v, q, groups, bit)
    assert _rel(o, ref.float().view(Bq, D)) < 5e-3


@pytest.mark.parametrize("bit,large", [(4, 11008), (8, 6144)])
@pytest.mark.parametrize("step_launch", [True, False])
def test_a_cache_of_either_capacity(bit, large, step_launch):
    """The same tokens in a small and in a large cache: every wavefront has one block in both, so the partials are the same
    numbers.  The window's stand further back among the slots of the large one and meet the others in another order: a few
    2^-24 of the largest weighted value, and one fp16 rounding (2^-11) to either side."""
    from mustafar_amd.cache import QuantSparseKVCache
    bs, n_kv, g, L = 6, 4, 4, 1309
    gen = torch.Generator(device="cuda")
    gen.manual_seed(bit)
    K = torch.randn((bs, n_kv, L, D), generator=gen, device="cuda", dtype=torch.float16)
    V = torch.randn((bs, n_kv, L, D), generator=gen, device="cuda", dtype=torch.float16)
    proj = torch.randn((bs, (g + 2) * n_kv * D), generator=gen, device="cuda", dtype=torch.float16)
    cos = torch.ones(D, device="cuda", dtype=torch.float16)
    outs = []
    for max_tokens in (1280, large):
        c = QuantSparseKVCache(g, D, 0.7, 0.7, 256, bit=bit, window_kernel=True, max_tokens=max_tokens)
        c.step_launch = step_launch
        c.prefill(K, V)
        nq, nk = g * n_kv * D, n_kv * D
        outs.append(c.decode_device_proj(proj[:, :nq], proj[:, nq:nq + nk], proj[:, nq + nk:], cos, cos * 0))
    a, b = outs[0].float(), outs[1].float()
    assert ((a - b).abs() <= 2.0 ** -10 * a.abs() + 2.0 ** -20 * a.abs().amax()).all()
