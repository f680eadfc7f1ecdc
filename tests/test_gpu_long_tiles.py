"""Tiles of more than 32 survivors in the fused attention over codes (StageRank, csrc/quant_device.hpp): with 2 bits a stage of 32
tiles with at most two of them is gathered from an image with zeros in front of every tile's values and those two are fetched
one by one; with more, and until a stage without any, the stages go under exec masks.  Stages with 0 to 32 such tiles follow each
other here in every order, of 33, 48, 49, 63 and 64 survivors beside tiles of 32, 31, one and none, and one, two and several
blocks a wavefront.  Reference: dense attention over the oracle's dequantised rows; the bound is the one of the fp16 path (scores
rounded to fp16 in front of the softmax, and small here)."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu
D = 128


def rows(rng, heads, tokens, is_value):
    """Values whose tiles hold a chosen number of survivors, by stage: `long` of 33 .. 64, the others 0, 1, 31 or 32."""
    x = rng.standard_normal((heads, tokens // 64, 256 // 2, 64)).astype(np.float16)      # [head, block, tile, element]
    x[x == 0] = 1
    for h in range(heads):
        for b in range(tokens // 64):
            for st in range(4):
                many = [0, 2, 1, 3, 0, 32, 1, 0, 2, 8][(h + 4 * b + st) % 10]
                for t in range(32):
                    n = rng.choice([33, 48, 49, 63, 64]) if t in (5 * many % 32,) or t < many - 1 else rng.choice([0, 1, 31, 32, 19])
                    x[h, b, st * 32 + t, rng.permutation(64)[n:]] = 0
    if not is_value:     # tile = channel, element = token
        return np.ascontiguousarray(x.transpose(0, 1, 3, 2)).reshape(heads, tokens, D)
    x = x.reshape(heads, tokens // 64, 2, 64, 64)    # [head, block, half, token, channel]
    return np.ascontiguousarray(x.transpose(0, 1, 3, 2, 4)).reshape(heads, tokens, D)


@pytest.mark.parametrize("bit,group_size", [(2, 64), (2, 32), (4, 64), (8, 64)])
@pytest.mark.parametrize("heads,groups,tokens", [(2, 4, 640), (3, 1, 128), (2, 8, 576), (3, 7, 64)])
def test_stages_with_and_without_long_tiles(bit, group_size, heads, groups, tokens):
    check(bit, group_size, heads, groups, tokens)


@pytest.mark.parametrize("heads,tokens", [(224, 1088), (300, 1024)])
def test_several_blocks_a_wavefront(heads, tokens):
    check(2, 64, heads, 4, tokens, repeat=4)


def check(bit, group_size, heads, groups, tokens, repeat=None):
    from mustafar_amd import compression_quant as cq
    from mustafar_amd import mustafar_package_quant as mq
    rng = np.random.default_rng(heads * tokens)
    base = repeat or heads       # (a few heads repeated where there are many: the oracle is slow)
    K, V = rows(rng, base, tokens, False), rows(rng, base, tokens, True)
    q = (0.25 * rng.standard_normal((base * groups, D))).astype(np.float16)
    dense = []
    for x, is_value in ((K, 0), (V, 1)):
        fn = cq.convert_value_batched_quant if is_value else cq.convert_key_batched_quant
        host = [t.cpu().numpy() for t in fn(torch.from_numpy(x).cuda(), True, bit, group_size)] if not is_value else [
            t.cpu().numpy() for t in fn(torch.from_numpy(x).cuda(), bit, group_size)]
        dense.append(np.stack([orc.decode_quant(host[0], host[2], host[1], host[5], host[6], h, tokens, D, is_value, bit, 0)
                               for h in range(base)]).astype(np.float16))
    want = orc.dense_masked_attention(q, dense[0], dense[1], groups)[2].astype(np.float64)
    n = -(-heads // base)
    tile = lambda a: torch.from_numpy(np.tile(a, (n,) + (1,) * (a.ndim - 1))).cuda()     # noqa: E731
    k = cq.convert_key_batched_quant(tile(K)[:heads].contiguous(), True, bit, group_size)
    v = cq.convert_value_batched_quant(tile(V)[:heads].contiguous(), bit, group_size)
    got = mq.decode_attention_quant(k, v, tile(q)[:heads * groups].contiguous(), groups, bit).float().cpu().numpy()
    want = np.tile(want, (n, 1))[:heads * groups]
    err = np.abs(got - want).max(-1) / np.abs(want).max(-1)
    assert err.max() < 2e-3, (err.max(), int(err.argmax()))
