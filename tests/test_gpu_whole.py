"""A workgroup of sixteen wavefronts per head, without a merge (fused_whole_head, csrc/fused_common.hpp): the two splits of a
head in one workgroup, or up to eight blocks shared by pairs of wavefronts.  Sums and their order are those of the split form
and its merge, so the output must be the same numbers, bit for bit, as from the two-phase entry points, which never take it.
Sizes: one block to sixteen, more than that at head counts on both sides of the rule, up to eight query heads; blocks that
hold nothing (pruned to one value in another block's favour) and infinities."""
import pytest
import torch

pytestmark = pytest.mark.gpu
D = 128


def sides(heads, tokens, seed=1):
    g = torch.Generator(device="cuda").manual_seed(seed)
    K, V = (torch.randn((heads, tokens, D), generator=g, device="cuda", dtype=torch.float16) for _ in range(2))
    K[:, :, 7] *= 10
    return K, V, g


def compare(K, V, q, groups, kth=89, infinite=False):
    from mustafar_amd import ops
    heads, tokens = K.shape[:2]
    ck, cv = ops.compress(K, False, kth=kth), ops.compress(V, True, kth=kth)
    o = ops.decode_attention(ck, cv, q, groups)
    if tokens <= 512 and infinite:  # (one split: the merge of the two phases would multiply its infinite outputs by zero)
        o2 = ops.decode_attention(ck, cv, q, groups, lse=torch.empty((heads * groups, 2), device="cuda"))
    else:
        ws = ops.decode_attention_partial(ck, cv, q, groups, ws=ops.Workspace("cuda", 64 << 20))
        o2 = ops.decode_attention_merge(ws, tokens, D, heads * groups, groups)
    odd = o.isnan()
    assert torch.equal(odd, o2.isnan()) and torch.equal(o.view(torch.int16)[~odd], o2.view(torch.int16)[~odd])


SHAPES = [(1, 1, 1), (1, 4, 2), (2, 3, 3), (8, 4, 8), (8, 2, 7), (256, 4, 8), (257, 4, 5), (1, 4, 9), (3, 8, 9), (5, 5, 15), (64, 4, 16),
          (8, 8, 16), (256, 8, 12), (257, 4, 16), (223, 1, 17), (224, 4, 17), (256, 4, 40), (230, 8, 21), (256, 1, 33)]


@pytest.mark.parametrize("heads,groups,blocks", SHAPES)
def test_the_same_numbers_as_in_two_phases(heads, groups, blocks):
    K, V, g = sides(heads, blocks * 64)
    q = torch.randn((heads * groups, D), generator=g, device="cuda", dtype=torch.float16)
    compare(K, V, q, groups)


@pytest.mark.parametrize("heads,groups,blocks", [(2, 4, 6), (2, 4, 13), (1, 8, 10)])
def test_empty_blocks_and_infinities(heads, groups, blocks):
    """A block of zeros (its tiles are empty), one with an infinite value, one with an infinite key."""
    K, V, g = sides(heads, blocks * 64, 2)
    K[:, 64:128], V[:, 64:128] = 0, 0
    q = torch.randn((heads * groups, D), generator=g, device="cuda", dtype=torch.float16)
    compare(K, V, q, groups, kth=0)
    V[0, 200, 3] = float("inf")
    compare(K, V, q, groups, kth=0, infinite=True)
    K[0, 300, 5] = float("-inf")
    compare(K, V, q, groups, kth=0, infinite=True)


@pytest.mark.parametrize("bit,group_size", [(2, 64), (2, 32), (4, 64), (4, 32), (8, 64)])
@pytest.mark.parametrize("heads,groups,blocks", [(1, 4, 9), (3, 4, 16), (256, 4, 12), (224, 2, 18), (256, 4, 20), (2, 8, 13)])
def test_quantised_the_same_numbers_as_with_max_and_sum(bit, group_size, heads, groups, blocks):
    """The call that also returns (max, sum) goes by way of the splits."""
    from mustafar_amd import compression_quant as cq, mustafar_package_quant as mpq
    K, V, g = sides(heads, blocks * 64, 3)
    k = cq.convert_key_batched_quant(K, True, bit, group_size, kth=89)
    v = cq.convert_value_batched_quant(V, bit, group_size, kth=89)
    q = torch.randn((heads * groups, D), generator=g, device="cuda", dtype=torch.float16)
    lse = torch.empty((heads * groups, 2), device="cuda")
    a, b = mpq.decode_attention_quant(k, v, q, groups, bit), mpq.decode_attention_quant(k, v, q, groups, bit, lse=lse)
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("heads,groups,blocks", [(1, 4, 4), (8, 4, 8), (3, 8, 1), (80, 4, 8), (81, 4, 8), (2, 7, 6)])
def test_recorded_calls_give_the_same_numbers(heads, groups, blocks):
    """Calls without a split share blocks when they are recorded; the workspace may be too small for that."""
    from mustafar_amd import ops
    K, V, g = sides(heads, blocks * 64, 4)
    ck, cv = ops.compress(K, False, kth=89), ops.compress(V, True, kth=89)
    q = torch.randn((heads * groups, D), generator=g, device="cuda", dtype=torch.float16)
    small = torch.empty(ops.attention_workspace_least(blocks * 64, 0, heads * groups), dtype=torch.uint8, device="cuda")
    for ws in (ops.Workspace("cuda"), small):
        ops.decode_attention(ck, cv, q, groups, ws=ws)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            o = ops.decode_attention(ck, cv, q, groups, ws=ws)
        for _ in range(3):
            q.copy_(torch.randn(q.shape, generator=g, device="cuda", dtype=torch.float16))
            graph.replay()
            assert torch.equal(o.view(torch.int16), ops.decode_attention(ck, cv, q, groups, ws=ws).view(torch.int16))


@pytest.mark.parametrize("heads,groups,blocks", [(160, 8, 1), (161, 8, 1), (112, 5, 3), (113, 5, 3), (128, 8, 5), (129, 8, 5), (128, 5, 2),
                                                 (129, 5, 2), (257, 5, 2), (640, 5, 1), (641, 5, 1)])
def test_recorded_calls_at_the_lines_of_their_rule(heads, groups, blocks):
    test_recorded_calls_give_the_same_numbers(heads, groups, blocks)
