"""Which quantised attention calls over few blocks share them (quant_shares, csrc/fused_quant.hip): not those over many heads of one to
four blocks, where one launch without a merge is the faster form.  Seen by the workspace, which only the shared form writes to where
neither a window nor (max, sum) asks for a merge; either way the numbers are those of the calls that do merge."""
import pytest
import torch

pytestmark = pytest.mark.gpu
D = 128


@pytest.mark.parametrize("bit,group_size,heads,groups,blocks,shares", [
    (2, 64, 256, 4, 4, False), (2, 64, 192, 4, 4, True), (2, 64, 512, 3, 2, False), (2, 64, 512, 2, 2, True), (2, 64, 128, 4, 8, True),
    (8, 64, 256, 4, 4, False), (8, 64, 257, 4, 3, True), (4, 64, 256, 4, 4, True),
    (2, 64, 512, 8, 1, False), (2, 64, 341, 8, 1, True), (2, 64, 513, 8, 1, True), (2, 64, 256, 8, 3, False), (2, 64, 128, 8, 4, True), (2, 64, 160, 8, 4, False),
    (2, 32, 512, 8, 1, False), (2, 32, 256, 8, 3, True), (4, 64, 256, 8, 3, False), (4, 64, 257, 8, 2, True), (8, 64, 256, 8, 3, True), (4, 32, 256, 8, 3, True)])
def test_route(bit, group_size, heads, groups, blocks, shares):
    from mustafar_amd import compression_quant as cq, mustafar_package_quant as mq, ops
    g = torch.Generator(device="cuda").manual_seed(heads * blocks + bit)
    tokens, rows = blocks * 64, heads * groups
    K, V = (torch.randn((heads, tokens, D), generator=g, device="cuda", dtype=torch.float16) for _ in range(2))
    q = 0.25 * torch.randn((rows, D), generator=g, device="cuda", dtype=torch.float16)
    kth = 89 if bit < 8 else 40
    k = cq.convert_key_batched_quant(K, True, bit, group_size, kth=kth)
    v = cq.convert_value_batched_quant(V, bit, group_size, kth=kth)
    room = torch.full((rows * blocks * 520 + 256,), 255, dtype=torch.uint8, device="cuda")
    got = mq.decode_attention_quant(k, v, q, groups, bit, ws=room)
    assert bool((room != 255).any()) == shares
    merged = mq.decode_attention_quant(k, v, q, groups, bit, ws=room, lse=torch.empty((rows, 2), device="cuda"))
    assert torch.equal(got.view(torch.int16), merged.view(torch.int16))
