"""Sizes that the producers hand over before their last values are stored (ops.compress_kv, compress_proj, the quantised
converters): the arrays are complete where their stream has come to, as with any torch call - for another stream behind an event
or wait_stream made after the call."""
import pytest
import torch

pytestmark = pytest.mark.gpu
D, KTH = 128, 89


def test_another_stream_behind_the_call():
    from mustafar_amd import compression_quant as cq, ops
    g = torch.Generator(device="cuda").manual_seed(9)
    heads, tokens = 64, 2048
    x = [torch.randn((heads, tokens, D), generator=g, device="cuda", dtype=torch.float16) for _ in range(2)]
    cos, sin = (torch.randn((tokens, D), generator=g, device="cuda").clamp(-1, 1).half() for _ in range(2))
    rows = x[0].view(1, heads, tokens, D).transpose(1, 2)

    def results():
        k, v = ops.compress_kv(*x, KTH, KTH)
        p, rot = ops.compress_proj(rows, False, KTH, tokens - 64, cos, sin, torch.empty_like(rows))
        q = cq.convert_value_batched_quant(x[1], 2, kth=KTH)
        return [k.packed(), v.packed(), k.idx, v.bmp, p.nz, p.idx, rot, q[0], q[1], q[2], q[5]]

    want = [t.clone() for t in results()]
    torch.cuda.synchronize()
    producer, consumer = torch.cuda.Stream(), torch.cuda.Stream()
    for _ in range(20):
        with torch.cuda.stream(producer):
            got = results()
        consumer.wait_stream(producer)
        with torch.cuda.stream(consumer):
            copies = [t.clone() for t in got]
        producer.wait_stream(consumer)
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(copies, want))
