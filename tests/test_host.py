"""The native calls in front of the C ABI (csrc/host.cpp): what they refuse, with the error types and texts of the reference's
own checks, and what they do with the scratch memory that they are given."""
import pytest
import torch

D = 128


def fp16_args():
    return [torch.zeros((1, 128), dtype=torch.int64), torch.zeros(8, dtype=torch.float16), torch.zeros((1, 129), dtype=torch.int32),
            torch.zeros(1, dtype=torch.int32), torch.zeros((1, 8, D), dtype=torch.float16)]


@pytest.mark.parametrize("at,to,text", [(0, torch.int32, "Tensor bmp must be of type int64."),
                                        (1, torch.float32, "Tensor NZ must be of type float16."),
                                        (2, torch.int64, "Tensor idx must be of type int."),
                                        (3, torch.int64, "Tensor NZ_Offset must be of type int."),
                                        (4, torch.float32, "Tensor B must be of type float16."),
                                        (None, None, "must be on CUDA device.")])
def test_operators_refuse_as_the_reference_does(at, to, text):
    from mustafar_amd import mustafar_package as mp
    for fn, tail in ((mp.mustafar_key_formulation, (64, D, 1, 1)), (mp.mustafar_value_formulation, (None, D, 64, 1, 1))):
        args = fp16_args()
        if at is not None:
            args[at] = args[at].to(to)
        with pytest.raises(RuntimeError, match=text.replace(".", r"\.")):
            fn(*args, *tail)


def test_quantised_operators_refuse_as_the_reference_does():
    from mustafar_amd import mustafar_package_quant as mpq
    i32 = torch.zeros((1, 128), dtype=torch.int32)
    half = torch.zeros((1, 128), dtype=torch.float16)
    good = [torch.zeros((1, 128), dtype=torch.int64), torch.zeros(8, dtype=torch.int32), i32, i32, i32, half, half,
            torch.zeros((1, 8, D), dtype=torch.float16)]
    for at, to, text in ((0, torch.int32, "bmp must be of type int64"), (1, torch.float16, "NZ_quant must be of type int32"),
                         (2, torch.int64, "tile_offsets must be of type int32"), (3, torch.int64, "tile_counts must be of type int32"),
                         (4, torch.int64, "tile_units must be of type int32"), (5, torch.float32, "scales must be of type float16"),
                         (6, torch.float32, "zeros must be of type float16"), (7, torch.float32, "B must be of type float16"),
                         (0, torch.int64, "must be on CUDA device")):
        args = list(good)
        args[at] = args[at].to(to)
        with pytest.raises(RuntimeError, match=text):
            mpq.mustafar_key_formulation_quant_meta(*args, 64, D, 1, 1, 2, 16)


def test_arguments_that_are_no_tensors_or_of_the_wrong_kind():
    from mustafar_amd import ops
    from mustafar_amd._lib import host
    with pytest.raises(TypeError):
        host().scale_softmax(3, D, None)
    with pytest.raises(TypeError):
        host().scale_softmax(torch.zeros((1, 64), dtype=torch.float16), D)
    with pytest.raises(AssertionError):
        ops.scale_softmax(torch.zeros((1, 64)), D)
    with pytest.raises(AssertionError):
        ops.compress_kv(torch.zeros((1, 64, D)), torch.zeros((1, 64, D)))
    with pytest.raises(OverflowError):
        host().scale_softmax(torch.zeros((1, 64), dtype=torch.float16), 1 << 40, None)


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [64, 640, 4096])
def test_scratch_memory(tokens):
    """A buffer that is too small is refused as such, a Workspace grows, none at all means the stream's own: same numbers."""
    from mustafar_amd import compression_quant as cq, mustafar_package_quant as mpq, ops
    g = torch.Generator(device="cuda").manual_seed(tokens)
    k, v = (torch.randn((2, tokens, D), generator=g, device="cuda", dtype=torch.float16) for _ in range(2))
    q = torch.randn((8, D), generator=g, device="cuda", dtype=torch.float16)
    ck, cv = ops.compress(k, False, 89), ops.compress(v, True, 89)
    qk, qv = cq.convert_key_batched_quant(k, True, 4, kth=89), cq.convert_value_batched_quant(v, 4, kth=89)
    for call in (lambda ws: ops.decode_attention(ck, cv, q, 4, ws=ws),
                 lambda ws: mpq.decode_attention_quant(qk, qv, q, 4, 4, ws=ws),
                 lambda ws: ops.compress_kv(k, v, 89, 89, ws=ws)[1].packed()):
        with pytest.raises(RuntimeError, match="workspace"):
            call(torch.empty(64, dtype=torch.uint8, device="cuda"))
        small = ops.Workspace("cuda", 256)
        want = call(None)
        assert torch.equal(call(small), want) and torch.equal(call(small), want) and small.tensor.numel() > 256
        assert torch.equal(call(torch.empty(1 << 22, dtype=torch.uint8, device="cuda")), want)
    with pytest.raises(AssertionError):
        ops.decode_attention(ck, cv, q.float(), 4)
    out = torch.empty_like(q)
    lse = torch.empty((8, 2), device="cuda")
    assert ops.decode_attention(ck, cv, q, 4, out=out, lse=lse) is not None
    assert torch.equal(out, ops.decode_attention(ck, cv, q, 4)) and bool((lse[:, 1] > 0).all())


@pytest.mark.parametrize("heads,tokens,sides", [(1, 64, 1), (3, 192, 2), (60, 4800, 1), (128, 4096, 2)])
def test_status_words(heads, tokens, sides):
    from mustafar_amd import ops
    from mustafar_amd._lib import lib
    assert 8 * ops.status_words(heads * (tokens // 64), sides) == lib().mstf_status_bytes(heads, tokens, sides)
