"""What the Python layer in front of the native calls (csrc/host.cpp) refuses itself."""
import pytest
import torch

D = 128


def test_wrong_number_of_dimensions():
    from mustafar_amd import compression_quant as cq, ops
    for shape in ((D,), (64, D)):
        x = torch.zeros(shape, dtype=torch.float16)
        for call in (lambda: ops.compress_kv(x, x), lambda: ops.compress_proj(x, True, 0, 64), lambda: cq.convert_value_batched_quant(x)):
            with pytest.raises(AssertionError):
                call()


def test_negative_capacity():
    from mustafar_amd import ops
    k, rows = torch.zeros((1, 64, D), dtype=torch.float16), torch.zeros((1, 64, 1, D), dtype=torch.float16)
    for capacity in (-1, -8):
        with pytest.raises(RuntimeError, match="capacity"):
            ops.compress_kv(k, k, capacity_halfs=capacity)
        with pytest.raises(RuntimeError, match="capacity"):
            ops.compress_proj(rows, True, 0, 64, capacity_halfs=capacity)


@pytest.mark.gpu
def test_units_without_counts_are_not_looked_at():
    from mustafar_amd import compression_quant as cq, mustafar_package_quant as mpq
    from mustafar_amd._lib import host
    x = torch.randn((1, 64, D), device="cuda", dtype=torch.float16)
    b = torch.randn((1, 8, D), device="cuda", dtype=torch.float16)
    bmp, off, packed, counts, units, scales, zeros = cq.convert_key_batched_quant(x, True, 4, kth=89)
    tail = (scales, zeros, b, 64, D, 1, 1, 4, 8, 0)
    want = host().key_formulation_quant(bmp, packed, off, counts, units, *tail)
    assert torch.equal(host().key_formulation_quant(bmp, packed, off, None, units.long().cpu(), *tail), want)
    assert torch.equal(mpq.mustafar_key_formulation_quant(bmp, packed, off, scales, zeros, b, 64, D, 1, 1, 4, 8), want)
