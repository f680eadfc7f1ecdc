"""Drop-in for the reference's kernel_quant/compression_quant.py (convert_key_batched_quant :159-264,
convert_value_batched_quant :425-529): same arguments and return tuples.  The reference hard-codes
2-bit codes; `bit` is exposed here as an extra keyword (2, 4 or 8; capacity = 32 // bit), and `group_size`
(64 = one scale / zero pair per tile as in the reference; 32 = two, scales and zeros then [B, T, 2]).

inputs: [B, M, N] fp16 on the GPU, already pruned (or pruned here: `kth`), M % 64 == 0.  The converters wait for the size of
the packed words and copy these out by a launch behind that, as the reference does: results are complete in the order of the
current stream.
"""
import torch

from . import ops
from ._lib import host


def _produce(inputs, is_value, bit, kth=0, group_size=64, ws=None, room=None, sized=False):
    """One call of the producer.  room: int32 tensor that takes the packed words (tile offsets count from its start;
    a tile whose words would pass its end is not written, and the total then exceeds room.numel());
    default: a fresh buffer with room for the worst case.  Returns the per-tile arrays, the buffer and the word total
    as a device tensor (all ones should a wait of the one-pass producer have run out) - nothing is read on the host.
    sized: the total as an int instead."""
    assert inputs.dim() == 3
    B, M, _ = inputs.shape
    own = ops._own_workspace(ws, inputs.device) if sized else None
    words = own.status(ops.status_words(B * (M // 64))) if own else None
    out = ops._call(host().produce_quant, ws, inputs.device, None, inputs, int(bool(is_value)), int(bit), int(kth),
                    int(group_size), room, ops._landing_word()[1] if sized else 0, words)
    if sized and out[-1] < 0:
        ops.gave_up(own, words, _GAVE_UP)
    return out


_GAVE_UP = "the quantised producer gave up waiting for an earlier workgroup; the packed words are incomplete"


def words_written(total):
    """The producer's word total on the host (one read, as the reference's .item()); raises if the producer gave up."""
    n = ops.read_word(total)
    if n < 0:   # all ones: a workgroup of the one-pass producer gave up waiting (ruled out by the dispatch order)
        raise RuntimeError(_GAVE_UP)
    return n


def _convert(inputs, is_value, bit, kth=0, group_size=64, ws=None):
    bmp, tile_off, room, counts, units, scales, zeros, total = _produce(inputs, is_value, bit, kth, group_size, ws, sized=True)
    # the used part is copied out so that the large buffer goes back to the allocator
    packed = room[:words_written(total)].clone()
    return bmp, tile_off, packed, counts, units, scales, zeros


def convert_key_batched_quant(inputs: torch.Tensor, return_metadata: bool = False, bit: int = 2, group_size: int = 64,
                              ws=None, kth: int = 0):
    """kth > 0 (an extra of this build): the rows are pruned to that rank inside the producer, as dh_prune_key would
    have done in front of it (models/llama_mustafar_quant_kernel.py), with one read of the dense rows."""
    bmp, tile_off, packed, counts, units, scales, zeros = _convert(inputs, False, bit, kth, group_size, ws)
    if return_metadata:
        return bmp, tile_off, packed, counts, units, scales, zeros
    return bmp, tile_off, packed, scales, zeros


def convert_value_batched_quant(inputs: torch.Tensor, bit: int = 2, group_size: int = 64, ws=None, kth: int = 0):
    return _convert(inputs, True, bit, kth, group_size, ws)
