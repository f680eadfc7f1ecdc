"""How a value product numbers its workgroups (value_index): one to 157 token splits per head, powers of two and not, one and two
halves of the channels, surplus workgroups of the rounded grid."""
import pytest
import torch

from test_gpu_walk import close, product, pruned

pytestmark = pytest.mark.gpu


# (up to eight rows a split covers 512 tokens here, so that tokens / 512, rounded up, is the number of splits)
@pytest.mark.parametrize("heads,tokens", [(5, 512), (7, 576), (3, 1536), (5, 2496), (9, 3584), (3, 4096), (2, 5696), (1, 80384)])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bit,groups,n_rows", [(0, 4, 1), (0, 2, 8), (4, 4, 1)])
def test_every_split_finds_its_tokens(heads, tokens, D, bit, groups, n_rows):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(tokens + D)
    V = pruned(gen, heads, tokens, D)
    p = torch.rand((heads, groups * n_rows, tokens), generator=gen, device="cuda").half() / 64
    out, rows = product(V, p, True, bit, groups, n_rows)
    close(out, p, rows)
