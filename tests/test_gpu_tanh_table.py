"""The tanh activations of large bf16 tensors, whose tanh comes from a table,
are bit for bit those of small ones, over every bf16 value."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

EVERY = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)


def same(got, want):
    got, want = got.cpu(), want.cpu()
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(got), nan)
    assert torch.equal(got.view(torch.int16)[~nan], want.view(torch.int16)[~nan])


# the smallest that takes the table, with a remainder, past one vector a
# thread, past the growing grid
@pytest.mark.parametrize("n", [1 << 20, (1 << 20) + 3, (1 << 22) + 8 * 1024 + 5, (1 << 25) + (1 << 16) + 1])
def test_large_calls_equal_small_ones(n, no_fallback):
    x = EVERY.repeat(n // 65536 + 1)[:n].to("supa")
    dy = torch.randn(n, generator=torch.Generator().manual_seed(1)).bfloat16().to("supa")
    step = (1 << 20) - 8
    gelu = lambda a: F.gelu(a, approximate="tanh")
    for fn in (gelu, torch.tanh):
        same(fn(x), torch.cat([fn(x[i:i + step]) for i in range(0, n, step)]))
    bwd = lambda g, a: torch.ops.aten.gelu_backward(g, a, approximate="tanh")
    same(bwd(dy, x), torch.cat([bwd(dy[i:i + step], x[i:i + step]) for i in range(0, n, step)]))
    want = torch.tanh(x)
    x.tanh_()  # in place
    same(x, want)
