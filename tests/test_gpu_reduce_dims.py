"""sum and mean over dims where the tensor lies: columns, rows and a channel's
planes, at the edges of the vector, of the row groups and of the chunks, in
every dim order that is dense, and orders that are not."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float64: 0.0}


def seeded(shape, seed, dtype=torch.float32):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(dtype)


def check(x, dx, dims, keepdim=False):
    want = x.double().sum(dims, keepdim)
    n = x.numel() // max(want.numel(), 1)
    # float32 sums, each element in at most n / 256 + 40 of the additions one
    # after another: columns add trees of 8, eight of those, a thread's eights
    # (n / 256 with four row groups), then the groups; rows eight of a vector,
    # a thread's vectors (n / 1024), then the threads; a chunk's rows and the
    # chunks likewise.  Then one rounding
    u = 2.0 ** -53 if x.dtype == torch.float64 else 2.0 ** -24
    tol = x.double().abs().sum(dims, keepdim) * (n / 256 + 40) * u
    got = dx.sum(dims, keepdim)
    assert got.shape == want.shape and got.dtype == x.dtype
    err = (got.cpu().double() - want).abs()
    assert (err <= tol + EPS[x.dtype] * want.abs()).all(), float(err.max())
    err = (dx.mean(dims, keepdim).cpu().double() - want / n).abs()
    assert (err <= (tol + 2 * 2.0 ** -24 * want.abs()) / n + EPS[x.dtype] * want.abs() / n).all(), float(err.max())
    assert torch.equal(got.cpu(), dx.sum(dims, keepdim).cpu())  # the same bits again


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16, torch.float64])
@pytest.mark.parametrize("shape", [(1, 9), (2, 7), (16, 64), (17, 257), (33, 1023), (4099, 130), (8192, 40), (100003, 3),
                                   (70001, 17), (3, 70001), (3, 32769), (4100, 2051)])
def test_columns_and_rows(shape, dtype, no_fallback):
    x = seeded(shape, 1, dtype)
    for dx, cx in ((x.to("supa"), x), (x.to("supa").t(), x.t())):
        check(cx, dx, 0)
        check(cx, dx, 1, True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(2, 3, 5), (5, 4099, 6), (64, 31, 49), (300, 2, 8), (3, 16, 8192), (2, 1, 40000)])
def test_three_dims(shape, dtype, no_fallback):
    x = seeded(shape, 2, dtype)
    dx = x.to("supa")
    for dims in (0, 1, 2, (0, 1), (0, 2), (1, 2)):
        check(x, dx, dims)
    p = dx.permute(2, 0, 1)  # dense in another order: kept dims in and out of their own order
    for dims in (0, 1, 2, (0, 2), (1, 2)):
        check(x.permute(2, 0, 1), p, dims)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows", [300, 4096, 9000])
def test_precision_of_many_columns(rows, dtype, no_fallback):
    """Columns that fill the chip alone, so that a thread adds a quarter of the
    rows: against 64 bits.  The squared rounding errors of a sum of n equal
    variances add up to about (n / 512 + 16) / 3 of 2^-48 with chains of n / 256
    (one chain of n / 4 additions: n / 8 / 3)."""
    x = seeded((rows, 128), 6, dtype)
    want = x.double().sum(0)
    wide = x.to("supa").unsqueeze(1).expand(rows, 1040, 128).reshape(rows, -1)
    got = wide.sum(0, dtype=torch.float32).view(-1, 128)
    assert bool((got == got[0]).all())
    err = (got[0].cpu().double() - want).norm() / want.norm()
    assert err <= ((rows / 512 + 16) / 3) ** 0.5 * 2.0 ** -24, float(err)


def test_other_layouts_and_types(no_fallback):
    x = seeded((6, 7, 8, 9), 3)
    dx = x.to("supa")
    for dims in ((1, 3), (0, 2), 0, 3, (0, 1, 2)):  # kept, reduced, kept, reduced
        check(x, dx, dims)
    check(x[:, ::2], dx[:, ::2], 1)
    check(x[:, 1:5, 2:, 1:], dx[:, 1:5, 2:, 1:], (0, 3))
    check(x[:1].expand(5, 7, 8, 9), dx[:1].expand(5, 7, 8, 9), 0)
    buf = torch.empty(7 * 13 + 1, dtype=torch.bfloat16, device="supa")
    odd = buf[1:].view(7, 13)
    y = seeded((7, 13), 4, torch.bfloat16)
    odd.copy_(y.to("supa"))
    check(y, odd, 0)
    check(y, odd, 1)
    for dt in (torch.int64, torch.int32, torch.int8, torch.bool):
        i = (seeded((300, 77), 5) * 3).to(dt)
        for d in (0, 1):
            assert torch.equal(i.to("supa").sum(d).cpu(), i.sum(d))
    z = dx.clone()
    torch.sum(z, 0, out=z[1])  # the result over a part of the input
    np.testing.assert_allclose(z[1].cpu().numpy(), x.sum(0).numpy(), rtol=1e-5, atol=1e-5)
    for special in (float("nan"), float("inf")):
        w = x.clone()
        w[2, 3, 4, 5] = special
        got, want = w.to("supa").sum(0).cpu(), w.sum(0)
        assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))


@pytest.mark.parametrize("shape, dim", [((1 << 22, 64 + 1, 2), 2), ((1 << 23, 64, 17, 2), 2)])
def test_more_results_than_one_launch(shape, dim, no_fallback):
    """More threads than a launch holds: 2^28 rows, and 2^30 columns in planes of two."""
    if torch.supa.mem_get_info()[0] < 80 << 30:
        pytest.skip("takes 45 GiB of device memory")
    small = seeded(shape[1:], 7, torch.bfloat16).to("supa")
    x = torch.empty(shape, dtype=torch.bfloat16, device="supa")
    x.copy_(small)
    want = small.sum(dim - 1)
    got = x.view(-1, *shape[2:]).sum(dim - 1).view(shape[0], *want.shape)
    del x
    assert bool((got == want).all())
    del got
    torch.supa.empty_cache()
