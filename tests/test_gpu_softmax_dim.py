"""log_softmax and softmax over a dim that is not the last one (the spatial
kernels): class counts around the edges of each split of the classes over
class groups, planes of every remainder of the vector, special values, and
the output written over the input."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import bf16_ulp_dist

pytestmark = pytest.mark.gpu

LSM_BWD = torch.ops.aten._log_softmax_backward_data
SM_BWD = torch.ops.aten._softmax_backward_data


def seeded(shape, seed, scale=1.0, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(dtype)


def rows_of(t):
    """[outer, cols, inner] -> [outer * inner, cols] float32."""
    return np.ascontiguousarray(np.moveaxis(t.float().numpy(), 1, 2)).reshape(-1, t.shape[1])


def planes_of(a, shape):
    return np.moveaxis(a.reshape(shape[0], shape[2], shape[1]), 2, 1)


def check_forward(got, ref, dtype):
    got = got.cpu()
    if dtype == torch.float32:
        np.testing.assert_allclose(got.numpy(), ref, rtol=1e-5, atol=1e-6)
    else:  # one rounding to the storage type of a float32 value: at most one unit in the last place
        r = torch.from_numpy(np.ascontiguousarray(ref)).to(dtype)
        a, b = (v.view(torch.int16).numpy().view(np.uint16) for v in (got.contiguous(), r))
        assert bf16_ulp_dist(a, b).max() <= 1


# a 16-bit gradient is one rounding too, of a difference whose terms' sum moves
# by `atol`: one unit in the last place, relative, on top of that
ULP = {torch.float32: 1e-5, torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}
# the smallest gradients: float32's own floor, half a unit of a float16 subnormal
FLOOR = {torch.float32: 1e-6, torch.bfloat16: 0.0, torch.float16: 2.0 ** -24}


def check_gradient(got, ref, dtype, atol):
    err = np.abs(got.cpu().float().numpy() - ref)
    assert (err <= ULP[dtype] * np.abs(ref) + FLOOR[dtype] + (1 + ULP[dtype]) * atol).all(), float(err.max())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(3, 1, 2), (2, 2, 3), (2, 7, 5), (3, 8, 64), (2, 9, 257), (5, 19, 1030), (2, 32, 33),
                                   (2, 33, 12), (1, 128, 71), (2, 129, 9), (2, 256, 15), (2, 257, 11), (2, 300, 8201),
                                   (70, 21, 4)])
def test_spatial_softmax_matches_oracle(shape, dtype, no_fallback):
    x = seeded(shape, 1, 2.0, dtype)
    g = seeded(shape, 2, 1.0, dtype)
    dx, dg = x.to("supa"), g.to("supa")
    for log, fwd, bwd, ofwd, obwd in ((True, torch.log_softmax, LSM_BWD, O.log_softmax, O.log_softmax_backward),
                                      (False, torch.softmax, SM_BWD, O.softmax, O.softmax_backward)):
        y = fwd(dx, 1)
        assert y.is_contiguous()
        check_forward(y, planes_of(ofwd(rows_of(x)), shape), dtype)
        gi = bwd(dg, y, 1, dtype)
        # a gradient is p (g - S) or g - p S: two float32 sums of the same C
        # terms differ by at most 2 (chain) 2^-24 sum|term|, chains of at most
        # C / 16 + 8 additions (or all C up to the 16 classes one thread holds)
        yc = y.cpu().double().numpy()
        p, terms = (np.exp(yc), g.double().numpy()) if log else (yc, g.double().numpy() * yc)
        atol = 2 * (shape[1] / 16 + 16) * 2.0 ** -24 * np.abs(terms).sum(1, keepdims=True) * p
        check_gradient(gi, planes_of(obwd(rows_of(g), rows_of(y.cpu())), shape), dtype, atol)


@pytest.mark.parametrize("shape", [(2, 19, 37), (2, 300, 4101), (2, 5, 3)])
def test_spatial_softmax_over_its_input(shape, no_fallback):
    x, g = seeded(shape, 3, 2.0), seeded(shape, 4)
    want = torch.log_softmax(x.to("supa"), 1)
    dx = x.to("supa")
    torch.ops.aten._log_softmax.out(dx, 1, False, out=dx)
    assert torch.equal(dx.cpu(), want.cpu())
    gi = LSM_BWD(g.to("supa"), want, 1, torch.float32)
    dg = g.to("supa")
    LSM_BWD.out(dg, want, 1, torch.float32, out=dg)
    assert torch.equal(dg.cpu(), gi.cpu())


def test_spatial_softmax_layouts_and_special_values(no_fallback):
    x = seeded((2, 5, 6, 7), 5, 2.0)
    x[0, 1, 0, 0] = float("nan")
    x[0, 2, 0, 1] = float("inf")
    x[0, :, 0, 2] = -float("inf")
    x[1, 3, 2, 3] = -float("inf")
    for f in (torch.log_softmax, torch.softmax):
        want = f(x, 1)
        for dx in (x.to("supa"), x.to("supa").to(memory_format=torch.channels_last),
                   x.transpose(2, 3).contiguous().to("supa").transpose(2, 3)):
            got = f(dx, 1).cpu()
            assert torch.equal(torch.isnan(got), torch.isnan(want))
            np.testing.assert_allclose(got.numpy(), want.numpy(), rtol=1e-5, atol=1e-6)
    h = torch._log_softmax(seeded((2, 5, 9), 6, 2.0, torch.bfloat16).to("supa"), 1, True)
    assert h.dtype == torch.float32
    np.testing.assert_allclose(h.cpu().numpy(), torch.log_softmax(seeded((2, 5, 9), 6, 2.0, torch.bfloat16).float(), 1),
                               rtol=1e-5, atol=1e-6)


def test_spatial_softmax_over_a_shifted_view(no_fallback):
    """An output that overlaps the input out of step is written after the input is read."""
    n, shape = 2 * 19 * 515, (2, 19, 515)
    x, g = seeded(shape, 7, 2.0), seeded(shape, 8)
    want = torch.softmax(x.to("supa"), 1)
    gwant = SM_BWD(g.to("supa"), want, 1, torch.float32)
    for off in (1, 515):
        buf = torch.empty(n + off, device="supa")
        src, dst = buf[:n].view(shape), buf[off:].view(shape)
        src.copy_(x.to("supa"))
        torch.ops.aten._softmax.out(src, 1, False, out=dst)
        assert torch.equal(dst.cpu(), want.cpu())
        src.copy_(g.to("supa"))
        SM_BWD.out(src, want, 1, torch.float32, grad_input=dst)
        assert torch.equal(dst.cpu(), gwant.cpu())


@pytest.mark.parametrize("shape", [(1, 4096, 128, 128), (1, 1000, 64, 128)])
def test_spatial_gradient_precision(shape, no_fallback):
    """The sums over many streamed classes against 64 bits.  A sum of n equal
    variances whose thread chains are n / 128 steps of 8 additions, then 16
    groups, carries about (n / 256 + 16) / 3 squared roundings of 2^-24; one
    chain of n / 16 additions, as before, n / 32 / 3 of them."""
    n, reps = shape[1], shape[3]
    g, y = (seeded(shape[:3], 9 + i) for i in range(2))
    p = y.double()
    want = p * (g.double() - (g.double() * p).sum(1, keepdim=True))
    dg, dy = (t.repeat(1, 1, reps).to("supa") for t in (g, y))
    got = SM_BWD(dg, dy, 1, torch.float32)
    err = (got[:, :, :shape[2]].cpu().double() - want).norm() / want.norm()
    assert err <= ((n / 256 + 16) / 3) ** 0.5 * 2.0 ** -24, float(err)
    assert torch.equal(got[:, :, -shape[2]:].cpu(), got[:, :, :shape[2]].cpu())


@pytest.mark.parametrize("shape", [(4, 1000, 2048), (2, 128, 4096), (2, 256, 2049)])
def test_spatial_softmax_precision(shape, no_fallback):
    """Over a middle dim, against 64 bits, as near as the same rows laid out last:
    there the maximum is known before the exponentials are added.  A rescale of
    each group's sum costs it two more roundings (3 to 8 % in all); the order of
    the additions, and the draw, 1 %."""
    x = torch.cat([seeded((1,) + shape[1:], 40 + i) for i in range(shape[0])])
    want = torch.softmax(x.double(), 1)

    def error(y):
        return float((y.cpu().double() - want).norm() / want.norm())

    mid = error(torch.softmax(x.to("supa"), 1))
    last = error(torch.softmax(x.transpose(1, 2).contiguous().to("supa"), 2).transpose(1, 2))
    assert mid <= 1.02 * last, (mid, last)


@pytest.mark.parametrize("log", [True, False])
def test_more_positions_than_one_launch(log, no_fallback):
    """2^28 positions of 33 classes: more threads than a launch holds."""
    if torch.supa.mem_get_info()[0] < 80 << 30:
        pytest.skip("takes 54 GiB of device memory")
    f = torch.log_softmax if log else torch.softmax
    small = seeded((64, 33, 2), 12, 2.0, torch.bfloat16).to("supa")
    want = f(small, 1)
    x = torch.empty(1 << 21, 64, 33, 2, dtype=torch.bfloat16, device="supa")
    x.copy_(small)
    y = f(x.view(-1, 33, 2), 1).view_as(x)
    for i in (0, (1 << 20) - 1, 1 << 20, (1 << 21) - 3, (1 << 21) - 1):
        assert torch.equal(y[i].cpu(), want.cpu())
    del x
    assert bool((y == want).all())
    del y
    torch.supa.empty_cache()
