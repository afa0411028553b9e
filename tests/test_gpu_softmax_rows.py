"""Row softmax, log_softmax and their gradients at the edges of the row
kernels: the longest row of each thread split and one element more, rows of
every remainder of the vector, rows whose base is not 16-byte aligned, the
output over the input, special values in every position of a short row."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import bf16_ulp_dist

pytestmark = pytest.mark.gpu

LSM_BWD = torch.ops.aten._log_softmax_backward_data
SM_BWD = torch.ops.aten._softmax_backward_data
ULP = {torch.float32: 1e-5, torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}


def seeded(shape, seed, scale=1.0, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(dtype)


def shifted(t):
    """The same values in a contiguous supa tensor one element off its allocation's alignment."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device="supa")
    v = buf[1:].view(t.shape)
    v.copy_(t.to("supa"))
    return v


# the smallest gradients: float32's own floor, half a unit of a float16 subnormal
FLOOR = {torch.float32: 1e-6, torch.bfloat16: 0.0, torch.float16: 2.0 ** -24}


def check_forward(got, ref, dtype, atol):
    got = got.cpu()
    if dtype == torch.float32:
        np.testing.assert_allclose(got.numpy(), ref, rtol=1e-5, atol=1e-6 + atol)
    else:  # one rounding to the storage type of a float32 value: at most one unit in the last place
        r = torch.from_numpy(np.ascontiguousarray(ref)).to(dtype)
        a, b = (v.view(torch.int16).numpy().view(np.uint16) for v in (got.contiguous(), r))
        assert bf16_ulp_dist(a, b).max() <= 1


def check(got, ref, dtype, atol):
    err = np.abs(got.cpu().float().numpy() - ref)
    assert (err <= ULP[dtype] * np.abs(ref) + FLOOR[dtype] + (1 + ULP[dtype]) * atol).all(), float(err.max())


def compare(x, g, dtype, to):
    cols = x.shape[1]
    dx, dg = to(x), to(g)
    for log, fwd, bwd, ofwd, obwd in ((True, torch.log_softmax, LSM_BWD, O.log_softmax, O.log_softmax_backward),
                                      (False, torch.softmax, SM_BWD, O.softmax, O.softmax_backward)):
        y = fwd(dx, 1)
        # log p carries the relative error of the sum: cols 2^-24 at most
        check_forward(y, ofwd(x.float().numpy()), dtype, cols * 2.0 ** -24 if log else 0.0)
        yc = y.cpu()
        gi = bwd(dg, to(yc), 1, dtype)
        # two float32 sums of the same terms, in chains of at most cols / 16 + 16 additions
        yd = yc.double().numpy()
        p, t = (np.exp(yd), g.double().numpy()) if log else (yd, g.double().numpy() * yd)
        atol = 2 * (cols / 16 + 16) * 2.0 ** -24 * np.abs(t).sum(1, keepdims=True) * p
        check(gi, obwd(g.float().numpy(), yc.float().numpy()), dtype, atol)


# vectors a row: the last of each thread split, and one more
VECS = [1, 2, 16, 17, 64, 65, 128, 129, 256, 257, 512, 513, 1024, 1025, 2048, 2049, 2560, 2561, 5121]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("vecs", VECS)
def test_rows_at_the_edges(vecs, dtype, no_fallback):
    v = 16 // torch.empty(0, dtype=dtype).element_size()
    for cols, rows in ((vecs * v, 5), (vecs * v - 1, 3), (vecs * v - v + 1, 19)):
        x, g = seeded((rows, cols), cols, 2.0, dtype), seeded((rows, cols), cols + 1, 1.0, dtype)
        compare(x, g, dtype, lambda t: t.to("supa"))
        compare(x, g, dtype, shifted)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("vecs, rows", [(128, 1535), (129, 1535), (129, 1536), (256, 1535), (256, 1536), (257, 1023),
                                        (257, 1024), (512, 3071), (512, 3072), (513, 599), (513, 600), (1024, 600),
                                        (1025, 599), (1025, 600), (2048, 600), (2049, 599), (2049, 600), (2560, 600)])
def test_rows_by_their_number(rows, vecs, dtype, no_fallback):
    """The thread splits that depend on the number of rows, on both sides of
    each line: every row as the same row is among few."""
    v = 16 // torch.empty(0, dtype=dtype).element_size()
    for cols in (vecs * v, vecs * v - 1):
        x, g = seeded((5, cols), cols, 2.0, dtype), seeded((5, cols), cols + 1, 1.0, dtype)
        dx, dg = (t.to("supa").expand(-(-rows // 5), 5, cols).reshape(-1, cols)[:rows] for t in (x, g))
        for log, fwd, bwd, ofwd, obwd in ((True, torch.log_softmax, LSM_BWD, O.log_softmax, O.log_softmax_backward),
                                          (False, torch.softmax, SM_BWD, O.softmax, O.softmax_backward)):
            last = slice(rows // 5 * 5 - 5, rows // 5 * 5)
            y = fwd(dx, 1)
            gi = bwd(dg, y, 1, dtype)
            for at in (slice(0, 5), last):
                yc = y[at].cpu()
                check_forward(yc, ofwd(x.float().numpy()), dtype, cols * 2.0 ** -24 if log else 0.0)
                yd = yc.double().numpy()
                p, t = (np.exp(yd), g.double().numpy()) if log else (yd, g.double().numpy() * yd)
                atol = 2 * (cols / 16 + 16) * 2.0 ** -24 * np.abs(t).sum(1, keepdims=True) * p
                check(gi[at], obwd(g.float().numpy(), yc.float().numpy()), dtype, atol)
            if cols % v == 0:  # rows of one alignment add in one order: as the rows repeat, so do the results
                for r in (y, gi):
                    same = bool((r[5:] == r[:-5]).all())
                    assert same


def test_more_rows_than_one_launch(no_fallback):
    """2^28 rows of 8: more threads than a launch holds."""
    if torch.supa.mem_get_info()[0] < 30 << 30:
        pytest.skip("takes 14 GiB of device memory")
    small, g = (seeded((64, 8), 12 + i, 2.0, torch.bfloat16).to("supa") for i in range(2))
    x = torch.empty(1 << 22, 64, 8, dtype=torch.bfloat16, device="supa")
    for f, b in ((torch.log_softmax, LSM_BWD), (torch.softmax, SM_BWD)):
        want = f(small, 1)
        x.copy_(small)
        y = f(x.view(-1, 8), 1)
        assert bool((y.view_as(x) == want).all())
        x.copy_(g)
        gi = b(x.view(-1, 8), y, 1, torch.bfloat16)
        assert bool((gi.view_as(x) == b(g, want, 1, torch.bfloat16)).all())
        del y, gi
    del x
    torch.supa.empty_cache()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("cols", [1, 3, 10, 16, 50257, 262147, 700001])
def test_ragged_rows(cols, dtype, no_fallback):
    x, g = seeded((3, cols), 5, 2.0, dtype), seeded((3, cols), 6, 1.0, dtype)
    compare(x, g, dtype, lambda t: t.to("supa"))


@pytest.mark.parametrize("cols", [50257, 128258])
def test_ragged_split_fallback_is_bit_identical(cols, no_fallback, monkeypatch):
    x, g = seeded((6, cols), 7, 2.0, torch.bfloat16).to("supa"), seeded((6, cols), 8, 1.0, torch.bfloat16).to("supa")
    y = torch.log_softmax(x, 1)
    gi = LSM_BWD(g, y, 1, torch.bfloat16)
    monkeypatch.setenv("SUPA_AMD_ROW_SPLIT_SPIN", "0")
    for _ in range(3):
        assert torch.equal(torch.log_softmax(x, 1).cpu(), y.cpu())
        assert torch.equal(LSM_BWD(g, y, 1, torch.bfloat16).cpu(), gi.cpu())


@pytest.mark.parametrize("cols", [13, 130, 1000, 9001, 50257])
def test_rows_over_their_input(cols, no_fallback):
    x, g = seeded((9, cols), 9, 2.0), seeded((9, cols), 10)
    want = torch.softmax(x.to("supa"), 1)
    dx = x.to("supa")
    torch.ops.aten._softmax.out(dx, 1, False, out=dx)
    np.testing.assert_allclose(dx.cpu().numpy(), want.cpu().numpy(), rtol=1e-5, atol=1e-12)
    gi = SM_BWD(g.to("supa"), want, 1, torch.float32)
    dg = g.to("supa")
    SM_BWD.out(dg, want, 1, torch.float32, grad_input=dg)
    np.testing.assert_allclose(dg.cpu().numpy(), gi.cpu().numpy(), rtol=1e-5, atol=1e-9)


@pytest.mark.parametrize("cols", [5, 37, 515, 4099, 50257, 600001])
@pytest.mark.parametrize("at", [0, -1])
def test_special_values(cols, at, no_fallback):
    """NaN, +inf, -inf and an all -inf row, at the first element and in the rest."""
    x = seeded((6, cols), 11, 2.0)
    x[0, at] = float("nan")
    x[1, at] = float("inf")
    x[2, at] = -float("inf")
    x[3, :] = -float("inf")
    x[4, :] = -float("inf")
    x[4, at] = float("nan")
    for f in (torch.log_softmax, torch.softmax):
        want, got = f(x, 1), f(x.to("supa"), 1).cpu()
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        ok = ~torch.isnan(want)
        np.testing.assert_allclose(got[ok].numpy(), want[ok].numpy(), rtol=1e-5, atol=1e-5)
