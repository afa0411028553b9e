"""Elementwise ops and full reductions over runs whose length is no multiple of
the vector, at any alignment: bias broadcasts, slices of rows, misaligned
views, in-place forms, and the losses over them; the nll and cross-entropy
gradients of odd class counts."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def seeded(shape, seed, dtype=torch.float32):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(dtype)


def exact(got, want):
    assert got.shape == want.shape and got.dtype == want.dtype
    assert torch.equal(got.cpu(), want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("cols", [1, 3, 4, 5, 7, 8, 9, 15, 17, 255, 1021])
def test_broadcasts_over_odd_runs(cols, dtype, no_fallback):
    x, row, col = seeded((37, cols), 1, dtype), seeded((cols,), 2, dtype), seeded((37, 1), 3, dtype)
    dx, drow, dcol = x.to("supa"), row.to("supa"), col.to("supa")
    exact(dx + drow, x + row)
    exact(dx * dcol, x * col)
    exact(drow - dx, row - x)
    exact(torch.where(dx > dcol, dx, drow), torch.where(x > col, x, row))
    if dtype != torch.float32:
        exact(dx + drow.float(), x + row.float())
    y = seeded((5, 7, cols), 4, dtype)
    ch = seeded((7, 1), 5, dtype)
    exact(y.to("supa") + ch.to("supa"), y + ch)
    z = dx.clone()
    z += drow  # in place over overlapping vectors
    z *= 2
    exact(z, (x + row) * 2)
    m = seeded((cols,), 6) > 0
    exact(dx.masked_fill(m.to("supa"), -3.5), x.masked_fill(m, -3.5))
    exact(dx.masked_fill((dx > 0), 1), x.masked_fill(x > 0, 1))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.bool, torch.uint8])
@pytest.mark.parametrize("off", [1, 3, 7])
def test_misaligned_and_sliced(off, dtype, no_fallback):
    n = 1003
    base = (seeded((6, n + 8), 7) * 3).to(dtype)
    db = base.to("supa")
    for v, dv in ((base[:, off:off + n], db[:, off:off + n]), (base.view(-1)[off:off + 5000], db.view(-1)[off:off + 5000]),
                  (base[::2, off:], db[::2, off:])):
        exact(dv.clone(), v.clone())
        exact(dv.contiguous(), v.contiguous())
        if dtype.is_floating_point:
            exact(dv * 2 + dv, v * 2 + v)
            exact(torch.relu(dv), torch.relu(v))
            w = torch.zeros_like(db)
            wv = w[:, off:off + n]
            if dv.shape == wv.shape:
                wv.copy_(dv)  # a misaligned destination
                exact(w[:, off:off + n].contiguous(), v.contiguous())
                assert (w[:, :off] == 0).all().item() and (w[:, off + n:] == 0).all().item()
    h = base[:, :n - 1].chunk(2, -1)
    dh = db[:, :n - 1].chunk(2, -1)
    exact(torch.cat(dh, -1), torch.cat(h, -1))


@pytest.mark.parametrize("dtype", [torch.float64, torch.int64, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("cols", [2, 5, 16, 31, 32, 33, 510, 511, 512, 513])
def test_slices_by_run_length(cols, dtype, no_fallback):
    """Whole vectors aligned and not, and for 8-byte types the run lengths on
    both sides of the line between vectors and single elements, with one and
    with several full-size inputs."""
    x, y = (seeded((9, 2 * cols + 3), 21) * 50).to(dtype), (seeded((9, cols + 1), 22) * 50).to(dtype)
    m = seeded((9, cols), 23) > 0
    dx, dy, dm = x.to("supa"), y.to("supa"), m.to("supa")
    for o in (0, 1, 2, cols):
        exact(-dx[:, o:o + cols], -x[:, o:o + cols])
        exact(dx[:, o:o + cols] * dy[:, 1:], x[:, o:o + cols] * y[:, 1:])
        exact(dx[:, o:o + cols] + dy[0, :cols], x[:, o:o + cols] + y[0, :cols])
        exact(torch.where(dm, dx[:, o:o + cols], dy[:, :cols]), torch.where(m, x[:, o:o + cols], y[:, :cols]))
    w, dw = x.clone(), dx.clone()
    w[:, 1:1 + cols] *= y[:, :cols]
    dw[:, 1:1 + cols] *= dy[:, :cols]
    exact(dw, w)


def test_masked_fill_shapes_and_errors(no_fallback):
    x = seeded((4, 1, 6), 8)
    m = seeded((5, 6), 9) > 0
    got = x.to("supa").masked_fill(m.to("supa"), float("-inf"))
    exact(got, x.masked_fill(m, float("-inf")))
    assert got.is_contiguous()
    exact(x.to("supa").masked_fill(m.to("supa"), torch.tensor(2.0)), x.masked_fill(m, torch.tensor(2.0)))
    i = torch.arange(12).view(3, 4)
    exact(i.to("supa").masked_fill(i.to("supa") > 5, -1), i.masked_fill(i > 5, -1))
    with pytest.raises(RuntimeError, match="boolean masks"):
        x.to("supa").masked_fill(x.to("supa"), 1.0)
    p = x.to("supa").requires_grad_()
    p.masked_fill(m.to("supa"), 0.0).sum().backward()
    q = x.clone().requires_grad_()
    q.masked_fill(m, 0.0).sum().backward()
    exact(p.grad, q.grad)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("cols", [1, 3, 5, 8, 13, 8193])
@pytest.mark.parametrize("reduction", ["mean", "sum", "none"])
def test_losses_over_odd_runs(cols, dtype, reduction, no_fallback):
    x, t, pw = seeded((19, cols), 10, dtype), (seeded((19, cols), 11) > 0).to(dtype), seeded((cols,), 12, dtype).abs() + 0.5
    dx = x.to("supa").requires_grad_()
    cx = x.double().requires_grad_()
    loss = F.binary_cross_entropy_with_logits(dx, t.to("supa"), pos_weight=pw.to("supa"), reduction=reduction)
    want = F.binary_cross_entropy_with_logits(cx, t.double(), pos_weight=pw.double(), reduction=reduction)
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    torch.testing.assert_close(loss.detach().cpu().double(), want.detach(), rtol=tol, atol=tol)
    loss.sum().backward()
    want.sum().backward()
    torch.testing.assert_close(dx.grad.cpu().double(), cx.grad, rtol=tol, atol=tol / max(1, x.numel() if reduction == "mean" else 1))
    torch.testing.assert_close(F.mse_loss(dx.detach(), t.to("supa"), reduction=reduction).cpu().double(),
                               F.mse_loss(x.double(), t.double(), reduction=reduction), rtol=tol, atol=tol)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float64])
@pytest.mark.parametrize("c", [1, 2, 3, 7, 8, 9, 100, 2047, 2048, 2049, 5003])
def test_nll_backward_of_odd_classes(c, dtype, no_fallback):
    n = 301
    t = torch.randint(0, c, (n,), generator=torch.Generator().manual_seed(13))
    t[::7] = -100
    lp = seeded((n, c), 14, dtype)
    w = (seeded((c,), 15).abs() + 0.5).to(dtype)
    for red, weight in (("mean", None), ("sum", w), ("none", w)):
        d = lp.to("supa").requires_grad_()
        r = lp.clone().requires_grad_()
        ld = F.nll_loss(d, t.to("supa"), None if weight is None else weight.to("supa"), reduction=red)
        lr = F.nll_loss(r, t, weight, reduction=red)
        g = seeded((n,), 16, dtype) if red == "none" else torch.ones((), dtype=dtype)
        ld.backward(g.to("supa"))
        lr.backward(g)
        tol = 1e-2 if dtype == torch.bfloat16 else 1e-5
        torch.testing.assert_close(d.grad.cpu(), r.grad, rtol=tol, atol=0)


def test_nll_backward_flags_a_bad_target(no_fallback):
    for c in (5, 3001):
        t = torch.tensor([0, c, 1], device="supa")
        with pytest.raises(IndexError):
            torch.ops.aten.nll_loss_backward(torch.ones((), device="supa"), torch.zeros(3, c, device="supa"), t, None, 2,
                                             -100, torch.ones((), device="supa")).cpu()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("c", [3, 9, 1001, 50257])
def test_fused_cross_entropy_of_odd_classes(c, dtype, no_fallback, fused_ce):
    n = 33
    x = (seeded((n, c), 17) * 2).to(dtype)
    t = torch.randint(0, c, (n,), generator=torch.Generator().manual_seed(18))
    t[5] = -100
    prob = torch.softmax(seeded((n, c), 19), 1).to(dtype)
    for target in (t, prob):
        d, r = x.to("supa").requires_grad_(), x.double().requires_grad_()
        ld = F.cross_entropy(d, target.to("supa"))
        lr = F.cross_entropy(r, target if target is t else target.double())
        ld.backward()
        lr.backward()
        tol = 1e-5 if dtype == torch.float32 else 1e-2
        torch.testing.assert_close(ld.detach().cpu().double(), lr.detach(), rtol=tol, atol=0)
        torch.testing.assert_close(d.grad.cpu().double(), r.grad, rtol=tol, atol=tol / n / 10)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("c", [1, 3, 7, 19, 255, 1001, 1024, 4100])
def test_fused_cross_entropy_special_values(c, dtype, no_fallback, fused_ce):
    """A NaN or +inf logit anywhere makes its row's loss and gradient NaN,
    also where every logit that one thread holds is one; -inf logits count
    nothing; a row of -inf alone is NaN.  Index and probability targets."""
    rows, nan, inf = [], float("nan"), float("inf")
    spans = sorted({(0, 1), (c // 2, c // 2 + 1), (c - 1, c), (0, min(c, 8)), (max(0, c - 9), c), (0, c)})
    for lo, hi in spans:  # (span, its value, whether every other logit is -inf)
        rows += [(lo, hi, nan, False), (lo, hi, nan, True), (lo, hi, inf, False), (lo, hi, -inf, False)]
    x = seeded((len(rows), c), 24).to(dtype)
    for i, (lo, hi, v, alone) in enumerate(rows):
        if alone:
            x[i] = -inf
        x[i, lo:hi] = v
    for at in (0, c - 1, c // 3):
        t = torch.full((len(rows),), at)
        prob = torch.softmax(seeded((len(rows), c), 25), 1).to(dtype)
        for target in (t, prob):
            d, r = x.to("supa").requires_grad_(), x.double().requires_grad_()
            ld = F.cross_entropy(d, target.to("supa"), reduction="none")
            lr = F.cross_entropy(r, target if target is t else target.double(), reduction="none")
            ld.sum().backward()
            lr.sum().backward()
            tol = 1e-5 if dtype == torch.float32 else 1e-2
            torch.testing.assert_close(ld.detach().cpu().double(), lr.detach(), rtol=tol, atol=tol, equal_nan=True)
            torch.testing.assert_close(d.grad.cpu().double(), r.grad, rtol=tol, atol=tol, equal_nan=True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float64])
@pytest.mark.parametrize("n", [65535, 65536, 70001])
def test_nll_loss_of_many_rows(n, dtype, no_fallback):
    """Both sides of the line between one launch and two."""
    lp = -seeded((n, 5), 26).abs().to(dtype)
    t = torch.randint(0, 5, (n,), generator=torch.Generator().manual_seed(27))
    t[::11] = -100
    w = (seeded((5,), 28).abs() + 0.5).to(dtype)
    for red in ("mean", "sum"):
        for weight in (None, w):
            got = F.nll_loss(lp.to("supa"), t.to("supa"), None if weight is None else weight.to("supa"), reduction=red)
            want = F.nll_loss(lp.double(), t, None if weight is None else weight.double(), reduction=red)
            # chains of at most n / 1024 + 64 float32 additions of one sign, then one rounding
            tol = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float64: 0.0}[dtype]
            tol += 2 * (n / 1024 + 64) * 2.0 ** (-53 if dtype == torch.float64 else -24)
            torch.testing.assert_close(got.cpu().double(), want, rtol=tol, atol=0)
    t[-1] = 5
    with pytest.raises(IndexError):
        F.nll_loss(lp.to("supa"), t.to("supa")).cpu()


def test_losses_of_short_odd_runs(no_fallback):
    """Runs of a few vectors with a broadcast weight, from one workgroup to all of them."""
    for shape in ((1, 9), (3, 100), (700, 13), (8192, 100), (40000, 33)):
        for dtype in (torch.float32, torch.bfloat16):
            x, t = seeded(shape, 29, dtype), (seeded(shape, 30) > 0).to(dtype)
            w = (seeded(shape[1:], 31).abs() + 0.5).to(dtype)
            got = F.binary_cross_entropy_with_logits(x.to("supa"), t.to("supa"), pos_weight=w.to("supa"))
            want = F.binary_cross_entropy_with_logits(x.double(), t.double(), pos_weight=w.double())
            torch.testing.assert_close(got.cpu().double(), want, rtol=1e-5 if dtype == torch.float32 else 1e-2, atol=0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_losses_of_whole_runs_beside_a_weight(dtype, no_fallback):
    """Whole aligned vectors beside an operand that is read again, below and above
    the size from which the others stream.  The mean of equal rows is that of one;
    bounds: n / 2^24 additions of one sign for float32, half a step for bfloat16."""
    for rows, cols in ((3, 8), (64, 264), (1000, 4096), (40, 1 << 20), (72, 1 << 20)):
        x, t = seeded((cols + 8,), 34, dtype), (seeded((cols,), 35) > 0).to(dtype)
        w = (seeded((cols,), 36).abs() + 0.5).to(dtype)
        xs = torch.empty(rows, cols + 8, dtype=dtype, device="supa")
        ts = torch.empty(rows, cols, dtype=dtype, device="supa")
        xs.copy_(x.to("supa"))
        ts.copy_(t.to("supa"))
        rtol = 1e-5 if dtype == torch.float32 else 2.0 ** -8
        for view in (xs[:, 8:], xs[:, 8:].contiguous()):
            got = F.binary_cross_entropy_with_logits(view, ts, pos_weight=w.to("supa"))
            want = F.binary_cross_entropy_with_logits(x[8:].double(), t.double(), pos_weight=w.double())
            torch.testing.assert_close(got.cpu().double(), want, rtol=rtol, atol=0)
            got = F.mse_loss(view, w.to("supa").expand_as(view))
            want = F.mse_loss(x[8:].double(), w.double())
            torch.testing.assert_close(got.cpu().double(), want, rtol=rtol, atol=0)
        del xs, ts, view
    torch.supa.empty_cache()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_fused_cross_entropy_gradient_at_any_alignment(dtype, no_fallback, fused_ce):
    """Rows of whole vectors that start at a boundary and off it: the same bits."""
    for n, c in ((1, 8), (37, 64), (5, 1000), (9, 4104)):
        flat = seeded((n * c + 8,), 37, dtype).to("supa")
        t = (torch.arange(n) * 7 % c).to("supa")
        for off in (0, 1, 3, 8):
            x = flat[off:off + n * c].view(n, c)
            grads = []
            for logits in (x, x.clone()):
                logits = logits.detach().requires_grad_()
                F.cross_entropy(logits, t).backward()
                grads.append(logits.grad)
            assert torch.equal(grads[0].cpu(), grads[1].cpu()), (n, c, off)


@pytest.mark.parametrize("prob", [False, True])
def test_cross_entropy_of_more_rows_than_one_launch(prob, no_fallback, fused_ce):
    """2^26 rows (2^24 with probability targets): more threads than a launch holds."""
    if torch.supa.mem_get_info()[0] < 20 << 30:
        pytest.skip("takes 4 GiB of device memory")
    n = 1 << (18 if prob else 20)
    small = seeded((65, 4), 32).to("supa")
    st = torch.softmax(seeded((65, 4), 33), 1).to("supa") if prob else (torch.arange(65) % 4).to("supa")
    x = torch.empty(n, 65, 4, device="supa")
    x.copy_(small)
    t = torch.empty(n, *st.shape, dtype=st.dtype, device="supa")
    t.copy_(st)
    got = F.cross_entropy(x.view(-1, 4), t.flatten(0, 1), reduction="none")
    assert bool((got.view(n, 65) == F.cross_entropy(small, st, reduction="none")).all())
    del x, t, got
    torch.supa.empty_cache()


def test_fused_cross_entropy_mean_precision(no_fallback):
    """The mean over rows of one sign against 64 bits.  30 classes put the sum
    of 2048 rows, 7950, near the top of its binade, so that an addition rounds by
    at most u = 2^-12 and is worth 0.52 2^-24 of the sum.  In a tree each addition of two sums of one
    step falls on a multiple of u half the time: its error is 0 or u, u^2/2 on
    average, and with the levels below, at a half of it each, u^2: 0.52 2^-24.
    Sixteen partial sums one after another make eight additions in the top
    binade and four in the one below, of u^2/3 and u^2/12: 0.9 2^-24.  48 draws
    give a root mean square to a tenth: three of them make 0.68.  (40 classes
    put the sum just above a power of two, where the last addition alone rounds
    by up to 2^-24 of it, either way.)"""
    err = []
    for seed in range(48):
        x = seeded((2048, 30), 100 + seed)
        t = torch.randint(0, 30, (2048,), generator=torch.Generator().manual_seed(seed))
        want = F.cross_entropy(x.double(), t)
        err.append(float((F.cross_entropy(x.to("supa"), t.to("supa")).cpu().double() - want) / want))
    rms = (sum(e * e for e in err) / len(err)) ** 0.5
    assert rms <= 0.68 * 2.0 ** -24, rms
