"""``agmi_lse_rows_fused``: a row-wise logsumexp, its cotangent and what consumes it in one pass over the operand.

Sizes sit at the edges of the kernel's variants (64 ... 8192 vectors of 16 bytes to a row, one more and one less) and at numbers
of rows that leave blocks and row groups part empty; the oracle is NumPy in float64.
"""

import numpy as onp
import pytest
import scipy.special

pytestmark = pytest.mark.gpu

F32, F64 = onp.float32, onp.float64
# (vectors to a row, what is added to the elements they hold, rows)
EDGES = [(1, -1, 3), (1, 0, 33), (64, -1, 5), (64, 1, 700), (128, 0, 2500), (128, 1, 2049), (256, -1, 2100), (256, -3, 70), (256, 1, 9),
         (512, 1, 1100), (1024, 0, 1030), (1024, -1, 300), (1024, 1, 37), (2048, 1, 261), (4096, 0, 5), (4096, 1, 300), (8192, -1, 3)]


def _tolerance(dtype, cols):
    # x - ans is rounded before the exponential (|x - ans| < 32 here: 32 half-ulps of relative error at most), sums add
    # a handful of roundings on top
    return 64 * onp.finfo(dtype).eps


def _fits(cols, dtype, staged):
    """Whether ``staged`` column vectors beyond the first fit the LDS beside the padded row (as ``include/agmi.h`` states it)."""
    vectors = -(-cols * onp.dtype(dtype).itemsize // 16)
    padded = next(n for n in (64, 128, 256, 512, 1024, 2048, 4096, 8192) if vectors <= n)
    return 16 * (staged * vectors + padded) <= 144 * 1024


@pytest.mark.parametrize("dtype", [F32, F64])
@pytest.mark.parametrize("vectors,extra,rows", EDGES)
def test_every_result_at_the_edges_of_the_variants(dtype, vectors, extra, rows):
    import torch

    from autograd_amd import _lib

    cols = vectors * (16 // onp.dtype(dtype).itemsize) + extra
    rs = onp.random.RandomState(cols + rows)
    dev, code = _lib.device(), _lib.DTYPE_CODE[onp.dtype(dtype)]
    pitch = cols + 3  # rows of the operand and of the copy lie apart: what is between them is not touched
    mem = rs.randn(rows, pitch).astype(dtype)
    by_col, by_row, g = rs.uniform(0.5, 1.5, cols).astype(dtype), rs.randn(rows, 1).astype(dtype), rs.uniform(0.5, 2.0, (rows, 1)).astype(dtype)
    put = lambda a: torch.from_numpy(onp.ascontiguousarray(a)).to(dev)
    t_mem = put(mem)[:, :cols]
    t_col, t_row, t_g = put(by_col), put(by_row), put(g)
    wide = lambda t: t.expand(rows, cols)
    # operand, its value, column vectors staged beyond the first: with the copy's factor, without one, without the copy
    forms = {
        "A*b + c": (_lib.Affine(t_mem, 1.0, wide(t_row), wide(t_col)), mem[:, :cols].astype(F64) * by_col + by_row, (0, 1, 0)),
        "-A + b": (_lib.Affine(t_mem, -1.0, wide(t_col)), -mem[:, :cols].astype(F64) + by_col, (2, 1, 1)),
        "A": (t_mem, mem[:, :cols].astype(F64), (1, 0, 0)),
    }
    tol = _tolerance(dtype, cols)
    for name, (operand, x, staged) in forms.items():
        ans = scipy.special.logsumexp(x, axis=1, keepdims=True)
        S = g.astype(F64) * onp.exp(x - ans)
        for factor in (t_col, None):
            kind = dict(dtype=t_mem.dtype, device=dev)
            out = torch.full((rows, pitch), 7.0, **kind)
            t_ans, row_sums, col_sums = torch.empty((rows, 1), **kind), torch.empty((rows, 1), **kind), torch.empty((1, cols), **kind)
            taken = _lib.lse_rows(code, operand, t_g, ans=t_ans, row_sums=row_sums, col_factor=factor, scaled=out[:, :cols], col_sums=col_sums)
            assert taken == _fits(cols, dtype, staged[factor is None]), name
            if not taken:
                continue
            want = S * by_col if factor is not None else S
            got = out.cpu().numpy()
            assert onp.all(got[:, cols:] == 7.0), name
            for what, have, ref in (("copy", got[:, :cols], want), ("ans", t_ans.cpu().numpy(), ans),
                                    ("row sums", row_sums.cpu().numpy(), S.sum(1, keepdims=True)),
                                    ("column sums", col_sums.cpu().numpy(), (mem[:, :cols] * S).sum(0, keepdims=True))):
                scale = onp.abs(mem[:, :cols] * S).sum(0, keepdims=True) if what == "column sums" else onp.maximum(onp.abs(ref), tol)
                assert onp.all(onp.abs(have - ref) <= tol * scale), (name, what, factor is None)
            # each result on its own, too (other instantiations)
            alone = torch.empty((rows, cols), **kind)
            assert _lib.lse_rows(code, operand, t_g, col_factor=factor, scaled=alone)
            assert onp.array_equal(alone.cpu().numpy(), got[:, :cols]), name
            taken = _lib.lse_rows(code, operand, t_g, col_sums=(again := torch.empty_like(col_sums)))
            assert taken == _fits(cols, dtype, staged[2]), name
            assert not taken or torch.equal(again, col_sums), name


@pytest.mark.parametrize("dtype", [F32, F64])
@pytest.mark.parametrize("fits", [0, 1, 2.5, 40])  # rows of partial column sums that the workspace holds (none: one block)
def test_a_smaller_workspace_is_met_with_fewer_blocks(dtype, fits):
    import ctypes

    import torch

    from autograd_amd import _lib

    rows, cols = 5003, 259
    rs = onp.random.RandomState(11)
    dev, code, size = _lib.device(), _lib.DTYPE_CODE[onp.dtype(dtype)], onp.dtype(dtype).itemsize
    mem, g = rs.randn(rows, cols).astype(dtype), rs.uniform(0.5, 2.0, (rows, 1)).astype(dtype)
    t_mem, t_g = torch.from_numpy(mem).to(dev), torch.from_numpy(g).to(dev)
    t_ans, row_sums, scaled = torch.empty_like(t_g), torch.empty_like(t_g), torch.empty_like(t_mem)
    col_sums = torch.empty((1, cols), dtype=t_mem.dtype, device=dev)
    c = _lib._fill_lse_cotangent(t_mem, t_g, row_sums, None, scaled, col_sums)
    held = int(fits * cols) * size
    workspace = torch.full((held + 4096,), 7, dtype=torch.uint8, device=dev)
    _lib.lib()
    rc = _lib._LIB.agmi_lse_rows_fused(code, ctypes.byref(c), t_ans.data_ptr(), 1, workspace.data_ptr() if held else None, held, _lib._stream())
    assert rc == 0
    assert bool((workspace[held:] == 7).all())  # nothing is written past the workspace
    x = mem.astype(F64)
    ans = scipy.special.logsumexp(x, axis=1, keepdims=True)
    S = g * onp.exp(x - ans)
    tol = _tolerance(dtype, cols)
    assert onp.all(onp.abs(t_ans.cpu().numpy() - ans) <= tol * onp.maximum(onp.abs(ans), 1))
    assert onp.all(onp.abs(scaled.cpu().numpy() - S) <= tol * S) and onp.all(onp.abs(row_sums.cpu().numpy() - g) <= tol * g)
    # (a block's rows are added one after the other: up to 5003 / 8 of them, and one round per block)
    assert onp.all(onp.abs(col_sums.cpu().numpy() - (x * S).sum(0)) <= (tol + (rows / 8 + 256) * onp.finfo(dtype).eps) * onp.abs(x * S).sum(0))


@pytest.mark.parametrize("dtype", [F32, F64])
@pytest.mark.parametrize("cols", [7, 600, 5000, 16001])
def test_rows_with_infinities_and_nans(dtype, cols):
    """Special values, in the rows and in their cotangents, travel as through the two separate kernels (scipy's logsumexp, then
    g * exp(x - ans)): an infinite g times an exponential that vanishes is NaN, in the matrix and in the row's sum, wherever
    in the row it lies."""
    import torch

    from autograd_amd import _lib

    rs = onp.random.RandomState(cols)
    dev, code = _lib.device(), _lib.DTYPE_CODE[onp.dtype(dtype)]
    x = rs.randn(20, cols).astype(dtype)
    x[1], x[2, 3], x[3, 0], x[4, cols - 1], x[5] = -onp.inf, onp.inf, onp.nan, -onp.inf, onp.nan
    x[6, 1], x[6, 2] = onp.inf, onp.nan
    x[7] = -onp.inf
    x[7, cols // 2] = -1000.0
    x[8, :] = 80.0
    x[9, : cols // 2] = -onp.inf
    g = onp.full((20, 1), 2.0, dtype)
    g[11:20, 0] = onp.inf, onp.inf, -onp.inf, onp.nan, onp.inf, onp.nan, onp.inf, -onp.inf, onp.nan
    x[12, cols - 1] = x[13, 0] = -1000.0  # (exp(x - ans) is 0 in both precisions)
    x[14, : cols // 2] = x[15, : cols // 2] = -onp.inf
    x[17], x[18, 1], x[19, 2] = -onp.inf, onp.inf, onp.nan
    t_x, t_g = torch.from_numpy(x).to(dev), torch.from_numpy(g).to(dev)
    t_ans, row_sums, out = torch.empty_like(t_g), torch.empty_like(t_g), torch.empty_like(t_x)
    assert _lib.lse_rows(code, t_x, t_g, ans=t_ans, row_sums=row_sums, scaled=out)
    with onp.errstate(all="ignore"):
        m = onp.max(x.astype(F64), axis=1, keepdims=True)
        safe = onp.where(onp.isfinite(m), m, 0.0)
        ans = onp.log(onp.sum(onp.exp(x.astype(F64) - safe), axis=1, keepdims=True)) + safe
        S = g.astype(F64) * onp.exp(x.astype(F64) - ans)
        sums = S.sum(1, keepdims=True)
    alone = torch.empty_like(row_sums)
    assert _lib.lse_rows(code, t_x, t_g, row_sums=alone) and onp.array_equal(alone.cpu().numpy(), row_sums.cpu().numpy(), equal_nan=True)
    for have, ref in ((t_ans, ans), (out, S), (row_sums, sums)):
        have = have.cpu().numpy().astype(F64)
        assert onp.array_equal(onp.isnan(have), onp.isnan(ref)) and onp.array_equal(onp.isinf(have), onp.isinf(ref))
        assert onp.array_equal(have[onp.isinf(ref)], ref[onp.isinf(ref)])
        fine = onp.isfinite(ref)
        # (80 and -1000 bring the error of |ans| ulps that rounding ans leaves in exp(x - ans))
        assert onp.all(onp.abs(have[fine] - ref[fine]) <= 2048 * onp.finfo(dtype).eps * onp.maximum(onp.abs(ref[fine]), 1e-30))


def test_a_pending_logsumexp_is_formed_by_the_pass_that_differentiates_it():
    import autograd_amd as ag
    import autograd_amd.numpy as dnp
    from autograd_amd import _lib
    from autograd_amd.scipy.special import logsumexp

    rs = onp.random.RandomState(3)
    a, b, c = rs.randn(301, 1003), rs.uniform(0.5, 1.5, 1003), rs.randn(301)
    A, B, C = (dnp.asarray(v) for v in (a, b, c))
    f = lambda A, B, C: dnp.sum(logsumexp(A * B[None, :] + C[:, None], axis=1) ** 2)
    g = lambda A, B, C: dnp.sum(logsumexp(A * B[None, :] + C[:, None], axis=1))
    x = a * b + c[:, None]
    lse = scipy.special.logsumexp(x, axis=1, keepdims=True)
    S = onp.exp(x - lse)
    with _lib.KernelTimer() as kt:
        dA, dB, dC = ag.grad(g, (0, 1, 2))(A, B, C)
    assert sum(row["launches"] for row in kt.summary().values()) == 1
    for have, ref in ((dA, S * b), (dB, (a * S).sum(0)), (dC, S.sum(1))):
        assert onp.allclose(have.numpy(), ref, rtol=1e-12, atol=1e-12)
    value, dA = ag.value_and_grad(f)(A, B, C)  # a reader of the value first: the reduction runs, the rule finds it
    assert onp.allclose(float(value), (lse**2).sum(), rtol=1e-13)
    assert onp.allclose(dA.numpy(), 2 * lse * S * b, rtol=1e-12, atol=1e-12)
    untraced = logsumexp(A, axis=1)
    assert type(untraced).__name__ == "DevArray"


def test_values_handed_to_the_caller_do_not_follow_later_writes():
    import autograd_amd as ag
    import autograd_amd.numpy as dnp
    from autograd_amd.scipy.special import logsumexp

    rs = onp.random.RandomState(5)
    for cols in (100, 101):
        a, b, g = rs.randn(100, cols), rs.randn(100, cols), rs.randn(100)
        want = scipy.special.logsumexp(a, axis=1)
        A = dnp.array(a)
        V = A[:50]
        vjp, val = ag.make_vjp(lambda A: logsumexp(A, axis=1))(A)
        V[:] = dnp.array(b[:50])
        A[50:] = dnp.array(b[50:])
        cotangent = vjp(dnp.array(g)).numpy()
        assert onp.allclose(val.numpy(), want, rtol=1e-13)
        assert onp.allclose(cotangent, g[:, None] * onp.exp(b - want[:, None]), rtol=1e-12)
        A = dnp.array(a)
        gradient, aux = ag.grad_and_aux(lambda A: (dnp.sum(A * A), logsumexp(A, axis=1)))(A)
        A._t.fill_(5.0)
        assert onp.allclose(aux.numpy(), want, rtol=1e-13) and onp.allclose(gradient.numpy(), 2 * a, rtol=1e-13)
        A = dnp.array(a)
        C = A * 2.0
        value, gradient = ag.value_and_grad(lambda A: dnp.sum(logsumexp(A, axis=1)))(A)
        A[:] = 0.0
        assert onp.allclose(C.numpy(), 2 * a) and onp.allclose(float(value), want.sum())


@pytest.mark.parametrize("of", ["sum", "sum of squares"])  # the one pass; the reduction and the pass that reads its value
def test_a_kernel_is_timed_under_the_key_it_reports(of):
    """What ``bench.py`` does: find a kernel in an unrestricted timing, then time launches with its key only."""
    import autograd_amd as ag
    import autograd_amd.numpy as dnp
    from autograd_amd import _lib
    from autograd_amd.scipy.special import logsumexp

    rs = onp.random.RandomState(3)
    A, B, C = (dnp.asarray(v) for v in (rs.randn(300, 1000), rs.uniform(0.5, 1.5, 1000), rs.randn(300)))
    lse = lambda A, B, C: logsumexp(A * B[None, :] + C[:, None], axis=1)
    f = ag.grad((lambda *a: dnp.sum(lse(*a))) if of == "sum" else (lambda *a: dnp.sum(lse(*a) ** 2)), (0, 1, 2))
    with _lib.KernelTimer() as kt:
        f(A, B, C)
    seen = kt.summary()
    assert any(name.startswith("lse_cotangent_tile") for name in seen)
    for name, row in seen.items():
        with _lib.KernelTimer(only={row["key"]}) as kt:
            f(A, B, C)
        assert kt.summary()[name]["launches"] == row["launches"], (name, row["key"])


@pytest.mark.parametrize("asked_on_default", [False, True])
def test_a_waiting_value_is_formed_on_the_stream_it_was_asked_for_on(asked_on_default):
    import torch

    import autograd_amd.numpy as dnp
    from autograd_amd import core
    from autograd_amd.scipy.special import logsumexp

    a = onp.random.RandomState(7).randn(1024, 1024).astype(F32)
    A, B = dnp.array(a), dnp.array(a)
    side, default = torch.cuda.Stream(), torch.cuda.current_stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(default if asked_on_default else side):
        X = A
        for _ in range(50):  # the operand is a while in the making
            X = dnp.dot(X, A) * F32(1 / 32)
        X = dnp.settle(X)
        _, val = core.make_vjp(lambda X: logsumexp(X, axis=1), X)
    with torch.cuda.stream(side if asked_on_default else default):
        B[0] = A[1]
    torch.cuda.synchronize()
    assert onp.allclose(val.numpy(), scipy.special.logsumexp(X.numpy().astype(F64), axis=1), rtol=1e-5)


@pytest.mark.parametrize("cols", [1003, 8193, 12001])  # (the longer ones ask for more than 64 KB of LDS)
def test_the_one_pass_is_recorded_and_replayed(cols):
    import torch

    import autograd_amd as ag
    import autograd_amd.numpy as dnp
    from autograd_amd.scipy.special import logsumexp

    rs = onp.random.RandomState(cols)
    f = ag.grad(lambda A, B, C: dnp.sum(logsumexp(A * B[None, :] + C[:, None], axis=1)), (0, 1, 2))
    args = [dnp.array(v) for v in (rs.randn(40, cols), rs.uniform(0.5, 1.5, cols), rs.randn(40))]
    replayed = ag.capture(f, *args)
    for _ in range(3):
        args = [dnp.array(v) for v in (rs.randn(40, cols), rs.uniform(0.5, 1.5, cols), rs.randn(40))]
        got = [r.numpy() for r in replayed(*args)]
        torch.cuda.synchronize()
        for have, want in zip(got, f(*args)):
            assert onp.array_equal(have, want.numpy())
