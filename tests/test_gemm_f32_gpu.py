"""GPU parity of the fp32 products, which run on the bf16 matrix cores, against 64 bits: every tile, ragged edges, loads of single
floats, ranges of K, and inputs that have no sum of three bf16 values."""
import math

import pytest
import torch

from conftest import randn

pytestmark = pytest.mark.gpu

OPS = ["nt", "nn", "tn"]


def _operands(op, M, N, K, dev, pad=0):
    """op(A), op(B) in 64 bits and the tensors of a call; pad: extra columns, the view starts one element in (no 16-byte rows)."""
    def make(rows, cols, seed):
        t = randn((rows, cols + pad), seed).to(dev)
        return t[:, 1:1 + cols] if pad else t

    a = make(*((K, M) if op == "tn" else (M, K)), 1)
    b = make(*((N, K) if op == "nt" else (K, N)), 2)
    return (a.double().t() if op == "tn" else a.double()), (b.double().t() if op == "nt" else b.double()), a, b


def _gemm(op, a, b, **kw):
    from odysseus_transformer_amd import ops
    return ops.gemm({"nt": ops.GEMM_NT, "nn": ops.GEMM_NN, "tn": ops.GEMM_TN}[op], a, b, **kw)


def _bound(K):
    """What rounding the running sum of K products of N(0, 1) values after every addition gives: 2^-25 sqrt(k) at the k-th addition,
    2^-25.5 K over all, of a result of size sqrt(K).  Leaving out one of the six products costs 2^-16 and more."""
    return 2.0 ** -25.5 * math.sqrt(K) + 2.0 ** -24


@pytest.mark.parametrize("pad", [0, 7], ids=["vectors", "floats"])
@pytest.mark.parametrize("shape", [(1, 4, 4), (64, 64, 32), (65, 68, 36), (60, 132, 100), (128, 64, 128), (300, 516, 132),
                                   (512, 512, 2048), (2048, 1376, 96), (1000, 2752, 68), (2300, 4100, 40)], ids=lambda s: "M%d_N%d_K%d" % s)
@pytest.mark.parametrize("op", OPS)
def test_products_against_64_bits(op, shape, pad, dev):
    M, N, K = shape
    print(f"op={op} shape={shape} pad={pad}", flush=True)
    if op == "tn" and not pad:
        M = (M + 3) // 4 * 4
    A, B, a, b = _operands(op, M, N, K, dev, pad)
    ref = A @ B
    y = _gemm(op, a, b)
    assert (y.double() - ref).norm() <= _bound(K) * ref.norm()
    again = _gemm(op, a, b)
    assert torch.equal(y, again)
    bias, c0 = randn((N,), 3).to(dev), randn((M, N), 4).to(dev)
    y = _gemm(op, a, b, bias=bias, out=c0.clone(), accumulate=True)
    ref = ref + bias.double() + c0.double()
    assert (y.double() - ref).norm() <= (_bound(K) + 2.0 ** -23) * ref.norm()


@pytest.mark.parametrize("shape", [(96, 64, 40), (520, 200, 2048), (2048, 2752, 36)], ids=lambda s: "M%d_N%d_K%d" % s)
@pytest.mark.parametrize("op", OPS)
def test_infinities_nan_and_the_largest_values(op, shape, dev):
    """What fp32 arithmetic gives for them, in their rows and columns and nowhere else."""
    M, N, K = shape
    A, B, a, b = _operands(op, M, N, K, dev)
    at = a.t() if op == "tn" else a      # (M, K) views
    bt = b.t() if op == "nt" else b      # (K, N)
    big = torch.finfo(torch.float32).max
    at[3, 5], at[9, 0], at[9, 1], at[17, K - 1] = math.inf, math.inf, -math.inf, math.nan
    at[33, :], at[33, 7] = 0.0, big      # rounds to infinity in bf16; its products with values below one are finite
    bt[2, 11], bt[K - 1, 40] = -math.inf, math.nan
    bt[7, :].clamp_(-0.9, 0.9)
    bt[:, 50] = 2.0 ** -3                # exact in bf16: the lower parts are zero
    ref = at.double() @ bt.double()
    y = _gemm(op, a, b)
    assert torch.equal(y.isnan(), ref.isnan())
    assert torch.equal(y.isinf(), ref.isinf()) and torch.equal(y[ref.isinf()] > 0, ref[ref.isinf()] > 0)
    ok = ref.isfinite()
    ok[33] = False
    assert (y.double() - ref)[ok].norm() <= _bound(K) * ref[ok].norm()
    row = ref[33].isfinite()
    assert ((y[33].double() - ref[33])[row].abs() <= 2.0 ** -22 * ref[33][row].abs()).all()


@pytest.mark.parametrize("scale", [2.0 ** -60, 2.0 ** 60], ids=["small", "large"])
def test_values_far_from_one(scale, dev):
    A, B, a, b = _operands("nt", 256, 192, 512, dev)
    y = _gemm("nt", a * scale, b)
    ref = (A @ B) * scale
    assert (y.double() - ref).norm() <= _bound(512) * ref.norm()


@pytest.mark.parametrize("ea,eb", [(-112, 0), (0, -118), (-122, 100), (-130, 20), (-145, 60), (-60, -70), (100, -60), (113, -113), (-119, 119),
                                   (60, 50), (-148, 100)], ids=lambda v: str(v))
@pytest.mark.parametrize("shape", [(65, 68, 36), (512, 512, 2048), (2300, 4100, 40)], ids=lambda s: "M%d_N%d_K%d" % s)
@pytest.mark.parametrize("op", OPS)
def test_operands_of_any_size_keep_their_bits(op, shape, ea, eb, dev):
    """Operands of 2^ea and 2^eb, down to denormals and up to where the parts overflow, each as exact as the type holds it: the bound of
    operands near one, and the spacing of denormals where the result is one."""
    M, N, K = shape
    M = (M + 3) // 4 * 4 if op == "tn" else M
    _, _, a, b = _operands(op, M, N, K, dev)
    a, b = (t * 2.0 ** (e // 2) * 2.0 ** (e - e // 2) for t, e in ((a, ea), (b, eb)))
    A, B = (a.double().t() if op == "tn" else a.double()), (b.double().t() if op == "nt" else b.double())
    ref = A @ B
    y = _gemm(op, a, b).double()
    assert ((y - ref).norm() - 2.0 ** -149 * math.sqrt(M * N) * math.sqrt(K)) <= _bound(K) * ref.norm()
