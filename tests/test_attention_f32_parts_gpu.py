"""GPU parity: fp32 attention of head_dim 64 in three bf16 parts per value (attn_f32_parts.hip) against the CPU oracle."""
import math

import pytest
import torch

import odysseus_oracle as oracle
from conftest import TOL_F32, assert_parity, randn

pytestmark = pytest.mark.gpu

# edges of the 32-row tiles and of blocks of 32, 64 and 128 rows; turns that leave some groups without a tile; groups of heads; key offsets of
# either sign; with each, the rows of a block of the three kernels (0: the forward of so few keys runs on the fp32 instruction)
CASES = [((1, 33, 257, 2, 2, True), (32, 32, 128)), ((1, 65, 289, 4, 1, False), (32, 32, 32)), ((1, 300, 300, 8, 2, True), (32, 32, 32)),
         ((1, 129, 65, 4, 4, True), (0, 32, 32)), ((1, 1, 300, 2, 1, True), (32, 32, 128)), ((4, 484, 484, 16, 16, True), (128, 128, 128)),
         ((2, 300, 301, 16, 4, False), (64, 64, 32)), ((2, 1025, 1025, 16, 16, True), (128, 64, 64)), ((1, 1500, 700, 32, 8, False), (128, 64, 32)),
         ((2, 1100, 260, 16, 16, True), (128, 128, 32))]

SHAPES = pytest.mark.parametrize("shape", [(1, 300, 320, 2), (4, 484, 484, 16), (2, 300, 301, 16)], ids=lambda s: "B%d_Lq%d_Lk%d_H%d" % s)


def _inputs(B, Lq, Lk, Hq, Hkv, seed):
    return [randn(s, seed + n) for n, s in enumerate([(B, Lq, Hq, 64), (B, Lk, Hkv, 64), (B, Lk, Hkv, 64), (B, Lq, Hq, 64)])]


def _run(fn):
    from odysseus_transformer_amd import _lib
    _lib.profile_enable(True)
    try:
        _lib.profile_collect()
        r = fn()
        torch.cuda.synchronize()
        return r, set(_lib.profile_collect())
    finally:
        _lib.profile_enable(False)


def _names(fwd, dq, dkdv):
    return {f"attn_fwd_f32_parts{fwd}" if fwd else "attn_fwd_f32_split", f"attn_bwd_dq_f32_parts{dq}", f"attn_bwd_dkdv_f32_parts{dkdv}"}


@pytest.mark.parametrize("case,rows", CASES, ids=lambda c: "B%d_Lq%d_Lk%d_H%d_%d_c%d" % c if len(c) == 6 else "x".join(map(str, c)))
def test_fp32_attention_in_parts(case, rows):
    from odysseus_transformer_amd import ops
    B, Lq, Lk, Hq, Hkv, causal = case
    print(f"case={case}", flush=True)
    q, k, v, do = _inputs(B, Lq, Lk, Hq, Hkv, Lq + 3 * Lk)
    o_ref, lse_ref = oracle.attention_fwd(q, k, v, causal=causal)
    grads = oracle.attention_bwd(q, k, v, o_ref, lse_ref, do, causal=causal)
    # every other row of larger buffers: the row strides are not those of a packed tensor
    qg, kg, vg, dog = (torch.stack([t, t + 1], 2).flatten(1, 2).cuda()[:, ::2] for t in (q, k, v, do))
    (o, lse), ran = _run(lambda: ops.attn_fwd(qg, kg, vg, causal=causal))
    got, more = _run(lambda: ops.attn_bwd(qg, kg, vg, o, lse, dog, causal=causal))
    assert _names(*rows) <= ran | more, (ran, more)
    assert_parity(o, o_ref, TOL_F32, "o")
    assert torch.allclose(lse.cpu(), lse_ref, atol=1e-5, rtol=1e-5)
    for name, a, b in zip(("dq", "dk", "dv"), got, grads):
        assert_parity(a, b, TOL_F32, name)
    again = (*ops.attn_fwd(qg, kg, vg, causal=causal), *ops.attn_bwd(qg, kg, vg, o, lse, dog, causal=causal))
    assert all(torch.equal(a, b) for a, b in zip(again, (o, lse, *got)))
    acc0 = randn(q.shape, 5).cuda()
    acc = acc0.clone()
    ops.attn_bwd(qg, kg, vg, o, lse, dog, causal=causal, dq=acc, accumulate_dq=True)
    assert_parity((acc - acc0).cpu(), grads[0], TOL_F32, "dq added to a buffer")


@SHAPES
def test_fp32_attention_beyond_the_range_of_the_parts(shape):
    """Values that bf16 rounds to infinity, and infinities: as the fp32 instruction gives them."""
    from odysseus_transformer_amd import ops
    B, Lq, Lk, H = shape
    q, k, v, do = _inputs(B, Lq, Lk, H, H, 11)
    big = 3.4e38
    assert torch.tensor(big).isfinite() and not torch.tensor(big).bfloat16().isfinite()
    v[0, 40, 1, 3], do[0, 100, 0, 5] = big, big
    v[0, 41, 0, 7] = float("inf")
    o_ref, lse_ref = oracle.attention_fwd(q, k, v, causal=False)
    assert o_ref[0, :, 1].isfinite().all() and (o_ref[0, :, 0, 7] == float("inf")).all()
    qg, kg, vg, dog = (t.cuda() for t in (q, k, v, do))
    o, lse = ops.attn_fwd(qg, kg, vg, causal=False)
    o = o.cpu()
    assert torch.equal(o == float("inf"), o_ref == float("inf")) and not o.isnan().any()
    live = o_ref.isfinite()
    assert torch.allclose(o[live], o_ref[live], rtol=TOL_F32, atol=TOL_F32)
    assert torch.allclose(lse.cpu(), lse_ref, atol=1e-5, rtol=1e-5)
    # dV holds no value of V, only P and dO
    v0 = torch.zeros_like(v)
    o0, lse0 = ops.attn_fwd(qg, kg, v0.cuda(), causal=False)
    dv = ops.attn_bwd(qg, kg, v0.cuda(), o0, lse0, dog, causal=False)[2].cpu()
    p = torch.softmax(torch.matmul(q.transpose(1, 2), k.permute(0, 2, 3, 1)) / 8, -1)
    dv_ref = torch.matmul(p.transpose(2, 3), do.transpose(1, 2)).transpose(1, 2)
    assert dv_ref.isfinite().all() and torch.allclose(dv, dv_ref, rtol=TOL_F32, atol=TOL_F32)


def _attention64(q, k, v, do, scale, causal=False):
    """out, dq, dk, dv in 64 bits"""
    q, k, v, do = (t.double().transpose(1, 2) for t in (q, k, v, do))
    s = (q @ k.transpose(2, 3)) * scale
    if causal:
        s = s.masked_fill(~torch.ones(s.shape[-2:], dtype=torch.bool).tril(s.shape[-1] - s.shape[-2]), float("-inf"))
    p = s.softmax(-1)
    o = p @ v
    ds = p * (do @ v.transpose(2, 3) - (do * o).sum(-1, keepdim=True)) * scale
    return [t.transpose(1, 2) for t in (o, ds @ k, ds.transpose(2, 3) @ q, p.transpose(2, 3) @ do)]


@SHAPES
@pytest.mark.parametrize("exps,what", [((0, 0, -122, 0), "out dv"), ((0, 0, -112, 0), "dq dk"), ((0, 0, 0, -122), "out dv"), ((0, 0, 0, -112), "dq dk"),
                                       ((-115, 90, 0, 0), "out dq dk dv"), ((90, -115, 0, 0), "out dq dk dv"), ((0, 0, 60, 50), "out dv"),
                                       ((0, 0, 114, 0), "out dv"), ((114, -114, 0, 0), "out dq dk dv")], ids=str)
def test_fp32_attention_of_operands_of_any_size(shape, exps, what):
    """q, k, v and dout times 2^exps: every operand as exact as fp32 holds it, where the results and what lies between are no denormals."""
    from odysseus_transformer_amd import ops
    B, Lq, Lk, H = shape
    ins = [t * 2.0 ** e for t, e in zip(_inputs(B, Lq, Lk, H, H, 3), exps)]
    scale = 2.0 ** -(exps[0] + exps[1]) / 8
    ref = dict(zip(("out", "dq", "dk", "dv"), _attention64(*ins, scale)))
    q, k, v, do = (t.cuda() for t in ins)
    o, lse = ops.attn_fwd(q, k, v, causal=False, scale=scale)
    got = dict(zip(("out", "dq", "dk", "dv"), (o, *ops.attn_bwd(q, k, v, o, lse, do, causal=False, scale=scale))))
    for n in what.split():
        err = ((got[n].cpu().double() - ref[n]).norm() / ref[n].norm()).item()
        print(n, err)
        assert err <= 2e-6, (n, err)


@SHAPES
def test_fp32_attention_of_a_key_that_nobody_attends_to(shape):
    """Probabilities near 2^-119 (a score of -76 under a log-sum-exp of 6): the gradients of such a key are as exact as the scores (half a unit of 2^-17 in 120)."""
    from odysseus_transformer_amd import ops
    B, Lq, Lk, H = shape
    q, k, v, do = _inputs(B, Lq, Lk, H, H, 13)
    q[..., 0], k[..., 0] = 8.0, 0.0
    k[:, 5, :, 0] = -76.0
    _, _, dk_ref, dv_ref = _attention64(q, k, v, do, 0.125)
    assert 0 < dv_ref[:, 5].abs().max() < 2.0 ** -100
    qg, kg, vg, dog = (t.cuda() for t in (q, k, v, do))
    o, lse = ops.attn_fwd(qg, kg, vg, causal=False)
    _, dk, dv = ops.attn_bwd(qg, kg, vg, o, lse, dog, causal=False)
    for a, b in ((dk, dk_ref), (dv, dv_ref)):
        err = ((a.cpu().double() - b)[:, 5].norm() / b[:, 5].norm()).item()
        print(err)
        assert err <= 1e-5


@SHAPES
def test_fp32_attention_of_scores_beyond_what_the_parts_hold(shape):
    """All scores of a row near -2^100, their differences multiples of the spacing there: the largest ones share the row."""
    from odysseus_transformer_amd import ops
    B, Lq, Lk, H = shape
    q, k, v, do = _inputs(B, Lq, Lk, H, H, 17)
    q.zero_(), k.zero_()
    q[..., 0], k[..., 0] = 2.0 ** 50, -(2.0 ** 50) * torch.randint(1, 3, k.shape[:3]).float()
    q[:, 7:9] *= -1.0      # and rows near 2^100
    scale = math.log(2.0)      # scores are whole numbers of the exponent's base, exact in fp32
    qg, kg, vg, dog = (t.cuda() for t in (q, k, v, do))
    o, lse = ops.attn_fwd(qg, kg, vg, causal=False, scale=scale)
    ref = _attention64(q, k, v, do, scale)
    _, _, dv = ops.attn_bwd(qg, kg, vg, o, lse, dog, causal=False, scale=scale)
    assert (o.cpu().double() - ref[0]).norm() <= 1e-5 * ref[0].norm()
    assert dv.isfinite().all() and o.isfinite().all()


@SHAPES
@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
def test_fp32_gradients_beyond_the_range_of_the_parts(causal, shape):
    """One value of dout and one of v too large for the parts, the gradients with them finite: every block that meets them walks again on the fp32
    instruction, in all three kernels, and the others are what they are without."""
    from odysseus_transformer_amd import ops
    B, Lq, Lk, H = shape
    q, k, v, do = _inputs(B, Lq, Lk, H, H, 19)
    do[0, 100, 0, 5] = 2.0 ** 115
    v[0, 40, 1, 3] = 2.0 ** 113
    ref = _attention64(q, k, v, do, 0.125, causal)
    assert all(t.abs().max() < 2.0 ** 125 for t in ref)
    qg, kg, vg, dog = (t.cuda() for t in (q, k, v, do))
    o, lse = ops.attn_fwd(qg, kg, vg, causal=causal)
    got = (o, *ops.attn_bwd(qg, kg, vg, o, lse, dog, causal=causal))
    for name, a, b in zip(("out", "dq", "dk", "dv"), got, ref):
        a = a.cpu().double()
        for h in range(H):
            whole = [(a[0, :, h], b[0, :, h])]
            if h == 0 and name == "dq":   # its large row, and the rest
                rest = torch.arange(Lq) != 100
                whole = [(a[0, 100, h], b[0, 100, h]), (a[0, rest, h], b[0, rest, h])]
            if h == 1 and name == "out":  # its large column, and the rest
                rest = torch.arange(64) != 3
                whole = [(a[0, :, h, 3], b[0, :, h, 3]), (a[0, :, h, rest], b[0, :, h, rest])]
            for x, y in whole:
                assert (x - y).norm() <= TOL_F32 * y.norm(), (name, h)
