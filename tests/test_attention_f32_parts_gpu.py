"""GPU parity: fp32 attention of head_dim 64 in three bf16 parts per value (attn_f32_parts.hip) against the CPU oracle."""
import pytest
import torch

import odysseus_oracle as oracle
from conftest import TOL_F32, assert_parity, randn

pytestmark = pytest.mark.gpu

# edges of the 32-row tiles and of blocks of 32, 64 and 128 rows; turns that leave some groups without a tile; groups of heads; key offsets of
# either sign; shapes that take each kind of block
CASES = [(1, 33, 257, 2, 2, True), (1, 65, 289, 4, 1, False), (1, 300, 300, 8, 2, True), (1, 129, 65, 4, 4, True), (1, 1, 300, 2, 1, True),
         (4, 484, 484, 16, 16, True), (2, 300, 301, 16, 4, False), (2, 1025, 1025, 16, 16, True), (1, 1500, 700, 32, 8, False), (2, 1100, 260, 16, 16, True)]


def _inputs(B, Lq, Lk, Hq, Hkv, seed):
    return [randn(s, seed + n) for n, s in enumerate([(B, Lq, Hq, 64), (B, Lk, Hkv, 64), (B, Lk, Hkv, 64), (B, Lq, Hq, 64)])]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B%d_Lq%d_Lk%d_H%d_%d_c%d" % c)
def test_fp32_attention_in_parts(case):
    from odysseus_transformer_amd import ops
    B, Lq, Lk, Hq, Hkv, causal = case
    print(f"case={case}", flush=True)
    q, k, v, do = _inputs(B, Lq, Lk, Hq, Hkv, Lq + 3 * Lk)
    o_ref, lse_ref = oracle.attention_fwd(q, k, v, causal=causal)
    grads = oracle.attention_bwd(q, k, v, o_ref, lse_ref, do, causal=causal)
    # every other row of larger buffers: the row strides are not those of a packed tensor
    qg, kg, vg, dog = (torch.stack([t, t + 1], 2).flatten(1, 2).cuda()[:, ::2] for t in (q, k, v, do))
    o, lse = ops.attn_fwd(qg, kg, vg, causal=causal)
    got = ops.attn_bwd(qg, kg, vg, o, lse, dog, causal=causal)
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


@pytest.mark.parametrize("shape", [(1, 300, 320, 2), (4, 484, 484, 16), (2, 300, 301, 16)], ids=lambda s: "B%d_Lq%d_Lk%d_H%d" % s)
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
