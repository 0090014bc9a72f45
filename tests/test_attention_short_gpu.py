"""GPU parity: the attention kernels of head_dim 128 for few blocks (attn_short.hip) against the CPU oracle."""
import pytest
import torch

import odysseus_oracle as oracle
from conftest import TOL_BF16, TOL_LSE, assert_parity, device_kernels, randn, rel_err

pytestmark = pytest.mark.gpu

# edges of the 32 rows of a wavefront, of the 64-row tiles, of the 128-row blocks and of a pair of tiles; groups of 1, 4 and 8; key
# offsets of either sign; the last causal and the last full shape that the kernels take
CASES = [(1, 65, 65, 2, 2, True), (2, 96, 33, 4, 1, False), (1, 127, 128, 4, 4, True), (1, 128, 129, 4, 1, False), (1, 129, 127, 2, 2, True),
         (3, 191, 193, 8, 1, True), (1, 257, 256, 8, 2, False), (1, 320, 64, 4, 4, True), (4, 331, 331, 8, 2, True), (1, 97, 900, 8, 2, True),
         (1, 1000, 1000, 32, 8, True), (4, 1024, 1024, 8, 8, False), (1, 2040, 2040, 5, 5, True)]


def _run(fn):
    from odysseus_transformer_amd import _lib
    _lib.profile_enable(True)
    try:
        r = fn()
        torch.cuda.synchronize()
        return r, set(_lib.profile_collect())
    finally:
        _lib.profile_enable(False)


def _inputs(B, Lq, Lk, Hq, Hkv, seed):
    return [randn(s, seed + n, dtype=torch.bfloat16) for n, s in enumerate([(B, Lq, Hq, 128), (B, Lk, Hkv, 128), (B, Lk, Hkv, 128), (B, Lq, Hq, 128)])]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B%d_Lq%d_Lk%d_H%d_%d_c%d" % c)
def test_attention_of_few_blocks(case):
    """Forward and every destination of dq, twice: results do not depend on the order of the blocks."""
    from odysseus_transformer_amd import ops
    B, Lq, Lk, Hq, Hkv, causal = case
    print(f"case={case}", flush=True)
    q, k, v, do = _inputs(B, Lq, Lk, Hq, Hkv, Lq + 3 * Lk)
    o_ref, lse_ref = oracle.attention_fwd(q.float(), k.float(), v.float(), causal=causal)
    dq_ref, dk_ref, dv_ref = oracle.attention_bwd(q.float(), k.float(), v.float(), o_ref, lse_ref, do.float(), causal=causal)
    # every other row of larger buffers: the row strides are not those of a packed tensor
    qg, kg, vg, dog = (torch.stack([t, t + 1], 2).flatten(1, 2).cuda()[:, ::2] for t in (q, k, v, do))
    (o, lse), ran = _run(lambda: ops.attn_fwd(qg, kg, vg, causal=causal))
    assert "attn_fwd_short" in ran, ran
    assert_parity(o, o_ref, TOL_BF16, "o")
    assert torch.allclose(lse.cpu(), lse_ref, atol=TOL_LSE, rtol=TOL_LSE)
    (dq, dk, dv), ran = _run(lambda: ops.attn_bwd(qg, kg, vg, o, lse, dog, causal=causal))
    assert "attn_bwd_short" in ran, ran
    assert_parity(dq, dq_ref, TOL_BF16, "dq", 1e-3)
    assert_parity(dk, dk_ref, TOL_BF16, "dk", 1e-3)
    assert_parity(dv, dv_ref, TOL_BF16, "dv")
    again = (*ops.attn_fwd(qg, kg, vg, causal=causal), *ops.attn_bwd(qg, kg, vg, o, lse, dog, causal=causal))
    assert all(torch.equal(a, b) for a, b in zip(again, (o, lse, dq, dk, dv)))
    acc0 = randn((B, Lq, Hq, 128), 5).cuda()
    acc = acc0.clone()
    ops.attn_bwd(qg, kg, vg, o, lse, dog, causal=causal, dq=acc, accumulate_dq=True)
    assert_parity((acc - acc0).cpu(), dq_ref, TOL_BF16, "dq added to an fp32 buffer", 1e-3)
    pos_q = (torch.arange(Lq).cuda() + max(Lk - Lq, 0)).repeat(B, 1)
    pos_k = torch.arange(Lk).cuda().repeat(B, 1)
    tables = ops.rope_table(pos_q, B * Lq, 128, 10000.0), ops.rope_table(pos_k, B * Lk, 128, 10000.0)
    dq_r, dk_r, _ = ops.attn_bwd(qg, kg, vg, o, lse, dog, causal=causal, rope_tables=tables)
    assert_parity(dq_r, oracle.apply_rope_bwd(dq_ref, *oracle.rope_cos_sin(pos_q.cpu(), 128, 10000.0)), TOL_BF16, "dq rotated back", 1e-3)
    assert_parity(dk_r, oracle.apply_rope_bwd(dk_ref, *oracle.rope_cos_sin(pos_k.cpu(), 128, 10000.0)), TOL_BF16, "dk rotated back", 1e-3)


@pytest.mark.parametrize("late", [4.0, 40.0], ids=["row_sum", "infinite"])
def test_scores_and_sums_beyond_a_fixed_reference(late):
    """Late scores far above a row's first tile, and with them sums of P V beyond fp32: the block walks its keys again."""
    from odysseus_transformer_amd import ops
    q, k, v, _ = _inputs(1, 300, 300, 2, 2, 29)
    q[:, :, 0], k[:, :, 0] = 2.0, -4.0
    k[:, 200:220, 0] = late
    v[:, 210, 0] = 1e30
    o_ref, lse_ref = oracle.attention_fwd(q.float(), k.float(), v.float(), causal=True)
    (o, lse), ran = _run(lambda: ops.attn_fwd(q.cuda(), k.cuda(), v.cuda(), causal=True))
    assert "attn_fwd_short" in ran and torch.isfinite(o).all()
    assert rel_err(o[:, :, 0], o_ref[:, :, 0]) <= TOL_BF16
    assert_parity(o[:, :, 1], o_ref[:, :, 1], TOL_BF16, "o of the ordinary head")
    assert torch.allclose(lse.cpu(), lse_ref, atol=TOL_LSE, rtol=TOL_LSE)


def test_query_side_of_few_blocks_serves_the_other_kernels():
    """The causal step of a ring, then a full one that takes its query-side scratch as it is and runs on the kernels for long rows."""
    from odysseus_transformer_amd import ops
    q, k, v, do = (t.cuda() for t in _inputs(1, 2200, 2200, 8, 2, 7))
    o, lse = ops.attn_fwd(q, k, v, causal=True)
    ws = ops.attn_bwd_workspace(q, k)
    _, ran = _run(lambda: ops.attn_bwd(q, k, v, o, lse, do, causal=True, workspace=ws))
    assert {"attn_bwd_short", "attn_bwd_prepass"} <= ran, ran
    reused, ran = _run(lambda: ops.attn_bwd(q, v, k, o, lse, do, causal=False, workspace=ws, reuse_query_side=True))
    assert "attn_bwd_dq_pipe" in ran and "attn_bwd_prepass" not in ran, ran
    assert all(torch.equal(a, b) for a, b in zip(reused, ops.attn_bwd(q, v, k, o, lse, do, causal=False)))


@pytest.mark.parametrize("case", [(1, 512, 512, 1, 1, True), (1, 512, 512, 2, 2, True), (1, 1024, 768, 1, 1, False)], ids=lambda c: "Lq%d_Lk%d_H%d_c%d" % (*c[1:4], c[5]))
def test_backward_of_one_or_two_heads(case):
    """The fewest blocks there are: on these kernels, and dK and dV the bits of a call that keeps dS."""
    from odysseus_transformer_amd import ops
    B, Lq, Lk, Hq, Hkv, causal = case
    print(f"case={case}", flush=True)
    q, k, v, do = (t.cuda() for t in _inputs(B, Lq, Lk, Hq, Hkv, 23))
    o, lse = ops.attn_fwd(q, k, v, causal=causal)
    got, ran = _run(lambda: ops.attn_bwd(q, k, v, o, lse, do, causal=causal))
    assert "attn_bwd_short" in ran, ran
    kept, ran = _run(lambda: ops.attn_bwd(q, k, v, o, lse, do, causal=causal, keep_ds=True))
    assert "attn_bwd_dq_kept" in ran and torch.equal(got[1], kept[1]) and torch.equal(got[2], kept[2])
    o_ref, lse_ref = oracle.attention_fwd(*(t.cpu().float() for t in (q, k, v)), causal=causal)
    for a, b, n in zip(got, oracle.attention_bwd(*(t.cpu().float() for t in (q, k, v)), o_ref, lse_ref, do.cpu().float(), causal=causal), ("dq", "dk", "dv")):
        assert_parity(a, b, TOL_BF16, n, 1e-3)


@pytest.mark.parametrize("L,H,short", [(1024, 96, True), (1000, 96, True), (1024, 97, False), (1025, 86, False), (1536, 42, True)])
def test_causal_backward_of_many_blocks(L, H, short):
    """At the line in blocks, which goes by the rows: on either side of it dK and dV are the bits of a call that keeps dS."""
    from odysseus_transformer_amd import ops
    print(f"L={L} H={H}", flush=True)
    q, k, v, do = (t.cuda() for t in _inputs(1, L, L, H, H, 27))
    o, lse = ops.attn_fwd(q, k, v, causal=True)
    got, ran = _run(lambda: ops.attn_bwd(q, k, v, o, lse, do, causal=True))
    assert ("attn_bwd_short" in ran) == short and ("attn_bwd_dq_pipe" in ran) != short, ran
    if L % 256 == 0:
        kept = ops.attn_bwd(q, k, v, o, lse, do, causal=True, keep_ds=True)
        assert torch.equal(got[1], kept[1]) and torch.equal(got[2], kept[2])
    q, k, v, do = (t[:, :, :2].cpu().float() for t in (q, k, v, do))
    for a, b, n in zip(got, oracle.attention_bwd(q, k, v, *oracle.attention_fwd(q, k, v, causal=True), do, causal=True), ("dq", "dk", "dv")):
        assert_parity(a[:, :, :2], b, TOL_BF16, n, 1e-3)


# the forward's ring: fewer and more tiles than it holds, odd and even counts, ragged last sub-tiles, wavefronts and groups without a key, blocks without
# one, and calls on either side of its lines
@pytest.mark.parametrize("case", [(1, 512, 512, 2, 1, True), (1, 511, 511, 2, 2, True), (1, 61, 513, 3, 3, True), (1, 700, 545, 2, 2, True), (2, 900, 577, 2, 1, True),
                                  (1, 1023, 1023, 4, 4, True), (1, 130, 320, 2, 2, False), (1, 130, 319, 2, 2, False), (1, 257, 353, 2, 1, False), (1, 97, 991, 2, 2, False),
                                  (1, 2561, 4100, 7, 7, True), (1, 2049, 1536, 17, 17, True)], ids=lambda c: "B%d_Lq%d_Lk%d_H%d_%d_c%d" % c)
@pytest.mark.parametrize("late", [1.0, 40.0], ids=["unit", "outgrown"])
def test_forward_ring(case, late):
    from odysseus_transformer_amd import ops
    B, Lq, Lk, Hq, Hkv, causal = case
    print(f"case={case} late={late}", flush=True)
    q, k, v, _ = _inputs(B, Lq, Lk, Hq, Hkv, 7 * Lq + Lk)
    k[:, Lk // 2:] *= late
    (o, lse), ran = _run(lambda: ops.attn_fwd(q.cuda(), k.cuda(), v.cuda(), causal=causal))
    assert "attn_fwd_short" in ran, ran
    o_ref, lse_ref = oracle.attention_fwd(q.float(), k.float(), v.float(), causal=causal)
    assert_parity(o, o_ref, TOL_BF16, "o")
    assert torch.allclose(lse.cpu(), lse_ref, atol=TOL_LSE, rtol=TOL_LSE)


# the backward's rings likewise: either side of their line, in one direction only, few and many tiles, wavefronts without a query or a key
@pytest.mark.parametrize("case", [(1, 511, 512, 2, 1, True), (1, 511, 511, 2, 2, True), (1, 33, 545, 3, 3, True), (1, 700, 31, 2, 2, True), (2, 900, 577, 2, 1, True),
                                  (1, 130, 513, 2, 2, False), (1, 577, 65, 4, 1, False), (1, 1023, 1025, 4, 4, True), (1, 97, 991, 2, 2, False),
                                  (1, 3401, 3400, 1, 1, True), (1, 1601, 3500, 3, 3, False), (1, 959, 959, 17, 17, True), (1, 961, 960, 17, 17, True)],
                         ids=lambda c: "B%d_Lq%d_Lk%d_H%d_%d_c%d" % c)
def test_backward_rings(case):
    from odysseus_transformer_amd import ops
    B, Lq, Lk, Hq, Hkv, causal = case
    print(f"case={case}", flush=True)
    q, k, v, do = _inputs(B, Lq, Lk, Hq, Hkv, 11 * Lq + Lk)
    o_ref, lse_ref = oracle.attention_fwd(q.float(), k.float(), v.float(), causal=causal)
    refs = oracle.attention_bwd(q.float(), k.float(), v.float(), o_ref, lse_ref, do.float(), causal=causal)
    qg, kg, vg, dog = (t.cuda() for t in (q, k, v, do))
    o, lse = ops.attn_fwd(qg, kg, vg, causal=causal)
    grads, ran = _run(lambda: ops.attn_bwd(qg, kg, vg, o, lse, dog, causal=causal))
    assert "attn_bwd_short" in ran, ran
    for got, ref, name in zip(grads, refs, ("dq", "dk", "dv")):
        assert_parity(got, ref, TOL_BF16, name, 1e-3)
    assert all(torch.equal(a, b) for a, b in zip(grads, ops.attn_bwd(qg, kg, vg, o, lse, dog, causal=causal)))


def test_backward_ring_has_the_sums_of_the_kernels_for_long_rows():
    """dK and dV do not depend on whether dS is kept, which those kernels do."""
    from odysseus_transformer_amd import ops
    q, k, v, do = (t.cuda() for t in _inputs(1, 1024, 1024, 16, 4, 77))
    o, lse = ops.attn_fwd(q, k, v, causal=True)
    got, ran = _run(lambda: ops.attn_bwd(q, k, v, o, lse, do, causal=True))
    assert "attn_bwd_short" in ran, ran
    kept, ran = _run(lambda: ops.attn_bwd(q, k, v, o, lse, do, causal=True, keep_ds=True))
    assert "attn_bwd_short" not in ran, ran
    assert torch.equal(got[1], kept[1]) and torch.equal(got[2], kept[2])


@pytest.mark.parametrize("stride", [(1 << 24) - 16, (1 << 24) - 8], ids=str)
def test_rows_beyond_a_tiles_offsets_go_to_the_other_kernels(stride):
    from odysseus_transformer_amd import ops
    q, k, v, _ = _inputs(1, 200, 130, 1, 1, 3)
    far = torch.empty(stride * 129 + 128, dtype=torch.bfloat16, device="cuda").as_strided((1, 130, 1, 128), (0, stride, 128, 1))
    far.copy_(v)
    (o, lse), ran = _run(lambda: ops.attn_fwd(q.cuda(), k.cuda(), far, causal=True))
    assert ("attn_fwd_short" in ran) == (stride < (1 << 24) - 8), ran
    o_ref, lse_ref = oracle.attention_fwd(q.float(), k.float(), v.float(), causal=True)
    assert_parity(o, o_ref, TOL_BF16, "o")
    assert torch.allclose(lse.cpu(), lse_ref, atol=TOL_LSE, rtol=TOL_LSE)


def _instance(names, kernel):
    """The one instance of `kernel` among the launched ones: its template arguments, "" if it has none, None if it did not run."""
    ran = {n.split(kernel, 1)[1].split("(", 1)[0] for n in names if kernel in n}
    assert len(ran) <= 1, names
    return ran.pop() if ran else None


# loop or ring, on both sides of the forward's lines
@pytest.mark.parametrize("case,ring", [
    ((1, 512, 512, 2, 1, True), True), ((1, 511, 511, 2, 2, True), False), ((1, 61, 513, 3, 3, True), True), ((1, 700, 545, 2, 2, True), True),
    ((2, 900, 577, 2, 1, True), True), ((1, 1023, 1023, 4, 4, True), True), ((1, 130, 320, 2, 2, False), True), ((1, 130, 319, 2, 2, False), False),
    ((1, 257, 353, 2, 1, False), True), ((1, 97, 991, 2, 2, False), True), ((1, 2561, 4100, 7, 7, True), True), ((1, 2049, 1536, 17, 17, True), True),
    ((1, 2049, 1535, 17, 17, True), False), ((1, 1664, 320, 16, 8, False), True), ((1, 1665, 959, 15, 5, False), False), ((1, 1665, 960, 15, 15, False), True)],
    ids=lambda c: "B%d_Lq%d_Lk%d_H%d_%d_c%d" % c if isinstance(c, tuple) else "ring" if c else "loop")
def test_forward_on_the_instance_of_its_sizes(case, ring):
    from odysseus_transformer_amd import ops
    B, Lq, Lk, Hq, Hkv, causal = case
    print(f"case={case}", flush=True)
    q, k, v, _ = _inputs(B, Lq, Lk, Hq, Hkv, 7 * Lq + Lk)
    (o, lse), ran = device_kernels(lambda: ops.attn_fwd(q.cuda(), k.cuda(), v.cuda(), causal=causal))
    assert _instance(ran, "attn_fwd_short") == ("_ring_kernel" if ring else "_kernel"), ran
    o_ref, lse_ref = oracle.attention_fwd(q.float(), k.float(), v.float(), causal=causal)
    assert_parity(o, o_ref, TOL_BF16, "o")
    assert torch.allclose(lse.cpu(), lse_ref, atol=TOL_LSE, rtol=TOL_LSE)


# and of the backward's (test_backward_rings compares their results)
@pytest.mark.parametrize("case,ring", [
    ((1, 511, 512, 2, 1, True), True), ((1, 511, 511, 2, 2, True), False), ((1, 33, 545, 3, 3, True), True), ((1, 700, 31, 2, 2, True), True),
    ((2, 900, 577, 2, 1, True), True), ((1, 130, 513, 2, 2, False), True), ((1, 577, 65, 4, 1, False), True), ((1, 1023, 1025, 4, 4, True), True),
    ((1, 97, 991, 2, 2, False), True), ((1, 3401, 3400, 1, 1, True), True), ((1, 1601, 3500, 3, 3, False), True), ((1, 959, 959, 17, 17, True), False),
    ((1, 961, 960, 17, 17, True), True)],
    ids=lambda c: "B%d_Lq%d_Lk%d_H%d_%d_c%d" % c if isinstance(c, tuple) else "ring" if c else "loop")
def test_backward_on_the_instance_of_its_sizes(case, ring):
    from odysseus_transformer_amd import ops
    B, Lq, Lk, Hq, Hkv, causal = case
    print(f"case={case}", flush=True)
    q, k, v, do = (t.cuda() for t in _inputs(B, Lq, Lk, Hq, Hkv, 11 * Lq + Lk))
    o, lse = ops.attn_fwd(q, k, v, causal=causal)
    _, ran = device_kernels(lambda: ops.attn_bwd(q, k, v, o, lse, do, causal=causal))
    assert _instance(ran, "attn_bwd_short_kernel") == f"<{str(Hq != Hkv).lower()}, {str(ring).lower()}>", ran


@pytest.mark.parametrize("stride", [(1 << 24) - 16, (1 << 24) - 8], ids=str)
@pytest.mark.parametrize("far", ["keys", "queries"])
def test_rings_over_rows_far_apart(far, stride):
    """Keys and values, or queries and the gradient of the output, with the last row stride whose tile fits 32-bit offsets and the first one beyond: the
    rings, and the kernels with 64-bit ones."""
    from odysseus_transformer_amd import ops
    Lq, Lk = (130, 545) if far == "keys" else (545, 130)
    near = stride < (1 << 24) - 8
    print(f"{far=} {stride=}", flush=True)
    q, k, v, do = _inputs(1, Lq, Lk, 1, 1, 5)
    o_ref, lse_ref = oracle.attention_fwd(q.float(), k.float(), v.float(), causal=False)
    refs = oracle.attention_bwd(q.float(), k.float(), v.float(), o_ref, lse_ref, do.float(), causal=False)
    rows = max(Lq, Lk)
    apart = torch.empty(stride * (rows - 1) + 256, dtype=torch.bfloat16, device="cuda")
    pair = [apart.as_strided((1, rows, 1, 128), (0, stride, 128, 1), 128 * n).copy_(t) for n, t in enumerate((k, v) if far == "keys" else (q, do))]
    q, k, v, do = (t.cuda() for t in (q, k, v, do))
    if far == "keys":
        k, v = pair
        (o, lse), ran = device_kernels(lambda: ops.attn_fwd(q, k, v, causal=False))
        assert _instance(ran, "attn_fwd_short") == ("_ring_kernel" if near else None), ran
        assert_parity(o, o_ref, TOL_BF16, "o")
        assert torch.allclose(lse.cpu(), lse_ref, atol=TOL_LSE, rtol=TOL_LSE)
    else:
        q, do = pair
    new = {n: torch.empty((1, L, 1, 128), dtype=torch.bfloat16, device="cuda") for n, L in (("dq", Lq), ("dk", Lk), ("dv", Lk))}
    grads, ran = device_kernels(lambda: ops.attn_bwd(q, k, v, o_ref.bfloat16().cuda(), lse_ref.cuda(), do, causal=False, **new))
    assert _instance(ran, "attn_bwd_short_kernel") == f"<false, {str(near).lower()}>", ran
    for got, ref, name in zip(grads, refs, ("dq", "dk", "dv")):
        assert_parity(got, ref, TOL_BF16, name, 1e-3)
