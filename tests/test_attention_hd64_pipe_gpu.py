"""GPU parity of the head_dim-64 kernels for many blocks (csrc/attn_hd64_pipe.hip) at the edges of their tiles, rings, blocks and dispatch, against
the oracle, and of the calls that stay with the kernels for few."""
import pytest
import torch

from conftest import TOL_BF16, TOL_LSE, assert_parity, device_kernels, randn
import odysseus_oracle as oracle

pytestmark = pytest.mark.gpu
FWD, DKDV = "attn_fwd_hd64_pipe", "attn_bwd_hd64_dkdv_pipe"


def _ran(f):
    from odysseus_transformer_amd import _lib
    _lib.profile_enable(True)
    try:
        _lib.profile_collect()
        out = f()
        torch.cuda.synchronize()
        return out, set(_lib.profile_collect())
    finally:
        _lib.profile_enable(False)


def _inputs(B, Lq, Lk, Hq, Hkv, seed):
    shapes = ((Lq, Hq), (Lk, Hkv), (Lk, Hkv), (Lq, Hq))
    return [randn((B, L, H, 64), seed + n, dtype=torch.bfloat16) for n, (L, H) in enumerate(shapes)]


def _check(B, Lq, Lk, Hq, Hkv, causal, fwd, dkdv, dev, seed=61, heads=None, stretch=1.0):
    """All of a call; the oracle for the first `heads` kv heads only, which see the others' blocks as neighbours."""
    from odysseus_transformer_amd import ops
    print(f"{B=} {Lq=} {Lk=} {Hq=} {Hkv=} {causal=} {stretch=}", flush=True)
    q, k, v, do = _inputs(B, Lq, Lk, Hq, Hkv, seed)
    k = (k.float() * torch.linspace(1.0, stretch, Lk)[None, :, None, None]).bfloat16()
    qg, kg, vg, dog = (t.to(dev) for t in (q, k, v, do))
    (o, lse), ran = _ran(lambda: ops.attn_fwd(qg, kg, vg, causal=causal))
    assert (FWD in ran) == fwd, ran
    grads, ran = _ran(lambda: ops.attn_bwd(qg, kg, vg, o, lse, dog, causal=causal))
    assert (DKDV in ran) == dkdv, ran
    n, G = heads or Hkv, Hq // Hkv
    q, k, v, do, o, lse = q[:, :, :n * G], k[:, :, :n], v[:, :, :n], do[:, :, :n * G], o[:, :, :n * G].cpu(), lse[:, :n * G].cpu()
    o_ref, lse_ref = oracle.attention_fwd(q.float(), k.float(), v.float(), causal=causal)
    assert_parity(o, o_ref, TOL_BF16, "o")
    assert torch.allclose(lse, lse_ref, atol=TOL_LSE, rtol=TOL_LSE)
    # gradients from the o and lse that the kernels had: one-hot rows leave dS little but the rounding of out
    refs = oracle.attention_bwd(q.float(), k.float(), v.float(), o.float(), lse, do.float(), causal=causal)
    for got, ref, name, count in zip(grads, refs, ("dq", "dk", "dv"), (n * G, n, n)):
        assert_parity(got[:, :, :count], ref, TOL_BF16, name, 1e-3)
    return o


# keys from the fewest that the forward takes on: whole and ragged last tiles, rings that wrap; queries: whole blocks, half a last one
@pytest.mark.parametrize("stretch", [1.0, 60.0], ids=["unit", "moving_reference"])
@pytest.mark.parametrize("Lq,Lk", [(512, 512), (505, 513), (1024, 575), (1000, 639), (2049, 641)])
def test_full(Lq, Lk, stretch, dev):
    H = 512 // ((Lq + 255) // 256)   # two whole rounds of 256 blocks
    _check(1, Lq, Lk, H, H, False, True, True, dev, heads=3, stretch=stretch)


# at the lines of the causal forward: 768 blocks, 1024 blocks of 2048 keys; more keys than queries, more queries than keys
@pytest.mark.parametrize("L,Lk,Hq,Hkv", [(4096, 4096, 48, 12), (2000, 2048, 128, 128), (1991, 2111, 128, 32), (4091, 2731, 48, 48), (4099, 4096, 46, 46),
                                         (4500, 4096, 44, 22)])
def test_causal(L, Lk, Hq, Hkv, dev):
    _check(1, L, Lk, Hq, Hkv, True, True, True, dev, heads=1)


# 6 tiles of queries and a few keys: fewer tiles than the ring holds for the last key blocks, wavefronts without a query, ranges of one key
@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("B,Lq,Lk,Hq,Hkv", [(1, 321, 1, 64, 64), (2, 321, 127, 32, 32), (1, 383, 129, 4, 1), (1, 385, 700, 4, 2), (1, 700, 385, 16, 16), (1, 1031, 1031, 2, 1)])
def test_few_keys_or_queries(B, Lq, Lk, Hq, Hkv, causal, dev):
    _check(B, Lq, Lk, Hq, Hkv, causal, False, True, dev)


@pytest.mark.parametrize("Lq,Lk,H,causal", [(320, 320, 2, False), (512, 511, 128, False), (128, 512, 256, False), (640, 512, 86, False),
                                            (2048, 2048, 127, True), (4096, 4096, 47, True), (1000, 1000, 7, True), (1000, 1000, 8, False)])
def test_calls_that_stay_with_the_kernels_for_few_blocks(Lq, Lk, H, causal, dev):
    _check(1, Lq, Lk, H, H, causal, False, Lq > 320 and H * ((Lk + 127) // 128) >= 64, dev, heads=2)


# at the lines that rounds draw: forward, a last round that is full, more or less than half full, of few rounds and of many; dK / dV, 512 key blocks
# and more of few and of many queries
@pytest.mark.parametrize("Lq,Lk,H,causal,fwd,dkdv", [(1000, 600, 75, False, False, True), (1000, 600, 98, False, True, True), (1000, 650, 64, False, True, True),
                                                     (1000, 600, 64, False, False, True), (2100, 600, 44, False, False, True), (260, 520, 512, False, False, False),
                                                     (512, 1024, 258, False, False, True), (512, 1024, 514, False, True, True), (1000, 550, 385, False, False, True),
                                                     (708, 708, 128, True, False, False), (961, 961, 65, True, False, True), (708, 708, 85, True, False, True),
                                                     (448, 600, 128, False, False, False), (449, 600, 128, False, False, True)])
def test_last_rounds(Lq, Lk, H, causal, fwd, dkdv, dev):
    _check(1, Lq, Lk, H, H, causal, fwd, dkdv, dev, heads=2)


def test_the_same_bits_again_and_a_reused_query_side(dev):
    from odysseus_transformer_amd import ops
    q, k, v, do = (t.to(dev) for t in _inputs(1, 900, 1100, 8, 4, 71))
    o, lse = ops.attn_fwd(q, k, v, causal=False)
    ws = ops.attn_bwd_workspace(q, k)
    first = ops.attn_bwd(q, k, v, o, lse, do, causal=False, workspace=ws)
    for reuse in (True, False, True):
        again, ran = _ran(lambda: ops.attn_bwd(q, k, v, o, lse, do, causal=False, workspace=ws, reuse_query_side=reuse))
        assert DKDV in ran and ("attn_bwd_hd64_rows" in ran) != reuse, ran
        assert all(torch.equal(a, b) for a, b in zip(first, again))


@pytest.mark.parametrize("Hkv,first", [(8, 100), (4, 1100), (8, 1100)])
def test_a_reused_query_side_behind_other_keys(Hkv, first, dev):
    """Every call with the workspace of its own size, from one buffer: the one before had fewer keys and took the other dK / dV kernel, or the same
    one, which left start values of another scale."""
    from odysseus_transformer_amd import ops
    q, k, v, do = (t.to(dev) for t in _inputs(1, 900, 1100, 8, Hkv, 75))
    o, lse = ops.attn_fwd(q, k, v, causal=False)
    want = ops.attn_bwd(q, k, v, o, lse, do, causal=False)
    whole = torch.full_like(ops.attn_bwd_workspace(q, k), 255)
    few, fewv = k[:, :first], v[:, :first]
    part = whole[:ops.attn_bwd_workspace_bytes(q, few)]
    ops.attn_bwd(q, few, fewv, o, lse, do, causal=False, workspace=part, scale=0.1)
    got, ran = _ran(lambda: ops.attn_bwd(q, k, v, o, lse, do, causal=False, workspace=whole, reuse_query_side=True))
    assert DKDV in ran and "attn_bwd_hd64_rows" not in ran, ran
    assert all(torch.equal(a, b) for a, b in zip(want, got))


@pytest.mark.parametrize("stride", [64, 1 << 23, (1 << 24) - 16, (1 << 24) - 8], ids=str)
def test_rows_far_apart(stride, dev):
    """Row strides up to the last one whose tile fits 32-bit offsets, and the first one beyond: keys of the forward, queries of dK / dV."""
    from odysseus_transformer_amd import ops
    near = stride < (1 << 24) - 8
    q, k, v, do = _inputs(1, 513 * 256, 520, 1, 1, 81)
    q, do = q[:, :131072 - 7], do[:, :131072 - 7]

    def far(t):
        out = torch.empty(stride * (t.shape[1] - 1) + 64, dtype=torch.bfloat16, device=dev).as_strided(t.shape, (0, stride, 64, 1))
        return out.copy_(t)
    fk = far(k)
    (o, lse), ran = _ran(lambda: ops.attn_fwd(q.to(dev), fk, v.to(dev), causal=False))
    assert (FWD in ran) == near, ran
    o_ref, lse_ref = oracle.attention_fwd(q[:, -300:].float(), k.float(), v.float(), causal=False)
    assert_parity(o[:, -300:], o_ref, TOL_BF16, "o")
    del fk
    q, k, v, do = _inputs(1, 330, 200, 1, 1, 82)
    o_ref, lse_ref = oracle.attention_fwd(q.float(), k.float(), v.float(), causal=True)
    refs = oracle.attention_bwd(q.float(), k.float(), v.float(), o_ref, lse_ref, do.float(), causal=True)
    grads, ran = _ran(lambda: ops.attn_bwd(far(q), k.to(dev), v.to(dev), o_ref.bfloat16().to(dev), lse_ref.to(dev), do.to(dev), causal=True,
                                           dq=torch.empty(q.shape, dtype=torch.bfloat16, device=dev),
                                           workspace=torch.empty(1 << 14, dtype=torch.uint8, device=dev)))   # with room for its row values
    assert (DKDV in ran) == near, ran
    for got, ref, name in zip(grads, refs, ("dq", "dk", "dv")):
        assert_parity(got, ref, TOL_BF16, name)


@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
def test_large_values_behind_an_outgrown_reference(causal, dev):
    """Scores 56 above a row's first tile with |v| around 2^48: the blocks walk their keys once more, and nothing may overflow on the way."""
    from odysseus_transformer_amd import ops
    L, H = (4096, 48) if causal else (1000, 64)
    q, k, v, _ = _inputs(1, L, L, H, H, 91)
    q[..., 0], k[..., 0] = 8.0, 0.0
    k[:, -(L // 4):, :, 0] = 56.0
    v = (v.float() * 2.0 ** 48).bfloat16()
    (o, lse), ran = _ran(lambda: ops.attn_fwd(q.to(dev), k.to(dev), v.to(dev), causal=causal))
    assert FWD in ran, ran
    assert bool(o.isfinite().all())
    o_ref, lse_ref = oracle.attention_fwd(q[:, :, :2].float(), k[:, :, :2].float(), v[:, :, :2].float(), causal=causal)
    assert_parity(o[:, :, :2], o_ref, TOL_BF16, "o")
    assert torch.allclose(lse[:, :2].cpu(), lse_ref, atol=TOL_LSE, rtol=TOL_LSE)


# blocks of 128 queries on either side of the lines of the dispatch; half and whole last sub-tiles and tiles, rings that wrap, wavefronts and blocks
# without a key, queries past the end; every form of dq
@pytest.mark.parametrize("form", ["new", "added", "fp32"])
@pytest.mark.parametrize("Lq,Lk,Hq,Hkv,causal,pipe", [
    (1, 1, 2, 1, True, True), (127, 31, 2, 2, False, True), (129, 33, 4, 2, True, True), (200, 96, 3, 3, True, True), (300, 257, 2, 1, False, True),
    (257, 100, 2, 2, True, True), (500, 130, 1, 1, True, True), (161, 700, 2, 1, True, True), (128, 511, 512, 512, False, False),
    (128, 512, 512, 256, False, True), (121, 999, 512, 512, True, False), (256, 1000, 256, 64, True, True)])
def test_dq(Lq, Lk, Hq, Hkv, causal, pipe, form, dev):
    from odysseus_transformer_amd import ops
    print(f"{Lq=} {Lk=} {Hq=} {Hkv=} {causal=} {form=}", flush=True)
    q, k, v, do = _inputs(1, Lq, Lk, Hq, Hkv, 101)
    qg, kg, vg, dog = (t.to(dev) for t in (q, k, v, do))
    o, lse = ops.attn_fwd(qg, kg, vg, causal=causal)
    start = randn((1, Lq, Hq, 64), 105, dtype=torch.bfloat16)
    dq = {"new": None, "added": start.to(dev), "fp32": start.float().to(dev)}[form]
    (got, _, _), ran = _ran(lambda: ops.attn_bwd(qg, kg, vg, o, lse, dog, causal=causal, dq=dq, accumulate_dq=form != "new"))
    assert ("attn_bwd_hd64_dq_pipe" in ran) == pipe, ran
    n, G = min(2, Hkv), Hq // Hkv
    ref = oracle.attention_bwd(q[:, :, :n * G].float(), k[:, :, :n].float(), v[:, :, :n].float(), o[:, :, :n * G].float().cpu(),
                               lse[:, :n * G].cpu(), do[:, :, :n * G].float(), causal=causal)[0]
    assert_parity(got[:, :, :n * G], ref + (0 if form == "new" else start[:, :, :n * G].float()), TOL_BF16, "dq", 1e-3)


def test_keys_behind_a_sub_tile_of_the_mask_do_not_reach_dq(dev):
    """Masked keys 32 and more behind a wavefront's last query are not read into its products, whatever they hold."""
    from odysseus_transformer_amd import ops
    L = 192
    q, k, v, do = (t.to(dev) for t in _inputs(1, L, L, 2, 2, 111))
    o, lse = ops.attn_fwd(q, k, v, causal=True)
    (want, _, _), ran = _ran(lambda: ops.attn_bwd(q, k, v, o, lse, do, causal=True))
    assert "attn_bwd_hd64_dq_pipe" in ran, ran
    for last in (32, 64, 96, 128, 160):
        bk, bv = k.clone(), v.clone()
        bk[:, last:], bv[:, last:] = float("nan"), float("inf")
        got = ops.attn_bwd(q, bk, bv, o, lse, do, causal=True)[0]
        assert torch.equal(got[:, :last], want[:, :last]), last


# forward with eight wavefronts a block: odd counts of tiles, ragged last ones, blocks of 0, 1 and 2 tiles (fewer keys than queries), queries past the end,
# references that a later half outgrows, and the lines of its dispatch (pipe: the kernel with 256-row blocks, with one group of wavefronts or two)
@pytest.mark.parametrize("stretch", [1.0, 60.0], ids=["unit", "moving_reference"])
@pytest.mark.parametrize("Lq,Lk,Hq,Hkv,causal,pipe", [
    (512, 768, 65, 13, False, True), (505, 831, 127, 127, False, True), (2049, 1024, 28, 14, False, True), (512, 767, 65, 65, False, False),
    (512, 1023, 128, 32, False, True), (256, 2048, 128, 128, False, False), (4096, 4096, 32, 8, True, True), (3000, 3000, 22, 22, True, True),
    (6401, 4001, 14, 14, True, True), (8192, 3969, 8, 4, True, True), (4096, 4096, 33, 33, True, False), (3000, 2999, 22, 22, True, False),
    (3000, 4096, 24, 24, True, False)])
def test_forward_in_two_groups(Lq, Lk, Hq, Hkv, causal, pipe, stretch, dev):
    from odysseus_transformer_amd import ops
    print(f"{Lq=} {Lk=} {Hq=} {Hkv=} {causal=} {stretch=}", flush=True)
    q, k, v, _ = _inputs(1, Lq, Lk, Hq, Hkv, 121)
    k = (k.float() * torch.linspace(1.0, stretch, Lk)[None, :, None, None]).bfloat16()
    (o, lse), ran = _ran(lambda: ops.attn_fwd(q.to(dev), k.to(dev), v.to(dev), causal=causal))
    assert (FWD in ran) == pipe, ran
    G = Hq // Hkv
    o_ref, lse_ref = oracle.attention_fwd(q[:, :, :G].float(), k[:, :, :1].float(), v[:, :, :1].float(), causal=causal)
    assert_parity(o[:, :, :G], o_ref, TOL_BF16, "o")
    assert torch.allclose(lse[:, :G].cpu(), lse_ref, atol=TOL_LSE, rtol=TOL_LSE)


@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
def test_large_values_in_two_groups(causal, dev):
    """Keys 56 above the first ones from a quarter in front of the end on, |v| around 2^48: in the second group's tiles, whose reference is among the low ones."""
    from odysseus_transformer_amd import ops
    L, H = (4096, 16) if causal else (1536, 40)
    q, k, v, _ = _inputs(1, L, L, H, H, 131)
    q[..., 0], k[..., 0] = 8.0, 0.0
    k[:, -(L // 4):, :, 0] = 56.0
    v = (v.float() * 2.0 ** 48).bfloat16()
    (o, lse), ran = _ran(lambda: ops.attn_fwd(q.to(dev), k.to(dev), v.to(dev), causal=causal))
    assert FWD in ran, ran
    assert bool(o.isfinite().all())
    o_ref, lse_ref = oracle.attention_fwd(q[:, :, :2].float(), k[:, :, :2].float(), v[:, :, :2].float(), causal=causal)
    assert_parity(o[:, :, :2], o_ref, TOL_BF16, "o")
    assert torch.allclose(lse[:, :2].cpu(), lse_ref, atol=TOL_LSE, rtol=TOL_LSE)


# Which of the forwards runs, on both sides of every line (groups of four wavefronts in a block of 256 rows; 0: the kernel with 128-row blocks)
@pytest.mark.parametrize("Lq,Lk,Hq,Hkv,causal,groups", [
    (512, 768, 65, 13, False, 2), (512, 767, 65, 65, False, 0), (512, 1023, 128, 32, False, 1), (512, 1024, 128, 32, False, 2), (256, 2048, 128, 128, False, 0),
    (4096, 4096, 32, 8, True, 2), (4096, 4096, 33, 33, True, 0), (3000, 3000, 22, 22, True, 2), (3000, 2999, 22, 22, True, 0), (3000, 4096, 24, 24, True, 0)])
def test_forward_on_the_instance_of_its_sizes(Lq, Lk, Hq, Hkv, causal, groups, dev):
    from odysseus_transformer_amd import ops
    print(f"{Lq=} {Lk=} {Hq=} {Hkv=} {causal=}", flush=True)
    q, k, v, _ = _inputs(1, Lq, Lk, Hq, Hkv, 151)
    (o, lse), ran = device_kernels(lambda: ops.attn_fwd(q.to(dev), k.to(dev), v.to(dev), causal=causal))
    assert [g for g in (1, 2) if any(f"attn_fwd_hd64_pipe_kernel<{g}>" in n for n in ran)] == ([groups] if groups else []), ran
    G = Hq // Hkv
    o_ref, lse_ref = oracle.attention_fwd(q[:, :, :G].float(), k[:, :, :1].float(), v[:, :, :1].float(), causal=causal)
    assert_parity(o[:, :, :G], o_ref, TOL_BF16, "o")
    assert torch.allclose(lse[:, :G].cpu(), lse_ref, atol=TOL_LSE, rtol=TOL_LSE)


@pytest.mark.parametrize("stride", [(1 << 24) - 16, (1 << 24) - 8], ids=str)
@pytest.mark.parametrize("H,groups", [(2, 2), (256, 1)])
def test_dq_over_keys_far_apart(H, groups, stride, dev):
    """Keys and values with the last row stride whose tile fits 32-bit offsets and the first one beyond, which the kernels with 64-bit ones take, with two
    sets of wavefronts where blocks are few and with one."""
    from odysseus_transformer_amd import ops
    Lq, Lk = 200, 1000 if H == 256 else 130
    print(f"{H=} {stride=}", flush=True)
    q, k, v, do = _inputs(1, Lq, Lk, H, 1, 141)
    o_ref, lse_ref = oracle.attention_fwd(q[:, :, :2].float(), k.float(), v.float(), causal=True)
    ref = oracle.attention_bwd(q[:, :, :2].float(), k.float(), v.float(), o_ref, lse_ref, do[:, :, :2].float(), causal=True)[0]
    q, k, v, do = (t.to(dev) for t in (q, k, v, do))
    o, lse = ops.attn_fwd(q, k, v, causal=True)
    apart = torch.empty(stride * (Lk - 1) + 128, dtype=torch.bfloat16, device=dev)
    k, v = (apart.as_strided((1, Lk, 1, 64), (0, stride, 64, 1), 64 * n).copy_(t) for n, t in enumerate((k, v)))
    new = {n: torch.empty((1, L, h, 64), dtype=torch.bfloat16, device=dev) for n, L, h in (("dq", Lq, H), ("dk", Lk, 1), ("dv", Lk, 1))}
    got, ran = device_kernels(lambda: ops.attn_bwd(q, k, v, o, lse, do, causal=True, **new)[0])
    kernel = "attn_bwd_hd64_dq_pipe_kernel" if stride < (1 << 24) - 8 else f"attn_bwd_hd64_dq_kernel<{groups}>"
    assert [n for n in ran if "hd64_dq" in n and kernel in n] and len([n for n in ran if "hd64_dq" in n]) == 1, ran
    assert_parity(got[:, :, :2], ref, TOL_BF16, "dq", 1e-3)
