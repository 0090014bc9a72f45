"""GPU parity of the long-sequence backward (csrc/attn_bwd_pipe.hip) where its rings and its order of units can go wrong: one tile on the streamed
side, fewer than the rings hold and one more, ragged last tiles, wavefronts and whole blocks that see nothing, strided rows."""
import pytest
import torch

from conftest import TOL_BF16, assert_parity, randn
import odysseus_oracle as oracle

pytestmark = pytest.mark.gpu
LONG = 3700   # rows beyond the kernels for few blocks


def _ran(f):
    from odysseus_transformer_amd import _lib
    f()
    torch.cuda.synchronize()
    _lib.profile_enable(True)
    out = f()
    torch.cuda.synchronize()
    ran = set(_lib.profile_collect())
    _lib.profile_enable(False)
    return out, ran


def _compare(Lq, Lk, Hq, Hkv, causal, dev, seed):
    from odysseus_transformer_amd import ops
    print(f"Lq={Lq} Lk={Lk} heads={Hq}/{Hkv} causal={causal}", flush=True)
    q, do = (randn((1, Lq, Hq, 128), seed + n, dtype=torch.bfloat16) for n in range(2))
    k, v = (randn((1, Lk, Hkv, 128), seed + 2 + n, dtype=torch.bfloat16) for n in range(2))
    o_ref, lse_ref = oracle.attention_fwd(q.float(), k.float(), v.float(), causal=causal)
    ref = oracle.attention_bwd(q.float(), k.float(), v.float(), o_ref, lse_ref, do.float(), causal=causal)
    qg, kg, vg, dog = (t.to(dev) for t in (q, k, v, do))
    o, lse = ops.attn_fwd(qg, kg, vg, causal=causal)
    got, ran = _ran(lambda: ops.attn_bwd(qg, kg, vg, o, lse, dog, causal=causal))
    assert {"attn_bwd_dkdv_pipe", "attn_bwd_dq_pipe"} <= ran, ran
    floor = 1.0 if Lk == 1 else 1e-3   # a single key: dS is identically zero, compared on the scale of the inputs
    for a, r, n in zip(got, ref, ("dq", "dk", "dv")):
        assert_parity(a, r, TOL_BF16, n, 1e-3 if n == "dv" else floor)


@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("Lq", [1, 31, 64, 65, 128, 129, 193, 257])
def test_few_query_tiles(Lq, causal, dev):
    _compare(Lq, LONG, 2, 1 if Lq % 2 else 2, causal, dev, 61)


@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("Lk", [1, 33, 64, 65, 128, 130, 192, 259])
def test_few_key_tiles(Lk, causal, dev):
    _compare(LONG, Lk, 2, 1 if Lk % 2 else 2, causal, dev, 71)


@pytest.mark.parametrize("L", [3649, 3839, 3840, 4033])
def test_causal_rows_of_every_block_position(L, dev):
    _compare(L, L, 2, 1, True, dev, 81)


@pytest.mark.parametrize("stride", [1 << 23, (1 << 24) - 16, 1 << 24], ids=str)
def test_keys_far_apart(stride, dev):
    """Row strides up to the last one whose tile fits 32-bit offsets, and one beyond, which the kernels with 64-bit ones take."""
    from odysseus_transformer_amd import ops
    Lk = 67
    q, do = (randn((1, LONG, 2, 128), 91 + n, dtype=torch.bfloat16).to(dev) for n in range(2))
    k, v = (randn((1, Lk, 1, 128), 93 + n, dtype=torch.bfloat16).to(dev) for n in range(2))
    far = torch.empty(stride * (Lk - 1) + 128, dtype=torch.bfloat16, device=dev).as_strided((1, Lk, 1, 128), (0, stride, 128, 1))
    far.copy_(k)
    print(f"stride={stride}", flush=True)
    o, lse = ops.attn_fwd(q, k, v, causal=False)
    got, ran = _ran(lambda: ops.attn_bwd(q, far, v, o, lse, do, causal=False))
    assert ("attn_bwd_short" if stride >= 1 << 24 else "attn_bwd_dq_pipe") in ran, ran
    for a, r, n in zip(got, ops.attn_bwd(q, k, v, o, lse, do, causal=False), ("dq", "dk", "dv")):
        assert_parity(a, r.float().cpu(), TOL_BF16, n)


@pytest.mark.parametrize("keep", [False, True], ids=["recomputed", "kept"])
@pytest.mark.parametrize("Hkv", [1, 2])
@pytest.mark.parametrize("which", ["q", "k", "v", "do"])
def test_any_operand_far_apart(which, Hkv, keep, dev):
    """Every operand of these kernels, with grouped heads and where dS would be kept: beyond 32-bit offsets all go to the kernels with 64-bit ones."""
    from odysseus_transformer_amd import ops
    L, stride = 256, 1 << 24
    t = {n: randn((1, L, H, 128), 95 + m, dtype=torch.bfloat16).to(dev) for m, (n, H) in enumerate((("q", 2), ("k", Hkv), ("v", Hkv), ("do", 2)))}
    o, lse = ops.attn_fwd(t["q"], t["k"], t["v"], causal=True)
    want = ops.attn_bwd(t["q"], t["k"], t["v"], o, lse, t["do"], causal=True, keep_ds=True)
    H = t[which].shape[2]
    far = torch.empty(stride * (L - 1) + 128 * H, dtype=torch.bfloat16, device=dev).as_strided((1, L, H, 128), (0, stride, 128, 1))
    t[which] = far.copy_(t[which])
    print(f"{which} far apart, {Hkv} kv heads, keep_ds={keep}", flush=True)
    new = {n: torch.empty((1, L, h, 128), dtype=torch.bfloat16, device=dev) for n, h in (("dq", 2), ("dk", Hkv), ("dv", Hkv))}
    got, ran = _ran(lambda: ops.attn_bwd(t["q"], t["k"], t["v"], o, lse, t["do"], causal=True, keep_ds=keep, **new))
    assert "attn_bwd_short" in ran and "attn_bwd_dq_kept" not in ran, ran
    for a, r, n in zip(got, want, ("dq", "dk", "dv")):
        assert_parity(a, r.float().cpu(), TOL_BF16, n)
