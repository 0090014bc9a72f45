"""GPU parity of the long-sequence forward (csrc/attn_fwd_pipe.hip) where its ring and its phases can go wrong: key ranges of one tile, of fewer
tiles than the ring holds and of one more, ragged last tiles, wavefronts without a key, first tiles that need the mask, strided keys."""
import math

import pytest
import torch

from conftest import TOL_BF16, TOL_LSE, assert_parity, randn
import odysseus_oracle as oracle

pytestmark = pytest.mark.gpu


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


# more than 640 (causal) / 256 blocks of 128 queries keep these off the kernel for few blocks
@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("Lk", [1, 31, 33, 64, 65, 128, 130, 192, 193, 256, 319, 321, 385])
def test_few_key_tiles(Lk, causal, dev):
    from odysseus_transformer_amd import ops
    Hq, Lq = (16, 5136) if causal else (8, 4137)
    print(f"Lk={Lk} causal={causal}", flush=True)
    q, k, v = (randn((1, L, H, 128), 31 + n, dtype=torch.bfloat16) for n, (L, H) in enumerate(((Lq, Hq), (Lk, 2), (Lk, 2))))
    (o, lse), ran = _ran(lambda: ops.attn_fwd(q.to(dev), k.to(dev), v.to(dev), causal=causal))
    assert "attn_fwd_pipe" in ran, ran
    o_ref, lse_ref = oracle.attention_fwd(q.float(), k.float(), v.float(), causal=causal)
    assert_parity(o, o_ref, TOL_BF16, "o")
    assert torch.allclose(lse.cpu(), lse_ref, atol=TOL_LSE, rtol=TOL_LSE)


@pytest.mark.parametrize("L", [2049, 2303, 2560, 3001])
def test_causal_rows_of_every_block_position(L, dev):
    """First tiles with and without a mask, key ranges cut into parts and not, four heads on one."""
    from odysseus_transformer_amd import ops
    for Hq in (4, 44):
        print(f"L={L} Hq={Hq}", flush=True)
        q, k, v = (randn((1, L, H, 128), 41 + n, dtype=torch.bfloat16) for n, H in enumerate((Hq, Hq // 4, Hq // 4)))
        (o, lse), ran = _ran(lambda: ops.attn_fwd(q.to(dev), k.to(dev), v.to(dev), causal=True))
        assert "attn_fwd_pipe" in ran, ran
        heads = slice(0, 4)   # of the first kv head
        o_ref, lse_ref = oracle.attention_fwd(q[:, :, heads].float(), k[:, :, :1].float(), v[:, :, :1].float(), causal=True)
        assert_parity(o[:, :, heads], o_ref, TOL_BF16, "o")
        assert torch.allclose(lse.cpu()[:, heads], lse_ref, atol=TOL_LSE, rtol=TOL_LSE)


@pytest.mark.parametrize("stride", [128, 1 << 23, (1 << 24) - 8, 1 << 24], ids=str)
def test_keys_far_apart(stride, dev):
    """Row strides up to the last one whose tile fits 32-bit offsets, and the first one beyond, which the kernel behind takes."""
    from odysseus_transformer_amd import ops
    Lq, Lk, Hq = 8200, 67, 4
    q, k, v = (randn((1, L, H, 128), 51 + n, dtype=torch.bfloat16) for n, (L, H) in enumerate(((Lq, Hq), (Lk, 1), (Lk, 1))))
    far = torch.empty(stride * (Lk - 1) + 128, dtype=torch.bfloat16, device=dev).as_strided((1, Lk, 1, 128), (0, stride, 128, 1))
    far.copy_(k.to(dev))
    print(f"stride={stride}", flush=True)
    (o, lse), ran = _ran(lambda: ops.attn_fwd(q.to(dev), far, v.to(dev), causal=False))
    assert "attn_fwd_pipe" in ran, ran
    near = ops.attn_fwd(q.to(dev), k.to(dev), v.to(dev), causal=False)
    assert_parity(o, near[0].float().cpu(), TOL_BF16, "o")
    assert torch.allclose(lse, near[1], atol=TOL_LSE, rtol=TOL_LSE)


@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("D", [64, 128])
def test_row_sums_of_many_small_weights(D, causal, dev):
    """The first key has weight 1, every other one 2^-24.5, less than half of the last bit of 1: what is added to a sum that holds the first key is
    lost.  A row is summed in four chains by each half of a wavefront, so that this is an eighth of the keys (0.15: with the roundings of lse,
    below 1e-6); with two chains it is a quarter."""
    from odysseus_transformer_amd import ops
    L, H = (4096, 48) if causal else (256, 256)
    Lk = max(L, 8192)
    q, k = torch.zeros((1, L, H, D)), torch.zeros((1, Lk, 1, D))
    q[..., 0], k[:, 1:, :, 0] = 1.0, -24.5
    v = randn((1, Lk, 1, D), 45, dtype=torch.bfloat16)
    (o, lse), ran = _ran(lambda: ops.attn_fwd(q.bfloat16().to(dev), k.bfloat16().to(dev), v.to(dev), causal=causal, scale=math.log(2.0)))
    assert ("attn_fwd_pipe" if D == 128 else "attn_fwd_hd64_pipe") in ran, ran
    seen = torch.arange(Lk - L + 1, Lk + 1) if causal else torch.full((L,), Lk)
    small = (seen - 1).double() * 2.0 ** -24.5
    assert bool(((lse.cpu().double() - small.log1p()).abs() <= 0.15 * small + 1e-6).all())
