"""The host path in C++ against the one in Python: the same results bit for bit over the forms that it takes, and the same answers to
what it leaves alone."""
import pytest
import torch

from conftest import randn

pytestmark = pytest.mark.gpu


class _Off:
    """Stands for the module where it answers None to everything."""

    def __getattr__(self, name):
        return lambda *a: None


def _both(monkeypatch, fn):
    """fn() on either path, and how many calls the C++ one answered."""
    from odysseus_transformer_amd import ops
    taken = []

    class Counting:
        def __getattr__(self, name):
            def call(*a):
                r = getattr(ops_native, name)(*a)
                if r is not None:
                    taken.append(name)
                return r
            return call

    ops_native = ops.native
    with monkeypatch.context() as m:
        m.setattr(ops, "native", Counting())
        here = fn()
    with monkeypatch.context() as m:
        m.setattr(ops, "native", _Off())
        there = fn()
    torch.cuda.synchronize()
    return here, there, taken


def _same(a, b):
    a, b = (x if isinstance(x, (tuple, list)) else (x,) for x in (a, b))
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert x.shape == y.shape and x.dtype == y.dtype and x.stride() == y.stride() and x.requires_grad == y.requires_grad
        assert torch.equal(x, y)


def _matrix(rows, cols, seed, dtype, form, dev):
    """A (rows, cols) matrix: dense, with padded rows, or starting off a 16-byte boundary (fp32: off any vector)."""
    pad = {"dense": 0, "padded": 16, "shifted": 16}[form]
    t = randn((rows, cols + pad), seed, std=0.1, dtype=dtype).to(dev)
    off = 0 if form != "shifted" else (1 if dtype == torch.float32 else 8)
    return t[:, off:off + cols]


@pytest.mark.parametrize("form", ["dense", "padded", "shifted"])
@pytest.mark.parametrize("rows", [1, 7, 300])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
def test_linears(dtype, rows, form, dev, monkeypatch):
    from odysseus_transformer_amd import ops
    K, N, I = 256, 384, 256
    x, w = _matrix(rows, K, 1, dtype, form, dev), _matrix(N, K, 2, dtype, form, dev)
    r, wgu = _matrix(rows, N, 3, dtype, form, dev), _matrix(2 * I, K, 4, dtype, form, dev)
    wd, gu, dy = _matrix(K, I, 5, dtype, form, dev), _matrix(rows, 2 * I, 6, dtype, form, dev), _matrix(rows, N, 7, dtype, form, dev)
    calls = {"nt": lambda: ops.gemm(ops.GEMM_NT, x, w), "nn": lambda: ops.gemm(ops.GEMM_NN, dy, w),
             "residual": lambda: ops.linear_residual(x, w, r), "swiglu": lambda: ops.linear_swiglu(x, wgu),
             "swiglu_h": lambda: ops.linear_swiglu_h(x, wgu), "dgrad": lambda: ops.linear_dgrad_swiglu(x, wd, gu)}
    if dtype == torch.float32 and form == "shifted":   # refused on either path: the SwiGLU backward wants vectors
        del calls["dgrad"]
    if dtype == torch.float32 or rows % 8 == 0:
        calls["tn"] = lambda: ops.gemm(ops.GEMM_TN, dy, x)
    if dtype == torch.bfloat16:
        table = ops.rope_table(torch.arange(rows, device=dev)[None], rows, 128)
        calls["rope"] = lambda: ops.linear_rope(x, w, table, 2, 128)
    for name, fn in calls.items():
        print(f"{name} rows={rows} {dtype} {form}", flush=True)
        here, there, taken = _both(monkeypatch, fn)
        _same(here, there)
        assert taken or name in ("swiglu_h", "dgrad"), name


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
def test_norm_and_rotation(dtype, dev, monkeypatch):
    from odysseus_transformer_amd import ops
    x, w = randn((1, 33, 512), 1, dtype=dtype).to(dev), randn((512,), 2, dtype=dtype).to(dev)
    dy, add = randn((1, 33, 512), 3, dtype=dtype).to(dev), randn((1, 33, 512), 4, dtype=dtype).to(dev)
    here, there, taken = _both(monkeypatch, lambda: ops.rmsnorm_fwd(x, w, 1e-6))
    _same(here, there)
    rstd = here[1]
    for a in (None, add):
        h, t, k = _both(monkeypatch, lambda: ops.rmsnorm_bwd(x, w, rstd, dy, a))
        _same(h, t)
        taken += k
    assert taken == ["rmsnorm_fwd", "rmsnorm_bwd", "rmsnorm_bwd"]
    # rows that are not dense: the copies are Python's
    here, there, taken = _both(monkeypatch, lambda: ops.rmsnorm_fwd(x[..., :256], w[:256], 1e-6))
    _same(here, there)
    assert not taken
    for B, pos in ((1, None), (1, torch.arange(5, 38, device=dev)[None]), (2, torch.arange(33, device=dev)[None]),
                   (2, torch.randint(0, 99, (2, 33), device=dev)), (1, torch.arange(33, device=dev, dtype=torch.int32)[None])):
        q = randn((B, 33, 6, 64), 5, dtype=dtype).to(dev)

        def rotated(inverse):
            y = q.clone()
            ops.rope_(y, 4, pos, inverse=inverse)
            return y

        for inverse in (False, True):
            here, there, taken = _both(monkeypatch, lambda: rotated(inverse))
            _same(here, there)
            assert bool(taken) == (pos is None or (pos.dtype == torch.int64 and pos.numel() == B * 33))


@pytest.mark.parametrize("packed", [False, True], ids=["dense", "packed"])
@pytest.mark.parametrize("shape", [(1, 1, 200, 4, 1, 128), (2, 65, 65, 4, 2, 128), (1, 130, 130, 2, 2, 64), (1, 300, 170, 4, 4, 64)],
                         ids=lambda s: "B%d_Lq%d_Lk%d_H%d_%d_D%d" % s)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
def test_attention(dtype, shape, packed, dev, monkeypatch):
    from odysseus_transformer_amd import ops
    B, Lq, Lk, Hq, Hkv, D = shape
    print(f"shape={shape} {dtype} packed={packed}", flush=True)
    if packed:
        L = max(Lq, Lk)
        qkv = randn((B, L, Hq + 2 * Hkv, D), 1, dtype=dtype).to(dev)
        q, k, v = qkv[:, :Lq, :Hq], qkv[:, :Lk, Hq:Hq + Hkv], qkv[:, :Lk, Hq + Hkv:]
    else:
        q, k, v = (randn((B, L, H, D), s, dtype=dtype).to(dev) for L, H, s in ((Lq, Hq, 1), (Lk, Hkv, 2), (Lk, Hkv, 3)))
    dout = randn((B, Lq, Hq, D), 4, dtype=dtype).to(dev)
    for causal in (False, True):
        here, there, taken = _both(monkeypatch, lambda: ops.attn_fwd(q, k, v, causal=causal, scale=None if causal else 0.1))
        _same(here, there)
        out, lse = here
        for keep in (None, False):
            h, t, kk = _both(monkeypatch, lambda: ops.attn_bwd(q, k, v, out, lse, dout, causal=causal, keep_ds=keep))
            _same(h, t)
            taken += kk
        assert taken == ["attn_fwd", "attn_bwd", "attn_bwd"]
        if dtype == torch.bfloat16 and D == 128 and packed and Lq == Lk:
            tables = (ops.rope_table(None, B * Lq, D, device=dev),) * 2

            def into():
                d = torch.zeros_like(qkv)
                ops.attn_bwd(q, k, v, out, lse, dout, causal=causal, dq=d[:, :, :Hq], dk=d[:, :, Hq:Hq + Hkv], dv=d[:, :, Hq + Hkv:],
                             rope_tables=tables)
                return d

            h, t, kk = _both(monkeypatch, into)
            _same(h, t)
            assert kk == ["attn_bwd"]


def test_what_it_leaves_alone(dev, monkeypatch):
    """Errors, transforms, budgets and the arena go the way they went."""
    from odysseus_transformer_amd import _lib, ops
    from odysseus_transformer_amd.utils import globals as g
    x, w = randn((16, 64), 1).to(dev), randn((64, 64), 2).to(dev)
    for bad, err in ((lambda: ops.gemm(ops.GEMM_NT, x, w[:, :32]), ValueError), (lambda: ops.gemm(7, x, w), ValueError),
                     (lambda: ops.gemm(ops.GEMM_NT, x, w.bfloat16()), TypeError), (lambda: ops.gemm(ops.GEMM_NT, x, w.cpu()), RuntimeError),
                     (lambda: ops.gemm(ops.GEMM_NT, x.double(), w.double()), TypeError),
                     (lambda: ops.gemm(ops.GEMM_NT, x.t(), w), ValueError),
                     (lambda: ops.gemm(ops.GEMM_NT, x.bfloat16()[:, :60], w.bfloat16()[:, :60]), _lib.OdysseusHipError),
                     (lambda: ops.rmsnorm_fwd(x, w[0].bfloat16()), TypeError), (lambda: ops.linear_residual(x, w, x[:, :8]), ValueError)):
        with pytest.raises(err):
            bad()

    class Sub(torch.Tensor):
        pass

    q = randn((1, 256, 2, 128), 3, dtype=torch.bfloat16).to(dev)
    for t in (q.as_subclass(Sub), q.cpu(), None, torch._neg_view(q)):
        assert ops.native.attn_fwd(t, q, q, True, 0.1) is None
    assert ops.native.attn_fwd(q, q, q, 1, 0.1) is None and ops.native.attn_fwd(q, q, q, True) is None
    side = torch.cuda.Stream()
    assert ops.native.current_stream() == ops._stream()
    with torch.cuda.stream(side):
        assert ops.native.current_stream() == ops._stream() == side.cuda_stream
    out, lse = ops.attn_fwd(q, q, q)
    ops.set_keep_ds_max_bytes(1 << 30)
    try:
        _, _, taken = _both(monkeypatch, lambda: ops.attn_bwd(q, q, q, out, lse, out))
        assert not taken
    finally:
        ops.set_keep_ds_max_bytes(None)
    g._set_global_memory_buffer(dev)
    try:
        a, b = randn((2048, 512), 4).to(dev), randn((2048, 512), 5).to(dev)
        here, there, taken = _both(monkeypatch, lambda: ops.gemm(ops.GEMM_TN, a, b))
        assert taken == ["gemm"] and torch.equal(here, there)
        assert g.get_global_memory_buffer().buffer[("gemm_workspace", torch.uint8)].numel() > 0
    finally:
        g._destroy_global_memory_buffer()


@pytest.mark.parametrize("rows", [1, 3, 4, 5])
@pytest.mark.parametrize("K", [8, 40, 512, 4096, 9000], ids=lambda k: "K%d" % k)
def test_norm_inside_a_product_of_few_rows(K, rows, dev, monkeypatch):
    """One kernel against the norm, the table and the product: the same but for the order of the norm's sum (an ulp of 1 / rms, which
    can move a rounding of the normalised row); beyond 4 rows and 64 KiB the three of them."""
    from odysseus_transformer_amd import ops
    print(f"K={K} rows={rows}", flush=True)
    x, nw = randn((rows, K), 1, dtype=torch.bfloat16).to(dev), (1 + 0.1 * randn((K,), 2)).bfloat16().to(dev)
    wq, wg = randn((640, K), 3, std=0.05, dtype=torch.bfloat16).to(dev), randn((96, K), 4, std=0.05, dtype=torch.bfloat16).to(dev)
    pos = torch.tensor([0, 70001, 5, 1 << 20, 9], device=dev)[:rows]
    for fn, one in ((lambda: ops.norm_linear_rope(x, nw, 1e-6, wq, 3, 128, pos), "norm_linear_rope"),
                    (lambda: ops.norm_linear_swiglu_h(x, nw, 1e-6, wg), "norm_linear_swiglu_h")):
        here, there, taken = _both(monkeypatch, fn)
        assert (one in taken) == (rows <= 4 and 2 * rows * (K + 8) <= 1 << 16)
        assert here.shape == there.shape and here.dtype == there.dtype
        assert (here.float() - there.float()).norm() <= 2.0 ** -9 * there.float().norm()
    n = (x.double() * (x.double().square().mean(-1, keepdim=True) + 1e-6).rsqrt() * nw.double())
    g, u = (n @ wg.double().t()).chunk(2, -1)
    ref = torch.nn.functional.silu(g) * u
    assert (ops.norm_linear_swiglu_h(x, nw, 1e-6, wg).double() - ref).norm() <= 1e-2 * ref.norm()


def test_norm_inside_a_product_with_infinities(dev):
    from odysseus_transformer_amd import ops
    x, nw = randn((3, 256), 1, dtype=torch.bfloat16), torch.ones(256, dtype=torch.bfloat16)
    x[0, 3], x[1, 7] = float("inf"), float("nan")
    w = randn((64, 256), 2, std=0.05, dtype=torch.bfloat16)
    w[5, 250] = float("inf")
    x, nw, w = x.to(dev), nw.to(dev), w.to(dev)
    here, there = ops.norm_linear_swiglu_h(x, nw, 1e-6, w), ops.linear_swiglu_h(ops.rmsnorm_fwd(x, nw)[0], w)
    assert torch.equal(here.isnan(), there.isnan()) and torch.equal(here.isinf(), there.isinf())
    ok = there.isfinite()
    assert (here[ok].float() - there[ok].float()).norm() <= 2.0 ** -9 * there[ok].float().norm()


def test_decoding_layer_folds_its_norms_and_gives_hooks_what_they_had(dev):
    import types
    from transformers import DynamicCache
    from odysseus_transformer_amd import _lib, ops
    from odysseus_transformer_amd.decoder.odysseus import OdysseusDecoderLayer
    cfg = types.SimpleNamespace(hidden_size=512, num_attention_heads=4, num_key_value_heads=2, head_dim=128, intermediate_size=1408,
                                hidden_act="silu", attention_dropout=0.0, rms_norm_eps=1e-6, rope_theta=10000.0, pretraining_tp=1)
    torch.manual_seed(0)
    layer = OdysseusDecoderLayer(cfg).bfloat16().to(dev)
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0 if p.dim() > 1 else 1.0, 0.05)
    x = randn((1, 34, 512), 1, dtype=torch.bfloat16).to(dev)

    def step(hooked):
        cache = DynamicCache()
        with torch.no_grad():
            layer(x[:, :33], position_ids=torch.arange(33, device=dev)[None], past_key_values=cache)
            seen = []
            h = layer.self_attn.register_forward_pre_hook(lambda m, a: seen.append(a[0])) if hooked else None
            _lib.profile_enable(True)
            _lib.profile_collect()
            try:
                y = layer(x[:, 33:], position_ids=torch.arange(33, 34, device=dev)[None], past_key_values=cache)
                ran = set(_lib.profile_collect())
            finally:
                _lib.profile_enable(False)
                if h is not None:
                    h.remove()
        return y, ran, seen

    y, ran, _ = step(False)
    assert {"gemm_skinny_norm_rope", "gemm_skinny_norm_swiglu"} <= ran and "rmsnorm_fwd" not in ran
    z, ran, seen = step(True)
    assert "rmsnorm_fwd" in ran and torch.equal(seen[0], ops.rmsnorm(x[:, 33:], layer.input_layernorm.weight, 1e-6))
    assert (y.float() - z.float()).norm() <= 1e-2 * z.float().norm()


def _refused(fn):
    try:
        fn()
    except Exception as e:  # noqa: BLE001  (its type is the answer)
        return type(e)
    return None


def test_what_either_path_refuses(dev, monkeypatch):
    """One definition of what an op takes: the same exception with the module and without it, for operands that no kernel may see."""
    from odysseus_transformer_amd import ops
    bf = torch.bfloat16
    x, w, r = (randn(s, n, dtype=bf).to(dev) for n, s in enumerate([(16, 64), (256, 64), (16, 256)]))
    f = randn((16, 64), 5).to(dev)
    n = torch.ones(64, dtype=bf, device=dev)
    rstd = torch.ones(16, device=dev)
    table = ops.rope_table(torch.arange(16, device=dev), 16, 128)
    q, k = randn((2, 8, 4, 128), 6, dtype=bf).to(dev), randn((2, 8, 2, 128), 7, dtype=bf).to(dev)
    out, lse = ops.attn_fwd(q, k, k)
    y = randn((2, 8, 4, 64), 8, dtype=bf).to(dev)
    one = randn((1, 8, 4, 64), 9, dtype=bf).to(dev)
    pos, inv = torch.arange(8, device=dev), torch.ones(32, device=dev)
    calls = {
        "norm: weight of another size": lambda: ops.rmsnorm_fwd(x, n[:32]),
        "norm: weight of another type": lambda: ops.rmsnorm_fwd(x, n.float()),
        "norm: strided weight": lambda: ops.rmsnorm_fwd(x[:, :32].contiguous(), n[::2]),
        "norm: weight of two dimensions": lambda: ops.rmsnorm_fwd(x, n[None]),
        "norm: rows of another count": lambda: ops.rmsnorm_bwd(x, n, rstd[:8], x),
        "norm: rstd of another type": lambda: ops.rmsnorm_bwd(x, n, rstd.double(), x),
        "norm: dy of another shape": lambda: ops.rmsnorm_bwd(x, n, rstd, x[:8]),
        "norm: dx_add of another type": lambda: ops.rmsnorm_bwd(x, n, rstd, x, f),
        "gemm: inner extents": lambda: ops.gemm(ops.GEMM_NT, x, r),
        "gemm: three dimensions": lambda: ops.gemm(ops.GEMM_NT, x[None], w),
        "gemm: column stride": lambda: ops.gemm(ops.GEMM_NN, x, w.t()),
        "gemm: op": lambda: ops.gemm(3, x, w),
        "gemm: odd extent": lambda: ops.gemm(ops.GEMM_NT, x[:, :60], w[:, :60]),
        "gemm: off a 16-byte boundary": lambda: ops.gemm(ops.GEMM_NT, x[:, 1:57], w[:, 1:57]),
        "gemm: rows closer than their length": lambda: ops.gemm(ops.GEMM_NT, x.as_strided((4, 64), (8, 1)), w),
        "residual: shape": lambda: ops.linear_residual(x, w, r[:8]),
        "residual: type": lambda: ops.linear_residual(x, w, r.float()),
        "rope: table's rows": lambda: ops.linear_rope(x, w, table[:8], 1, 128),
        "rope: table's type": lambda: ops.linear_rope(x, w, table.float(), 1, 128),
        "rope: heads": lambda: ops.linear_rope(x, w, table, 3, 128),
        "rope: head_dim": lambda: ops.linear_rope(x, w, table, 1, 64),
        "rope: fp32": lambda: ops.linear_rope(f, w.float(), table, 1, 128),
        "swiglu: odd rows of the weight": lambda: ops.linear_swiglu(x, w[:255]),
        "swiglu: inner extents": lambda: ops.linear_swiglu(x, r),
        "dgrad: gate_up's shape": lambda: ops.linear_dgrad_swiglu(x, w.t().contiguous(), r),
        "attention: kv shapes": lambda: ops.attn_fwd(q, k, k[:, :7]),
        "attention: type": lambda: ops.attn_fwd(q, k, k.float()),
        "attention: heads": lambda: ops.attn_fwd(q, q[:, :, :3], q[:, :, :3]),
        "attention: head_dim": lambda: ops.attn_fwd(q[..., :32], k[..., :32], k[..., :32]),
        "attention: stride of head_dim": lambda: ops.attn_fwd(q.transpose(2, 3).contiguous().transpose(2, 3), k, k),
        "attention: rows off 16 bytes": lambda: ops.attn_fwd(q[..., 4:68], k[..., :64], k[..., :64]),
        "attention: scale": lambda: ops.attn_fwd(q, k, k, scale=-1.0),
        "attention: three dimensions": lambda: ops.attn_fwd(q[0], k[0], k[0]),
        "backward: lse's shape": lambda: ops.attn_bwd(q, k, k, out, lse[:1], out),
        "backward: lse's type": lambda: ops.attn_bwd(q, k, k, out, lse.double(), out),
        "backward: dout": lambda: ops.attn_bwd(q, k, k, out, lse, out[:, :4]),
        "backward: dk": lambda: ops.attn_bwd(q, k, k, out, lse, out, dk=torch.empty_like(q)),
        "backward: tables": lambda: ops.attn_bwd(q, k, k, out, lse, out, rope_tables=(table[:8], table)),
        "rotation: positions of three dimensions": lambda: ops.rope_(one, 2, pos[None, None]),
        "rotation: positions of another batch": lambda: ops.rope_(y, 2, pos.repeat(3, 1)),
        "rotation: positions of no dimension": lambda: ops.rope_(one, 2, pos[0]),
        "rotation: positions of another type": lambda: ops.rope_(one, 2, pos.float()[None]),
        "rotation: all positions in a row": lambda: ops.rope_(y, 2, torch.arange(16, device=dev)),
        "rotation: frequencies of two dimensions": lambda: ops.rope_(one, 2, pos[None], inv_freq=inv[None]),
        "rotation: frequencies of another count": lambda: ops.rope_(one, 2, pos[None], inv_freq=inv[:16]),
        "rotation: heads": lambda: ops.rope_(one, 5, pos[None]),
        "rotation: odd head_dim": lambda: ops.rope_(one[..., :63], 2, pos[None]),
        "rotation: three dimensions": lambda: ops.rope_(one[0], 2, pos[None]),
        "table: positions": lambda: ops.rope_table(pos, 12, 128, inv_freq=torch.ones(64, device=dev)),
        "table: frequencies": lambda: ops.rope_table(pos, 8, 128, inv_freq=inv),
        "folded norm: positions": lambda: ops.norm_linear_rope(x[:3], n, 1e-6, w, 1, 128, pos[:2]),
        "folded norm: weight": lambda: ops.norm_linear_swiglu_h(x[:3], n.float(), 1e-6, w),
    }
    for name, fn in calls.items():
        here = _refused(fn)
        with monkeypatch.context() as m:
            m.setattr(ops, "native", _Off())
            there = _refused(fn)
        assert here is not None and here == there, (name, here, there)
    for p in (pos, pos[None]):   # one sequence, either way to write it
        a, b = one.clone(), one.clone()
        ops.rope_(a, 4, p)
        ops.rope_(b, 4, None)
        assert torch.equal(a, b)


def test_threads_and_autocast(dev):
    """Calls of several threads, each on a stream of its own, and calls under autocast, which the ops themselves do not look at."""
    import threading
    from odysseus_transformer_amd import ops
    q, k, v = (randn((1, 70, h, 128), h, dtype=torch.bfloat16).to(dev) for h in (4, 2, 2))
    want = (*ops.attn_fwd(q, k, v),)
    want += (*ops.attn_bwd(q, k, v, *want, want[0]),)
    torch.cuda.synchronize()
    wrong = []

    def work():
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(20):
                got = (*ops.attn_fwd(q, k, v),)
                got += (*ops.attn_bwd(q, k, v, *got, got[0]),)
                stream.synchronize()
                wrong.extend(1 for a, b in zip(got, want) if not torch.equal(a, b))

    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    x, w = randn((16, 64), 1).to(dev), randn((32, 64), 2).to(dev)
    y = ops.gemm(ops.GEMM_NT, x, w)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert torch.equal(ops.gemm(ops.GEMM_NT, x, w), y) and y.dtype == torch.float32


def test_arena_without_room_for_all_of_the_scratch(dev, monkeypatch):
    """The backward of head_dim 64 goes on with the least workspace, as without the module; the products, which have no other way, raise."""
    from odysseus_transformer_amd import _lib, ops
    from odysseus_transformer_amd.utils import globals as g
    q, k, v, do = (randn((1, 300, h, 64), n, dtype=torch.bfloat16).to(dev) for n, h in enumerate((8, 2, 2, 8)))
    out, lse = ops.attn_fwd(q, k, v)
    want = ops.attn_bwd(q, k, v, out, lse, do, keep_ds=False)
    sizes = 1, 300, 300, 8, 2, 64, _lib.ODY_BF16
    least, full = _lib.load().ody_attn_bwd_workspace_least_bytes(*sizes), _lib.load().ody_attn_bwd_workspace_bytes(*sizes)
    assert least < full

    class Small(g.GlobalMemoryBuffer):
        refused = 0

        def get_tensor(self, shape, dtype, name):
            if shape[0] > least:
                self.refused += 1
                raise torch.OutOfMemoryError("no room for that")
            return super().get_tensor(shape, dtype, name)

    monkeypatch.setattr(g._Arena, "instance", Small(dev))
    here, there, _ = _both(monkeypatch, lambda: ops.attn_bwd(q, k, v, out, lse, do, keep_ds=False))
    assert g._Arena.instance.refused >= 2
    _same(here, there)
    for a, b in zip(here, want):
        assert (a.float() - b.float()).norm() <= 1e-2 * b.float().norm()
    x, w = randn((512, 64 * 512), 4).to(dev), randn((512, 64 * 512), 5).to(dev)
    assert _lib.load().ody_gemm_workspace_bytes(ops.GEMM_NT, 512, 512, 64 * 512, _lib.ODY_F32) > least
    with pytest.raises(torch.OutOfMemoryError):
        ops.gemm(ops.GEMM_NT, x, w)


def _flash_inputs(dev, dtype=torch.bfloat16, L=197, hq=8, hkv=2, D=128, needs=(True, True, True)):
    big = randn((2, L, hq + 2 * hkv, D), 71, dtype=dtype).to(dev)
    q, k, v = (t.detach() for t in big.split([hq, hkv, hkv], dim=2))   # heads of one packed buffer: rows far apart
    return [t.requires_grad_(n) for t, n in zip((q, k, v), needs)]


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.bfloat16, 64), (torch.float32, 64)], ids=["bf16_128", "bf16_64", "f32_64"])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("needs", [(True, True, True), (False, True, False), (True, False, False)], ids=lambda n: "".join("nq"[x] for x in n))
def test_attention_routine_as_a_node_of_its_own(dtype, D, causal, needs, dev, monkeypatch):
    """The routine through the node in C++ and through FlashAttnFunc: outputs, gradients and what requires one, bit for bit; a gradient that arrives
    with a strided head dimension, expanded, or not at all; a graph that is kept and walked twice."""
    from odysseus_transformer_amd import ops

    def run():
        q, k, v = _flash_inputs(dev, dtype, D=D, needs=needs)
        out, lse = ops.flash_attn_func(q, k, v, softmax_scale=0.1, causal=causal, return_lse=True)
        assert out.requires_grad and not lse.requires_grad and out.grad_fn is not None
        got = [out.detach(), lse]
        inputs = [t for t, n in zip((q, k, v), needs) if n]
        for dout in (randn(out.shape, 72, dtype=dtype).to(dev), randn((2, D, 197, 8), 73, dtype=dtype).to(dev).permute(0, 2, 3, 1),
                     torch.ones((), dtype=dtype, device=dev).expand(out.shape)):
            got += torch.autograd.grad(out, inputs, dout, retain_graph=True)
        return got

    here, there, taken = _both(monkeypatch, run)
    assert taken[0] == "flash" and "attn_bwd" not in taken
    _same(here, there)


def test_attention_node_keeps_what_autograd_promises(dev, monkeypatch):
    """Hooks on saved tensors, modification in place, a graph walked twice without being kept, a budget of kept dS set between forward and backward,
    transforms and forward mode: as through FlashAttnFunc."""
    from odysseus_transformer_amd import _lib, ops
    q, k, v = _flash_inputs(dev)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t.cpu())[1], lambda t: t.to(dev)):
        out = ops.flash_attn_func(q, k, v, causal=True)
    assert "FlashNode" in out.grad_fn.name() and len(packed) == 5
    dout = randn(out.shape, 74, dtype=torch.bfloat16).to(dev)
    offloaded = torch.autograd.grad(out, (q, k, v), dout)
    plain = torch.autograd.grad(ops.flash_attn_func(q, k, v, causal=True), (q, k, v), dout)
    _same(offloaded, plain)

    out = ops.flash_attn_func(q, k, v, causal=True)
    torch.autograd.grad(out, q, dout)
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out, q, dout)
    out = ops.flash_attn_func(q, k, v, causal=True)
    with torch.no_grad():
        v.mul_(1.0)
    with pytest.raises(RuntimeError, match="inplace"):
        torch.autograd.grad(out, q, dout)

    q, k, v = (t.requires_grad_(True) for t in randn((3, 1, 2048, 4, 128), 75, dtype=torch.bfloat16).to(dev))
    dout = randn((1, 2048, 4, 128), 76, dtype=torch.bfloat16).to(dev)
    lib = _lib.load()

    def names(fn):
        import ctypes
        lib.ody_profile_enable(1)
        fn()
        torch.cuda.synchronize()
        buf = ctypes.create_string_buffer(1 << 16)
        lib.ody_profile_collect(buf, 1 << 16)
        lib.ody_profile_enable(0)
        return buf.value.decode()

    out = ops.flash_attn_func(q, k, v, causal=True)
    ops.set_keep_ds_max_bytes(1 << 30)
    try:
        assert "attn_bwd_dq_kept" in names(lambda: torch.autograd.grad(out, (q, k, v), dout))
    finally:
        ops.set_keep_ds_max_bytes(None)
    fails = []
    for call in (lambda: torch.func.vmap(lambda t: ops.flash_attn_func(t, t, t))(q.detach()[None]),
                 lambda: torch.func.jvp(lambda t: ops.flash_attn_func(t, k, v), (q,), (q.detach(),))):
        for native in (ops.native, _Off()):
            with monkeypatch.context() as m:
                m.setattr(ops, "native", native)
                with pytest.raises(Exception) as e:
                    call()
            fails.append(type(e.value))
    assert fails[0] is fails[1] and fails[2] is fails[3]


def test_an_error_inside_the_attention_node_reaches_the_caller(dev, monkeypatch):
    """The node calls attn_bwd of ops.py where its plain form is not the one to be taken; what that raises comes out of backward()."""
    from odysseus_transformer_amd import ops
    q, k, v = _flash_inputs(dev)
    out = ops.flash_attn_func(q, k, v)
    with monkeypatch.context() as m:
        m.setattr(ops, "_never_keeps_ds", lambda: False)
        m.setattr(ops, "attn_bwd", lambda *args: (_ for _ in ()).throw(ValueError("from inside")))
        with pytest.raises(ValueError, match="from inside"):
            out.backward(torch.ones_like(out))


class _NoGradient(torch.autograd.Function):
    """Passes its input on and no gradient back."""

    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, grad):
        return None


@pytest.mark.parametrize("needs", [(True, True, True), (False, True, False)], ids=lambda n: "".join("nq"[x] for x in n))
def test_attention_node_without_a_gradient(needs, dev, monkeypatch):
    """No gradient arrives at the node at all: those of its inputs are zeros, as from FlashAttnFunc."""
    from odysseus_transformer_amd import ops

    def run():
        q, k, v = _flash_inputs(dev, needs=needs)
        out = ops.flash_attn_func(q, k, v, causal=True)
        return torch.autograd.grad(_NoGradient.apply(out).sum(), [t for t, n in zip((q, k, v), needs) if n])

    here, there, taken = _both(monkeypatch, run)
    assert taken[0] == "flash" and all(not g.any() for g in here)
    _same(here, there)


@pytest.mark.parametrize("reentrant", [False, True])
def test_attention_node_under_checkpointing(reentrant, dev, monkeypatch):
    """The forward is formed again in backward(); without reentry it is left by an exception from a hook on saved tensors as soon as all are there."""
    from odysseus_transformer_amd import ops
    from torch.utils.checkpoint import checkpoint

    def run():
        q, k, v = _flash_inputs(dev)
        out = checkpoint(lambda *qkv: ops.flash_attn_func(*qkv, causal=True), q, k, v, use_reentrant=reentrant)
        out.backward(randn(out.shape, 77, dtype=torch.bfloat16).to(dev))
        return [out.detach(), q.grad, k.grad, v.grad]

    here, there, taken = _both(monkeypatch, run)
    assert "flash" in taken
    _same(here, there)
