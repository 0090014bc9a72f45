"""GPU parity: the three products of a linear layer through ody_gemm vs. the CPU oracle."""
import pytest
import torch

from conftest import TOL_BF16, TOL_F32, device_kernels, randn, rel_err
import odysseus_oracle as oracle

pytestmark = pytest.mark.gpu

SHAPES = [
    # M, N, K
    (64, 64, 64),
    (256, 256, 256),
    (128, 128, 64),        # interior tiles, a single K slab
    (256, 384, 192),       # interior tiles, odd number of K slabs
    (300, 136, 72),        # ragged in every direction (multiples of 8)
    (2048, 1536, 512),     # the fp32 configuration's QKV projection
    (520, 2752, 512),      # gate_up of the fp32 configuration, ragged M
    (1024, 768, 4096),
    (4096, 4096, 512),     # enough tiles for the 256 x 256 kernel
    (1000, 1096, 256),     # whole tiles plus a ragged strip on the right and at the bottom
    (4104, 3848, 128),     # the same with 256 x 256 tiles
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "M%d_N%d_K%d" % s)
def test_linear_fwd_dgrad_wgrad(shape, dtype, dev):
    from odysseus_transformer_amd import ops
    M, N, K = shape
    print(f"shape={shape} dtype={dtype}", flush=True)
    tol = TOL_BF16 if dtype == torch.bfloat16 else TOL_F32
    x = randn((M, K), 1, dtype=dtype)
    w = randn((N, K), 2, std=0.02, dtype=dtype)
    dy = randn((M, N), 3, dtype=dtype)
    y_ref = oracle.linear_fwd(x.float(), w.float())
    dx_ref, dw_ref, _ = oracle.linear_bwd(x.float(), w.float(), dy.float())
    xg, wg, dyg = x.to(dev), w.to(dev), dy.to(dev)
    y = ops.gemm(ops.GEMM_NT, xg, wg)              # X W^T
    dx = ops.gemm(ops.GEMM_NN, dyg, wg)            # dY W
    dw = ops.gemm(ops.GEMM_TN, dyg, xg)            # dY^T X
    torch.cuda.synchronize()
    assert rel_err(y, y_ref) <= tol, "fwd"
    assert rel_err(dx, dx_ref) <= tol, "dgrad"
    assert rel_err(dw, dw_ref) <= tol, "wgrad"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
def test_bias_accumulate_and_strides(dtype, dev):
    from odysseus_transformer_amd import ops
    tol = TOL_BF16 if dtype == torch.bfloat16 else TOL_F32
    M, N, K = 200, 264, 136
    x = randn((M, K + 24), 4, dtype=dtype)[:, 8:8 + K]          # row stride > K, offset start
    w = randn((N, K), 5, std=0.05, dtype=dtype)
    b = randn((N,), 6, dtype=dtype)
    c0 = randn((M, N), 7, dtype=dtype)
    ref = oracle.linear_fwd(x.float(), w.float(), b.float()) + c0.float()
    xg = randn((M, K + 24), 4, dtype=dtype).to(dev)[:, 8:8 + K]
    out = c0.to(dev).clone()
    ops.gemm(ops.GEMM_NT, xg, w.to(dev), bias=b.to(dev), out=out, accumulate=True)
    assert rel_err(out, ref) <= tol


@pytest.mark.parametrize("op", ["nt", "nn", "tn"])
def test_bias_accumulate_and_strides_on_interior_tiles(op, dev):
    """The kernel for full tiles: padded leading dimensions, bias and accumulation into C."""
    from odysseus_transformer_amd import ops
    dt = torch.bfloat16
    M, N, K = 512, 256, 320
    shape_a = {"nt": (M, K), "nn": (M, K), "tn": (K, M)}[op]
    shape_b = {"nt": (N, K), "nn": (K, N), "tn": (K, N)}[op]
    a = randn((shape_a[0], shape_a[1] + 40), 11, dtype=dt)[:, 16:16 + shape_a[1]]
    b = randn((shape_b[0], shape_b[1] + 8), 12, std=0.05, dtype=dt)[:, :shape_b[1]]
    bias = randn((N,), 13, dtype=dt)
    c0 = randn((M, N + 16), 14, dtype=dt)[:, 8:8 + N]
    af = a.float().t() if op == "tn" else a.float()
    bf = b.float().t() if op == "nt" else b.float()
    ref = af @ bf + bias.float() + c0.float()
    ag = randn((shape_a[0], shape_a[1] + 40), 11, dtype=dt).to(dev)[:, 16:16 + shape_a[1]]
    bg = randn((shape_b[0], shape_b[1] + 8), 12, std=0.05, dtype=dt).to(dev)[:, :shape_b[1]]
    out = randn((M, N + 16), 14, dtype=dt).to(dev)[:, 8:8 + N]
    code = {"nt": ops.GEMM_NT, "nn": ops.GEMM_NN, "tn": ops.GEMM_TN}[op]
    ops.gemm(code, ag, bg, bias=bias.to(dev), out=out, accumulate=True)
    assert rel_err(out, ref) <= TOL_BF16


@pytest.mark.parametrize("shape", [(77, 53, 41), (130, 66, 33), (5, 3, 1), (259, 131, 100), (2901, 2903, 37)],
                         ids=lambda s: "M%d_N%d_K%d" % s)
def test_fp32_any_shape_and_alignment(shape, dev):
    """fp32 takes extents that are not multiples of 4 and views that start on odd elements."""
    from odysseus_transformer_amd import ops
    M, N, K = shape
    print(f"shape={shape}", flush=True)
    x = randn((M, K + 3), 21)[:, 1:1 + K]
    w = randn((N, K), 22, std=0.05)
    dy = randn((M, N + 1), 23)[:, 1:]
    b = randn((N,), 24)
    c0 = randn((M, N), 25)
    xg, wg, dyg = randn((M, K + 3), 21).to(dev)[:, 1:1 + K], w.to(dev), randn((M, N + 1), 23).to(dev)[:, 1:]
    out = c0.to(dev).clone()
    ops.gemm(ops.GEMM_NT, xg, wg, bias=b.to(dev), out=out, accumulate=True)
    assert rel_err(out, x @ w.T + b + c0) <= TOL_F32, "fwd"
    assert rel_err(ops.gemm(ops.GEMM_NN, dyg, wg), dy @ w) <= TOL_F32, "dgrad"
    assert rel_err(ops.gemm(ops.GEMM_TN, dyg, xg), dy.T @ x) <= TOL_F32, "wgrad"


def test_linearity_at_full_size(dev):
    """Size-independent property at a rank-shard shape: X (W1 + W2)^T == X W1^T + X W2^T
    up to bf16 rounding, and the wgrad of a row-permuted batch is unchanged."""
    from odysseus_transformer_amd import ops
    M, N, K = 8192, 1536, 4096
    x = randn((M, K), 11, dtype=torch.bfloat16).to(dev)
    w1 = randn((N, K), 12, std=0.02, dtype=torch.bfloat16).to(dev)
    w2 = randn((N, K), 13, std=0.02, dtype=torch.bfloat16).to(dev)
    y12 = ops.gemm(ops.GEMM_NT, x, (w1.float() + w2.float()).bfloat16())
    y1, y2 = ops.gemm(ops.GEMM_NT, x, w1), ops.gemm(ops.GEMM_NT, x, w2)
    assert rel_err(y12, y1.float() + y2.float()) <= TOL_BF16
    dy = randn((M, N), 14, dtype=torch.bfloat16).to(dev)
    perm = torch.randperm(M, generator=torch.Generator().manual_seed(0)).to(dev)
    dw = ops.gemm(ops.GEMM_TN, dy, x)
    dwp = ops.gemm(ops.GEMM_TN, dy[perm].contiguous(), x[perm].contiguous())
    assert rel_err(dwp, dw.float()) <= 5e-3
    # spot check rows against fp64
    rows = torch.tensor([0, 1, 777, M - 1], device=dev)
    ref = x[rows].double() @ w1.double().T
    assert rel_err(y1[rows], ref) <= TOL_BF16


def test_gemm_errors(dev):
    from odysseus_transformer_amd import ops
    from odysseus_transformer_amd._lib import OdysseusHipError
    a = torch.zeros(16, 20, dtype=torch.bfloat16, device=dev)   # K = 20 is not a multiple of 8
    with pytest.raises(OdysseusHipError):
        ops.gemm(ops.GEMM_NT, a, a)
    with pytest.raises(ValueError):
        ops.gemm(ops.GEMM_NT, a, torch.zeros(16, 24, dtype=torch.bfloat16, device=dev))


@pytest.mark.parametrize("M", [1, 15, 16, 17, 32, 33, 64, 65])
@pytest.mark.parametrize("N,K", [(264, 136), (128, 4096), (512, 2056), (16512, 64)], ids=lambda v: str(v))
def test_products_with_few_rows(M, N, K, dev):
    """The kernel for few rows of A: edges of its 16-row groups on both sides, K that is no multiple of 32 or of the
    wavefronts' shares, bias, accumulation and padded leading dimensions."""
    from odysseus_transformer_amd import ops
    print(f"few rows M={M} N={N} K={K}", flush=True)
    x = randn((M, K + 8), 31, dtype=torch.bfloat16)[:, :K]
    w = randn((N, K), 32, std=0.05, dtype=torch.bfloat16)
    bias = randn((N,), 33, dtype=torch.bfloat16)
    ref = x.float() @ w.float().t()
    xd, wd = x.to(dev), w.to(dev)
    assert rel_err(ops.gemm(ops.GEMM_NT, xd, wd), ref) <= TOL_BF16, "y"
    out = torch.ones((M, N), dtype=torch.bfloat16, device=dev)
    ops.gemm(ops.GEMM_NT, xd, wd, bias=bias.to(dev), out=out, accumulate=True)
    assert rel_err(out, ref + bias.float() + 1.0) <= TOL_BF16, "y + bias + C"


@pytest.mark.parametrize("op", ["nt", "nn", "tn"])
@pytest.mark.parametrize("M,N,K", [(72, 8, 8), (128, 264, 72), (136, 248, 64), (248, 256, 1000), (264, 520, 200), (1000, 1096, 2056),
                                   (2056, 4104, 136), (4104, 5128, 72), (4360, 4104, 136)], ids=lambda v: str(v))
def test_tile_edges(op, M, N, K, dev):
    """The tile kernel around its edges in all three extents: rows and columns on both sides of 64, 128 and 256, a partial last
    slab of K, K cut into ranges, a last round in half tiles (289 and more tiles of 256 x 256), padded pitches whose padding is
    not a number, bias and accumulation."""
    from odysseus_transformer_amd import ops
    print(f"tile edges {op} M={M} N={N} K={K}", flush=True)
    nan = float("nan")

    def padded(r, c, seed, std=1.0):
        t = torch.full((r, c + 8), nan, dtype=torch.bfloat16, device=dev)
        t[:, :c] = randn((r, c), seed, std=std, dtype=torch.bfloat16).to(dev)
        return t[:, :c]
    a = padded(*((K, M) if op == "tn" else (M, K)), 41)
    b = padded(*((N, K) if op == "nt" else (K, N)), 42, 0.05)
    code = {"nt": ops.GEMM_NT, "nn": ops.GEMM_NN, "tn": ops.GEMM_TN}[op]
    ref = (a.float().t() if op == "tn" else a.float()) @ (b.float().t() if op == "nt" else b.float())
    assert rel_err(ops.gemm(code, a, b), ref) <= TOL_BF16
    bias = randn((N,), 43, dtype=torch.bfloat16).to(dev)
    for pad in (8, 4):                                  # rows of C with and without 16-byte alignment
        out = torch.ones((M, N + pad), dtype=torch.bfloat16, device=dev)
        ops.gemm(code, a, b, bias=bias, out=out[:, :N], accumulate=True)
        assert rel_err(out[:, :N], ref + bias.float() + 1.0) <= TOL_BF16
        assert bool((out[:, N:] == 1).all()), "columns beyond N were written"


def test_row_pitch_beyond_the_tile_kernels_offsets(dev):
    """A pitch of more than 2^22 elements takes the kernel with 64-bit offsets."""
    from odysseus_transformer_amd import ops
    M, N, K, pitch = 72, 136, 64, (1 << 22) + 8
    flat = torch.zeros(M * pitch, dtype=torch.bfloat16, device=dev)
    a = flat.as_strided((M, K), (pitch, 1))
    a.copy_(randn((M, K), 44, dtype=torch.bfloat16))
    w = randn((N, K), 45, std=0.05, dtype=torch.bfloat16).to(dev)
    assert rel_err(ops.gemm(ops.GEMM_NT, a, w), a.float() @ w.float().t()) <= TOL_BF16


@pytest.mark.parametrize("op", ["nt", "nn", "tn"])
@pytest.mark.parametrize("M,N,K", [(64, 64, 4096), (68, 132, 1028), (129, 64, 640), (1111, 132, 516), (132, 1028, 2049)], ids=lambda v: str(v))
def test_fp32_ranges_of_k(op, M, N, K, dev):
    """fp32 products whose K is cut into ranges, ragged rows beside vector loads, and extents that vector loads cannot take."""
    from odysseus_transformer_amd import ops
    a = randn((K, M) if op == "tn" else (M, K), 46).to(dev)
    b = randn((N, K) if op == "nt" else (K, N), 47).to(dev)
    code = {"nt": ops.GEMM_NT, "nn": ops.GEMM_NN, "tn": ops.GEMM_TN}[op]
    ref = ((a.double().t() if op == "tn" else a.double()) @ (b.double().t() if op == "nt" else b.double()))
    bias, out = randn((N,), 48).to(dev), torch.ones((M, N), device=dev)
    assert rel_err(ops.gemm(code, a, b), ref) <= 1e-5
    assert rel_err(ops.gemm(code, a, b, bias=bias, out=out, accumulate=True), ref + bias.double() + 1.0) <= 1e-5


@pytest.mark.parametrize("op", ["nt", "nn", "tn"])
@pytest.mark.parametrize("K", [4, 32, 36, 64, 68, 96, 100, 132, 160])
@pytest.mark.parametrize("M,N", [(64, 64), (68, 132), (2052, 4100)], ids=lambda v: str(v))
def test_fp32_slab_pipeline(op, M, N, K, dev):
    """One to five slabs of 32 k, whole and ragged, through 64 and 128 wide tiles, inside buffers whose other elements are NaN: each
    element within the bound of a sum of K products in fp32, (K + 2) 2^-24 sum |a| |b|."""
    from odysseus_transformer_amd import ops
    print(f"op={op} M={M} N={N} K={K}", flush=True)
    a, b = randn((M, K), 11), randn((N, K), 12)

    def inside(t):
        big = torch.full((t.shape[0] + 8, t.shape[1] + 8), float("nan"), device=dev)
        big[4:4 + t.shape[0], 4:4 + t.shape[1]] = t.to(dev)
        return big[4:4 + t.shape[0], 4:4 + t.shape[1]]

    ag = inside(a.t() if op == "tn" else a)
    bg = inside(b if op == "nt" else b.t())
    got = ops.gemm({"nt": ops.GEMM_NT, "nn": ops.GEMM_NN, "tn": ops.GEMM_TN}[op], ag, bg)
    ad, bd = a.double().to(dev), b.double().to(dev)
    want, bound = ad @ bd.t(), (K + 2) * 2.0 ** -24 * (ad.abs() @ bd.abs().t())
    assert ((got.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("M", [4100, 4104, 4216, 4360, 8200], ids=lambda m: "M%d" % m)
@pytest.mark.parametrize("what", ["nt", "nn", "tn", "rope", "swiglu", "residual"])
def test_tiles_of_a_nearly_empty_last_round(what, M, dev):
    """272 to 528 tiles of 256 x 256 on 256 compute units: the last ones run in halves or quarters, some of them past the edge.  Same
    bits as a call whose tiles fill its one round, and right beyond it."""
    from odysseus_transformer_amd import ops
    dt, K, N = torch.bfloat16, 192, 3968
    print(f"what={what} M={M}", flush=True)
    M = (M + 7) // 8 * 8 if what == "tn" else M
    x, w = randn((M, K), 1, dtype=dt).to(dev), randn((N, K), 2, std=0.05, dtype=dt).to(dev)
    r = randn((M, N), 3, dtype=dt).to(dev)
    table = ops.rope_table(torch.arange(M, device=dev), M, 128)

    def run(x, r, table):
        if what == "nt":
            return ops.gemm(ops.GEMM_NT, x, w)
        if what == "nn":
            return ops.gemm(ops.GEMM_NN, x, w.t().contiguous())
        if what == "tn":
            return ops.gemm(ops.GEMM_TN, x.t().contiguous(), w.t().contiguous())
        if what == "rope":
            return ops.linear_rope(x, w, table, 20, 128)
        if what == "swiglu":
            return ops.linear_swiglu(x, w)[1]
        return ops.linear_residual(x, w, r)

    y = run(x, r, table)
    assert torch.equal(y[:4096], run(x[:4096], r[:4096], table[:4096]))
    ref = x.float() @ w.float().t()
    if what == "rope":   # (cos, sin) of a frequency side by side in the table, columns j and j + 64 of a head in the product
        cos, sin = table.float().view(M, 1, 64, 2).unbind(-1)
        a, b = ref[:, :20 * 128].reshape(M, 20, 2, 64).unbind(2)
        ref[:, :20 * 128] = torch.stack([a * cos - b * sin, b * cos + a * sin], 2).reshape(M, -1)
    if what == "swiglu":
        g, u = ref.chunk(2, -1)
        ref = torch.nn.functional.silu(g.to(dt).float()) * u.to(dt).float()
    if what == "residual":
        ref = ref + r.float()
    assert rel_err(y, ref.cpu()) <= TOL_BF16
    assert rel_err(y[4096:], ref[4096:].cpu()) <= TOL_BF16


@pytest.mark.parametrize("op", ["nt", "nn", "tn"])
@pytest.mark.parametrize("M,N,K", [(4096, 8192, 64), (4096, 8192, 72), (4096, 8192, 128), (4104, 8200, 136), (4224, 8200, 192), (6152, 8184, 200),
                                   (5384, 12296, 1000), (12296, 4872, 264)], ids=lambda v: str(v))
def test_several_tiles_a_block(op, M, N, K, dev):
    """512 and more tiles of 256 x 256: odd and even numbers of slabs from one on, a partial last one, rounds that are full, short, and left to
    halves and quarters of tiles.  Same bits as with a bias of zero, where every block has one tile; rows of C some way apart."""
    from odysseus_transformer_amd import ops
    print(f"op={op} M={M} N={N} K={K}", flush=True)
    dt = torch.bfloat16
    a = randn((K, M) if op == "tn" else (M, K), 1, dtype=dt).to(dev)
    b = randn((N, K) if op == "nt" else (K, N), 2, std=0.05, dtype=dt).to(dev)
    code = {"nt": ops.GEMM_NT, "nn": ops.GEMM_NN, "tn": ops.GEMM_TN}[op]
    y = ops.gemm(code, a, b)
    assert torch.equal(y, ops.gemm(code, a, b, bias=torch.zeros(N, dtype=dt, device=dev)))
    ref = (a.float().t() if op == "tn" else a.float()) @ (b.float().t() if op == "nt" else b.float())
    assert rel_err(y, ref) <= TOL_BF16
    out = torch.ones((M, N + 8), dtype=dt, device=dev)
    ops.gemm(code, a, b, out=out[:, :N])
    assert torch.equal(out[:, :N], y) and bool((out[:, N:] == 1).all())


@pytest.mark.parametrize("M,K", [(8192, 136), (8456, 192), (12288, 200), (12296, 1000)], ids=lambda v: str(v))
@pytest.mark.parametrize("what", ["rope", "swiglu", "swiglu_h", "dgrad_swiglu"])
def test_several_tiles_a_block_with_an_epilogue(what, M, K, dev):
    """512 and more tiles of 256 x 256 with an epilogue, several of them a block for the forward of SwiGLU: same bits as calls on 4096 rows at
    a time, whose blocks have one tile."""
    from odysseus_transformer_amd import ops
    print(f"what={what} M={M} K={K}", flush=True)
    dt, N = torch.bfloat16, 4096
    x, w = randn((M, K), 1, dtype=dt).to(dev), randn((N, K), 2, std=0.05, dtype=dt).to(dev)
    if what == "rope":
        table = ops.rope_table(torch.arange(M, device=dev), M, 128)
        run = lambda r: [ops.linear_rope(x[r], w, table[r], 20, 128)]
    elif what == "swiglu":
        run = lambda r: ops.linear_swiglu(x[r], w)
    elif what == "swiglu_h":
        run = lambda r: [ops.linear_swiglu_h(x[r], w)]
    else:
        gate_up, down = randn((M, 2 * N), 3, dtype=dt).to(dev), w.t().contiguous()
        run = lambda r: [ops.linear_dgrad_swiglu(x[r], down, gate_up[r])]
    whole = run(slice(0, M))
    for m in range(0, M - 4095, 4096):
        for got, want in zip(whole, run(slice(m, m + 4096))):
            assert torch.equal(got[m:m + 4096], want)
    for got, want in zip(whole, run(slice(M - 264, M))):   # K in ranges there, perhaps
        assert rel_err(got[M - 264:], want.float()) <= TOL_BF16


@pytest.mark.parametrize("op", ["nn", "tn"])
@pytest.mark.parametrize("M,N,K", [(72, 136, 8), (256, 256, 56), (264, 512, 72), (136, 128, 120), (1000, 264, 1544), (264, 1032, 4104), (8200, 4616, 136),
                                   (5640, 6152, 4168)], ids=lambda v: str(v))
def test_slabs_that_k_does_not_fill(op, M, N, K, dev):
    """Operands with rows of K inside buffers whose other rows and columns are not numbers: one slab, a whole number of them and a part, K in ranges, one tile and
    several a block (short K and long).  What lies behind K is read as zeros and by nobody."""
    from odysseus_transformer_amd import ops
    print(f"op={op} M={M} N={N} K={K}", flush=True)

    def inside(t):
        big = torch.full((t.shape[0] + 136, t.shape[1] + 16), float("nan"), dtype=t.dtype, device=dev)
        big[8:8 + t.shape[0], 8:8 + t.shape[1]] = t.to(dev)
        return big[8:8 + t.shape[0], 8:8 + t.shape[1]]

    a = inside(randn((K, M) if op == "tn" else (M, K), 51, dtype=torch.bfloat16))
    b = inside(randn((K, N), 52, std=0.05, dtype=torch.bfloat16))
    y = ops.gemm({"nn": ops.GEMM_NN, "tn": ops.GEMM_TN}[op], a, b)
    assert rel_err(y, (a.float().t() if op == "tn" else a.float()) @ b.float()) <= TOL_BF16


@pytest.mark.parametrize("M", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("N,K", [(4992, 72), (5120, 2056), (5120, 2048), (16256, 136), (16384, 72)], ids=lambda v: str(v))
@pytest.mark.parametrize("what", ["plain", "residual", "swiglu", "rope"])
def test_few_rows_around_the_lines_between_instances(what, N, K, M, dev):
    """312 and 320, 1016 and 1024 groups of 16 rows of W, rows of A on both sides of 4 and 8, K on both sides of 2048: one or two groups a block on 4 or 8
    wavefronts, the pairs of an epilogue inside a group or in two."""
    from odysseus_transformer_amd import ops
    print(f"what={what} M={M} N={N} K={K}", flush=True)
    dt = torch.bfloat16
    x, w = randn((M, K), 61, dtype=dt).to(dev), randn((N, K), 62, std=0.05, dtype=dt).to(dev)
    ref = x.float() @ w.float().t()
    if what == "plain":
        assert rel_err(ops.gemm(ops.GEMM_NT, x, w), ref) <= TOL_BF16
    elif what == "residual":
        r = randn((M, N), 63, dtype=dt).to(dev)
        assert rel_err(ops.linear_residual(x, w, r), ref + r.float()) <= TOL_BF16
    elif what == "swiglu":
        g, u = ref.to(dt).float().chunk(2, -1)
        want = torch.nn.functional.silu(g) * u
        gate_up, h = ops.linear_swiglu(x, w)
        assert rel_err(gate_up, ref) <= TOL_BF16 and rel_err(h, want) <= TOL_BF16
        assert torch.equal(ops.linear_swiglu_h(x, w), h)
    else:
        table = ops.rope_table(torch.arange(7, 7 + M, device=dev), M, 128)
        n_rot = N // 128 - 3
        cos, sin = table.float().view(M, 1, 64, 2).unbind(-1)
        a, b = ref[:, :n_rot * 128].reshape(M, n_rot, 2, 64).unbind(2)
        ref[:, :n_rot * 128] = torch.stack([a * cos - b * sin, b * cos + a * sin], 2).reshape(M, -1)
        assert rel_err(ops.linear_rope(x, w, table, n_rot, 128), ref) <= TOL_BF16


@pytest.mark.parametrize("op", ["nt", "nn", "tn"])
@pytest.mark.parametrize("M,N,K,ranges", [(8, 264, 40960, 16), (72, 1032, 30720, 12), (136, 1280, 41032, 16), (168, 4096, 40968, 16), (40, 392, 30656, 8),
                                          (128, 3072, 40960, 8)], ids=lambda v: str(v))
def test_ranges_of_a_long_k(op, M, N, K, ranges, dev):
    """More than eight ranges of K at their lines (`ranges`: the most there may be; fewer rows than a tile, a last slab that K does not fill, a last range
    shorter than the others), and a workspace with room for eight ranges, for one, and for none: the same product each time."""
    from odysseus_transformer_amd import _lib, ops
    print(f"long K {op} {M}x{N}x{K}", flush=True)
    if op == "nt" and M <= 16:
        pytest.skip("kernels for few rows have no ranges")
    code, lib = {"nt": ops.GEMM_NT, "nn": ops.GEMM_NN, "tn": ops.GEMM_TN}[op], _lib.load()
    a = randn((K, M) if op == "tn" else (M, K), 61, dtype=torch.bfloat16).to(dev)
    b = randn((N, K) if op == "nt" else (K, N), 62, std=0.05, dtype=torch.bfloat16).to(dev)
    ref = (a.double().t() if op == "tn" else a.double()) @ (b.double().t() if op == "nt" else b.double())
    need = lib.ody_gemm_workspace_bytes(code, M, N, K, _lib.ODY_BF16)
    assert need <= ranges * M * N * 4
    assert need > 8 * M * N * 4 or ranges == 8
    assert rel_err(ops.gemm(code, a, b), ref) <= TOL_BF16
    for room in (need, 8 * M * N * 4, need // ranges):
        ws = torch.full((room // 4 + 64,), float("nan"), dtype=torch.float32, device=dev)
        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)
        rc = lib.ody_gemm(code, a.data_ptr(), b.data_ptr(), y.data_ptr(), None, M, N, K, a.stride(0), b.stride(0), N, 0, _lib.ODY_BF16, ws.data_ptr(), room,
                          torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        assert rel_err(y, ref) <= TOL_BF16
        assert torch.isnan(ws[room // 4:]).all()


@pytest.mark.parametrize("op", ["nn", "tn"])
@pytest.mark.parametrize("M,N,K", [(264, 520, 64), (8200, 4616, 64), (136, 264, 128)], ids=lambda v: str(v))
def test_slabs_behind_a_k_of_whole_slabs(op, M, N, K, dev):
    test_slabs_that_k_does_not_fill(op, M, N, K, dev)


# groups of 16 rows of W a block, steps of K in flight, wavefronts: on both sides of every line of the choice
@pytest.mark.parametrize("what,N,K,M,instance", [
    ("plain", 2048, 1024, 9, "1, 8, 4"), ("plain", 2048, 1032, 9, "1, 4, 8"), ("residual", 2048, 2048, 9, "1, 4, 8"), ("plain", 2048, 2056, 9, "1, 8, 4"),
    ("plain", 4080, 4104, 2, "1, 4, 8"), ("plain", 4096, 4104, 2, "1, 8, 4"), ("plain", 4096, 4096, 2, "1, 4, 8"), ("plain", 4096, 4104, 1, "1, 4, 8"),
    ("residual", 4096, 4096, 5, "1, 4, 8"), ("residual", 4096, 4104, 5, "1, 8, 4"), ("plain", 4080, 4104, 5, "1, 8, 4"), ("residual", 4112, 72, 5, "1, 8, 4"),
    ("residual", 4112, 2056, 5, "2, 4, 4"), ("plain", 4112, 72, 9, "2, 4, 4"), ("rope", 4096, 72, 4, "1, 4, 8"), ("rope", 4224, 2048, 4, "2, 8, 8"),
    ("rope", 4224, 2048, 8, "2, 8, 8"), ("rope", 4224, 2048, 9, "2, 8, 8"), ("swiglu", 4128, 2048, 8, "2, 8, 8"), ("swiglu", 4128, 2048, 9, "2, 4, 4"),
    ("rope", 4224, 2056, 4, "2, 8, 8"), ("swiglu", 4224, 2056, 5, "2, 4, 4"), ("rope", 7168, 2056, 1, "2, 8, 8"), ("rope", 7296, 2056, 1, "1, 4, 8"),
    ("swiglu", 7200, 2056, 4, "1, 4, 8"), ("rope", 8192, 136, 16, "2, 8, 8"), ("rope", 8320, 136, 1, "1, 8, 4"), ("swiglu", 8192, 72, 1, "2, 8, 8"),
    ("swiglu", 8224, 72, 3, "1, 8, 4"), ("plain", 8192, 72, 4, "1, 4, 8"), ("plain", 8208, 72, 4, "1, 8, 4"), ("plain", 8208, 2056, 16, "1, 8, 4"),
    ("plain", 12784, 72, 9, "1, 8, 4"), ("plain", 12800, 72, 9, "2, 4, 4"), ("residual", 12800, 72, 8, "1, 8, 4"), ("residual", 12800, 2056, 8, "2, 4, 4")],
    ids=lambda v: str(v))
def test_few_rows_on_the_instance_of_their_sizes(what, N, K, M, instance, dev):
    _, ran = device_kernels(lambda: test_few_rows_around_the_lines_between_instances(what, N, K, M, dev))
    ran = [name for name in ran if "gemm_skinny_kernel<" in name]
    assert ran and all(f"gemm_skinny_kernel<{instance}, " in name for name in ran), ran


@pytest.mark.parametrize("what,N,K,M,instance", [
    ("plain", 16384, 1792, 5, "2, 4, 4"), ("plain", 16384, 1800, 5, "2, 4, 8"), ("residual", 16392, 2048, 8, "2, 4, 8"), ("plain", 16384, 2048, 12, "2, 4, 8"), ("plain", 16384, 2048, 13, "2, 4, 4"),
    ("plain", 16384, 2048, 4, "1, 8, 4"), ("swiglu", 16384, 2056, 8, "2, 4, 4"), ("swiglu", 16416, 2040, 6, "2, 4, 8"), ("rope", 16384, 1920, 7, "2, 4, 8"),
    ("plain", 16352, 2048, 5, "1, 8, 4")], ids=lambda v: str(v))
def test_few_rows_of_two_batches(what, N, K, M, instance, dev):
    test_few_rows_on_the_instance_of_their_sizes(what, N, K, M, instance, dev)


@pytest.mark.parametrize("op", ["nt", "nn", "tn"])
@pytest.mark.parametrize("M,N,K", [(72, 1032, 30720), (136, 1280, 41032), (40, 392, 30656)], ids=lambda v: str(v))
def test_a_long_k_without_a_workspace(op, M, N, K, dev):
    from odysseus_transformer_amd import _lib, ops
    print(f"long K, no workspace {op} {M}x{N}x{K}", flush=True)
    code = {"nt": ops.GEMM_NT, "nn": ops.GEMM_NN, "tn": ops.GEMM_TN}[op]
    a = randn((K, M) if op == "tn" else (M, K), 61, dtype=torch.bfloat16).to(dev)
    b = randn((N, K) if op == "nt" else (K, N), 62, std=0.05, dtype=torch.bfloat16).to(dev)
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)
    rc = _lib.load().ody_gemm(code, a.data_ptr(), b.data_ptr(), y.data_ptr(), None, M, N, K, a.stride(0), b.stride(0), N, 0, _lib.ODY_BF16, None, 0,
                              torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert rel_err(y, (a.double().t() if op == "tn" else a.double()) @ (b.double().t() if op == "nt" else b.double())) <= TOL_BF16
