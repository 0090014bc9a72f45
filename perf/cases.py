"""What a user of this framework has it compute, as timed cases: decoder layers in training and in inference, the attention
routine and the ring step on their own, the two shards of a tensor- / sequence-parallel rank, the loss head and the optimizer.

`listed()` names the standing cases, `draw(rng)` gives another one of the same ranges; a case is a dict of plain values whose
"kind" selects one of the families below.  `prepare(case, seed)` makes what a program holds before the call, `run(state)` is one
pass through the public entry points, `work(case)` the bytes and operations it cannot do without, and `tolerance(case)` the
relative error another correct implementation at the same precision would show.

Families (the model sizes are those of the training driver, the benchmark and the tests of this repository: hidden 4096 with
32 query heads on 8 or 32 key heads of 128 and an MLP of 11008 or 14336; hidden 2048 and 1024 beside them; the fp32 layer of
hidden 512 with 8 heads of 64 and an MLP of 1376):

  cached     forward of a decoder layer on few new tokens with earlier content in the key / value cache: one token is a step of
             autoregressive decoding, more are a chunk of a long prompt
  prefill    forward of a decoder layer on a whole prompt into an empty cache
  train      forward and backward of a decoder layer (bf16, or fp32 for the parity configuration)
  attn_rank  forward and backward of the attention block of one tensor-parallel rank: few heads, the whole gathered sequence
  mlp_rank   forward and backward of the second half of a layer (norm, SwiGLU MLP, residual add) on a rank's sequence shard
  flash      forward and backward of the attention routine alone, as the host models patched for it call it
  ring       forward and backward of one rank's share of zigzag ring attention, from the blocks the ring would bring
  head       the end of a training step: final norm, vocabulary projection, cross-entropy, and back
  adamw      one optimizer step over the parameters of decoder layers
"""
import math
import types

import torch

from odysseus_transformer_amd import ops
from odysseus_transformer_amd.decoder.odysseus import LlamaFlashAttention2TPSP, LlamaMLPZeRO, LlamaRMSNorm, OdysseusDecoderLayer
from odysseus_transformer_amd.decoder.ring import zigzag_ring_rank_attn
from odysseus_transformer_amd.losses.cross_entropy import CrossEntropyLoss
from odysseus_transformer_amd.optim import AdamW
from odysseus_transformer_amd.train import NativeLinear

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # one decoding step of the training driver's model behind a prompt of eight thousand tokens: latency and weight reads
        dict(name="decode_c8191", kind="cached", new=1, cache=8191, d=4096, hq=32, hkv=8, hd=128, i=11008),
        # a prompt of ordinary, ragged length
        dict(name="prefill_L3001", kind="prefill", L=3001, d=4096, hq=32, hkv=8, hd=128, i=11008),
        # the fp32 parity configuration: what the correctness of everything else is held against
        dict(name="train_fp32_L2048", kind="train", dtype="f32", L=2048, d=512, hq=8, hkv=8, hd=64, i=1376),
        # fine-tuning on documents of their own length
        dict(name="train_L1000", kind="train", dtype="bf16", L=1000, d=4096, hq=32, hkv=8, hd=128, i=11008),
        # the training driver's default: 16384 tokens, GQA 32/8
        dict(name="train_L16384", kind="train", dtype="bf16", L=16384, d=4096, hq=32, hkv=8, hd=128, i=11008),
        # the benchmark's rank of eight: 4 heads of 128 over 32768 gathered tokens
        dict(name="attn_rank_L32768", kind="attn_rank", L=32768, d=4096, hq=4, hkv=4, hd=128),
        # the same rank's MLP shard
        dict(name="mlp_rank_T4096", kind="mlp_rank", T=4096, d=4096, i=11008),
        # short sequences of a patched host model: a few small launches
        dict(name="flash_B4_L331", kind="flash", B=4, L=331, hq=8, hkv=2, hd=128, causal=True),
        # head_dim 64, the other head size that the routine takes
        dict(name="flash_hd64_L8192", kind="flash", B=1, L=8192, hq=16, hkv=16, hd=64, causal=True),
        # one rank of a ring of eight over 131072 tokens
        dict(name="ring_rank3_of_8", kind="ring", rank=3, world=8, chunk=8192, hq=4, hkv=4, hd=128),
        # norm, vocabulary projection and loss of a training step
        dict(name="head_T4096_V32000", kind="head", T=4096, d=4096, V=32000),
        # the optimizer on two layers of the 7B shape
        dict(name="adamw_2_layers", kind="adamw", layers=2, d=4096, hq=32, hkv=32, hd=128, i=11008),
    ]


def _log_int(rng, lo, hi, multiple=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(multiple, int(round(v / multiple)) * multiple)


def _model(rng):
    d, hq, i = rng.choice([(4096, 32, 11008), (4096, 32, 14336), (2048, 16, 5632), (2048, 16, 5464), (1024, 8, 2816)])
    return dict(d=d, hq=hq, hkv=max(1, hq // rng.choice([1, 4, 4, 8])), hd=128, i=i)


def draw(rng):
    kind = rng.choice(["cached", "prefill", "train", "train", "train_f32", "attn_rank", "mlp_rank", "flash", "flash", "ring",
                       "head", "adamw"])
    if kind == "cached":
        return dict(kind=kind, new=rng.choice([1, 1, 1, _log_int(rng, 2, 1024)]), cache=_log_int(rng, 64, 32768), **_model(rng))
    if kind == "prefill":
        return dict(kind=kind, L=_log_int(rng, 32, 16384), **_model(rng))
    if kind == "train":
        return dict(kind=kind, dtype="bf16", L=_log_int(rng, 64, 12000, rng.choice([1, 1, 64, 256])), **_model(rng))
    if kind == "train_f32":
        heads, hd = rng.choice([(8, 64), (4, 128), (16, 64)])
        return dict(kind="train", dtype="f32", L=_log_int(rng, 64, 4096), d=heads * hd, hq=heads, hkv=max(1, heads // rng.choice([1, 1, 4])),
                    hd=hd, i=rng.choice([1376, 2736]))
    if kind == "attn_rank":
        hq = rng.choice([2, 4, 8])
        return dict(kind=kind, L=_log_int(rng, 2048, 32768, rng.choice([1, 256])), d=4096, hq=hq, hkv=max(1, hq // rng.choice([1, 4])), hd=128)
    if kind == "mlp_rank":
        d, i = rng.choice([(4096, 11008), (4096, 14336), (2048, 5632), (2048, 5464)])
        return dict(kind=kind, T=_log_int(rng, 128, 8192, rng.choice([1, 1, 256])), d=d, i=i)
    if kind == "flash":
        hd = rng.choice([64, 64, 128])
        hq = rng.choice([4, 8, 16, 32])
        return dict(kind=kind, B=rng.choice([1, 1, 2, 4]), L=_log_int(rng, 96, 8192, rng.choice([1, 1, 128])), hq=hq,
                    hkv=max(1, hq // rng.choice([1, 1, 4])), hd=hd, causal=rng.choice([True, True, False]))
    if kind == "ring":
        world = rng.choice([2, 4, 8])
        return dict(kind=kind, rank=rng.randrange(world), world=world, chunk=_log_int(rng, 512, 8192, rng.choice([1, 256])), hq=4,
                    hkv=rng.choice([1, 4]), hd=128)
    if kind == "head":
        d = rng.choice([1024, 2048, 4096])
        return dict(kind=kind, T=_log_int(rng, 128, 8192), d=d, V=rng.choice([32000, 32000, 32008, 50264]))
    return dict(kind="adamw", layers=rng.choice([1, 2, 4]), **_model(rng))


# ------------------------------------------------------------------------------------------------- inputs
def _config(c):
    """The fields of a Llama configuration that the modules read."""
    return types.SimpleNamespace(hidden_size=c["d"], num_attention_heads=c.get("hq", 1), num_key_value_heads=c.get("hkv", 1),
                                 head_dim=c.get("hd", 128), intermediate_size=c.get("i", 8), hidden_act="silu", attention_dropout=0.0,
                                 rms_norm_eps=1e-6, rope_theta=10000.0, max_position_embeddings=1 << 20, pretraining_tp=1,
                                 num_hidden_layers=1)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, shape, dtype, std=1.0):
    t = torch.empty(shape, dtype=dtype, device=DEV)
    return t.normal_(0.0, std, generator=g)


def _filled(make, g, dtype):
    """A module made on the GPU with matrices of N(0, 0.02) and norm weights around one."""
    with torch.device(DEV):
        m = make().to(dtype)
    with torch.no_grad():
        for p in m.parameters():
            if p.dim() > 1:
                p.normal_(0.0, 0.02, generator=g)
            else:
                p.normal_(1.0, 0.1, generator=g)
    return m


class _Cache:
    """Key / value cache of one sequence and one layer in buffers allocated once.  Every pass of a case starts from the same
    `filled` tokens, so that it can be repeated."""

    def __init__(self, filled, room, hkv, hd, dtype, g):
        self.filled = filled
        self.k = _normal(g, (1, hkv, filled + room, hd), dtype)
        self.v = _normal(g, (1, hkv, filled + room, hd), dtype)

    def get_seq_length(self, layer_idx=0):
        return self.filled

    def update(self, k, v, layer_idx, cache_kwargs=None):
        a, b = self.filled, self.filled + k.shape[2]
        self.k[:, :, a:b].copy_(k)
        self.v[:, :, a:b].copy_(v)
        return self.k[:, :, :b], self.v[:, :, :b]

    def written(self, n):
        return self.k[:, :, self.filled:self.filled + n], self.v[:, :, self.filled:self.filled + n]


def prepare(case, seed):
    c, g = case, _gen(seed)
    kind = c["kind"]
    dt = DTYPES[c.get("dtype", "bf16")]
    s = types.SimpleNamespace(kind=kind, case=c)
    if kind in ("cached", "prefill"):
        n, filled = (c["new"], c["cache"]) if kind == "cached" else (c["L"], 0)
        s.layer = _filled(lambda: OdysseusDecoderLayer(_config(c)), g, dt)
        s.cache = _Cache(filled, n, c["hkv"], c["hd"], dt, g)
        s.x = _normal(g, (1, n, c["d"]), dt)
        s.pos = torch.arange(filled, filled + n, device=DEV)[None]
    elif kind == "train":
        s.layer = _filled(lambda: OdysseusDecoderLayer(_config(c)), g, dt)
        s.params = list(s.layer.parameters())
        s.x = _normal(g, (1, c["L"], c["d"]), dt).requires_grad_(True)
        s.dy = _normal(g, (1, c["L"], c["d"]), dt)
        s.pos = torch.arange(c["L"], device=DEV)[None]
    elif kind == "attn_rank":
        s.attn = _filled(lambda: LlamaFlashAttention2TPSP(_config(c), 0), g, dt)
        s.params = list(s.attn.parameters())
        s.x = _normal(g, (1, c["L"], c["d"]), dt).requires_grad_(True)      # the gathered, normalised activation
        s.dy = _normal(g, (1, c["L"], c["d"]), dt)
        s.pos = torch.arange(c["L"], device=DEV)[None]
    elif kind == "mlp_rank":
        s.norm = _filled(lambda: LlamaRMSNorm(c["d"]), g, dt)
        s.mlp = _filled(lambda: LlamaMLPZeRO(_config(c)), g, dt)
        s.params = list(s.norm.parameters()) + list(s.mlp.parameters())
        s.x = _normal(g, (1, c["T"], c["d"]), dt).requires_grad_(True)
        s.dy = _normal(g, (1, c["T"], c["d"]), dt)
    elif kind == "flash":
        shape = lambda h: (c["B"], c["L"], h, c["hd"])  # noqa: E731
        s.q, s.k, s.v = (_normal(g, shape(h), dt).requires_grad_(True) for h in (c["hq"], c["hkv"], c["hkv"]))
        s.do = _normal(g, shape(c["hq"]), dt)
    elif kind == "ring":
        shape = lambda h: (1, 2 * c["chunk"], h, c["hd"])  # noqa: E731
        s.q = _normal(g, shape(c["hq"]), dt).requires_grad_(True)
        s.ks = [_normal(g, shape(c["hkv"]), dt).requires_grad_(True) for _ in range(c["world"])]
        s.vs = [_normal(g, shape(c["hkv"]), dt).requires_grad_(True) for _ in range(c["world"])]
        s.do = _normal(g, shape(c["hq"]), dt)
    elif kind == "head":
        s.norm = _filled(lambda: LlamaRMSNorm(c["d"]), g, dt)
        s.lm_head = _filled(lambda: NativeLinear(torch.nn.Linear(c["d"], c["V"], bias=False)), g, dt)
        s.params = list(s.norm.parameters()) + list(s.lm_head.parameters())
        s.loss = CrossEntropyLoss(inplace_backward=True)
        s.x = _normal(g, (1, c["T"], c["d"]), dt).requires_grad_(True)
        s.labels = torch.randint(0, c["V"], (c["T"],), generator=g, device=DEV)
    elif kind == "adamw":
        s.layers = [_filled(lambda: OdysseusDecoderLayer(_config(c)), g, dt) for _ in range(c["layers"])]
        s.params = [p for m in s.layers for p in m.parameters()]
        s.optim = AdamW(s.params, lr=1e-3)
        for p in s.params:
            p.grad = _normal(g, p.shape, dt, 1e-2)
    else:
        raise ValueError(f"unknown kind {kind!r}")
    return s


# ------------------------------------------------------------------------------------------------- one pass
def _clear(*tensors):
    for t in tensors:
        t.grad = None


def run(s):
    c = s.case
    if s.kind in ("cached", "prefill"):
        with torch.no_grad():
            y = s.layer(s.x, position_ids=s.pos, past_key_values=s.cache)
        return (y, *s.cache.written(s.x.shape[1]))
    if s.kind == "train":
        _clear(s.x, *s.params)
        y = s.layer(s.x, position_ids=s.pos)
        y.backward(s.dy)
        return (y, s.x.grad, *(p.grad for p in s.params))
    if s.kind == "attn_rank":
        _clear(s.x, *s.params)
        y = s.attn(s.x, position_ids=s.pos)[0]
        y.backward(s.dy)
        return (y, s.x.grad, *(p.grad for p in s.params))
    if s.kind == "mlp_rank":
        _clear(s.x, *s.params)
        n, skip = ops.rmsnorm_fork(s.x, s.norm.weight, s.norm.variance_epsilon)
        y = s.mlp(n, residual=skip)
        y.backward(s.dy)
        return (y, s.x.grad, *(p.grad for p in s.params))
    if s.kind == "flash":
        _clear(s.q, s.k, s.v)
        out = ops.flash_attn_func(s.q, s.k, s.v, causal=c["causal"])
        out.backward(s.do)
        return (out, s.q.grad, s.k.grad, s.v.grad)
    if s.kind == "ring":
        _clear(s.q, *s.ks, *s.vs)
        out, lse = zigzag_ring_rank_attn(s.q, s.ks, s.vs, c["rank"], c["world"])
        out.backward(s.do)
        return (out, lse, s.q.grad, *(t.grad for t in s.ks), *(t.grad for t in s.vs))
    if s.kind == "head":
        _clear(s.x, *s.params)
        logits = s.lm_head(s.norm(s.x))
        loss = s.loss(logits.reshape(-1, logits.shape[-1]), s.labels)
        loss.backward()
        return (loss, s.x.grad, *(p.grad for p in s.params))
    if s.kind == "adamw":
        s.optim.step()
        st = [s.optim.state[p] for p in s.params]
        return [t for p, q in zip(s.params[:16], st) for t in (p, q["exp_avg"], q["exp_avg_sq"])]
    raise ValueError(f"unknown kind {s.kind!r}")


# ------------------------------------------------------------------------------------------------- what it cannot do without
def _pairs(new, cache, causal=True):
    """Visible (query, key) pairs of `new` queries behind `cache` earlier keys."""
    return new * cache + new * (new + 1) / 2 if causal else new * (cache + new)


def work(case):
    c, kind = case, case["kind"]
    es = 4 if c.get("dtype") == "f32" else 2
    hd = c.get("hd", 0)
    qkv = c.get("hq", 0) + 2 * c.get("hkv", 0)
    if kind in ("cached", "prefill", "train"):
        n = c["new"] if kind == "cached" else c["L"]
        cache = c["cache"] if kind == "cached" else 0
        mats = c["d"] * hd * (qkv + c["hq"]) + 3 * c["d"] * c["i"]
        attn = 4 * hd * c["hq"] * _pairs(n, cache)
        if kind == "train":
            return {"flops": 6 * n * mats + 3.5 * attn, "bytes": es * (2 * mats + 4 * n * c["d"])}
        return {"flops": 2 * n * mats + attn, "bytes": es * (mats + 2 * n * c["d"] + 2 * (cache + n) * c["hkv"] * hd)}
    if kind == "attn_rank":
        mats = c["d"] * hd * (qkv + c["hq"])
        return {"flops": 6 * c["L"] * mats + 3.5 * 4 * hd * c["hq"] * _pairs(c["L"], 0), "bytes": es * (2 * mats + 4 * c["L"] * c["d"])}
    if kind == "mlp_rank":
        mats = 3 * c["d"] * c["i"]
        return {"flops": 6 * c["T"] * mats, "bytes": es * (2 * mats + 4 * c["T"] * c["d"])}
    if kind == "flash":
        rows = c["B"] * c["L"] * hd
        return {"flops": 3.5 * 4 * hd * c["B"] * c["hq"] * _pairs(c["L"], 0, c["causal"]), "bytes": es * rows * (4 * c["hq"] + 4 * c["hkv"])}
    if kind == "ring":
        n = c["chunk"]
        pairs = _pairs(2 * n, 0) + 2 * n * n * (c["world"] - 1)
        return {"flops": 3.5 * 4 * hd * c["hq"] * pairs, "bytes": es * 2 * n * hd * (4 * c["hq"] + 4 * c["hkv"] * c["world"])}
    if kind == "head":
        return {"flops": 6 * c["T"] * c["d"] * c["V"], "bytes": es * (2 * c["V"] * c["d"] + 2 * c["T"] * c["d"])}
    if kind == "adamw":
        params = c["layers"] * (c["d"] * hd * (qkv + c["hq"]) + 3 * c["d"] * c["i"])
        return {"flops": 12 * params, "bytes": 7 * es * params}
    raise ValueError(f"unknown kind {kind!r}")


def tolerance(case):
    """Measured: bf16 against the same pass in fp32 on the same values, fp32 against fp64.  Largest over the outputs: the layers
    1.1e-2 (gradients behind the softmax; 6e-3 the others), the attention routine, ring and loss head 2.3e-3 to 2.9e-3, AdamW 2.0e-3,
    fp32 layer 1.4e-6.  About four times these, twice for the layers, whose roundings are mostly shared by any bf16 implementation."""
    if case.get("dtype") == "f32":
        return {"rel": 6e-6}
    return {"rel": {"flash": 1e-2, "ring": 1e-2, "head": 1e-2, "adamw": 8e-3}.get(case["kind"], 2e-2)}
