"""What a serving process has this framework do, as cases that can be timed and compared.

Five kinds of work, each through the entry points a program calls:

* ``linear`` - one ``Int8Linear.forward``: a projection of a decoder layer, from a single
  decoded token to a whole prompt (prefill passes one prompt's tokens as the rows);
* ``gateup`` - ``int8_gateup_swiglu``: the MLP's gate and up projections with SwiGLU;
* ``decode`` - ``paged_attention_decode_batched``: one decode step's attention over the block pool;
* ``prefill`` - one layer's attention over a prompt (or over the rest of one whose first ``past``
  tokens are in the pool already): the cache layer's ``update``, which writes K and V to the pool
  and returns the row gathered, then the ``block_paged`` attention hook;
* ``step`` - one whole native decode step (``Int8DecodeModel.step``) replayed from a HIP graph, as
  a decode loop runs it.

Shapes are the Llama-3-8B and Qwen2-0.5B ones of ``decode_step.py``; contexts are the benchmark's.
"""

from __future__ import annotations

import math
import os
import sys
from types import SimpleNamespace

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "llm-serving-runtime_amd"))

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
DEV = "cuda"


def listed() -> list[dict]:
    return [
        # One request decoding alone: a single row through a square projection (o), latency bound.
        dict(name="linear_m1_o", kind="linear", m=1, n=4096, k=4096, bias=False),
        # The benchmark's batch of 32 decoding rows through the widest-K projection (down).
        dict(name="linear_m32_down", kind="linear", m=32, n=4096, k=14336, bias=False),
        # Prefill of an odd-length prompt on the small model: q/k/v rows with their bias.
        dict(name="linear_m777_qkv_small", kind="linear", m=777, n=1152, k=896, bias=True),
        # Prefill of a long odd-length prompt on the large model.
        dict(name="linear_m1531_down", kind="linear", m=1531, n=4096, k=14336, bias=False),
        # The shared-prefix batch: 128 decoding rows through gate||up.
        dict(name="gateup_m128", kind="gateup", m=128, inter=14336, k=4096),
        # Prefill of a 2048-token prompt through gate||up, the largest matrix of a layer.
        dict(name="gateup_m2048", kind="gateup", m=2048, inter=14336, k=4096),
        # The benchmark's attention: 32 rows of U[128, 4096] tokens, Llama-3-8B heads.
        dict(name="decode_b32", kind="decode", b=32, lo=128, hi=4096, hkv=8, group=4, d=128, bs=16, dtype="fp16"),
        # A small bf16 batch with an odd group and odd lengths: latency and launches.
        dict(name="decode_b7_bf16", kind="decode", b=7, lo=97, hi=1501, hkv=2, group=7, d=64, bs=32, dtype="bf16"),
        # Attention of a 2048-token prompt, one layer of the large model.
        dict(name="prefill_2048", kind="prefill", p=2048, past=0, hkv=8, group=4, d=128, bs=16, dtype="fp16"),
        # The odd-length rest of a prompt whose prefix was in the pool already, small model, bf16.
        dict(name="prefill_509_past_bf16", kind="prefill", p=509, past=176, hkv=2, group=7, d=64, bs=16,
             dtype="bf16"),
        # A whole step of the small model at batch 16: about 190 dependent launches.
        dict(name="step_small_b16", kind="step", shape="small", layers=24, b=16, lo=512, hi=2048),
        # A step of the large model at batch 32, cut to 4 layers so that the states fit; the head is whole.
        dict(name="step_large_b32", kind="step", shape="large", layers=4, b=32, lo=128, hi=4096),
    ]


def _log(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng) -> dict:
    kind = rng.choice(["linear", "linear", "gateup", "decode", "decode", "prefill", "prefill", "step"])
    if kind == "linear":
        n, k = 16 * _log(rng, 32, 1024), 64 * _log(rng, 8, 224)
        most = max(1, min(4096, 2048 * 28672 * 4096 // (n * k)))
        return dict(kind=kind, m=_log(rng, 1, most), n=n, k=k, bias=rng.random() < 0.5)
    if kind == "gateup":
        inter, k = 64 * _log(rng, 16, 224), 64 * _log(rng, 8, 64)
        return dict(kind=kind, m=_log(rng, 1, 2048), inter=inter, k=k)
    if kind == "decode":
        hkv, group, d = rng.choice([(8, 4, 128), (2, 7, 64), (4, 8, 128), (8, 5, 128), (12, 1, 64), (1, 8, 128)])
        b = _log(rng, 1, 64)
        hi = _log(rng, 64, min(8192, max(128, 32 * 4096 // b)))
        return dict(kind=kind, b=b, lo=rng.randint(1, hi), hi=hi, hkv=hkv, group=group, d=d,
                    bs=rng.choice([16, 16, 32]), dtype=rng.choice(["fp16", "fp16", "bf16"]))
    if kind == "prefill":
        hkv, group, d = rng.choice([(8, 4, 128), (2, 7, 64), (4, 8, 128), (8, 1, 64)])
        return dict(kind=kind, p=_log(rng, 2, 1536), past=rng.choice([0, 0, 16 * rng.randint(1, 32)]), hkv=hkv,
                    group=group, d=d, bs=16, dtype=rng.choice(["fp16", "fp16", "bf16"]))
    small = rng.random() < 0.7
    b = _log(rng, 1, 64 if small else 32)
    hi = _log(rng, 64, 2048 if small else 4096)
    return dict(kind=kind, shape="small" if small else "large", layers=rng.randint(2, 12) if small else
                rng.randint(1, 3), b=b, lo=rng.randint(1, hi), hi=hi)


# ---------------------------------------------------------------------------------------------
# Inputs. Each from one generator in a fixed order, so that exact() can make the same ones.
# ---------------------------------------------------------------------------------------------
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _quantize(w: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """Per-channel symmetric int8 of ``w [N, K]``: q and the fp16 scale."""
    scale = (w.abs().amax(dim=1) / 127).to(torch.float16)
    return (w / scale.float()[:, None]).round().clamp(-127, 127).to(torch.int8), scale


def _rows(m: int, k: int, g: torch.Generator) -> torch.Tensor:
    """Normalised activations: unit normal with the few large channels that decoders show."""
    x = torch.randn(m, k, generator=g, device=DEV)
    return (x * (1 + 7 * (torch.rand(k, generator=g, device=DEV) < 0.005))).to(torch.float16)


def _linear_inputs(c: dict, seed: int) -> tuple:
    g = _gen(seed)
    q, scale = _quantize(torch.randn(c["n"], c["k"], generator=g, device=DEV) * 0.02)
    bias = (torch.randn(c["n"], generator=g, device=DEV) * 0.1).to(torch.float16) if c["bias"] else None
    return q, scale, bias, _rows(c["m"], c["k"], g)


def _gateup_inputs(c: dict, seed: int) -> tuple:
    g = _gen(seed)
    gate, up = (_quantize(torch.randn(c["inter"], c["k"], generator=g, device=DEV) * 0.02) for _ in range(2))
    return gate, up, _rows(c["m"], c["k"], g)


def _lengths(c: dict) -> list[int]:
    """``b`` lengths spread evenly over lo..hi: the same for every seed, so that the work is the case's."""
    return [c["lo"] + int((c["hi"] - c["lo"]) * (i + 0.5) / c["b"]) for i in range(c["b"])]


def _tables(lens: list[int], bs: int, headroom: int, seed: int) -> tuple[list[int], torch.Tensor, int]:
    """Lengths in a seeded order, disjoint block tables in a seeded block order, and the pool's blocks."""
    g = torch.Generator().manual_seed(seed)
    lens = [lens[i] for i in torch.randperm(len(lens), generator=g).tolist()]
    need = [-(-(n + headroom) // bs) for n in lens]
    blocks = sum(need) + 8
    perm = torch.randperm(blocks, generator=g).to(torch.int32)
    tables, used = torch.zeros(len(lens), max(need), dtype=torch.int32), 0
    for row, n in enumerate(need):
        tables[row, :n] = perm[used:used + n]
        used += n
    return lens, tables, blocks


def _pool(blocks: int, bs: int, layers: int, hkv: int, d: int, dtype: torch.dtype, g: torch.Generator):
    from runtime_amd.phase2.paged_kv_kernel import GpuKVBlockPool

    pool = GpuKVBlockPool(num_blocks=blocks, block_size_tokens=bs, num_layers=layers, num_kv_heads=hkv, head_dim=d,
                          dtype=dtype, device=DEV)
    for layer in range(layers):
        for view, kv in zip((pool.k_layer_view(layer), pool.v_layer_view(layer)), _kv(blocks, bs, hkv, d, dtype, g)):
            view.copy_(kv)
    return pool


def _kv(blocks: int, bs: int, hkv: int, d: int, dtype: torch.dtype, g: torch.Generator):
    """K and V of one layer's blocks."""
    return [torch.randn(blocks, hkv, bs, d, generator=g, device=DEV).to(dtype) for _ in range(2)]


def _prefill_inputs(c: dict, seed: int) -> tuple:
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    total = c["past"] + c["p"]
    _, tables, blocks = _tables([total], c["bs"], 0, seed)

    def states(heads: int) -> torch.Tensor:  # [1, heads, p, d] as a decoder layer makes it from its rows
        return torch.randn(1, c["p"], heads, c["d"], generator=g, device=DEV).to(dt).transpose(1, 2)

    q, k, v = states(c["hkv"] * c["group"]), states(c["hkv"]), states(c["hkv"])
    return g, tables[0], blocks, q, k, v


SHAPES = {
    "small": dict(hidden=896, heads=14, kv_heads=2, d=64, inter=4864, vocab=151936, theta=1e6, eps=1e-6, bias=True),
    "large": dict(hidden=4096, heads=32, kv_heads=8, d=128, inter=14336, vocab=128256, theta=5e5, eps=1e-5, bias=False),
}


def _step_weights(c: dict, g: torch.Generator):
    """The weights in the module layout that ``Int8DecodeModel.from_hf`` reads."""
    s = SHAPES[c["shape"]]
    h, qd, kd, inter = s["hidden"], s["heads"] * s["d"], s["kv_heads"] * s["d"], s["inter"]

    def w(n: int, k: int, bias: bool = False):
        return SimpleNamespace(weight=torch.randn(n, k, generator=g, device=DEV) * k ** -0.5,
                               bias=(torch.randn(n, generator=g, device=DEV) * 0.1).half() if bias else None)

    def norm():
        return SimpleNamespace(weight=(1 + 0.1 * torch.randn(h, generator=g, device=DEV)).half())

    layers = []
    for _ in range(c["layers"]):
        attn = SimpleNamespace(q_proj=w(qd, h, s["bias"]), k_proj=w(kd, h, s["bias"]), v_proj=w(kd, h, s["bias"]),
                               o_proj=w(h, qd))
        mlp = SimpleNamespace(gate_proj=w(inter, h), up_proj=w(inter, h), down_proj=w(h, inter))
        layers.append(SimpleNamespace(self_attn=attn, mlp=mlp, input_layernorm=norm(),
                                      post_attention_layernorm=norm()))
    embed = SimpleNamespace(weight=torch.randn(s["vocab"], h, generator=g, device=DEV).half())
    config = SimpleNamespace(hidden_size=h, num_hidden_layers=c["layers"], num_attention_heads=s["heads"],
                             num_key_value_heads=s["kv_heads"], head_dim=s["d"], intermediate_size=inter,
                             vocab_size=s["vocab"], rope_theta=s["theta"], rms_norm_eps=s["eps"])
    return SimpleNamespace(config=config, lm_head=w(s["vocab"], h),
                           model=SimpleNamespace(layers=layers, embed_tokens=embed, norm=norm()))


def _step_tokens(c: dict, g: torch.Generator) -> torch.Tensor:
    return torch.randint(0, SHAPES[c["shape"]]["vocab"], (c["b"],), generator=g, device=DEV)


def prepare(case: dict, seed: int):
    kind = case["kind"]
    if kind == "linear":
        from runtime_amd.phase2.int8_linear import Int8Linear

        q, scale, bias, x = _linear_inputs(case, seed)
        return SimpleNamespace(kind=kind, module=Int8Linear.from_quantized(q, scale, bias), x=x)
    if kind == "gateup":
        from runtime_amd.phase2.int8_linear import gateup_interleave, pack_weight

        gate, up, x = _gateup_inputs(case, seed)
        packed = pack_weight(gateup_interleave(gate[0], up[0]))
        return SimpleNamespace(kind=kind, packed=packed, scale=gateup_interleave(gate[1], up[1]),
                               inter=case["inter"], x=x)
    if kind == "decode":
        from runtime_amd.phase2.paged_attention_hip import PagedDecodeBatchMetadata

        g = _gen(seed)
        lens, tables, blocks = _tables(_lengths(case), case["bs"], 0, seed)
        dt = DTYPES[case["dtype"]]
        pool = _pool(blocks, case["bs"], 1, case["hkv"], case["d"], dt, g)
        query = torch.randn(case["b"], case["hkv"] * case["group"], 1, case["d"], generator=g, device=DEV).to(dt)
        meta = PagedDecodeBatchMetadata(pool=pool, layer_idx=0, block_tables=tables.to(DEV),
                                        seq_lens=torch.tensor(lens, dtype=torch.int32, device=DEV))
        return SimpleNamespace(kind=kind, query=query, meta=meta, group=case["group"], scaling=case["d"] ** -0.5)
    if kind == "prefill":
        from runtime_amd.phase2.paged_kv_cache import BlockPagedLayer

        g, table, blocks, q, k, v = _prefill_inputs(case, seed)
        pool = _pool(blocks, case["bs"], 1, case["hkv"], case["d"], DTYPES[case["dtype"]], g)
        return SimpleNamespace(kind=kind, layer=BlockPagedLayer(pool, 0), block_ids=table.tolist(),
                               table=table.to(DEV), past=case["past"], q=q, k=k, v=v, scaling=case["d"] ** -0.5,
                               module=SimpleNamespace(num_key_value_groups=case["group"], training=False))
    from runtime_amd.phase2.decode_step import Int8DecodeModel

    g = _gen(seed)
    model = Int8DecodeModel.from_hf(_step_weights(case, g), device=DEV, max_positions=8192)
    tokens = _step_tokens(case, g)
    lens, tables, blocks = _tables(_lengths(case), 16, 1, seed)
    s = SHAPES[case["shape"]]
    pool = _pool(blocks, 16, case["layers"], s["kv_heads"], s["d"], torch.float16, g)
    st = SimpleNamespace(kind=kind, model=model, pool=pool, tokens=tokens, tables=tables.to(DEV),
                         start=torch.tensor(lens, dtype=torch.int32, device=DEV))
    st.seq_lens = st.start.clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _step(st)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    st.graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(st.graph):
        _step(st)
    return st


def _step(st) -> None:
    """One step from the same lengths each time, so that every pass does the same work."""
    torch.add(st.start, 0, out=st.seq_lens)
    _, st.logits = st.model.step(st.tokens, st.pool, st.tables, st.seq_lens, return_logits=True)


@torch.no_grad()
def run(st):
    if st.kind == "linear":
        return st.module(st.x)
    if st.kind == "gateup":
        from runtime_amd.phase2.int8_linear import int8_gateup_swiglu

        return int8_gateup_swiglu(st.x, st.packed, st.scale, None, st.inter)
    if st.kind == "decode":
        from runtime_amd.phase2.paged_attention_hip import paged_attention_decode_batched

        return paged_attention_decode_batched(st.query, st.meta, st.group, st.scaling)
    if st.kind == "prefill":
        from runtime_amd.phase2.block_paged_attention import block_paged_attention_forward

        st.layer.reset()
        st.layer.set_block_ids(st.block_ids, st.table)
        if st.past:
            st.layer.set_seq_length(st.past)
        keys, values = st.layer.update(st.k, st.v)
        out, weights = block_paged_attention_forward(st.module, st.q, keys, values, None, st.scaling)
        return {"out": out, "weights": weights}
    st.graph.replay()
    return {"logits": st.logits, "seq_lens": st.seq_lens}


# ---------------------------------------------------------------------------------------------
# What a pass cannot do without, how far two correct passes may be apart, and the exact answer.
# ---------------------------------------------------------------------------------------------
def _linear_work(m: int, n: int, k: int, out: int | None = None) -> tuple[int, int]:
    return n * k + 2 * n + 2 * m * k + 2 * m * (n if out is None else out), 2 * m * n * k


def _decode_work(lens: list[int], hkv: int, group: int, d: int, bs: int) -> tuple[int, int]:
    total = sum(lens)
    io = 2 * len(lens) * hkv * group * d * 2 + sum(-(-n // bs) for n in lens) * 4 + 4 * len(lens)
    return total * hkv * d * 4 + io, total * hkv * group * d * 4


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "linear":
        b, f = _linear_work(case["m"], case["n"], case["k"])
        b += 2 * case["n"] if case["bias"] else 0
    elif kind == "gateup":
        b, f = _linear_work(case["m"], 2 * case["inter"], case["k"], case["inter"])
    elif kind == "decode":
        b, f = _decode_work(_lengths(case), case["hkv"], case["group"], case["d"], case["bs"])
    elif kind == "prefill":
        p, total, hq = case["p"], case["past"] + case["p"], case["hkv"] * case["group"]
        # q and the new k, v in; k, v to the pool; the past read; out and the whole weight matrix written
        b = 2 * (2 * p * hq * case["d"] + 4 * p * case["hkv"] * case["d"] + 2 * case["past"] * case["hkv"] * case["d"]
                 + hq * p * total)
        f = 4 * hq * case["d"] * (p * case["past"] + p * (p + 1) // 2)
    else:
        s, m = SHAPES[case["shape"]], case["b"]
        qkv = (s["heads"] + 2 * s["kv_heads"]) * s["d"]
        parts = [_linear_work(m, qkv, s["hidden"]), _linear_work(m, s["hidden"], s["heads"] * s["d"]),
                 _linear_work(m, 2 * s["inter"], s["hidden"], s["inter"]), _linear_work(m, s["hidden"], s["inter"]),
                 _decode_work([n + 1 for n in _lengths(case)], s["kv_heads"], s["heads"] // s["kv_heads"], s["d"], 16)]
        head = _linear_work(m, s["vocab"], s["hidden"])
        b = case["layers"] * sum(x[0] for x in parts) + head[0]
        f = case["layers"] * sum(x[1] for x in parts) + head[1]
    return {"bytes": b, "flops": f}


def tolerance(case: dict):
    """About four times what the path measures off its exact() value (fp16 rounds by 2**-11, bf16 by
    2**-8): linear 2.1e-4, gateup 4.3e-4, decode 4.5e-4 and 2.7e-3, prefill 6e-4 to 1.8e-3 (its scores
    pass through the 16-bit type too) and 5.5e-3, step 2.9e-3."""
    if case["kind"] in ("linear", "gateup"):
        return {"rel": 1e-3 if case["kind"] == "linear" else 1.7e-3}
    if case["kind"] == "decode":
        return {"rel": 1.8e-3 if case["dtype"] == "fp16" else 1.1e-2}
    if case["kind"] == "prefill":
        return {"rel": 6e-3 if case["dtype"] == "fp16" else 2.2e-2}
    return {"rel": 1.2e-2}


def _attend(q, k, v, scaling: float):
    """q [H, D] against k, v [S, Hkv, D] in float64."""
    h, d = q.shape
    hkv = k.shape[1]
    qg = q.view(hkv, h // hkv, d)
    p = torch.softmax(torch.matmul(qg, k.permute(1, 2, 0).contiguous()) * scaling, dim=-1)
    return torch.matmul(p, v.transpose(0, 1).contiguous()).reshape(h, d)


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "linear":
        q, scale, bias, x = _linear_inputs(case, seed)
        y = x.double() @ (q.double() * scale.double()[:, None]).T.contiguous()
        return y + bias.double() if bias is not None else y
    if kind == "gateup":
        gate, up, x = _gateup_inputs(case, seed)
        g, u = (x.double() @ (q.double() * s.double()[:, None]).T.contiguous() for q, s in (gate, up))
        return g * torch.sigmoid(g) * u
    if kind == "decode":
        g = _gen(seed)
        lens, tables, blocks = _tables(_lengths(case), case["bs"], 0, seed)
        dt, bs = DTYPES[case["dtype"]], case["bs"]
        k, v = _kv(blocks, bs, case["hkv"], case["d"], dt, g)
        query = torch.randn(case["b"], case["hkv"] * case["group"], 1, case["d"], generator=g, device=DEV).to(dt)
        rows = []
        for b, n in enumerate(lens):
            kb, vb = (_row(t, tables[b], n, bs) for t in (k, v))
            rows.append(_attend(query[b, :, 0].double(), kb, vb, case["d"] ** -0.5))
        return torch.stack(rows).unsqueeze(2)
    if kind == "prefill":
        g, table, blocks, q, k, v = _prefill_inputs(case, seed)
        k, v = (t.double() for t in (k, v))
        if case["past"]:
            held = _kv(blocks, case["bs"], case["hkv"], case["d"], DTYPES[case["dtype"]], g)
            k, v = (torch.cat([_row(t, table, case["past"], case["bs"]).transpose(0, 1)[None], new], dim=2)
                    for t, new in zip(held, (k, v)))
        k, v = (t.repeat_interleave(case["group"], dim=1) for t in (k, v))
        scores = torch.matmul(q.double(), k.transpose(2, 3).contiguous()) * case["d"] ** -0.5
        p, total = case["p"], case["past"] + case["p"]
        hidden = torch.ones(p, total, dtype=torch.bool, device=DEV).triu(total - p + 1)
        weights = torch.softmax(scores.masked_fill(hidden, float("-inf")), dim=-1)
        return {"out": torch.matmul(weights, v.contiguous()).transpose(1, 2), "weights": weights}
    return _exact_step(case, seed)


def _row(t: torch.Tensor, table: torch.Tensor, n: int, bs: int) -> torch.Tensor:
    """The first ``n`` tokens of one row, ``[n, Hkv, D]`` in float64, from blocks ``[nb, Hkv, bs, D]``."""
    ids = table[: -(-n // bs)].to(DEV).long()
    return t[ids].permute(0, 2, 1, 3).reshape(-1, t.shape[1], t.shape[3])[:n].double()


def _exact_step(case: dict, seed: int):
    s, g = SHAPES[case["shape"]], _gen(seed)
    hf = _step_weights(case, g)
    tokens = _step_tokens(case, g)
    lens, tables, blocks = _tables(_lengths(case), 16, 1, seed)
    hd, hq, hkv = s["d"], s["heads"], s["kv_heads"]

    def lin(x, mod):
        q, scale = _quantize(mod.weight)
        y = x @ (q.double() * scale.double()[:, None]).T.contiguous()
        return y + mod.bias.double() if mod.bias is not None else y

    def norm(x, mod):
        return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + s["eps"]) * mod.weight.double()

    inv = 1.0 / (s["theta"] ** (torch.arange(0, hd, 2, dtype=torch.int64).to(torch.float32) / hd))
    ang = (torch.tensor(lens, dtype=torch.float32)[:, None] * inv[None]).double().to(DEV)
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def rope(x):
        a, b = x[..., : hd // 2], x[..., hd // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)

    h = hf.model.embed_tokens.weight[tokens].double()
    for layer in hf.model.layers:
        held = _kv(blocks, 16, hkv, hd, torch.float16, g)
        x = norm(h, layer.input_layernorm)
        at = layer.self_attn
        q, k, v = (lin(x, m).view(case["b"], -1, hd) for m in (at.q_proj, at.k_proj, at.v_proj))
        q, k = rope(q), rope(k)
        rows = []
        for b, n in enumerate(lens):
            kb, vb = (torch.cat([_row(t, tables[b], n, 16), new[b][None]]) for t, new in zip(held, (k, v)))
            rows.append(_attend(q[b], kb, vb, hd ** -0.5).reshape(-1))
        h = h + lin(torch.stack(rows), at.o_proj)
        x = norm(h, layer.post_attention_layernorm)
        gate, up = lin(x, layer.mlp.gate_proj), lin(x, layer.mlp.up_proj)
        h = h + lin(gate * torch.sigmoid(gate) * up, layer.mlp.down_proj)
    return {"logits": lin(norm(h, hf.model.norm), hf.lm_head), "seq_lens": None}
