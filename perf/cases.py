"""The work a user of this framework has it do, as measurable cases.

Each case goes through public entry points: the fp8-weight linear (``hip.fp8_linear``), one decoder layer
(``workloads.DecoderLayer``) in decode and in prefill, with bf16 or fp8 weights, one diffusion-transformer
block (``workloads.DiTBlock``), the decode of a unit kept exponent-coded in HBM (``DeviceEncodedBlock``), the
batched scatter of a streamed chunk (``ScatterPlan``) and one decode step of a model whose layers stream
from host memory (``OffloadManager``).

``listed()`` names the cases, ``draw(rng)`` gives further ones of the same ranges, ``prepare`` builds what a
program holds before the call, ``run`` is one pass, ``work`` what the pass cannot do without, ``tolerance``
how far two correct implementations lie apart, and ``exact`` the result in 64 bits by plain torch.
"""

from __future__ import annotations

import math

import torch

from flextensor_amd import expcode, hip
from flextensor_amd import workloads as W
from flextensor_amd.config import OffloadConfig
from flextensor_amd.manager import OffloadManager
from flextensor_amd.scatter import ScatterPlan

MIB = 1 << 20
DEV = "cuda"

# The decoder shapes of the benchmark (7B in bf16, 70B in fp8), by their layer dimensions.
_7B = {"hidden": 4096, "heads": 32, "kv_heads": 32, "head_dim": 128, "inter": 11008}
_70B = {"hidden": 8192, "heads": 64, "kv_heads": 8, "head_dim": 128, "inter": 28672}


def _layer_case(shape: dict, fp8: bool, batch: int, tokens: int, pos: int, name: str | None = None) -> dict:
    c = {"kind": "layer", **shape, "fp8": fp8, "batch": batch, "tokens": tokens, "pos": pos}
    return {"name": name, **c} if name else c


def listed() -> list[dict]:
    return [
        # the smallest call: one token through a k or v projection of the fp8 decoder
        {"name": "linear_1_row", "kind": "linear", "m": 1, "n": 1024, "k": 8192},
        # a decode batch of odd size through a matrix whose sides fill no tile
        {"name": "linear_33_rows_ragged", "kind": "linear", "m": 33, "n": 5003, "k": 4080},
        # a prefill through the gate projection of the fp8 decoder, at the benchmark's 512 rows
        {"name": "linear_512_rows", "kind": "linear", "m": 512, "n": 28672, "k": 8192},
        # a prompt of odd length through the down projection
        {"name": "linear_777_rows_ragged", "kind": "linear", "m": 777, "n": 8192, "k": 28672},
        # one decode step of a layer: batch 8 fp8 in the middle of a long context
        _layer_case(_70B, True, 8, 1, 1023, "layer_fp8_decode"),
        # the prefill of that batch: 8 prompts of 64 tokens
        _layer_case(_70B, True, 8, 64, 0, "layer_fp8_prefill"),
        # one decode step of a layer of the bf16 model, batch 1, just after a 512-token prompt
        _layer_case(_7B, False, 1, 1, 527, "layer_bf16_decode"),
        # that 512-token prompt
        _layer_case(_7B, False, 1, 512, 0, "layer_bf16_prefill"),
        # one block of the diffusion transformer on a quarter of the benchmark's latent tokens
        {"name": "dit_block", "kind": "dit", "heads": 40, "ffn": 13824, "tokens": 8190, "text": 512},
        # a projection of the 7B decoder kept exponent-coded in HBM, rebuilt before it runs
        {"name": "hbm_unit_90mb", "kind": "hbm_unit", "nbytes": 90177536, "dense": True},
        # one 512 MiB chunk of small and large tensors placed in one launch
        {"name": "scatter_512mib", "kind": "scatter", "nbytes": 512 * MIB, "lo": 4096, "hi": 64 * MIB},
        # a whole call: one decode step of a six-layer model, four of whose layers stream from the host
        {"name": "streamed_decode", "kind": "streamed", "layers": 6, "resident": 2, "hidden": 2048, "heads": 16,
         "kv_heads": 16, "head_dim": 128, "inter": 5504, "vocab": 32000, "batch": 1, "pos": 100},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["linear_decode", "linear_decode", "linear_prefill", "layer_decode", "layer_decode",
                       "layer_prefill", "layer_prefill", "dit", "hbm_unit", "scatter", "streamed"])
    if kind == "linear_decode":  # up to 64 rows; k a multiple of 16, as the entry point asks
        return {"kind": "linear", "m": _log_int(rng, 1, 64), "n": _log_int(rng, 256, 28672),
                "k": 16 * _log_int(rng, 64, 1792)}
    if kind == "linear_prefill":
        n, k = _log_int(rng, 1024, 28672), 16 * _log_int(rng, 64, 1792)
        most = max(66, min(4096, int(3.0e11 / (2 * n * k))))
        return {"kind": "linear", "m": _log_int(rng, 65, most), "n": n, "k": k}
    if kind.startswith("layer"):
        fp8 = rng.random() < 0.5
        shape = dict(_70B if fp8 else _7B)
        if rng.random() < 0.5:  # a smaller decoder of other proportions
            d = rng.choice([64, 128, 128])
            kv = rng.choice([2, 4, 8])
            heads = kv * rng.choice([1, 2, 4])
            shape = {"hidden": d * heads, "heads": heads, "kv_heads": kv, "head_dim": d,
                     "inter": 16 * rng.randint(4 * heads * d // 32, 7 * heads * d // 32)}
        if kind == "layer_decode":
            return _layer_case(shape, fp8, _log_int(rng, 1, 32), 1, _log_int(rng, 8, 2047))
        tokens = _log_int(rng, 4, 768)
        batch = rng.choice([1, 1, 2, 4, 8])
        pos = 0 if rng.random() < 0.7 else _log_int(rng, 1, 512)  # a prompt, or one that continues a context
        while batch > 1 and batch * tokens > 768:
            batch //= 2
        return _layer_case(shape, fp8, batch, tokens, pos)
    if kind == "dit":
        heads = rng.randint(4, 40)
        return {"kind": "dit", "heads": heads, "ffn": 16 * rng.randint(16 * heads, 24 * heads),
                "tokens": _log_int(rng, 64, 8190), "text": _log_int(rng, 16, 512)}
    if kind == "hbm_unit":
        return {"kind": "hbm_unit", "nbytes": _log_int(rng, MIB, 400 * MIB), "dense": rng.random() < 0.75}
    if kind == "scatter":
        hi = _log_int(rng, 64 << 10, 64 * MIB)
        return {"kind": "scatter", "nbytes": _log_int(rng, 8 * MIB, 512 * MIB), "lo": 512, "hi": hi}
    heads = rng.choice([4, 8, 16])
    return {"kind": "streamed", "layers": rng.randint(4, 6), "resident": rng.randint(1, 3), "hidden": 128 * heads,
            "heads": heads, "kv_heads": heads // rng.choice([1, 2, 4]), "head_dim": 128,
            "inter": 128 * heads * 43 // 16, "vocab": rng.choice([1000, 32000]), "batch": rng.choice([1, 2, 4]),
            "pos": rng.randint(8, 200)}


# ---- inputs -----------------------------------------------------------------------------------------


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(gen: torch.Generator, *shape: int) -> torch.Tensor:
    return torch.randn(*shape, device=DEV, generator=gen).to(torch.bfloat16)


def _linear_inputs(c: dict, seed: int):
    """Activations of unit size, and a weight N(0, 0.02) in e4m3 with one bf16 scale per output channel."""
    gen = _gen(seed)
    x = _randn(gen, c["m"], c["k"])
    w = torch.randn(c["n"], c["k"], device=DEV, generator=gen).mul_(0.02)
    scale = (w.abs().amax(dim=1) / W.FP8_E4M3_MAX).clamp_min(1e-12).to(torch.bfloat16)
    return x, (w / scale.float()[:, None]).to(torch.float8_e4m3fn), scale


def _llama_shape(c: dict, n_layers: int, max_seq: int, vocab: int = 64) -> W.LlamaShape:
    return W.LlamaShape(n_layers=n_layers, hidden=c["hidden"], n_heads=c["heads"], n_kv_heads=c["kv_heads"],
                        head_dim=c["head_dim"], inter=c["inter"], vocab=vocab, max_seq=max_seq,
                        fp8=bool(c.get("fp8", False)))


def _norms_near_one(module: torch.nn.Module, gen: torch.Generator) -> None:
    """Norm weights around one: with the projections' N(0, 0.02) the attention then sees scores of unit size."""
    for mod in module.modules():
        if isinstance(mod, W.RMSNorm):
            p = mod.weight
            p.copy_((1 + 0.1 * torch.randn(p.shape, device=gen.device, generator=gen)).to(p.dtype))


def _rope(head_dim: int, n: int, dtype: torch.dtype):
    inv = 1.0 / (10000.0 ** (torch.arange(0, head_dim, 2, dtype=dtype, device=DEV) / head_dim))
    ang = torch.outer(torch.arange(n, dtype=dtype, device=DEV), inv)
    return torch.cat([ang.cos(), ang.cos()], -1), torch.cat([ang.sin(), ang.sin()], -1)


def _layer_state(c: dict, seed: int) -> dict:
    gen = _gen(seed)
    total = c["pos"] + c["tokens"]
    s = _llama_shape(c, 1, total)
    with torch.device("meta"):
        layer = W.DecoderLayer(s, torch.bfloat16)
    layer = layer.to_empty(device=DEV)
    with torch.no_grad():
        W.init_normal_(layer, seed, 0.02, init_device=DEV)
        _norms_near_one(layer, gen)
    cos, sin = _rope(c["head_dim"], total, torch.float32)
    shape = (c["batch"], total + 3, c["kv_heads"], c["head_dim"])
    cache_k, cache_v = (torch.zeros(shape, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    cache_k[:, : c["pos"]] = _randn(gen, c["batch"], c["pos"], c["kv_heads"], c["head_dim"])
    cache_v[:, : c["pos"]] = _randn(gen, c["batch"], c["pos"], c["kv_heads"], c["head_dim"])
    x = _randn(gen, c["batch"], c["tokens"], c["hidden"])
    return {"layer": layer, "x": x, "cos": cos, "sin": sin, "k": cache_k, "v": cache_v, "pos": c["pos"]}


def _dit_shape(c: dict) -> W.DiTShape:
    return W.DiTShape(n_blocks=1, dim=128 * c["heads"], n_heads=c["heads"], ffn=c["ffn"])


def _dit_state(c: dict, seed: int) -> dict:
    s = _dit_shape(c)
    with torch.device("meta"):
        block = W.DiTBlock(s, torch.bfloat16)
    block = block.to_empty(device=DEV)
    gen = _gen(seed)
    with torch.no_grad():
        W.init_normal_(block, seed, 0.02, init_device=DEV)
        _norms_near_one(block, gen)
        w = block.norm3.weight
        w.copy_((1 + 0.1 * torch.randn(w.shape, device=DEV, generator=gen)).to(w.dtype))
    x, e, ctx = W.dit_inputs(s, c["tokens"], c["text"], seed=seed, device=DEV)
    return {"block": block, "x": x, "e": e, "ctx": ctx}


def _scatter_state(c: dict, seed: int) -> dict:
    """A chunk of tensors with log-uniform byte sizes, 128-byte aligned in the chunk as the packer lays them,
    and their destinations, each at its own 512-byte aligned address as an allocator gives it. The table is
    the configuration's, not the seed's; the seed makes the bytes."""
    sizes, used = [], 0
    for n in W.scatter_sizes(100000, c["lo"], c["hi"], seed=1):
        n = min(n, c["nbytes"] - used)
        if n <= 0:
            break
        sizes.append(n)
        used += -(-n // 128) * 128
    src = dst = 0
    table = []
    for n in sizes:
        table.append((src, dst, n))
        src += -(-n // 128) * 128
        dst += -(-n // 512) * 512
    chunk = torch.randint(0, 256, (c["nbytes"],), dtype=torch.uint8, device=DEV, generator=_gen(seed))
    out = torch.zeros(dst, dtype=torch.uint8, device=DEV)
    plan = ScatterPlan([(s, out.data_ptr() + d, n) for s, d, n in table])
    return {"chunk": chunk, "out": out, "plan": plan, "payload": sum(sizes)}


class _Streamed:
    """A model under an offload manager past its discovery and profiling passes; released with the object."""

    def __init__(self, c: dict, seed: int) -> None:
        self.shape = s = _llama_shape(c, c["layers"], c["pos"] + 2, c["vocab"])
        self.model = W.build_llama(s, seed=seed, init_device=DEV)
        gen = _gen(seed)
        with torch.no_grad():
            _norms_near_one(self.model, torch.Generator().manual_seed(seed))
        params = sum(p.numel() * p.element_size() for p in self.model.parameters())
        streamed = c["layers"] - c["resident"]
        # room for everything but the streamed layers, plus the two ring slots, which hold a layer each
        budget = params - streamed * s.layer_bytes() + 2 * s.layer_bytes() + 8 * MIB
        self.mgr = OffloadManager(f"cases-{id(self)}")
        self.mgr.offload(self.model, OffloadConfig(include_patterns=["layers.*"], num_blocks=2, min_blocks=2,
                                                   discovery_iters=1, profiling_iters=1, max_gpu_mem_bytes=budget))
        self.tokens = torch.randint(0, c["vocab"], (c["batch"], 1), device=DEV, generator=gen)
        self.pos = c["pos"]
        with torch.no_grad():
            self.model.init_cache(c["batch"], c["pos"] + 2, torch.device(DEV))
            for k in range(2):  # discovery, then profiling: the plan and the loader are built at its end
                self.model(self.tokens, k)
        for cache in (*self.model.cache_k, *self.model.cache_v):
            cache.zero_()
            cache[:, : c["pos"]] = _randn(gen, c["batch"], c["pos"], c["kv_heads"], c["head_dim"])

    def __del__(self) -> None:
        mgr = getattr(self, "mgr", None)
        if mgr is not None:
            mgr.release(preserve_model=False)


def prepare(case: dict, seed: int):
    kind = case["kind"]
    if kind == "linear":
        x, w, scale = _linear_inputs(case, seed)
        return {"kind": kind, "x": x, "w": w, "scale": scale}
    if kind == "layer":
        return {"kind": kind, **_layer_state(case, seed)}
    if kind == "dit":
        return {"kind": kind, **_dit_state(case, seed)}
    if kind == "hbm_unit":  # weights N(0, 0.02) in bf16, an odd last byte included
        n = case["nbytes"]
        raw = (torch.randn(n // 2 + 1, device=DEV, generator=_gen(seed)) * 0.02).to(torch.bfloat16)
        raw = raw.view(torch.uint8)[:n].cpu()
        capacity = expcode.encoded_size(raw, case["dense"]) + max(64 << 10, n // 1000)
        block = expcode.DeviceEncodedBlock.from_raw(raw, capacity, torch.device(DEV, torch.cuda.current_device()),
                                                    dense=case["dense"])
        return {"kind": kind, "block": block, "dst": torch.empty(n, dtype=torch.uint8, device=DEV)}
    if kind == "scatter":
        return {"kind": kind, **_scatter_state(case, seed)}
    return {"kind": kind, "streamed": _Streamed(case, seed)}


@torch.no_grad()
def run(state):
    kind = state["kind"]
    if kind == "linear":
        return hip.fp8_linear(state["x"], state["w"], state["scale"])
    if kind == "layer":
        y = state["layer"](state["x"], state["pos"], state["cos"], state["sin"], state["k"], state["v"])
        return {"y": y, "cache_k": state["k"], "cache_v": state["v"]}
    if kind == "dit":
        return state["block"](state["x"], state["e"], state["ctx"])
    if kind == "hbm_unit":
        state["block"].decode(state["dst"])
        return state["dst"]
    if kind == "scatter":
        state["plan"].run(state["chunk"])
        return state["out"]
    s = state["streamed"]
    logits = s.model(s.tokens, s.pos)
    return {"logits": logits, "cache_k": list(s.model.cache_k), "cache_v": list(s.model.cache_v)}


# ---- what a pass cannot do without ------------------------------------------------------------------


def _layer_work(c: dict) -> tuple[float, float]:
    h, d, f = c["hidden"], c["head_dim"], c["inter"]
    q, kv = c["heads"] * d, c["kv_heads"] * d
    params = h * (q + 2 * kv) + q * h + 3 * h * f
    rows = c["batch"] * c.get("tokens", 1)
    t, pos = c.get("tokens", 1), c["pos"]
    keys = t * pos + t * (t + 1) // 2  # query-key pairs of one sequence
    weight_bytes = params + 2 * (q + 2 * kv + 2 * h + 2 * f) if c.get("fp8") else 2 * params
    nbytes = weight_bytes + 4 * h + 4 * rows * h + 4 * c["batch"] * (pos + 2 * t) * kv
    return float(nbytes), float(2 * params * rows + 4 * c["batch"] * q * keys)


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": float(n * k + 2 * m * k + 2 * m * n + 2 * n), "flops": 2.0 * m * n * k}
    if kind == "layer":
        b, f = _layer_work(case)
        return {"bytes": b, "flops": f}
    if kind == "dit":
        s = _dit_shape(case)
        return {"bytes": float(2 * s.block_params() + 4 * case["tokens"] * s.dim + 2 * case["text"] * s.dim),
                "flops": s.block_flops(case["tokens"], case["text"])}
    if kind == "hbm_unit":  # the encoded bytes (0.697 and 0.752 of bf16 weights) read, the raw bytes written
        return {"bytes": case["nbytes"] * (1.697 if case["dense"] else 1.752), "flops": 0.0}
    if kind == "scatter":
        return {"bytes": 2.0 * case["nbytes"], "flops": 0.0}
    b, f = _layer_work(case)
    head = 2 * case["vocab"] * case["hidden"]
    return {"bytes": case["layers"] * b + head, "flops": case["layers"] * f + head * case["batch"]}


def tolerance(case: dict):
    kind = case["kind"]
    if kind in ("hbm_unit", "scatter"):
        return "exact"  # bytes
    # Four times what was seen between this path and the same mathematics with its sums in another order (a
    # 32-bit matrix product, and attention with its scores kept in 32 bits, each rounded to bf16 once).
    if kind == "linear":  # 6.4e-5 seen: 32-bit sums that fall on the two sides of a bf16 rounding
        return {"rel": 3e-4, "max": 0.04}
    if kind == "layer":  # 4e-3 to 1.1e-2 seen: roundings of the scores and of every projection
        return {"rel": 0.025, "max": 0.4}
    if kind == "dit":  # 3.3e-3 seen
        return {"rel": 0.013, "max": 0.15}
    return {"rel": 0.03, "max": 0.4}  # 2.1e-2 seen: a rounding in one layer goes through all that follow


# ---- the same results in 64 bits, by plain torch ------------------------------------------------------


def _weight64(mod: torch.nn.Module) -> torch.Tensor:
    w = mod.weight.detach().to(DEV)
    return w.to(torch.float64) * mod.scale.detach().to(DEV).double()[:, None] if hasattr(mod, "scale") else w.double()


def _lin64(x: torch.Tensor, mod: torch.nn.Module) -> torch.Tensor:
    y = x @ _weight64(mod).t()
    bias = getattr(mod, "bias", None)
    return y if bias is None else y + bias.detach().to(DEV).double()


def _rms64(x: torch.Tensor, mod: torch.nn.Module) -> torch.Tensor:
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + mod.eps) * mod.weight.detach().to(DEV).double()


def _attend64(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, pos: int | None) -> torch.Tensor:
    """[b, t, h, d] queries over [b, s, kv, d] keys, head by head; causal from ``pos`` when given."""
    b, t, h, d = q.shape
    rep = h // k.shape[2]
    out = torch.empty_like(q)
    mask = None
    if pos is not None and t > 1:
        mask = torch.ones(t, k.shape[1], dtype=torch.bool, device=q.device).triu(diagonal=pos + 1)
    for i in range(b):
        for j in range(h):
            s = (q[i, :, j] @ k[i, :, j // rep].t().contiguous()) / math.sqrt(d)
            if mask is not None:
                s = s.masked_fill(mask, float("-inf"))
            out[i, :, j] = torch.softmax(s, -1) @ v[i, :, j // rep].contiguous()
    return out


def _layer64(layer: torch.nn.Module, s: W.LlamaShape, x, pos: int, cos, sin, cache_k, cache_v):
    """The layer's output and its caches after the call, all in 64 bits."""
    b, t, _ = x.shape

    def rotate(u):
        half = s.head_dim // 2
        c, sn = cos[pos: pos + t].view(1, t, 1, -1), sin[pos: pos + t].view(1, t, 1, -1)
        return u * c + torch.cat((-u[..., half:], u[..., :half]), -1) * sn

    a = layer.attn
    h = _rms64(x, layer.attn_norm)
    q = rotate(_lin64(h, a.wq).view(b, t, s.n_heads, s.head_dim))
    k = rotate(_lin64(h, a.wk).view(b, t, s.n_kv_heads, s.head_dim))
    v = _lin64(h, a.wv).view(b, t, s.n_kv_heads, s.head_dim)
    cache_k, cache_v = cache_k.double(), cache_v.double()
    cache_k[:b, pos: pos + t], cache_v[:b, pos: pos + t] = k, v
    o = _attend64(q, cache_k[:b, : pos + t], cache_v[:b, : pos + t], pos)
    x = x + _lin64(o.reshape(b, t, -1), a.wo)
    h = _rms64(x, layer.mlp_norm)
    g, u = _lin64(h, layer.gate), _lin64(h, layer.up)
    return x + _lin64(g * torch.sigmoid(g) * u, layer.down), cache_k, cache_v


def _dit64(block: torch.nn.Module, x, e, ctx):
    def norm(u, eps):
        u = u - u.mean(-1, keepdim=True)
        return u * torch.rsqrt(u.pow(2).mean(-1, keepdim=True) + eps)

    def attend(att, u, c):
        n, heads, d = u.shape[1], att.s.n_heads, att.s.head_dim
        q = _rms64(_lin64(u, att.q), att.norm_q).view(1, n, heads, d)
        k = _rms64(_lin64(c, att.k), att.norm_k).view(1, c.shape[1], heads, d)
        v = _lin64(c, att.v).view(1, c.shape[1], heads, d)
        return _lin64(_attend64(q, k, v, None).reshape(1, n, heads * d), att.o)

    x, e, ctx = x.double(), e.double(), ctx.double()
    m = (block.modulation.detach().double() + e).chunk(6, dim=1)
    h = norm(x, block.s.eps) * (1 + m[1]) + m[0]
    x = x + attend(block.self_attn, h, h) * m[2]
    w, b = block.norm3.weight.detach().double(), block.norm3.bias.detach().double()
    x = x + attend(block.cross_attn, norm(x, block.norm3.eps) * w + b, ctx)
    h = norm(x, block.s.eps) * (1 + m[4]) + m[3]
    y = _lin64(torch.nn.functional.gelu(_lin64(h, block.fc1), approximate="tanh"), block.fc2)
    return x + y * m[5]


@torch.no_grad()
def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "linear":
        x, w, scale = _linear_inputs(case, seed)
        return x.double() @ (w.double() * scale.double()[:, None]).t()
    if kind == "layer":
        st = _layer_state(case, seed)
        cos, sin = _rope(case["head_dim"], case["pos"] + case["tokens"], torch.float64)
        y, k, v = _layer64(st["layer"], st["layer"].attn.s, st["x"].double(), case["pos"], cos, sin, st["k"], st["v"])
        return {"y": y, "cache_k": k, "cache_v": v}
    if kind == "dit":
        st = _dit_state(case, seed)
        return _dit64(st["block"], st["x"], st["e"], st["ctx"])
    if kind == "streamed":
        st = _Streamed(case, seed)
        model, pos = st.model, st.pos
        caches = [(k.clone(), v.clone()) for k, v in zip(model.cache_k, model.cache_v)]
        st.mgr.release()  # the model again, whole, in host memory or on the GPU
        cos, sin = _rope(case["head_dim"], pos + 1, torch.float64)
        x = model.embed.weight.detach().to(DEV)[st.tokens].double()
        keys, vals = [], []
        for layer, (k, v) in zip(model.layers, caches):
            x, k, v = _layer64(layer, st.shape, x, pos, cos, sin, k, v)
            keys.append(k)
            vals.append(v)
        return {"logits": _lin64(_rms64(x[:, -1:], model.norm), model.lm_head), "cache_k": keys, "cache_v": vals}
    return None  # bytes
