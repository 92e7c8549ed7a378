"""The attention, norm, rotary and SwiGLU kernels against float64 restatements of the same operations.

Tolerances are relative 2-norms of bf16 roundings: bf16 has eight significant bits, so a value rounded once (half a
unit in the last place) is off by at most 2^-8 of itself, and an output whose last product's inputs were rounded as
well (attention's probabilities) by at most 2^-7.
"""

from __future__ import annotations

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

ONE_ROUNDING = 2.0 ** -8
TWO_ROUNDINGS = 2.0 ** -7


def _rel(got: torch.Tensor, want: torch.Tensor) -> float:
    return float((got.double() - want).norm() / want.norm())


def _randn(gpu, *shape: int, seed: int = 0) -> torch.Tensor:
    gen = torch.Generator(device=gpu).manual_seed(seed + sum(shape))
    return torch.randn(*shape, device=gpu, generator=gen).to(torch.bfloat16)


def _attend64(q, k, v, pos):
    b, t, h, d = q.shape
    rep = h // k.shape[2]
    q, k, v = (x.double().cpu() for x in (q, k, v))
    out = torch.empty_like(q)
    mask = torch.ones(t, k.shape[1], dtype=torch.bool).triu(pos + 1) if pos is not None else None
    for i in range(b):
        for j in range(h):
            s = q[i, :, j] @ k[i, :, j // rep].t() / math.sqrt(d)
            if mask is not None:
                s = s.masked_fill(mask, float("-inf"))
            out[i, :, j] = torch.softmax(s, -1) @ v[i, :, j // rep]
    return out


# batch, queries, keys, heads, kv heads, d, position of the first query (None: every key is seen).
_ATTENTION = [
    (1, 1, 1, 1, 1, 128, 0), (2, 1, 31, 4, 4, 64, 30), (1, 1, 528, 32, 32, 128, 527), (8, 1, 1024, 64, 8, 128, 1023),
    (3, 1, 97, 10, 2, 128, 96), (1, 2, 65, 8, 1, 64, 63),  # one wave, split over the keys or not
    (1, 7, 200, 8, 2, 128, 193), (1, 33, 33, 2, 2, 128, 0), (1, 100, 612, 8, 8, 64, 512),  # splits of causal rows
    (2, 64, 64, 256, 32, 128, 0), (4, 40, 40, 64, 64, 64, 0), (4, 127, 127, 64, 64, 128, 0),  # 2 and 4 waves
    (1, 257, 257, 128, 64, 128, 0), (1, 300, 301, 128, 128, 64, 1), (1, 512, 512, 128, 128, 128, 0),  # 8 waves
    (1, 64, 16, 4, 4, 128, None), (1, 200, 77, 40, 40, 128, None), (2, 520, 129, 64, 64, 64, None),
    (1, 1030, 1027, 64, 64, 128, None),
]


@pytest.mark.parametrize("b,t,s,h,kv,d,pos", _ATTENTION)
def test_attention_matches_float64(gpu, b, t, s, h, kv, d, pos):
    """Queries, a longer KV cache and a head-major layout are read in place; the keys past the last one hold
    infinities, which must not reach the result."""
    from flextensor_amd import hip

    print(f"attention b={b} t={t} s={s} h={h}/{kv} d={d} pos={pos}", flush=True)
    q = _randn(gpu, b, t, h, d)
    cache_k, cache_v = _randn(gpu, b, s + 5, kv, d, seed=1), _randn(gpu, b, s + 5, kv, d, seed=2)
    cache_k[:, s:], cache_v[:, s:] = float("inf"), float("inf")
    k, v = cache_k[:, :s], cache_v[:, :s]
    want = _attend64(q, k, v, pos)
    assert hip.attention_eligible(q, k, v)
    got = hip.attention(q, k, v, pos)
    assert got.is_contiguous() and _rel(got.cpu(), want) < TWO_ROUNDINGS
    head_major = [x.transpose(1, 2).contiguous().transpose(1, 2) for x in (q, k, v)]
    got = hip.attention(*head_major, pos)
    assert got.stride() == head_major[0].stride() and _rel(got.cpu(), want) < TWO_ROUNDINGS


def test_attention_with_large_scores_and_rising_maxima(gpu):
    """Keys that grow along the sequence raise the maximum at every tile; scores reach the hundreds."""
    from flextensor_amd import hip

    q, k, v = (_randn(gpu, 1, 300, 4, 128, seed=i) for i in range(3))
    k = (k.float() * torch.linspace(0.1, 12.0, 300, device=gpu).view(1, -1, 1, 1)).to(torch.bfloat16)
    for pos in (None, 0):
        assert _rel(hip.attention(q, k, v, pos).cpu(), _attend64(q, k, v, pos)) < TWO_ROUNDINGS


def test_attention_passes_nan_and_infinite_scores_on(gpu):
    """A NaN query row gives NaN in its row only, as softmax does; other rows are untouched."""
    from flextensor_amd import hip

    q, k, v = (_randn(gpu, 1, 40, 2, 128, seed=i) for i in range(3))
    clean = hip.attention(q, k, v)
    q[0, 5, 1] = float("nan")
    got = hip.attention(q, k, v)
    assert bool(got[0, 5, 1].isnan().all())
    got[0, 5, 1] = clean[0, 5, 1]
    assert torch.equal(got, clean)
    k[0, 7, 0] = float("inf")  # scores of both signs: infinite, so NaN or a weight of one or zero, as in torch
    s = torch.softmax((q[0, :, 0].double() @ k[0, :, 0].double().t()), -1)
    assert torch.equal(hip.attention(q, k, v)[0, :, 0].isnan().all(-1), s.isnan().any(-1))


@pytest.mark.parametrize("blank", [32, 64, 96])
@pytest.mark.parametrize("b,t,s,h,kv,d,pos", [
    (1, 1, 100, 4, 4, 128, None), (1, 3, 528, 2, 1, 64, 525),  # one wave: unsplit, split over the keys
    (2, 64, 128, 256, 32, 128, None), (4, 127, 127, 64, 64, 128, 0), (1, 257, 257, 128, 64, 64, 0),  # 2, 4, 8 waves
])
def test_attention_after_keys_that_all_score_minus_infinity(gpu, blank, b, t, s, h, kv, d, pos):
    """Whole tiles of -inf scores ahead of finite ones weigh nothing, on split and unsplit plans; a causal row that
    sees only such keys is NaN, as softmax gives."""
    from flextensor_amd import hip

    print(f"attention blank={blank} b={b} t={t} s={s} h={h}/{kv} d={d} pos={pos}", flush=True)
    q, k, v = _randn(gpu, b, t, h, d), _randn(gpu, b, s, kv, d, seed=1), _randn(gpu, b, s, kv, d, seed=2)
    q[..., 0] = q[..., 0].abs() + 1
    k[:, :blank, :, 0] = float("-inf")
    want, got = _attend64(q, k, v, pos), hip.attention(q, k, v, pos).cpu()
    nan = want.isnan()
    assert bool(nan.any()) == (pos == 0) and torch.equal(got.isnan(), nan)
    assert _rel(got[~nan], want[~nan]) < TWO_ROUNDINGS


@pytest.mark.parametrize("s,stride", [(1, 0), (1, 128), (5, 0), (33, 8), (40, 64), (600, 0)])
@pytest.mark.parametrize("t", [1, 70])
def test_attention_reads_no_value_past_the_last_key(gpu, s, stride, t):
    """Keys and values whose rows overlap (a single one, expanded ones, a stride below a row) and hold infinities:
    the rows that fill up the last tile stay out of the sum."""
    from flextensor_amd import hip

    print(f"attention s={s} stride={stride} t={t}", flush=True)
    q, k, v = _randn(gpu, 1, t, 2, 128), _randn(gpu, 2 * (s + 2) * 128, seed=1), _randn(gpu, 2 * (s + 2) * 128, seed=2)
    v[(s - 1) * stride + 127] = float("inf")  # the end of the last row: inside the rows that would follow it
    k, v = (x.as_strided((1, s, 2, 128), (0, stride, (s + 2) * 128, 1)) for x in (k, v))
    want, got = _attend64(q, k, v, None), hip.attention(q, k, v).cpu()
    inf = want.isinf()
    assert bool(inf.any()) and torch.equal(got.isinf(), inf) and not bool(got.isnan().any())
    assert _rel(got[~inf], want[~inf]) < TWO_ROUNDINGS


def test_attention_refuses_what_the_kernel_cannot_address(gpu):
    from flextensor_amd import _native as nat
    from flextensor_amd import hip

    q = _randn(gpu, 1, 8, 4, 128)
    assert not hip.attention_eligible(q, q[..., 1:], q[..., 1:])
    assert not hip.attention_eligible(q.float(), q.float(), q.float())
    assert not hip.attention_eligible(q[..., :96].contiguous(), q[..., :96].contiguous(), q[..., :96].contiguous())
    assert not hip.attention_eligible(q, q[:, :0], q[:, :0])
    shifted = torch.empty(q.numel() + 4, dtype=torch.bfloat16, device=gpu)[4:].view_as(q)
    assert not hip.attention_eligible(shifted, q, q)
    with pytest.raises(nat.FtxError, match="head dimensions"):
        hip.attention(*[q[..., :96].contiguous()] * 3)
    with pytest.raises(nat.FtxError, match="no keys"):
        hip.attention(q, q[:, :0], q[:, :0])


@pytest.mark.parametrize("rows", [1, 5, 513])
@pytest.mark.parametrize("dim", [8, 200, 2048, 2056, 5120, 8192, 8200, 32768])
def test_rms_norm_matches_float64(gpu, rows, dim):
    from flextensor_amd import workloads as W

    x, w = _randn(gpu, rows, dim), _randn(gpu, dim, seed=1)
    norm = W.RMSNorm(dim, 1e-5, torch.bfloat16).to(gpu)
    with torch.no_grad():
        norm.weight.copy_(w)
        got = norm(x)
    xd = x.double()
    want = xd * torch.rsqrt(xd.pow(2).mean(-1, keepdim=True) + 1e-5) * w.double()
    assert _rel(got, want) < ONE_ROUNDING


@pytest.mark.parametrize("b,n,dim", [(1, 1, 8), (2, 3, 512), (1, 9, 2056), (3, 5, 5120), (1, 2, 16384)])
@pytest.mark.parametrize("residual", ["none", "add", "gated"])
@pytest.mark.parametrize("norm", ["none", "affine", "adaln"])
def test_residual_norm_matches_float64(gpu, b, n, dim, residual, norm):
    """The sum rounds once; the norm of the sum as stored rounds once more."""
    from flextensor_amd import hip

    x, delta = _randn(gpu, b, n, dim) + 0.5, _randn(gpu, b, n, dim, seed=1)
    w, bias = _randn(gpu, dim, seed=2), _randn(gpu, dim, seed=3)
    mod, e = _randn(gpu, 1, 6, dim, seed=4), _randn(gpu, b, 6, dim, seed=5)
    total, y = hip.residual_norm(x, 1e-6, None if residual == "none" else delta, 2 if residual == "gated" else -1,
                                 (w, bias) if norm == "affine" else None, (mod, e),
                                 *((4, 3) if norm == "adaln" else ()))
    m = mod.double() + e.double()
    want = x.double()
    if residual != "none":
        want = want + delta.double() * (m[:, 2:3] if residual == "gated" else 1)
    assert _rel(total, want) < ONE_ROUNDING
    if norm == "none":
        assert y is None
        return
    u = total.double()
    u = u - u.mean(-1, keepdim=True)
    u = u * torch.rsqrt(u.pow(2).mean(-1, keepdim=True) + 1e-6)
    want = u * w.double() + bias.double() if norm == "affine" else u * (1 + m[:, 4:5]) + m[:, 3:4]
    assert _rel(y, want) < ONE_ROUNDING
    assert hip.residual_norm(x, 1e-6, delta[:, :, : dim // 2], adaln=(mod, e)) is None


@pytest.mark.parametrize("options", [{}, {"bias": False}, {"elementwise_affine": False}])
def test_dit_block_with_any_layer_norm(gpu, options):
    """A norm3 without a bias, or without weight and bias, runs as torch's module between the kernels."""
    from flextensor_amd import workloads as W

    s = W.DiTShape(n_blocks=1, dim=128, n_heads=2, ffn=256)
    block = W.build_dit(s, seed=3).blocks[0]
    block.norm3 = torch.nn.LayerNorm(s.dim, eps=s.eps, dtype=torch.bfloat16, **options)
    x, e, ctx = W.dit_inputs(s, 40, 8, seed=3)
    with torch.no_grad():
        for p in block.norm3.parameters():
            p.uniform_(0.5, 1.5)
        want = block.float()(x.float(), e.float(), ctx.float())
        got = block.to(gpu, torch.bfloat16)(x.to(gpu), e.to(gpu), ctx.to(gpu))
    assert _rel(got.cpu(), want.double()) < 1e-2  # a bf16 block


@pytest.mark.parametrize("dim,n", [(5120, 8000), (256, 40)])
def test_dit_block_has_the_same_bits_with_its_norm_called_as_a_module(gpu, dim, n):
    """A hook (as a streamed unit's trap does) makes the block call norm3 instead of folding it into the add."""
    from flextensor_amd import workloads as W

    s = W.DiTShape(n_blocks=1, dim=dim, n_heads=dim // 128, ffn=256)
    block = W.build_dit(s, seed=3).blocks[0].to(gpu)
    x, e, ctx = (t.to(gpu) for t in W.dit_inputs(s, n, 64, seed=3))
    with torch.no_grad():
        block.modulation.copy_(_randn(gpu, 1, 6, dim) * 0.3)
        block.norm3.weight.copy_(_randn(gpu, dim, seed=1) * 0.1 + 1)
        block.norm3.bias.copy_(_randn(gpu, dim, seed=2))
        want = block(x, e, ctx)
        seen = []
        block.norm3.register_forward_hook(lambda mod, args, out: seen.append(out))
        assert torch.equal(block(x, e, ctx), want) and len(seen) == 1


@pytest.mark.parametrize("b,t,h,kv,d,pos", [(1, 1, 1, 1, 16, 0), (2, 3, 8, 2, 64, 5), (1, 65, 5, 5, 128, 0), (3, 1, 64, 8, 128, 40)])
def test_rope_cache_matches_float64(gpu, b, t, h, kv, d, pos):
    """Rotated queries, and keys and values at their positions; the rest of the caches is left alone."""
    from flextensor_amd import hip

    q, k, v = _randn(gpu, b, t, h, d), _randn(gpu, b, t, kv, d, seed=1), _randn(gpu, b, t, kv, d, seed=2)
    ang = torch.rand(pos + t + 2, d, device=gpu, generator=torch.Generator(device=gpu).manual_seed(3)) * 6.3
    cos, sin = ang.cos(), ang.sin()
    ck, cv = torch.full((2, b + 1, pos + t + 3, kv, d), 7.0, dtype=torch.bfloat16, device=gpu)
    got = hip.rope_cache(q, k, v, cos, sin, pos, ck, cv)

    def rotate(x):
        x = x.double()
        half = d // 2
        c, s = (a[pos: pos + t].double().view(1, t, 1, d) for a in (cos, sin))
        return x * c + torch.cat((-x[..., half:], x[..., :half]), -1) * s

    assert _rel(got, rotate(q)) < ONE_ROUNDING
    assert _rel(ck[:b, pos: pos + t], rotate(k)) < ONE_ROUNDING
    assert torch.equal(cv[:b, pos: pos + t], v)
    for c in (ck, cv):
        assert bool((c[:b, :pos] == 7).all()) and bool((c[:b, pos + t:] == 7).all()) and bool((c[b:] == 7).all())
    assert hip.rope_cache(q, k, v, cos, sin, pos + 3, ck, cv) is None  # past the tables: torch raises for these
    assert hip.rope_cache(q, k, v, cos, sin, pos, ck[:, : pos], cv) is None


@pytest.mark.parametrize("n", [8, 2040, 2056, 1 << 20])
def test_silu_mul_matches_float64(gpu, n):
    from flextensor_amd import hip

    g, u = _randn(gpu, n), _randn(gpu, n, seed=1)
    gd = g.double()
    want = (gd / (1 + torch.exp(-gd))).to(torch.bfloat16).double() * u.double()
    assert _rel(hip.silu_mul(g, u), want) < TWO_ROUNDINGS
    assert hip.silu_mul(g[1:], u[1:]) is None


def test_small_kernels_stay_off_the_cus_of_a_ring_copy(gpu):
    """Beside a copy that holds its 16 CUs, a silu_mul or rotary launch takes 11 us (2.1 and 2.6 alone); where their
    workgroups may share those CUs and queue behind the copy's host reads, 26."""
    from flextensor_amd import _native as nat
    from flextensor_amd import hip

    g, q, kv = _randn(gpu, 64, 5504), _randn(gpu, 1, 64, 32, 128), _randn(gpu, 1, 64, 32, 128, seed=1)
    table, caches = torch.ones(64, 128, device=gpu), [torch.empty_like(kv) for _ in range(2)]
    host = torch.empty(256 << 20, dtype=torch.uint8, pin_memory=True)
    dst, side, policy = torch.empty_like(host, device=gpu), torch.cuda.Stream(), nat.copy_policy(0, 2**63 - 1, 1, 16)
    for name, call in (("silu_mul", lambda: hip.silu_mul(g, g)),
                       ("rope_cache", lambda: hip.rope_cache(q, kv, kv, table, table, 0, *caches))):
        graph = torch.cuda.CUDAGraph()
        call()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
            for _ in range(50):
                call()
        best = {}
        for beside in (False, True) * 4:
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            if beside:
                nat.copy_h2d(dst.data_ptr(), host.data_ptr(), dst.numel(), nat.COPY_MODES["kernel"], side.cuda_stream,
                             policy)
            start.record()
            graph.replay()
            end.record()
            torch.cuda.synchronize()
            best[beside] = min(best.get(beside, math.inf), start.elapsed_time(end) * 20)
        print(f"{name}: {best[False]:.2f} us alone, {best[True]:.2f} beside the copy", flush=True)
        assert best[True] < best[False] + 16
        del graph


@pytest.mark.parametrize("m", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("ns,k", [((1,), 8), ((17, 16), 120), ((15, 300, 64), 136), ((257,), 2056), ((4096,), 1024)])
def test_bf16_linear_matches_float64(gpu, m, ns, k):
    """One launch for a group; each output has the same bits alone (the sum's order depends on k only), also under
    the residual epilogue; SwiGLU rounds where the separate operations round."""
    from flextensor_amd import _native as nat
    from flextensor_amd import hip

    x = _randn(gpu, m, k)
    ws = [_randn(gpu, n, k, seed=i + 1) for i, n in enumerate(ns)]
    assert hip.bf16_linear_eligible(x, *ws)
    got = hip.bf16_linear(x, ws)
    for y, w in zip(got, ws):
        assert _rel(y, x.double() @ w.double().t()) < ONE_ROUNDING
        assert torch.equal(hip.bf16_linear(x, [w])[0], y)
        r = _randn(gpu, m, w.shape[0], seed=9)
        assert torch.equal(hip.bf16_linear(x, [w], nat.FP8_EPILOGUE_RESIDUAL, r)[0], r + y)
    up = _randn(gpu, ns[0], k, seed=7)
    act = hip.bf16_linear(x, [ws[0], up], nat.FP8_EPILOGUE_SWIGLU)[0]
    g, u = got[0].double(), hip.bf16_linear(x, [up])[0].double()
    assert _rel(act, (g / (1 + torch.exp(-g))).to(torch.bfloat16).double() * u) < TWO_ROUNDINGS


def test_bf16_linear_takes_decode_batches_of_plain_modules_only(gpu):
    from flextensor_amd import _native as nat
    from flextensor_amd import hip
    from flextensor_amd import workloads as W

    x, w = _randn(gpu, 16, 64), _randn(gpu, 32, 64)
    assert not hip.bf16_linear_eligible(_randn(gpu, 17, 64), w)
    assert not hip.bf16_linear_eligible(x[:, :60].contiguous(), w[:, :60].contiguous())
    assert not hip.bf16_linear_eligible(x, w[:, :60].contiguous())
    assert not hip.bf16_linear_eligible(x, _randn(gpu, 64, 64)[:, ::2])
    assert not hip.bf16_linear_eligible(x.float(), w)
    with pytest.raises(nat.FtxError, match="up to 16 rows"):
        hip.bf16_linear(_randn(gpu, 17, 64), [w])
    lin = W.Linear(64, 32, bias=False, dtype=torch.bfloat16).to(gpu)
    seen = []
    with torch.no_grad():
        alone = lin(x)
        assert torch.equal(W.linear_group(x, [lin])[0], alone)
        handle = lin.register_forward_hook(lambda mod, args, out: seen.append(out))
        assert W.linear_group(x, [lin]) is None and W.linear_residual(x, lin, alone) is None
        assert torch.equal(lin(x), alone) and len(seen) == 1
        handle.remove()
    y = lin(x)  # with autograd, torch's linear
    assert y.requires_grad and _rel(y.detach(), alone.double()) < TWO_ROUNDINGS


def test_public_kernel_functions_refuse_what_has_no_answer(gpu):
    """Host operands, layouts that cannot be read in place and calls that ask for a derivative are refused; the same
    call on plain operands runs."""
    import torch.autograd.forward_ad as fwd

    from flextensor_amd import hip

    q, x, w = _randn(gpu, 1, 8, 4, 128), _randn(gpu, 4, 64), _randn(gpu, 32, 64)
    hip.attention(q, q, q)
    hip.bf16_linear(x, [w])
    shifted = torch.empty(q.numel() + 4, dtype=torch.bfloat16, device=gpu)[4:].view_as(q)
    for args in ((q, q.cpu(), q.cpu()), (shifted, q, q), (q, shifted, q),
                 (q, q, q.transpose(2, 3).contiguous().transpose(2, 3))):
        with pytest.raises(ValueError):
            hip.attention(*args)
    for args in ((x, [w.cpu()]), (x[:, ::2], [w[:, :32].contiguous()]), (x, [w[:, :32].contiguous()]),
                 (x.view(-1)[1:65], [w])):
        with pytest.raises(ValueError):
            hip.bf16_linear(*args)
    for call in (lambda t: hip.attention(t(q), q, q), lambda t: hip.bf16_linear(x, [t(w)])):
        with pytest.raises(ValueError, match="no backward"):
            call(lambda a: a.clone().requires_grad_())
        with fwd.dual_level(), pytest.raises(ValueError, match="forward-mode"):
            call(lambda a: fwd.make_dual(a, torch.ones_like(a)))
        with torch.no_grad():
            call(lambda a: a.clone().requires_grad_())


def test_operations_that_must_be_seen_run_in_torch(gpu):
    """Autograd, forward-mode differentiation, function and dispatch modes, functorch transforms and autocast get
    torch's operations; a plain call gets the kernel."""
    import torch.autograd.forward_ad as fwd
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    from flextensor_amd import hip
    from flextensor_amd import workloads as W

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    norm = W.RMSNorm(64, 1e-5, torch.bfloat16).to(gpu)
    x = _randn(gpu, 4, 64)
    with torch.no_grad():
        assert hip.rms_norm(x, norm.weight, 1e-5) is not None
        for mode in (Function(), Dispatch(), torch.autocast("cuda", dtype=torch.bfloat16)):
            with mode:
                assert hip.rms_norm(x, norm.weight, 1e-5) is None
        with fwd.dual_level():
            dual = fwd.make_dual(x, torch.ones_like(x))
            assert fwd.unpack_dual(norm(dual)).tangent is not None
        assert torch.func.vmap(norm)(x.view(2, 2, 64)).shape == (2, 2, 64)
    assert hip.rms_norm(x, norm.weight, 1e-5) is None
    y = norm(x.requires_grad_())
    y.float().sum().backward()
    assert x.grad is not None and norm.weight.grad is not None


def test_decoder_layer_kernels_against_torch_operations(gpu, monkeypatch):
    """A small decoder's prompt and a decode step, with the kernels and with each call refused, against each
    other and captured in a graph."""
    from flextensor_amd import hip
    from flextensor_amd import workloads as W

    s = W.LlamaShape(n_layers=2, hidden=256, n_heads=4, n_kv_heads=2, head_dim=64, inter=512, vocab=300, max_seq=64)
    model = W.build_llama(s, seed=1).to(gpu)
    prompt = W.prompt_tokens(3, 17, s.vocab, seed=1).to(gpu)
    tok = W.prompt_tokens(3, 1, s.vocab, seed=2).to(gpu)

    def passes():
        model.init_cache(3, 40, torch.device(gpu))
        with torch.no_grad():
            return [model(prompt, 0), model(tok, 17)], [c.clone() for c in model.cache_k]

    got, cache = passes()
    with monkeypatch.context() as m:
        m.setattr(hip, "kernel_call", lambda *ts: False)
        want, want_cache = passes()
    for a, b in zip(got + cache, want + want_cache):
        assert _rel(a, b.double()) < 2e-2  # two bf16 layers
    passes()
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.stream(side):
        model(tok, 17)
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            static = model(tok, 17)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(static, got[1])
    del graph
