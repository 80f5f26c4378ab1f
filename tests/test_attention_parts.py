"""Decode attention over four workgroups per head with the output projection
that combines their partials, against the one-workgroup attention followed by
dequant_matmul and against float64: positions at the edges of a step (32 at
head_dim 128, 64 at 64), parts that see no position, a cache longer than one
pass of the waves (1536 positions), positions outside the cache."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def _case(dev, H, KVH, D, L, N, seed, amp=1.0):
    from metal_native.decoder import DecoderConfig, QLinear, rope_tables

    cos, sin = rope_tables(DecoderConfig(heads=H, kv_heads=KVH, head_dim=D, max_len=L), dev)
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    kc = torch.randn((KVH, L, D), device=dev, generator=g).half() * amp
    vc = torch.randn((KVH, L, D), device=dev, generator=g).half()
    qkv = torch.randn((1, (H + 2 * KVH) * D), device=dev, generator=g).half() * amp
    return cos, sin, kc, vc, qkv, QLinear.random(N, H * D, 128, g, dev)


@pytest.mark.parametrize("H,KVH,D,L,N", [(28, 4, 128, 576, 3584), (4, 2, 64, 513, 250), (8, 8, 64, 777, 768),
                                         (3, 1, 128, 257, 64), (16, 2, 128, 2100, 2048), (14, 2, 64, 4096, 896),
                                         (4, 2, 64, 512, 250), (3, 1, 128, 256, 64)])
@pytest.mark.parametrize("where", ["first", "step", "step+1", "last", "past", "before"])
def test_matches_one_workgroup_per_head(gpu, H, KVH, D, L, N, where):
    from metal_native import ops
    from metal_native import _lib

    step = 4096 // D
    pos = {"first": 0, "step": min(4 * step, L) - 1, "step+1": min(4 * step, L - 1), "last": L - 1, "past": L + 3,
           "before": -1}[where]
    cos, sin, kc, vc, qkv, o = _case(gpu, H, KVH, D, L, N, seed=L + D, amp=2.0)
    assert bool(_lib.lib.mq_attention_parts_supported(N, H, D, L, 128, 0)) == (L > 8 * step)
    p, scale = torch.tensor([pos], device=gpu), 1.0 / math.sqrt(D)
    k1, v1, k2, v2 = kc.clone(), vc.clone(), kc.clone(), vc.clone()
    a = ops.attention_decode_rope(qkv, cos, sin, p, k1, v1, H, KVH, D, scale)
    want = ops.dequant_matmul(a, *o.operands())
    got = ops.attention_decode_rope_linear(qkv, cos, sin, p, k2, v2, H, KVH, D, scale, *o.operands())
    assert torch.equal(k1, k2) and torch.equal(v1, v2)
    # The two attentions round to fp16 sums that differ in fp32 order only: at
    # most one fp16 step apart per element (2^-10 relative, 2^-24 below the
    # normals).  Through the product: that times |W|, the fp32 order of K
    # products, and one fp16 rounding of each result.
    W = ops.dequantize(*o.operands()).double().cpu()
    aw = a.double().abs().cpu()
    K = H * D
    bound = (aw * 2.0**-10 + 2.0**-24) @ W.abs().T + 2 * K * 2.0**-24 * (aw @ W.abs().T)
    bound = bound + 2.0**-10 * want.double().abs().cpu() + 2.0**-24
    assert bool(((got.double() - want.double()).abs().cpu() <= bound).all())


def _wider(t, by=16):
    big = torch.full((t.shape[0], t.shape[1] + by), 77, dtype=t.dtype, device=t.device)
    big[:, :t.shape[1]] = t
    return big[:, :t.shape[1]]


def _shifted(t):
    """The same matrix at an address that is not 16-byte aligned."""
    flat = torch.empty(t.numel() + 2, dtype=t.dtype, device=t.device)[2:]
    return flat.copy_(t.flatten()).view(t.shape)


@pytest.mark.parametrize("L", [576, 64])   # with and without the four-workgroup attention
@pytest.mark.parametrize("form", ["weights", "scales", "zeros", "columns strided", "weights shifted", "scales shifted",
                                  "rows expanded"])
def test_operands_of_every_layout(gpu, L, form):
    """Operands that are not contiguous or not aligned give what contiguous ones give."""
    from metal_native import ops

    H, KVH, D, N = 8, 2, 128, 640
    cos, sin, kc, vc, qkv, o = _case(gpu, H, KVH, D, L, N, seed=11)
    w, s, z, g, qt = o.operands()
    if form == "rows expanded":
        w, s, z = (t[:1].expand(t.shape) for t in (w, s, z))
    p, scale = torch.tensor([50], device=gpu), 1.0 / math.sqrt(D)
    a = ops.attention_decode_rope(qkv, cos, sin, p, kc, vc, H, KVH, D, scale)
    want = ops.attention_decode_rope_linear(qkv, cos, sin, p, kc, vc, H, KVH, D, scale, w.contiguous(), s.contiguous(),
                                            z.contiguous(), g, qt)
    # (the bound of two attentions that differ in fp32 order, in the loosest form that a wrong operand fails)
    assert float((want - ops.dequant_matmul(a, w, s, z, g, qt)).double().norm() / want.double().norm()) < 1e-2
    change = {"weights": (_wider, "w"), "scales": (_wider, "s"), "zeros": (_wider, "z"),
              "columns strided": (lambda t: torch.stack((t, t), -1)[..., 0], "wsz"), "weights shifted": (_shifted, "w"),
              "scales shifted": (_shifted, "sz"), "rows expanded": (lambda t: t, "")}[form]
    w, s, z = (change[0](t) if n in change[1] else t for n, t in zip("wsz", (w, s, z)))
    got = ops.attention_decode_rope_linear(qkv, cos, sin, p, kc, vc, H, KVH, D, scale, w, s, z, g, qt)
    if form in ("weights", "weights shifted"):   # the two calls, on another kernel: rows with gaps or not aligned
        assert torch.equal(got, ops.dequant_matmul(a, w, s, z, g, qt))
    else:
        assert torch.equal(got, want)


@pytest.mark.parametrize("L", [576, 64])
def test_refuses_what_dequant_matmul_refuses(gpu, L):
    import metal_native as mn
    from metal_native import ops

    H, KVH, D, N = 8, 2, 128, 640
    cos, sin, kc, vc, qkv, o = _case(gpu, H, KVH, D, L, N, seed=12)
    w, s, z, g, qt = o.operands()
    p = torch.tensor([50], device=gpu)
    before = kc.clone(), vc.clone()
    for args, match in [((w, s[:, 1:].contiguous(), z, g, qt), "scales must be"), ((w, s, z[:-1], g, qt), "zeros must be"),
                        ((w, s.float(), z, g, qt), "scales must be Float16"), ((w, s, None, g, qt), "zeros must be"),
                        ((w, s.cpu(), z, g, qt), "scales must be a GPU tensor"), ((w.half(), s, z, g, qt), "uint8"),
                        ((w[:, 1:], s, z, g, qt), "INT4 weights"), ((w, s, z, 48, qt), "group_size"),
                        ((w, s, z, g, "int8"), "INT8 weights"), ((w.flatten(), s, z, g, qt), "2D")]:
        with pytest.raises(mn.MetalNativeError, match=match):
            ops.attention_decode_rope_linear(qkv, cos, sin, p, kc, vc, H, KVH, D, 1.0, *args)
    assert torch.equal(kc, before[0]) and torch.equal(vc, before[1])


def test_error_against_float64_no_larger(gpu):
    """The error of the split attention + projection over the ranges of the
    decode step, against float64 from the same fp16 operands."""
    from metal_native import ops

    worst, total = [0.0, 0.0], [0.0, 0.0]
    shapes = [(28, 4, 128, 576, 512), (28, 4, 128, 576, 31), (28, 4, 128, 576, 575), (28, 4, 128, 4096, 4000),
              (14, 2, 64, 1024, 777), (14, 2, 64, 576, 100), (16, 2, 128, 2048, 1500), (32, 32, 128, 260, 200)]
    for seed, (H, KVH, D, L, pos) in enumerate(shapes):
        cos, sin, kc, vc, qkv, o = _case(gpu, H, KVH, D, L, H * D, seed)
        p, scale = torch.tensor([pos], device=gpu), 1.0 / math.sqrt(D)
        k0, v0 = kc.clone(), vc.clone()
        q = ops.rope_kv(qkv, cos, sin, p, k0, v0, H, KVH, D).double().cpu()
        k64 = k0.double().cpu()[:, : pos + 1].repeat_interleave(H // KVH, 0)
        v64 = v0.double().cpu()[:, : pos + 1].repeat_interleave(H // KVH, 0)
        w = torch.softmax((k64 * q[:, None, :]).sum(-1) * scale, -1)
        ref = (w[:, :, None] * v64).sum(1).reshape(1, -1) @ ops.dequantize(*o.operands()).double().cpu().T
        a = ops.attention_decode_rope(qkv, cos, sin, p, kc.clone(), vc.clone(), H, KVH, D, scale)
        one = ops.dequant_matmul(a, *o.operands())
        parts = ops.attention_decode_rope_linear(qkv, cos, sin, p, kc.clone(), vc.clone(), H, KVH, D, scale,
                                                 *o.operands())
        for i, y in enumerate((one, parts)):
            err = float((y.double().cpu() - ref).norm() / ref.norm())
            worst[i], total[i] = max(worst[i], err), total[i] + err
    print("relative error, one workgroup per head / four: worst", worst, "mean", [t / len(shapes) for t in total])
    # Both round the attention and the result to fp16 once, 2^-11 each; an
    # element of either may fall to the other side of a rounding, which moves
    # a norm over a thousand elements by well under a percent.
    assert worst[1] <= 2.0**-10 and worst[1] <= 1.01 * worst[0]


def test_fused_branch_runs_where_supported(gpu, monkeypatch):
    """The two-call form is not behind a supported shape's output."""
    from metal_native import ops

    H, KVH, D, L = 8, 2, 128, 576
    cos, sin, kc, vc, qkv, o = _case(gpu, H, KVH, D, L, 640, seed=6)
    args = (qkv, cos, sin, torch.tensor([500], device=gpu), kc, vc, H, KVH, D, 1.0 / math.sqrt(D))
    want = ops.dequant_matmul(ops.attention_decode_rope(*args), *o.operands())

    def refuse(*a, **k):
        raise AssertionError("the general branch ran")

    monkeypatch.setattr(ops, "attention_decode_rope", refuse)
    got = ops.attention_decode_rope_linear(*args, *o.operands())
    assert float((got - want).double().norm() / want.double().norm()) < 1e-3   # fp16 roundings, 2^-11 each
    with pytest.raises(AssertionError, match="general branch"):
        ops.attention_decode_rope_linear(*args, *o.operands(), bias=want[0])


def test_graph_replays(gpu):
    from metal_native import ops

    H, KVH, D, L = 28, 4, 128, 576
    cos, sin, kc, vc, qkv, o = _case(gpu, H, KVH, D, L, 3584, seed=5)
    p, scale = torch.tensor([40], device=gpu), 1.0 / math.sqrt(D)

    def run(k, v):
        return ops.attention_decode_rope_linear(qkv, cos, sin, p, k, v, H, KVH, D, scale, *o.operands())

    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    kg, vg = kc.clone(), vc.clone()
    with torch.cuda.stream(s):
        run(kg, vg)
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run(kg, vg)
    for pos in (40, 41, 200, 575):
        p.fill_(pos)
        want = run(kc, vc)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(kg, kc) and torch.equal(vg, vc)
