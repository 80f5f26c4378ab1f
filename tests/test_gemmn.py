"""The many-row prefill GEMM (mq_gemmn.hip) against the oracle: tile edges and
remainders, K tails, groups, epilogues, strided operands, K parts, special
scales, and the routing that chooses it."""

import numpy as np
import pytest
import torch

from oracle import mq_oracle as O

pytestmark = pytest.mark.gpu

TOL_ABS = 1e-2   # the contract's bound on a matmul output
TOL_REL = 1e-3


@pytest.fixture(scope="module")
def mn(gpu):
    import metal_native

    yield metal_native
    for key in ("force_path", "gemm_rows", "gemm_parts"):
        metal_native.set_option(key, 0)


def dev(x, gpu):
    return torch.from_numpy(np.ascontiguousarray(x)).to(gpu)


class forced:
    """The kernel with `rows` per tile and `parts` K parts, whatever the planner would take."""

    def __init__(self, mn, rows, parts):
        self.mn, self.opts = mn, {"force_path": 13, "gemm_rows": rows, "gemm_parts": parts}

    def __enter__(self):
        for k, v in self.opts.items():
            self.mn.set_option(k, v)

    def __exit__(self, *exc):
        for k in self.opts:
            self.mn.set_option(k, 0)


def problem(M, K, N, g, qt, seed):
    if qt == "int4":
        x, wp, s, z = O.make_int4_problem(M, K, N, g, seed=seed)
        return x, wp, s, z, g, O.matmul_f32acc(x, O.dequant_int4(wp, s, z, K, g))
    x, wp, s, z, g = O.make_int8_problem(M, K, N, seed=seed, g=g or None)
    z = np.random.default_rng(3).uniform(-0.01, 0.01, s.shape).astype(np.float16)
    return x, wp, s, z, g, O.matmul_f32acc(x, O.dequant_int8(wp, s, z, K, g))


def silu(v):
    with np.errstate(over="ignore"):
        return v / (1.0 + np.exp(-v))


def expected(acc, epi, bias, res):
    """(reference in float64, extra tolerance): SiLU's is its change across
    one fp16 (SwiGLU: of gate and up) or fp32 rounding of its argument."""
    v = acc.astype(np.float64)
    extra = 0.0
    if epi == "swiglu":
        F = v.shape[1] // 2
        gate, up = (v[:, i * F:(i + 1) * F].astype(np.float16).astype(np.float64) for i in range(2))
        ulp = np.spacing(np.maximum(np.abs(gate), np.abs(up)).astype(np.float16)).astype(np.float64)
        return silu(gate) * up, ulp * (1.1 * np.abs(up) + np.abs(silu(gate)) + 1.1 * ulp)
    if bias is not None:
        v = v + bias.astype(np.float64)[None, :]
    if res is not None:
        v = v + res.astype(np.float64)
    if epi == "bias_relu":
        v = np.maximum(v, 0.0)
    if epi == "bias_silu":
        v = silu(v)
    return v, extra


def check(y, acc, epi=None, bias=None, res=None, what=""):
    ref, extra = expected(acc, epi, bias, res)
    err = np.abs(y.astype(np.float64) - ref)
    bad = ~(err <= TOL_ABS + TOL_REL * np.abs(ref) + extra)
    assert not bad.any(), f"{what}: {bad.sum()} of {bad.size} outside tolerance; max abs err {np.nanmax(err):.3g}"


def epilogue_args(epi, M, N, gpu):
    rng = np.random.default_rng(M + N)
    if epi and epi.startswith("bias"):
        b = rng.standard_normal(N).astype(np.float16)
        return {"epilogue": epi, "bias": dev(b, gpu)}, b, None
    if epi == "residual":
        r = rng.standard_normal((M, N)).astype(np.float16)
        return {"epilogue": epi, "residual": dev(r, gpu)}, None, r
    return ({"epilogue": epi} if epi else {}), None, None


@pytest.mark.parametrize("rows", [64, 128, 256])
@pytest.mark.parametrize("parts", [1, 3])
@pytest.mark.parametrize("M,K,N,g,qt,epi", [
    (1, 64, 2, 32, "int4", None),              # one K-tile, one row
    (127, 256, 256, 64, "int4", "bias"),       # four K-tiles, last row short of a tile
    (129, 320, 257, 32, "int4", None),         # five K-tiles, odd N: 2-byte stores
    (257, 416, 520, 32, "int4", "residual"),   # K ends inside a K-tile
    (200, 896, 1030, 128, "int4", "bias_silu"),
    (64, 1184, 516, 32, "int4", "swiglu"),     # up rows of a partial tile; K tail
    (255, 384, 254, 0, "int8", None),          # per-channel
    (130, 160, 300, 32, "int8", "bias_relu"),
    (300, 512, 770, 64, "int8", "swiglu"),
    (31, 96, 96, 32, "int8", "residual"),
])
def test_against_oracle(mn, gpu, rows, parts, M, K, N, g, qt, epi):
    x, wp, s, z, g, acc = problem(M, K, N, g, qt, seed=M + K + N)
    kw, b, r = epilogue_args(epi, M, N, gpu)
    with forced(mn, rows, parts):
        run = lambda: mn.dequant_matmul(dev(x, gpu), dev(wp, gpu), dev(s, gpu), dev(z, gpu), g, qt, **kw)
        y = run()
        assert mn.last_path() == "gemmn"
        check(y.cpu().numpy(), acc, epi, b, r, f"rows={rows} parts={parts}")
        assert torch.equal(run(), y)   # a fixed summation order


@pytest.mark.parametrize("rows,parts", [(64, 1), (128, 1), (256, 1), (64, 2), (128, 2)])
@pytest.mark.parametrize("pad", [8, 3])
def test_strided_operands(mn, gpu, rows, parts, pad):
    """Activations, weights and output as column ranges of wider tensors, the
    residual in place: nothing is read or written outside them."""
    M, K, N, g = 150, 416, 266, 32
    x, wp, s, z, g, acc = problem(M, K, N, g, "int4", seed=9)
    xs = torch.full((M, K + 8), float("nan"), dtype=torch.float16, device=gpu)
    xs[:, :K] = dev(x, gpu)
    ws = torch.full((N, K // 2 + 16), 255, dtype=torch.uint8, device=gpu)
    ws[:, :K // 2] = dev(wp, gpu)
    big = torch.zeros((M, N + pad), dtype=torch.float16, device=gpu)
    r = np.random.default_rng(2).standard_normal((M, N)).astype(np.float16)
    out = big[:, :N]
    out.copy_(dev(r, gpu))
    with forced(mn, rows, parts):
        mn.dequant_matmul(xs[:, :K], ws[:, :K // 2], dev(s, gpu), dev(z, gpu), g, "int4", epilogue="residual",
                          residual=out, out=out)
        assert mn.last_path() == "gemmn"
    check(out.cpu().numpy(), acc, "residual", None, r, "strided")
    assert (big[:, N:] == 0).all()


# fp16 bit patterns: zero, subnormals, the ends of the normal scales that the
# four-operation dequant covers (exponents 1..16), their neighbours, large ones
SCALES = np.array([0x0000, 0x0001, 0x03FF, 0x0400, 0x0401, 0x1400, 0x2555, 0x3C00, 0x43FF, 0x4400, 0x5800, 0x6C00,
                   0x8400, 0xA4D3, 0xC3FF, 0xC400], dtype=np.uint16)
ZEROS = np.array([0x0000, 0x8000, 0x0001, 0x83FF, 0x2E66, 0xBC00, 0x5555, 0xE000], dtype=np.uint16)


@pytest.mark.parametrize("rows", [64, 128, 256])
@pytest.mark.parametrize("qt", ["int4", "int8"])
@pytest.mark.parametrize("mixed", [False, True])
def test_one_hot_selects_dequantized_weights(mn, gpu, rows, qt, mixed):
    """Every dequantized weight equals the oracle's two-rounding one (up to
    the sign of zero); `mixed`: scales outside the fast form's range among
    the others, else none."""
    rng = np.random.default_rng(5)
    N, K, g, M = 320, 1024, 32, 256
    pool = SCALES if mixed else SCALES[[3, 4, 5, 6, 7, 8, 12, 13, 14]]
    s = pool[rng.integers(0, len(pool), (N, K // g))].view(np.float16)
    if qt == "int8":   # keep the weights finite
        s = np.clip(s.astype(np.float32), -255.0, 255.0).astype(np.float16)
    if mixed:          # whole column blocks of both kinds, too
        s[32:96] = np.float16(0.0123)
    z = ZEROS[rng.integers(0, len(ZEROS), (N, K // g))].view(np.float16)
    if qt == "int4":
        wp = rng.integers(0, 256, (N, K // 2), dtype=np.uint8)
        want = O.dequant_int4(wp, s, z, K, g)
    else:
        wp = rng.integers(-127, 128, (N, K), dtype=np.int16).astype(np.int8)
        want = O.dequant_int8(wp, s, z, K, g)
    assert np.isfinite(want).all()
    order = rng.permutation(K)
    with forced(mn, rows, 1):
        for k0 in range(0, K, M):
            ks = order[k0:k0 + M]
            x = np.zeros((M, K), dtype=np.float16)
            x[np.arange(M), ks] = 1.0
            y = mn.dequant_matmul(dev(x, gpu), dev(wp, gpu), dev(s, gpu), dev(z, gpu), g, qt).cpu().numpy()
            bad = y != want[:, ks].T
            assert not bad.any(), f"{bad.sum()} differ, e.g. {y[bad][:4]} vs {want[:, ks].T[bad][:4]}"


@pytest.mark.parametrize("rows,parts,M,K,N", [
    (256, 32, 300, 2048, 514),     # more parts than that tile height takes
    (128, 17, 130, 1088, 256),
    (128, 16, 2048, 1024, 8192),   # partial sums beyond the bound on the workspace
])
def test_forced_plan_the_kernel_declines(mn, gpu, rows, parts, M, K, N):
    """Rows and parts that the kernel does not take: the automatic choice
    runs and writes every output."""
    x, wp, s, z, g, acc = problem(M, K, N, 64, "int4", seed=parts)
    out = torch.full((M, N), float("nan"), dtype=torch.float16, device=gpu)
    args = dev(x, gpu), dev(wp, gpu), dev(s, gpu), dev(z, gpu), g, "int4"
    with forced(mn, rows, parts):
        mn.dequant_matmul(*args, out=out)
        path = mn.last_path()
    check(out.cpu().numpy(), acc, what=path)
    assert torch.equal(mn.dequant_matmul(*args), out) and mn.last_path() == path


@pytest.mark.parametrize("M,K,N,g,qt,epi,want", [
    (777, 4096, 3584, 128, "int4", "swiglu", "gemmn"),
    (300, 8192, 2048, 32, "int4", None, "gemmn"),       # K parts; more groups than the other kernels' tables hold
    (1100, 2048, 8192, 2048, "int8", "bias", "gemmn"),
    (37, 18944, 3584, 128, "int4", "residual", "gemmn"),
    (512, 3072, 5120, 128, "int4", None, "gemm16"),     # one round of the other kernel's tiles
    (64, 3104, 256, 32, "int4", None, "gemmw_split"),
])
def test_routing(mn, gpu, M, K, N, g, qt, epi, want):
    x, wp, s, z, g, acc = problem(M, K, N, g, qt, seed=K)
    kw, b, r = epilogue_args(epi, M, N, gpu)
    y = mn.dequant_matmul(dev(x, gpu), dev(wp, gpu), dev(s, gpu), dev(z, gpu), g, qt, **kw)
    assert mn.last_path() == want, mn.last_path()
    check(y.cpu().numpy(), acc, epi, b, r, want)


@pytest.mark.parametrize("M,K,N,g,qt,epi", [          # us: the other kernel / this one
    (1091, 3072, 3072, 128, "int4", "residual"),      # 63.6 / 42.8: its epilogue works element by element
    (834, 3584, 4608, 64, "int8", "bias"),            # 69.0 / 52.6
    (293, 896, 9728, 64, "int4", "residual"),         # 42.8 / 19.1
    (19, 3584, 37888, 64, "int4", "residual"),        # 52.9 / 41.5
    (67, 18944, 3584, 128, "int4", "bias"),           # 60.1 / 33.6
    (440, 832, 18390, 32, "int4", "residual"),        # 100.7 / 39.1: 64-row tiles, rows that are not 16-byte aligned
    (589, 928, 5778, 32, "int8", "residual"),         # 45.6 / 30.0
    (640, 896, 4870, 64, "int4", "swiglu"),           # the last M of 64-row tiles, the last columns past a tile
])
def test_routing_takes_the_faster_kernel(mn, gpu, M, K, N, g, qt, epi):
    x, wp, s, z, g, acc = problem(M, K, N, g, qt, seed=M)
    kw, b, r = epilogue_args(epi, M, N, gpu)
    y = mn.dequant_matmul(dev(x, gpu), dev(wp, gpu), dev(s, gpu), dev(z, gpu), g, qt, **kw)
    assert mn.last_path() == "gemmn", mn.last_path()
    check(y.cpu().numpy(), acc, epi, b, r)


@pytest.mark.parametrize("M,K,N,g,qt,epi", [   # us: the kernel it is left to / this one
    (1941, 1120, 1298, 32, "int8", None),      # 21.0 / 28.1
    (117, 3424, 23562, 3424, "int8", None),    # 44.2 / 53.7
    (21, 2560, 23744, 64, "int8", None),       # 25.7 / 37.5
    (93, 4864, 896, 128, "int4", "swiglu"),    # 15.9 / 19.1: many K parts for few threads to add
    (93, 2304, 21770, 64, "int4", None),       # 27.6 / 31.9
    (452, 2336, 4572, 32, "int4", None),       # 28.2 / 32.1
])
def test_routing_leaves_the_faster_kernel(mn, gpu, M, K, N, g, qt, epi):
    x = torch.randn((M, K), device=gpu).half()
    w = torch.randint(0, 256, (N, K // 2 if qt == "int4" else K), dtype=torch.uint8, device=gpu)
    s = torch.full((N, K // g), 0.01, dtype=torch.float16, device=gpu)
    args = (x, w if qt == "int4" else w.view(torch.int8), s, s, g, qt)
    got = mn.dequant_matmul(*args, epilogue=epi)
    assert mn.last_path() in ("gemmw", "gemmw_split", "gemm16"), mn.last_path()
    if epi is None:
        ref = x.float() @ mn.dequantize(*args[1:]).float().t().contiguous()
        assert bool(((got.float() - ref).abs() <= TOL_ABS + TOL_REL * ref.abs()).all())


def test_capture_and_shared_workspace(mn, gpu):
    """K parts under capture: with the stream's workspace in place the graph
    replays them; on a fresh stream a kernel without one runs.  The split-K
    GEMV, whose counters share the workspace, stays right in between."""
    M, K, N, g = 300, 8192, 2048, 128
    x, wp, s, z, g, acc = problem(M, K, N, g, "int4", seed=4)
    args = (dev(x, gpu), dev(wp, gpu), dev(s, gpu), dev(z, gpu), g, "int4")
    v = O.make_int4_problem(1, 896, 4864, 64, seed=8)
    vref = O.matmul_f32acc(v[0], O.dequant_int4(v[1], v[2], v[3], 896, 64))
    vargs = tuple(dev(a, gpu) for a in v) + (64, "int4")
    eager = {True: mn.dequant_matmul(*args)}
    assert mn.last_path() == "gemmn"
    mn.set_option("gemm_split", 0)
    eager[False] = mn.dequant_matmul(*args)
    path = {True: "gemmn", False: mn.last_path()}
    mn.set_option("gemm_split", 1)
    assert not torch.equal(eager[True], eager[False])   # the parts show in the rounding
    for warm in (True, False):
        stream = torch.cuda.Stream(gpu)
        stream.wait_stream(torch.cuda.current_stream(gpu))
        if warm:
            with torch.cuda.stream(stream):
                mn.dequant_matmul(*args)
                assert mn.last_path() == "gemmn"
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            y = mn.dequant_matmul(*args)
            captured = mn.last_path()
        assert captured == path[warm]
        for _ in range(3):
            y.zero_()
            graph.replay()
            torch.cuda.synchronize()
            check(y.cpu().numpy(), acc, what=f"replay warm={warm}")
            assert torch.equal(y, eager[warm])
            with torch.cuda.stream(stream):
                got = mn.dequant_matmul(*vargs)
            torch.cuda.synchronize()
            check(got.cpu().numpy(), vref, what="split-K GEMV between replays")


@pytest.mark.parametrize("M,K,N,epi,parts_path", [(300, 8192, 2048, None, "gemmn"), (37, 18944, 3584, "residual", "gemmn"),
                                                  (64, 3104, 256, "bias", "gemmw_split")])
def test_no_memory_for_a_workspace(mn, gpu, M, K, N, epi, parts_path):
    """Where a stream's workspace cannot grow, a plan without K parts runs;
    once it can, the K parts again."""
    x, wp, s, z, g, acc = problem(M, K, N, 32, "int4", seed=N)
    kw, b, r = epilogue_args(epi, M, N, gpu)
    args = dev(x, gpu), dev(wp, gpu), dev(s, gpu), dev(z, gpu), g, "int4"
    mn.release_workspaces()
    # (bounds below each plan's partial sums; 1 MiB is the smallest)
    stream = torch.cuda.Stream(gpu)
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        mn.set_option("gemm_split", 0)
        want = mn.dequant_matmul(*args, **kw)
        path = mn.last_path()
        mn.set_option("gemm_split", 1)
        mn.set_option("workspace_mb", 1)
        try:
            got = mn.dequant_matmul(*args, **kw)
            without = mn.last_path()
        finally:
            mn.set_option("workspace_mb", 0)
        again = mn.dequant_matmul(*args, **kw)
        assert mn.last_path() == parts_path
    torch.cuda.synchronize()
    if parts_path == "gemmn":   # (the third plan's partial sums fit in 1 MiB)
        assert without == path and torch.equal(got, want)
    for y in (got, again):
        check(y.cpu().numpy(), acc, epi, b, r, path)


def test_release_workspaces(mn, gpu):
    M, K, N, g = 777, 18944, 3584, 128   # 43 MiB of partial sums
    args = tuple(dev(a, gpu) for a in O.make_int4_problem(M, K, N, g, seed=2)) + (g, "int4")
    want = mn.dequant_matmul(*args)
    assert mn.last_path() == "gemmn"
    torch.cuda.synchronize()
    held = torch.cuda.mem_get_info(gpu)[0]
    mn.release_workspaces()
    assert torch.cuda.mem_get_info(gpu)[0] - held >= 40 << 20
    assert torch.equal(mn.dequant_matmul(*args), want)


def test_threads_on_one_stream(mn, gpu):
    """Calls of several K parts (two launches that share the stream's
    workspace) from threads on one stream, among calls of the split-K GEMV on
    the same workspace: each gives what it gives alone."""
    import threading

    shapes = [(300, 8192, 2048, 128, "gemmn"), (130, 8192, 1024, 128, "gemmn"), (8, 8192, 3072, 128, None),
              (200, 18944, 512, 128, "gemmn")]
    calls, want = [], []
    for i, (M, K, N, g, path) in enumerate(shapes):
        args = tuple(dev(a, gpu) for a in O.make_int4_problem(M, K, N, g, seed=60 + i)) + (g, "int4")
        want.append(mn.dequant_matmul(*args))
        assert path is None or mn.last_path() == path
        calls.append(args)
    got = [[] for _ in shapes]
    start = threading.Barrier(len(shapes))

    def work(i):
        start.wait()
        for _ in range(150):
            got[i].append(mn.dequant_matmul(*calls[i]))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(shapes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for i, outs in enumerate(got):
        assert len(outs) == 150
        wrong = sum(not torch.equal(y, want[i]) for y in outs)
        assert not wrong, f"{wrong} of {len(outs)} calls of {shapes[i]} differ"
