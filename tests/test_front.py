"""The native front of dequant_matmul and matmul (csrc/mq_torch.cpp): what it
takes gives what the general Python path gives, what it does not take goes
that way, with its copies and its errors."""

import pytest
import torch


@pytest.fixture(scope="module")
def mn():
    import metal_native

    return metal_native


def test_declines_what_is_not_a_plain_gpu_tensor(mn):
    from metal_native import _mq_torch

    x, w = torch.zeros((1, 64), dtype=torch.float16), torch.zeros((8, 32), dtype=torch.uint8)
    s = torch.zeros((8, 2), dtype=torch.float16)
    for args in ((x, w, s, s), (x.to("meta"), w, s, s), (None, w, s, s), ([1.0], w, s, s)):
        assert _mq_torch.dequant_matmul(*args, 32, True, 0, None, None, 0) is None
    assert _mq_torch.vecmat(x, x, True, 0) is None
    with pytest.raises(mn.MetalNativeError, match="must be a GPU tensor"):
        mn.dequant_matmul(x, w, s, s, 32, "int4")


def test_front_has_no_thread_local_storage(mn):
    """No PT_TLS segment: loading one late slows every thread-local access of
    the importing thread (glibc's stale thread vector) until that thread
    touches the newest library's own variables."""
    import struct

    from metal_native import _mq_torch

    with open(_mq_torch.__file__, "rb") as f:
        head = f.read(64)
        assert head[:6] == b"\x7fELF\x02\x01"
        (phoff,) = struct.unpack_from("<Q", head, 32)
        size, count = struct.unpack_from("<HH", head, 54)
        f.seek(phoff)
        table = f.read(size * count)
    types = [struct.unpack_from("<I", table, size * i)[0] for i in range(count)]
    assert 1 in types and 7 not in types   # PT_LOAD, PT_TLS


class Marked(torch.Tensor):
    pass


def problem(gpu, M=3, K=512, N=384, g=64, quant="int4", seed=0):
    gen = torch.Generator(device=gpu)
    gen.manual_seed(seed)
    cols = K // 2 if quant == "int4" else K
    w = torch.randint(0, 256, (N, cols), dtype=torch.uint8, device=gpu, generator=gen)
    w = w if quant == "int4" else w.view(torch.int8)
    s = (torch.rand((N, K // g), device=gpu, generator=gen) * 0.02).half()
    z = torch.randn((N, K // g), device=gpu, generator=gen).half()
    return [torch.randn((M, K), device=gpu, generator=gen).half(), w, s, z]


def wider(t, by=16):
    big = torch.full((t.shape[0], t.shape[1] + by), 77, dtype=t.dtype, device=t.device)
    big[:, :t.shape[1]] = t
    return big[:, :t.shape[1]]


@pytest.mark.gpu
@pytest.mark.parametrize("quant,g", [("int4", 64), ("int8", 512), ("int8", 32)])
@pytest.mark.parametrize("epilogue", [None, "none", "bias", "bias_relu", "bias_silu", "residual", "swiglu"])
def test_front_equals_the_general_path(mn, gpu, quant, g, epilogue):
    """``out=`` keeps a call on the general path."""
    M, K, N = 3, 512, 384
    args = problem(gpu, M, K, N, g, quant)
    kw = {"epilogue": epilogue}
    if epilogue and epilogue.startswith("bias"):
        kw["bias"] = torch.randn(N, device=gpu).half()
    elif epilogue == "residual":
        kw["residual"] = torch.randn((M, N), device=gpu).half()
    nout = N // 2 if epilogue == "swiglu" else N
    forms = {
        "plain": lambda t: t,
        "wider rows": wider,                                       # row strides
        "parameter": lambda t: torch.nn.Parameter(t, requires_grad=False),
        "subclass": lambda t: t.as_subclass(Marked),               # general path
        "columns strided": lambda t: torch.stack((t, t), -1)[..., 0],
        "rows expanded": lambda t: t[:1].expand(t.shape),          # general path: copied
    }
    for name, form in forms.items():
        a = [form(t) for t in args]
        if "residual" in kw:
            kw["residual"] = form(kw["residual"])
        out = torch.empty((M, nout), dtype=torch.float16, device=gpu)
        want = mn.dequant_matmul(*[torch.Tensor(t) if type(t) is Marked else t for t in a], g, quant, out=out, **kw)
        got = mn.dequant_matmul(*a, g, quant, **kw)
        assert got.is_contiguous() and not got.requires_grad
        assert torch.equal(got, want), name


@pytest.mark.gpu
def test_front_takes_or_declines(gpu):
    """Which calls the front takes (an output) and which it leaves to the
    general path (None)."""
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    from metal_native import _mq_torch

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    x, w, s, z = problem(gpu)
    stream = torch.cuda.current_stream(gpu).cuda_stream
    a, b = torch.randn((2, 512), device=gpu).half(), torch.randn((300, 512), device=gpu).half()

    def linear(x=x, w=w, s=s, z=z, g=64, int4=True, epi=0, bias=None, resid=None):
        return _mq_torch.dequant_matmul(x, w, s, z, g, int4, epi, bias, resid, stream)

    def vecmat(a=a, b=b, tb=True):
        return _mq_torch.vecmat(a, b, tb, stream)

    strided = lambda t: torch.stack((t, t), -1)[..., 0]
    row = lambda t: torch.nn.Parameter(t, requires_grad=False)
    resid = torch.randn((3, 384), device=gpu).half()
    for take in (lambda: linear(), lambda: linear(wider(x), wider(w)), lambda: linear(row(x), row(w), row(s), row(z)),
                 lambda: linear(x.clone().requires_grad_()), lambda: linear(epi=5),
                 lambda: linear(epi=1, bias=resid[0].contiguous()), lambda: linear(epi=4, resid=wider(resid)),
                 lambda: vecmat(), lambda: vecmat(wider(a), wider(b)), lambda: vecmat(a, b.t().contiguous(), False),
                 lambda: vecmat(a.float(), b.float())):
        assert type(take()) is torch.Tensor
    for decline in (lambda: linear(x.as_subclass(Marked)), lambda: linear(strided(x)), lambda: linear(w=strided(w)),
                    lambda: linear(s=strided(s)), lambda: linear(s=wider(s)), lambda: linear(x[:1].expand(3, 512)),
                    lambda: linear(x[0]), lambda: linear(x.float()), lambda: linear(x.cpu()), lambda: linear(s=s[1:]),
                    lambda: linear(g=48), lambda: linear(int4=False), lambda: linear(epi=1), lambda: linear(bias=s[0]),
                    lambda: linear(epi=7), lambda: linear(epi=4, resid=strided(resid)), lambda: linear(x[:0]),
                    lambda: vecmat(a[0]), lambda: vecmat(strided(a)), lambda: vecmat(a.as_subclass(Marked)),
                    lambda: vecmat(a, b.float()), lambda: vecmat(a[:, :200], b[:, :200]), lambda: vecmat(a, b[:200]),
                    lambda: vecmat(a.repeat(5, 1)), lambda: vecmat(a, b.cpu())):
        assert decline() is None
    for mode in (Function(), Dispatch()):
        with mode:
            assert linear() is None and vecmat() is None
    seen = []
    torch.func.vmap(lambda v: (seen.append((linear(v), vecmat(a, v))), v)[1])(torch.stack((x, x)))
    assert seen == [(None, None)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("transpose_b", [True, False])
@pytest.mark.parametrize("M", [1, 8])
def test_vecmat_forms(mn, gpu, dtype, transpose_b, M):
    K, N = 264, 300
    a = torch.randn((M, K), device=gpu).to(dtype)
    b = torch.randn((N, K) if transpose_b else (K, N), device=gpu).to(dtype)
    want = mn.matmul(a[None], b, False, transpose_b)[0]   # three dimensions: the general path
    assert torch.equal(mn.matmul(a, b, False, transpose_b), want)
    assert torch.equal(mn.matmul(wider(a), wider(b), False, transpose_b), want)


@pytest.mark.gpu
def test_errors_and_streams(mn, gpu):
    x, w, s, z = problem(gpu)
    with pytest.raises(mn.MetalNativeError, match="group_size must be 32, 64, or 128"):
        mn.dequant_matmul(x, w, s, z, 48, "int4")
    with pytest.raises(mn.MetalNativeError, match="scales must be"):
        mn.dequant_matmul(x, w, s[:, 1:], z, 64, "int4")
    with pytest.raises(mn.MetalNativeError, match="needs bias"):
        mn.dequant_matmul(x, w, s, z, 64, "int4", epilogue="bias")
    with pytest.raises(mn.MetalNativeError, match="without a bias epilogue"):
        mn.dequant_matmul(x, w, s, z, 64, "int4", bias=s[:, 0])
    with pytest.raises(mn.MetalNativeError, match="unknown epilogue"):
        mn.dequant_matmul(x, w, s, z, 64, "int4", epilogue="gelu")
    assert mn.dequant_matmul(x[:0], w, s, z, 64, "int4").shape == (0, 384)
    # the current stream: work queued before the call on it is seen
    want = mn.dequant_matmul(x, w, s, z, 64, "int4")
    side = torch.cuda.Stream(gpu)
    late = torch.zeros_like(x)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        torch.cuda._sleep(20_000_000)
        late.copy_(x)
        got = mn.dequant_matmul(late, w, s, z, 64, "int4")
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    with torch.inference_mode():
        assert torch.equal(mn.dequant_matmul(x, w, s, z, 64, "int4"), want)
