"""The row-block GEMV's 13-op int4 dequant (twelve-wave builds, long weight
rows): every weight equals the oracle's two-rounding one, with all scales in
its range, with others among them, and with the arrays ending inside a staged
16-byte piece of scales; in the plain, the two-half (M = 9..16) and the
fused-norm builds."""

import numpy as np
import pytest
import torch

from oracle import mq_oracle as O

pytestmark = pytest.mark.gpu

# fp16 bit patterns: the ends of the range (exponents 1 and 16) and inside
INSIDE = np.array([0x0400, 0x0401, 0x1400, 0x2555, 0x3C00, 0x43FF, 0x8400, 0xA4D3, 0xC3FF], dtype=np.uint16)
# zero, subnormals, the neighbours above, large
OUTSIDE = np.array([0x0000, 0x0001, 0x03FF, 0x4400, 0x5800, 0x6C00, 0xC400, 0x83FF], dtype=np.uint16)
ZEROS = np.array([0x0000, 0x8000, 0x0001, 0x83FF, 0x2E66, 0xBC00, 0x5555, 0xE000], dtype=np.uint16)


@pytest.mark.parametrize("outside", ["none", "one in the last row", "many"])
@pytest.mark.parametrize("M,epilogue", [(1, None), (4, None), (4, "swiglu")])
def test_one_hot_selects_dequantized_weights(gpu, M, epilogue, outside):
    import metal_native as mn

    rng = np.random.default_rng(7)
    N, K, g = 2050, 16640, 128   # 8-9 rows of 8 KiB per workgroup; N * K / g ends 4 entries into a piece of 8
    G = K // g
    s = INSIDE[rng.integers(0, len(INSIDE), (N, G))]
    if outside == "many":
        at = rng.random((N, G)) < 0.02
        s = np.where(at, OUTSIDE[rng.integers(0, len(OUTSIDE), (N, G))], s)
    elif outside != "none":
        s[-1, -1] = OUTSIDE[5]
    s = s.astype(np.uint16).view(np.float16)
    z = ZEROS[rng.integers(0, len(ZEROS), (N, G))].view(np.float16)
    wp = rng.integers(0, 256, (N, K // 2), dtype=np.uint8)
    want = O.dequant_int4(wp, s, z, K, g)
    assert np.isfinite(want).all()
    t = [torch.from_numpy(a).to(gpu) for a in (wp, s, z)]
    ks_all = np.concatenate([[0, K - 1, K - 128, 16383, 16384], rng.integers(0, K, 27)])
    mn.set_option("force_path", 7)
    try:
        for i in range(0, len(ks_all) - M + 1, M):
            ks = ks_all[i:i + M]
            x = np.zeros((M, K), dtype=np.float16)
            x[np.arange(M), ks] = 1.0
            y = mn.dequant_matmul(torch.from_numpy(x).to(gpu), *t, g, "int4", epilogue=epilogue).cpu().numpy()
            assert mn.last_path() == "rows"
            ref = want[:, ks].T
            if epilogue is None:
                bad = y != ref   # -0 == +0
                assert not bad.any(), f"{bad.sum()} differ, e.g. {y[bad][:4]} vs {ref[bad][:4]}"
            else:
                gate, up = (ref[:, j * N // 2:(j + 1) * N // 2].astype(np.float64) for j in range(2))
                with np.errstate(over="ignore"):
                    v = gate / (1.0 + np.exp(-gate)) * up
                # fp32 arithmetic and one fp16 rounding of the exact gate and up
                ok = (np.abs(y - v) <= 2.0**-10 * np.abs(v) + 2.0**-24) | (np.abs(v) >= 65504)
                assert ok.all()
    finally:
        mn.set_option("force_path", 0)


def _weights(rng, N, K, g, outside):
    G = K // g
    s = INSIDE[rng.integers(0, len(INSIDE), (N, G))]
    if outside:
        at = rng.random((N, G)) < 0.001   # workgroups of both kinds
        at[:64] = False
        at[-1, -1] = True
        s = np.where(at, OUTSIDE[rng.integers(0, len(OUTSIDE), (N, G))], s)
    s = s.astype(np.uint16).view(np.float16)
    z = ZEROS[rng.integers(0, len(ZEROS), (N, G))].view(np.float16)
    return rng.integers(0, 256, (N, K // 2), dtype=np.uint8), s, z


@pytest.mark.parametrize("N", [13442, 8450, 1026])   # 112 and 68 KiB of weights per workgroup; eight waves at M = 1
@pytest.mark.parametrize("outside", [False, True])
@pytest.mark.parametrize("build", ["M=9", "M=13", "fused norm"])
def test_one_hot_in_the_other_builds(gpu, build, outside, N):
    import metal_native as mn
    from metal_native import ops

    rng = np.random.default_rng(N + outside)
    K, g = 4096, 128
    wp, s, z = _weights(rng, N, K, g, outside)
    t = [torch.from_numpy(a).to(gpu) for a in (wp, s, z)]
    M = 1 if build == "fused norm" else int(build[2:])
    ks_all = np.concatenate([[0, K - 1, K - 128, 127], rng.integers(0, K, 22)])
    want = O.dequant_int4(wp, s, z, K, g)[:, ks_all]
    assert np.isfinite(want).all()
    mn.set_option("force_path", 7)
    try:
        for i in range(0, len(ks_all) - M + 1, M):
            x = np.zeros((M, K), dtype=np.float16)
            x[np.arange(M), ks_all[i:i + M]] = 1.0
            xd = torch.from_numpy(x).to(gpu)
            if build == "fused norm":
                # the norm of a one-hot row: 1 / sqrt(1 / 4096) = 64, times a weight of 1/64
                w = torch.full((K,), 1.0 / 64, dtype=torch.float16, device=gpu)
                resid = torch.empty_like(xd)
                y = ops.rmsnorm_dequant_matmul(xd, None, w, 0.0, resid, *t, g, "int4")
                assert torch.equal(resid, xd)
            else:
                y = mn.dequant_matmul(xd, *t, g, "int4")
            assert mn.last_path() == "rows"
            y, ref = y.cpu().numpy(), want[:, i:i + M].T
            bad = y != ref   # -0 == +0
            assert not bad.any(), f"{bad.sum()} differ, e.g. {y[bad][:4]} vs {ref[bad][:4]}"
    finally:
        mn.set_option("force_path", 0)
