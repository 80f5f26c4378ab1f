"""The row-block GEMV's 13-op int4 dequant (twelve-wave builds, long weight
rows): every weight equals the oracle's two-rounding one, with all scales in
its range, with others among them, and with the arrays ending inside a staged
16-byte piece of scales."""

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
