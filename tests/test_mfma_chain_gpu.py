"""The chain property of the batched prefill's attention, over edge operands.

mynah_prefill_scores and mynah_prefill_pv* (csrc/decode.hip) take the
reference's FMA chains (src/kernels.c:39-62, 83-100) from
v_mfma_f32_16x16x4_f32: its four products join the accumulator one after the
other in k order, each with fmaf's one rounding. Held here against the VALU's
fmaf on 4096 waves of 256 chains of four: specials (zeros of both signs,
subnormals, the smallest and largest normals, infinities, NaN), any bit
pattern, products at the subnormal and overflow boundaries, and N(0, 1)
values, each with accumulators of their own kind; and unlike the same products
in the reverse order, or rounded before they are added, on many of them.
"""
from __future__ import annotations

import numpy as np
import pytest

from test_mfma_product_gpu import GROUP, SPECIALS, WAVES, f32, operands, same

pytestmark = pytest.mark.gpu


def accumulators():
    rng = np.random.default_rng(1)
    n = 256 * GROUP
    return np.concatenate([
        rng.choice(SPECIALS, n),
        f32(rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)),
        (rng.choice([-1.0, 1.0], n) * np.ldexp(rng.uniform(1.0, 2.0, n), rng.choice(
            [-149, -140, -126, 100, 126], n))).astype(np.float32),
        rng.standard_normal(n).astype(np.float32)])


def products(a, b):
    """a and b of every output's four products: [4, 256 * WAVES]."""
    out = np.arange(256 * WAVES)
    w, l, e = out // 256, (out % 256) // 4, out % 4
    k = 16 * np.arange(4)[:, None]
    return a[64 * w + k + 4 * (l // 16) + e], b[64 * w + k + l % 16]


def test_the_instruction_is_a_chain_of_fmaf():
    import mynah_amd as M
    M.check(M.lib.mynah_hip_init(0), "init")
    print(f"[case] v_mfma_f32_16x16x4_f32 on {WAVES} waves x 256 chains", flush=True)
    a, b, _ = operands()
    c = accumulators()
    bufs = [M.DeviceBuffer.from_array(v) for v in (a, b, c)]
    outs = [M.DeviceBuffer(4 * 256 * WAVES) for _ in range(2)]
    M.check(M.lib.mynah_hip_mfma_chain_probe(*[x.ptr for x in bufs], *[o.ptr for o in outs],
                                             WAVES, None), "mfma_chain_probe")
    M.sync()
    acc, fused = [o.download(np.float32, 256 * WAVES) for o in outs]
    for x in bufs + outs:
        x.free()
    ok = same(acc, fused)
    print(f"{int(ok.sum())} of {ok.size} chains equal; subnormal results "
          f"{int(((fused != 0) & (np.abs(fused) < np.float32(2.0 ** -126))).sum())}, infinite "
          f"{int(np.isinf(fused).sum())}, NaN {int(np.isnan(fused).sum())}; the first unequal "
          f"{acc[~ok][:4]}, {fused[~ok][:4]}", flush=True)
    assert ok.all()
    # fmaf in the reverse order (through doubles: all but its double roundings)
    # and products rounded on their own give other sums.
    x, y = products(a, b)
    with np.errstate(all="ignore"):
        back, apart = c.astype(np.float64), c.copy()
        for k in range(4):
            back = (x[3 - k].astype(np.float64) * y[3 - k] + back).astype(np.float32) \
                .astype(np.float64)
            apart = apart + x[k] * y[k]
    normal = slice(3 * 256 * GROUP, None)
    for other in (back.astype(np.float32), apart):
        assert (~same(acc, other)[normal]).mean() > 0.05
