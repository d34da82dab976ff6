"""The batched prefill's attention on the matrix cores against decode steps.

Its scores come from 16-key x 32-query tiles over a span of positions, its
weighted V sums from 16-query tiles over all or a quarter of the dimensions
(MYNAH_PREFILL_SPAN, MYNAH_PREFILL_PV_DIMS force either). Both must leave the
bits of the decode step's kernels, which run the reference's chains on the
VALU, one position after the other. Chunks at the edges of the query tiles (1,
15 .. 17, 31 .. 33), prefixes at the edges of the 32-position copies, head
groups that split unevenly over the four waves of a workgroup.
"""
from __future__ import annotations

import numpy as np
import pytest

import configs as CF
import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def M():
    import mynah_amd
    mynah_amd.check(mynah_amd.lib.mynah_hip_init(0), "init")
    mynah_amd.check(mynah_amd.lib.mynah_hip_set_gemv_order(0), "order")
    O.orc.orc_threads_init(0)
    return mynah_amd


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


@pytest.mark.parametrize("span,dims", [(32, 32), (64, 128), (128, 32), (512, 128)])
@pytest.mark.parametrize("group,prefix,tokens", [
    (2, 1, 1), (2, 31, 15), (3, 32, 17), (5, 62, 33), (7, 130, 31), (8, 257, 66), (2, 300, 48)])
def test_tiles_equal_steps(M, monkeypatch, span, dims, group, prefix, tokens):
    monkeypatch.setenv("MYNAH_PREFILL_SPAN", str(span))
    monkeypatch.setenv("MYNAH_PREFILL_PV_DIMS", str(dims))
    monkeypatch.setenv("MYNAH_PREFILL_CHUNK", "512")
    print(f"[case] span={span} dims={dims} group={group} {prefix}+{tokens}", flush=True)
    shape = CF.Qwen3Shape(2, 256, 256, 2 * group, 2, 128, 512)
    model = M.SynthQwen3(shape, 0)
    k, v = O.kv_prefill(O.substream, shape, 0, prefix)
    # Values 2^-126 times smaller in one key head: subnormal sums and products.
    v = v.copy()
    v[0].reshape(prefix, -1)[:, :128] *= np.float32(2.0 ** -126)
    prompt = M.synth_uniform(M.substream(9, tokens), tokens, shape.vocab)
    n = prefix + tokens
    a, b = M.Qwen3Decoder(model, n + 2), M.Qwen3Decoder(model, n + 2)
    a.set_kv(k, v, prefix)
    b.set_kv(k, v, prefix)
    for t in prompt:
        a.forward(int(t), want_logits=False)
    b.prefill(prompt)
    for x, y in zip(a.get_kv(n), b.get_kv(n)):
        assert np.array_equal(bits(x), bits(y))
    assert np.array_equal(bits(a.forward(3)), bits(b.forward(3)))
