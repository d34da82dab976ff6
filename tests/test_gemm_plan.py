"""The host side of the batched products (csrc/matmat.c, csrc/int8.c), on the
CPU: its launches and its workspace, recorded by oracle/plan_pin.c. For exact
products on both sides of one tile per CU, in both orders and every type:

* the launches cover every token once, in order, by the tiles of the kernel
  that takes them;
* a split launch's partial sums (the first split's running total and one sum
  per later super-block) fit the workspace, which holds nothing else, and a
  product of more than one tile per CU keeps to 256 MiB of it;
* where the workspace cannot be had, the same product runs unsplit.

The int8 lane's larger tiles address their rows in 32 bits: rows too long for
them take the smallest tile, also where the environment names another.
"""
from __future__ import annotations

import ctypes as C
import math
import os
import random

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PIN = C.CDLL(os.path.join(ROOT, "oracle", "libplan_pin.so"))
CUS = 256
Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14


class Launch(C.Structure):
    _fields_ = [("kernel", C.c_char * 48), ("gx", C.c_uint32), ("gy", C.c_uint32),
                ("gz", C.c_uint32), ("block", C.c_uint32), ("y", C.c_uint64),
                ("tokens", C.c_uint32), ("slots", C.c_uint32), ("has_part", C.c_uint32)]


PIN.orc_plan.restype = C.c_int
PIN.orc_plan.argtypes = [C.c_int, C.c_int, C.c_uint64, C.c_uint64, C.c_uint64, C.c_int, C.c_int,
                         C.POINTER(Launch), C.c_int, C.POINTER(C.c_uint64), C.POINTER(C.c_int),
                         C.POINTER(C.c_int)]
LANES = {"batched": 0, "matvec": 1, "int8": 2}


def plan(lane, qtype, rows, cols, tokens, fail=False):
    """(launches, workspace bytes, allocations tried)"""
    out, n = (Launch * 8)(), C.c_uint64()
    allocs, frees = C.c_int(), C.c_int()
    got = PIN.orc_plan(LANES[lane], qtype, rows, cols, tokens, CUS, int(fail), out, 8,
                       C.byref(n), C.byref(allocs), C.byref(frees))
    assert got > 0
    assert frees.value == (0 if fail else allocs.value)
    return [out[i] for i in range(got)], n.value, allocs.value


def cases():
    rng = random.Random(5)
    yield from ((2560, 9728, 832), (2560, 9728, 512), (4096, 12288, 640), (2048, 2048, 64),
                (1, 256, 1), (64, 256, 64), (9728, 4096, 218), (151936, 1024, 2))
    for _ in range(400):
        log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
        yield log(1, 16000), 256 * log(1, 64), log(1, 4096)


@pytest.mark.parametrize("lane", ["batched", "matvec"])
@pytest.mark.parametrize("qtype", [Q4_K, Q5_K, Q6_K, Q8_0])
def test_launches_and_workspace(lane, qtype):
    split_past = 0
    for rows, cols, tokens in cases():
        where, units = (rows, cols, tokens), cols // 256
        launches, bytes_, _ = plan(lane, qtype, rows, cols, tokens)
        done = need = 0
        gemms = [x for x in launches if b"fold" not in x.kernel]
        for i, g in enumerate(launches):
            if b"fold" in g.kernel:
                assert launches[i - 1].gz > 1 and g.y == launches[i - 1].y, where
                continue
            assert g.y == done * rows, where
            done += g.tokens
            assert g.gx == -(-rows // 64) and g.gy == -(-g.tokens // 64), where
            few = b"few" in g.kernel
            assert not few or g.tokens <= int(g.kernel[-2:]), where
            assert g.block == 256 * (1 if few else int(g.kernel[-1:])), where
            if g.gz > 1:
                # The kernel's last slot is its last super-block's: units - units / gz.
                slots = units - units // g.gz + 1
                fold = launches[i + 1]
                assert b"fold" in fold.kernel and g.has_part and fold.has_part, where
                assert fold.slots == slots and fold.tokens == g.tokens, where
                need = max(need, 4 * slots * rows * g.tokens)
        assert done == tokens and len(gemms) <= 2, where
        assert bytes_ == need, where
        if -(-rows // 64) * -(-tokens // 64) > CUS:
            assert bytes_ <= 256 << 20, where
            split_past += bytes_ > 0
    assert split_past or (lane == "matvec" and qtype == Q8_0)


@pytest.mark.parametrize("lane", ["batched", "matvec"])
@pytest.mark.parametrize("qtype", [Q4_K, Q5_K, Q6_K, Q8_0])
def test_runs_unsplit_without_the_workspace(lane, qtype):
    tried = 0
    for rows, cols, tokens in cases():
        launches, bytes_, allocs = plan(lane, qtype, rows, cols, tokens, fail=True)
        assert bytes_ == 0 and allocs <= 1
        assert all(x.gz == 1 and b"fold" not in x.kernel for x in launches)
        assert sum(x.tokens for x in launches) == tokens
        tried += allocs
    assert tried or (lane == "matvec" and qtype == Q8_0)


@pytest.mark.parametrize("tile", [None, "0", "1", "2", "3"])
@pytest.mark.parametrize("qtype", [Q4_K, Q5_K])
def test_int8_tiles_by_row_length(monkeypatch, qtype, tile):
    monkeypatch.delenv("MYNAH_INT8_TILE", raising=False)
    if tile is not None:
        monkeypatch.setenv("MYNAH_INT8_TILE", tile)
    names = [b"32x32", b"64x64", b"96x128", b"128x128"]
    quant, gemm = plan("int8", qtype, 9728, 4096, 2048)[0]
    assert gemm.kernel.split(b"_")[-1] in ([names[int(tile)]] if tile else names)
    for cols in (1 << 24, 1 << 26):
        quant, gemm = plan("int8", qtype, 256, cols, 128)[0]
        assert gemm.kernel.endswith(b"32x32") and (gemm.gx, gemm.gy) == (8, 4)
