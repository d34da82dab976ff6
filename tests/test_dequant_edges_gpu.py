"""The dequantiser (csrc/dequant.hip) at the edges of its workgroups (4,096
values each): matrices of one block, just under and over whole workgroups,
and destinations at every 4-byte alignment; bit for bit against the oracle,
nothing written past the end.
"""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def M():
    import mynah_amd
    mynah_amd.check(mynah_amd.lib.mynah_hip_init(0), "init")
    return mynah_amd


@pytest.mark.parametrize("rows,cols", [(1, 256), (15, 256), (16, 256), (17, 256), (3, 1280),
                                       (33, 2560), (129, 512)])
@pytest.mark.parametrize("qtype", [2, 8, 12, 13, 14])
def test_dequant_edges(M, qtype, rows, cols):
    if qtype == 2:
        cols += 32                       # Q4_0 takes any multiple of 32
    n = rows * cols
    w = M.synth_blocks(qtype, rows, rows, cols)
    ref = np.ascontiguousarray(O.dequant(qtype, w, rows, cols)).ravel()
    wd = M.DeviceBuffer.from_array(w)
    for skew in range(4):
        yd = M.DeviceBuffer.from_array(np.full(n + 8, 7.5, np.float32))
        M.dequant_dev(qtype, wd.ptr, rows, cols, yd.ptr + 4 * skew)
        M.sync()
        got = yd.download(np.float32, n + 8)
        assert np.array_equal(got[skew:skew + n].view(np.uint32), ref.view(np.uint32))
        assert (got[:skew] == 7.5).all() and (got[skew + n:] == 7.5).all()
        yd.free()
    wd.free()
