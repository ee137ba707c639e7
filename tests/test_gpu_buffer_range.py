"""Raw buffer loads past their resource read zero, whichever offset takes them there: kernels put the row or
block in the scalar offset and let the range check cover the ones past the end (attention's last key block,
ragged activation rows of the tiled GEMM, ragged block counts of the tile GEMV, 192-row tiles of the packed
GEMM). Every address the offsets could form lies inside the buffer here, so nothing is read out of it even
if the check did not hold."""
import ctypes as C
import os

import numpy as np
import pytest

from rehip import hip

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("records", [128, 256, 1008, 4096])
@pytest.mark.parametrize("soffset", [0, 64, 128, 256, 1008, 4096, 4112, 65536, 196608])
def test_scalar_offset_counts_in_the_range_check(records, soffset):
    L = C.CDLL(os.path.join(ROOT, "rusty-engine_amd", "librecalib.so"))
    L.cal_buffer_range.argtypes = [C.c_void_p, C.c_uint64, C.c_uint32, C.c_uint32, C.c_void_p, C.c_void_p]
    words = np.arange(1, 65537, dtype=np.uint32)
    buf, out = hip.DeviceBuffer.from_array(words), hip.DeviceBuffer(1024)
    assert L.cal_buffer_range(buf.ptr, words.nbytes, records, soffset, out.ptr, None) == 0
    hip.synchronize()
    got = out.download(np.uint32, 256).reshape(4, 64)
    lane = np.arange(64)
    for row, width, word in ((0, 4, 0), (1, 16, 0), (2, 16, 3), (3, 16, 0)):
        at = soffset + width * lane + 4 * word
        want = np.where(at + 4 <= records, words[at // 4], 0)
        assert np.array_equal(got[row], want), row
