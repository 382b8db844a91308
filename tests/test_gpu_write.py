"""ps_write: a few bytes to device memory as a kernel's argument."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 4, 8, 63, 64])
def test_write_bytes_in_stream_order(device, n):
    """Exactly the n bytes change, in order with what is queued around it;
    the host buffer may be reused at once."""
    from pysweep_amd import hip
    buf = hip.DeviceArray(80)
    buf.fill_bytes(7)
    data = bytearray(range(100, 100 + n))
    hip.write_bytes(buf.ptr + 8, data)
    for i in range(n):
        data[i] = 0
    got = buf.download(np.empty(80, np.uint8))
    want = np.full(80, 7, np.uint8)
    want[8:8 + n] = np.arange(100, 100 + n)
    assert np.array_equal(got, want)
    buf.close()


def test_longer_writes_take_a_copy_and_the_entry_refuses_them(device):
    from pysweep_amd import hip
    buf = hip.DeviceArray(200)
    data = bytes(range(200))
    hip.write_bytes(buf.ptr, data)
    assert buf.download(np.empty(200, np.uint8)).tobytes() == data
    with pytest.raises(hip.HipError, match="64 bytes"):
        hip.check(hip._write(buf.ptr, data, 65), "ps_write")
    buf.close()
