"""
How the host waits for a number that a kernel writes into pinned memory, with a stream that stands in for the GPU's.
"""
import numpy as np
import pytest

from heat_amd.cluster._kcluster import _wait_count


class _Stream:
    def __init__(self, count, delivers=None, error=None):
        self.count, self.delivers, self.error, self.waits = count, delivers, error, 0

    def synchronize(self):
        self.waits += 1
        if self.error is not None:
            raise self.error
        if self.delivers is not None:
            self.count[...] = self.delivers


def test_a_number_that_is_there_needs_no_wait():
    for number in (0, 1, 2**40):
        count = np.array(number, dtype=np.int64)
        stream = _Stream(count)
        assert _wait_count(count, stream) == number and stream.waits == 0


def test_long_work_is_waited_for_by_the_stream():
    count = np.array(-1, dtype=np.int64)
    stream = _Stream(count, delivers=17)
    assert _wait_count(count, stream) == 17 and stream.waits == 1


def test_errors_are_raised():
    count = np.array(-1, dtype=np.int64)
    with pytest.raises(RuntimeError, match="of the device"):
        _wait_count(count, _Stream(count, error=RuntimeError("of the device")))
    with pytest.raises(RuntimeError, match="without delivering"):
        _wait_count(count, _Stream(count))
