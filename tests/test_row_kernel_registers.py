"""Scalar registers of the sine rows' kernel for short butterflies (one per
thread).  Its rows of 1024 threads share a compute unit only with at most 80:
the eight waves a SIMD then holds take 96 of its 800 each (16 of them the
trap handler's); 81 round up to 112, seven waves, and one row fits."""
from pyaxisymflow_amd import _lib


def find_name(data, kernel):
    at = 0
    while True:
        at = data.index(b".name\xd9", at)
        start = at + len(b".name\xd9") + 1
        if data[start:start + len(kernel)] == kernel:
            return at
        at = start


def sgpr_count(kernel):
    """Scalar registers of the kernel whose mangled name starts with
    ``kernel``, from the code object's metadata (msgpack: a name's map has
    its keys in order, the register count after the name)."""
    with open(_lib.LIB_PATH, "rb") as f:
        data = f.read()
    key = b".sgpr_count"
    at = data.index(key, find_name(data, kernel)) + len(key)
    return data[at] if data[at] < 128 else data[at + 1]


def test_sine_rows_leave_room_for_two_rows():
    assert sgpr_count(b"_ZN3axs20any_dst1_rows_kernelILi1EEE") <= 80
