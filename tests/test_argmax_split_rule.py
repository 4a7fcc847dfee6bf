"""Into how many segments a row of logits is cut: arctic_argmax_workspace_bytes holds 16 bytes for each, and makes no HIP
call.  On both sides of every line the rule draws."""
import pytest

from arcticinference_amd import _native

BF16, F32 = _native.DTYPE_BF16, _native.DTYPE_F32
CHUNK = {BF16: 8, F32: 4}   # elements of 16 bytes


def parts(rows, chunks, dtype):
    return _native.load().arctic_argmax_workspace_bytes(rows, chunks * CHUNK[dtype], dtype) // (16 * rows)


@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("rows,chunks,segments", [
    (1, 10240, 10), (1, 10239, {BF16: 9, F32: 0}), (48, 8192, {BF16: 8, F32: 0}), (49, 9999, 0), (49, 10000, {BF16: 9, F32: 0}),
    (74, 10240, 8), (80, 11000, 8), (85, 11250, 8), (85, 10240, 8), (85, 18000, 6),   # 180 chunks for each row but 5100
    (86, 10379, 0), (86, 10380, 8), (128, 17939, 0), (128, 17940, 8), (129, 40000, 0)])
def test_rows_that_leave_cus_idle(rows, chunks, segments, dtype):
    assert parts(rows, chunks, dtype) == (segments[dtype] if isinstance(segments, dict) else segments)


@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("rows,chunks,segments", [
    (256, 40000, 0), (257, 12287, 0), (257, 12288, 8), (288, 12288, 8), (289, 12288, {BF16: 8, F32: 0}), (304, 24575, {BF16: 8, F32: 0}),
    (304, 24576, 8), (305, 40000, 0), (512, 40000, 0), (513, 9999, 0), (513, 10000, 8), (600, 10000, 8), (601, 28671, 0), (601, 28672, 8),
    (704, 28672, 8), (705, 40000, 0)])
def test_a_few_more_rows_than_cus(rows, chunks, segments, dtype):
    assert parts(rows, chunks, dtype) == (segments[dtype] if isinstance(segments, dict) else segments)


@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("rows,chunks,anywhere", [(1, 12000, True), (85, 12000, True), (128, 40000, True), (257, 30000, False),
                                                  (304, 30000, False), (513, 12000, False), (704, 30000, False), (400, 30000, True)])
def test_rows_that_start_between_16_byte_boundaries_ask_for_no_more_than_they_use(rows, chunks, anywhere, dtype):
    lib, cols, size = _native.load(), chunks * CHUNK[dtype], 16 // CHUNK[dtype]
    at = lambda address, pitch: lib.arctic_argmax_workspace_bytes_at(address, rows, cols, pitch, dtype)
    most = lib.arctic_argmax_workspace_bytes(rows, cols, dtype)
    assert at(4096, cols) == at(4096, cols + 8) == most
    assert at(4096 + size, cols) == (most if anywhere else 0)
    assert at(4096, cols + 1) == (most if anywhere or rows == 1 else 0)
    assert at(4096 + 1, cols) == 0   # no element boundary: one workgroup per row, element by element
