"""Host-side pieces of the transfer pipeline that need no GPU: chunk
planning, the streaming threshold and the threaded block copy."""

import numpy as np
import pytest

from algotom_amd import _host
from algotom_amd.rec import reconstruction as rec


@pytest.mark.parametrize("nslice,slice_bytes", [
    (64, 4 * (1801 * 2560 + 2560 * 2560)),   # the 64-slice stack: 8 x 8
    (11, 1 << 30),                           # one slice per chunk
    (7, 1),                                  # everything in one chunk
    (130, 3 << 20)])
def test_chunk_ranges_cover_every_slice_once(nslice, slice_bytes):
    ranges = rec._chunk_ranges(nslice, slice_bytes)
    assert ranges[0][0] == 0 and ranges[-1][1] == nslice
    for (a0, a1), (b0, b1) in zip(ranges, ranges[1:]):
        assert a1 == b0 and a1 > a0
    sizes = [b - a for a, b in ranges]
    assert all(s == sizes[0] for s in sizes[:-1]) and sizes[-1] <= sizes[0]
    if sizes[0] >= 8:
        assert sizes[0] % 4 == 0
    assert sizes[0] * slice_bytes <= max(rec._CHUNK_BYTES, slice_bytes)


def test_stack_chunks_are_eight_slices():
    assert rec._chunk_ranges(64, 4 * (1801 * 2560 + 2560 * 2560))[0] == (0, 8)


@pytest.mark.parametrize("nslice,nrow,ncol,sizes", [
    (40, 1801, 7192, [16, 16, 8]),           # 1 slice in _CHUNK_BYTES
    (6, 1801, 5120, [6]),
    (64, 1801, 2560, [16] * 4),              # 8
    (20, 721, 2560, [8, 8, 4]),              # transfers hide the idle half
    (128, 901, 1024, [48, 48, 32]),
    (40, 100, 16384, [1] * 40),              # few angles
    (9, 60000, 32768, [2, 2, 2, 2, 1])])     # no group in _GROUP_BYTES
def test_matrix_stacks_stream_in_whole_groups(nslice, nrow, ncol, sizes):
    ranges = rec._chunk_ranges(nslice, 4 * (nrow * ncol + ncol * ncol), nrow)
    assert [b - a for a, b in ranges] == sizes
    assert ranges[0][0] == 0 and ranges[-1][1] == nslice


def test_streaming_threshold():
    small = np.zeros((10, 3, 20), np.float32)
    assert not rec._streams(small, 20)
    big = np.lib.stride_tricks.as_strided(np.zeros(1, np.float32),
                                          (1801, 64, 2560), (0, 0, 0))
    assert rec._streams(big, 2560)
    one = np.lib.stride_tricks.as_strided(np.zeros(1, np.float32),
                                          (1801, 1, 8192), (0, 0, 0))
    assert not rec._streams(one, 8192)      # a single slice never streams


@pytest.mark.parametrize("shape,src_dtype,dst_dtype", [
    ((37, 20, 50), np.uint16, np.float32),   # rows >= workers, cast
    ((3, 700, 900), np.float32, np.float32), # rows < workers: split axis 1
    ((5000,), np.float64, np.float64),       # 1D
    ((2, 3), np.float32, np.float32)])       # below the threading size
def test_threaded_copy_strided_and_cast(shape, src_dtype, dst_dtype):
    rng = np.random.default_rng(len(shape))
    big = (rng.random(tuple(2 * n for n in shape)) * 1000).astype(src_dtype)
    src = big[tuple(slice(None, None, 2) for _ in shape)]
    dst_big = np.zeros(tuple(n + 1 for n in shape), dst_dtype)
    dst = dst_big[tuple(slice(1, None) for _ in shape)]
    _host._copy(dst, src)
    assert np.array_equal(dst, src.astype(dst_dtype))
    assert not dst_big[(0,) * len(shape)]


def test_to_host_of_host_tensor():
    import torch
    t = torch.arange(12, dtype=torch.float32).reshape(3, 4)
    out = _host.to_host(t)
    assert isinstance(out, np.ndarray) and np.array_equal(out, t.numpy())


@pytest.mark.parametrize("nrow,nslice,ncol,f32seq,f32,f16", [
    (128, 6, 64, True, False, False),
    (127, 64, 2560, False, False, True),
    (128, 5, 2560, False, False, False),
    (361, 9, 640, True, False, False),       # half-filled rounds of the chip
    (361, 17, 640, True, False, True),
    (361, 20, 640, True, False, True),
    (361, 21, 640, True, True, True),
    (128, 48, 640, True, True, False),
    (361, 16, 512, True, False, True),
    (361, 17, 512, True, True, True),
    (255, 12, 1024, True, False, True),
    (256, 9, 1024, True, True, True),
    (361, 8, 1024, True, False, False),
    (361, 12, 1500, True, False, True),
    (361, 13, 1024, True, True, True),
    (128, 24, 256, True, False, True),
    (128, 25, 256, True, False, False),
    (128, 48, 384, True, False, True),
    (256, 48, 256, True, False, True),
    (64, 9, 1000, False, False, True),
    (63, 9, 1000, False, False, False),
    (64, 16, 512, False, False, True),
    (64, 17, 512, False, False, False),
    (127, 17, 640, False, False, False),
    (128, 17, 640, True, False, True),
    (128, 33, 640, True, True, False),
    (256, 33, 640, True, True, True),
    (1801, 64, 32769, False, False, False),
    (65536, 64, 2560, False, False, False)])
def test_matrix_rule(nrow, nslice, ncol, f32seq, f32, f16):
    """Where stacks go to the matrix cores: only where they measured faster
    than the vector kernel there."""
    import torch
    from algotom_amd import _native as nat
    rule = rec._matrix_stack
    assert rule(nrow, nslice, ncol, nat.ACC_F32SEQ, torch.float32) == f32seq
    assert rule(nrow, nslice, ncol, nat.ACC_F32, torch.float32) == f32
    for dtype in (torch.float16, torch.bfloat16):
        assert rule(nrow, nslice, ncol, nat.ACC_F32, dtype) == f16
        assert not rule(nrow, nslice, ncol, nat.ACC_F32SEQ, dtype)
    assert not rule(nrow, nslice, ncol, nat.ACC_F64, torch.float32)
