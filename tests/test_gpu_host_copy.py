"""Copies between host arrays and the resident buffers: the packed path of small transfers, the staging ring at the edges
of its pieces, chunks and slots, unaligned offsets, pageable and pinned destinations (oracle: the bytes themselves, through
the library's device-to-device copy kernel)."""
import threading

import numpy as np
import pytest

import bfuse_project_amd as bf
from bfuse_project_amd import _lib

pytestmark = pytest.mark.gpu

N = 16777216                     # floats of copy_f32_16777216
SMALL, PIECE, FIRST, CHUNK, RING = (512 << 10) // 4, (64 << 10) // 4, (256 << 10) // 4, (2 << 20) // 4, (16 << 20) // 4


@pytest.fixture(scope="module")
def op():
    with bf.Operation("copy_f32_16777216", "bias_relu_4096") as o:
        yield o


@pytest.mark.parametrize("offset,count", [(0, 1), (3, 5), (1, SMALL), (0, SMALL + 1), (7, FIRST * 5 + 3), (0, 3 * FIRST), (4, 7 * FIRST + 1), (0, 9 * PIECE), (1, 9 * PIECE + 1),
                                          (3, 13 * PIECE - 1), (0, 4 * CHUNK), (2, 4 * CHUNK + 1), (0, RING), (5, RING + CHUNK + 1), (0, N)])
def test_a_part_goes_up_and_comes_back_unchanged(op, offset, count):
    rng = np.random.default_rng(count)
    x = rng.integers(0, 1 << 32, count, np.uint32).view(np.float32)
    zero = np.zeros(min(N, offset + count + 64), np.float32)
    op.upload_part(0, 0, 0, zero)
    op.upload_part(0, 0, offset, x)
    op.launch("kernel1")
    got = op.download_part(0, offset, count)                     # pinned when large
    assert np.array_equal(got.view(np.uint32), x.view(np.uint32))
    pageable = np.full(count, 7, np.float32)                     # memory of the caller's own
    _lib.check(op.l.bfuse_download_part(1, offset * 4, pageable.ctypes.data, pageable.nbytes))
    assert np.array_equal(pageable.view(np.uint32), x.view(np.uint32))
    rest = op.download_part(0, 0, zero.size)
    assert not rest[:offset].any() and not rest[offset + count:].any()


def test_the_last_of_many_uploads_without_a_wait_is_what_stands(op):
    count = SMALL + FIRST + 1
    for k in range(700):
        x = np.full(count, k, np.float32)
        op.upload_part(0, 0, 0, x)
    op.launch("kernel1")
    assert np.array_equal(op.download_part(0, 0, count), x)


def test_results_are_the_callers_own_and_may_be_operands(op):
    a = op.download(0)
    op.upload(0, np.arange(N, dtype=np.float32), np.zeros(1, np.float32))
    op.launch("kernel1")
    keep = a.copy()
    b = op.download(0)                                           # another buffer: `a` still holds the earlier result
    assert np.array_equal(a.view(np.uint32), keep.view(np.uint32)) and b.ctypes.data != a.ctypes.data
    address = a.ctypes.data
    del a
    op.upload(0, b[::-1], np.zeros(1, np.float32))
    op.upload(0, b, np.zeros(1, np.float32))                     # from pinned memory, in place
    op.launch("kernel1")
    c = op.download(0)                                           # the released buffer serves again
    assert c.ctypes.data == address and np.array_equal(c, np.arange(N, dtype=np.float32).reshape(c.shape))


def test_two_threads_each_with_a_side_of_its_own(op):
    """Uploads, single-kernel launches and downloads of one thread are not disturbed by another's, which waits at times of
    its own."""
    failures = []

    def work(side, mode, expect, sizes):
        rng = np.random.default_rng(side)
        try:
            for k in range(200):
                n = sizes[k % len(sizes)]
                x = rng.standard_normal(n).astype(np.float32)
                op.upload_part(side, 0, 0, x)
                op.launch(mode)
                got = op.download_part(side, 0, n)
                if not np.array_equal(got, expect(x)):
                    raise AssertionError(f"side {side}, repetition {k}, {n} floats")
        except Exception as e:
            failures.append(e)

    op.upload_part(1, 1, 0, np.zeros(op.k[1].shapes[1][0], np.float32))
    threads = [threading.Thread(target=work, args=a) for a in ((0, "kernel1", lambda x: x, (1000, 90000, 300000)), (1, "kernel2", lambda x: np.maximum(x, 0), (4096, 17, 2048)))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures
