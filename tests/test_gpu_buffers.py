"""Copies between host and device: the short forms (words that travel as kernel arguments, small
read-backs through pinned memory) at the edges where the long ones take over, and what a copy
promises to other contexts."""
import numpy as np
import pytest

import karume_amd as ka

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("entry", ["upload", "write"])
@pytest.mark.parametrize("nbytes", [1, 3, 4, 1020, 1022, 1023, 1024, 1025, 1028, 4092, 4094, 4096,
                                    4097, 4100])
@pytest.mark.parametrize("at", [0, 1, 2, 4])
def test_bytes_go_up_and_come_back_whole(gpu_ctx, entry, nbytes, at):
    rng = np.random.default_rng(nbytes * 8 + at)
    around = rng.integers(0, 256, size=nbytes + 32, dtype=np.uint8)
    data = rng.integers(0, 256, size=nbytes, dtype=np.uint8)
    buf = gpu_ctx.upload(around)
    getattr(buf, entry)(data, byte_offset=at)
    assert np.array_equal(buf.download(np.uint8, (nbytes,), byte_offset=at), data)
    want = around.copy()
    want[at:at + nbytes] = data
    assert np.array_equal(buf.download(np.uint8, want.shape), want)
    buf.free()


@pytest.mark.parametrize("words", [1, 256, 257])
def test_an_upload_is_there_for_another_context_when_it_returns(gpu_ctx, words):
    """The uploading context's stream has work in front of the copy; the other context's stream
    is idle and does not wait for it."""
    other = ka.acquire_gpu(0)
    try:
        backlog = gpu_ctx.alloc(1 << 28)
        buf = gpu_ctx.zeros(words * 4)
        for turn in range(1, 4):
            data = np.arange(words, dtype=np.int32) + 1000 * turn
            for _ in range(20):
                backlog.zero()
            buf.upload(data)
            seen = other.borrow(buf.address, buf.nbytes).download(np.int32, (words,))
            assert np.array_equal(seen, data), turn
        backlog.free()
        buf.free()
    finally:
        gpu_ctx.sync()
        other.destroy()


def test_writes_are_seen_by_what_is_queued_behind_them(gpu_ctx):
    src, dst = gpu_ctx.zeros(1024), gpu_ctx.zeros(4 * 1024)
    for i in range(4):     # four versions of the same words, copied away one after the other
        src.write(np.full(256, i + 1, dtype=np.int32))
        gpu_ctx.copy(dst.offset(1024 * i), src, 1024)
    got = dst.download(np.int32, (4, 256))
    assert np.array_equal(got, np.repeat(np.arange(1, 5, dtype=np.int32)[:, None], 256, axis=1))
    src.free()
    dst.free()
