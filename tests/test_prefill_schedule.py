"""The schedule of a batched prefill, replayed on the host (CPU).

The library's planning code and the piece arithmetic of its kernels are compiled
for the host and every work-group of a launch is walked: each step of the walk
has to advance, every page of every (KV head, row block) has to be taken exactly
once, and the merge has to name the pieces that were left.  Chunks of a few
tokens share the call with chunks long enough for tile images that do not fit
the workspace, in either order.
"""
from __future__ import annotations

import ctypes
import random
import shutil
import subprocess

import pytest

from conftest import REPO
from k8v4_v030 import _build

pytestmark = pytest.mark.skipif(shutil.which(_build.hipcc()) is None, reason="no hipcc")


@pytest.fixture(scope="module")
def replay(tmp_path_factory):
    so = tmp_path_factory.mktemp("schedule") / "replay.so"
    subprocess.run([_build.hipcc(), "-x", "hip", "--cuda-host-only", "-fuse-cuid=none", "-O1", "-std=c++17", "-fPIC",
                    "-shared", "-w", str(REPO / "tests" / "prefill_schedule_host.cpp"), "-o", str(so)],
                   check=True, capture_output=True, text=True)
    lib = ctypes.CDLL(str(so))
    lib.batch_workspace.restype = ctypes.c_int64
    lib.replay_message.restype = ctypes.c_char_p

    def run(hkv, d, chunks, cus=256, extra=0):
        """Sequences that shared a launch; ``extra`` workspace bytes beyond the least."""
        arr = ctypes.c_int64 * len(chunks)
        n = ctypes.c_int(-1)
        rc = lib.replay_batch(cus, hkv, d, len(chunks), arr(*[q for q, _ in chunks]), arr(*[s for _, s in chunks]),
                              ctypes.c_int64(lib.batch_workspace(cus, hkv, d) + extra), ctypes.byref(n))
        assert rc == 0, (hkv, d, chunks, lib.replay_message().decode())
        return n.value

    return run


@pytest.mark.parametrize("hkv,d,chunks", [
    (4, 128, [(64, 2048), (170, 16554)]), (4, 128, [(64, 2048), (2000, 4000)]),
    (4, 128, [(64, 564), (200, 17200)]), (2, 256, [(64, 2048), (512, 30000)]),
    (4, 256, [(1, 1), (4224, 20000), (33, 9000), (300, 70000)]),
])
def test_long_chunks_beside_short_ones(replay, hkv, d, chunks):
    assert replay(hkv, d, chunks) == len(chunks)
    assert replay(hkv, d, chunks[::-1]) == len(chunks)


@pytest.mark.parametrize("hkv,d,chunk,n,shared", [
    # one launch costs less than images of each chunk's own
    (2, 256, (150, 2150), 8, 8), (2, 256, (150, 5150), 2, 2), (4, 256, (300, 2300), 8, 8), (2, 256, (1000, 1000), 4, 4),
    (2, 256, (150, 9000), 4, 4), (4, 128, (1000, 9000), 8, 8),
    (4, 128, (150, 300), 8, 8), (2, 128, (300, 2300), 2, 2), (4, 128, (300, 65536), 1, 1), (4, 128, (2000, 2000), 4, 4),
    # images pay although a launch is shared, or the chunk is alone
    (2, 256, (150, 9000), 2, 0), (4, 128, (1000, 9000), 2, 0), (4, 256, (512, 8289), 4, 0), (2, 256, (150, 33000), 2, 0), (4, 256, (300, 2300), 1, 0), (4, 128, (4224, 32768), 2, 0),
    (4, 128, (1999, 1999), 1, 0),
])
def test_a_chunk_leaves_the_shared_launch_where_images_pay(replay, hkv, d, chunk, n, shared):
    room = 1 << 31
    assert replay(hkv, d, [chunk] * n, extra=room) == shared
    assert replay(hkv, d, [(0, 500)] + [chunk] * n, extra=room) == shared
    if n > 1:  # beside a short one
        assert replay(hkv, d, [chunk] * (n - 1) + [(17, 900)], extra=room) == (n if shared else 1)


@pytest.mark.parametrize("d", [128, 256])
def test_random_batches(replay, d):
    rng = random.Random(d)
    shared = 0
    for _ in range(300):
        chunks = []
        for _ in range(rng.randint(1, 13)):
            q = rng.choice((0, 1, rng.randint(1, 128), rng.randint(1, 128), rng.randint(129, 700), rng.randint(129, 4300)))
            chunks.append((q, q + rng.choice((0, rng.randint(0, 3000), rng.randint(0, 40000)))))
        shared += replay(rng.choice((2, 4)), d, chunks, cus=rng.choice((256, 256, 7, 100, 304)),
                         extra=rng.choice((0, 0, rng.randint(0, 1 << 27))))
    assert shared > 300
