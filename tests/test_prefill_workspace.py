"""A prefill workspace sized for the longest call serves every shorter one (CPU).

Scratch is allocated once for the longest chunk over the longest context, while
the library chooses by size how many KV heads' tile images share a launch: the
size it asks for must not shrink as a call grows.
"""
from __future__ import annotations

import pytest

from k8v4_v030.ops_api import load_library


@pytest.mark.parametrize("hkv,d", [(2, 128), (4, 128), (2, 256), (4, 256)])
def test_workspace_grows_with_the_call(hkv, d):
    lib = load_library()
    contexts = [64, 65, 1000, 4096, 30000, 62000, 63000, 63500, 64000, 100000, 127000, 128000, 200000, 400000]
    chunks = [1, 11, 64, 128, 129, 200, 512, 1999, 4224]
    batch = lib.k8v4_prefill_batch_workspace_bytes(hkv, d)

    def need(ctx, q):
        return max(batch, lib.k8v4_prefill_workspace_bytes(ctx, min(q, ctx), hkv, d))

    for a, b in zip(contexts, contexts[1:]):
        for q in chunks:
            assert need(a, q) <= need(b, q), (a, b, q)
    for ctx in contexts:
        for p, q in zip(chunks, chunks[1:]):
            assert need(ctx, p) <= need(ctx, q), (ctx, p, q)
