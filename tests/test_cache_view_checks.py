"""The one-expression checks of the cache views accept exactly what the rule-by-rule ones do (CPU)."""
from __future__ import annotations

import pytest
import torch

from k8v4_v030 import ops_api
from k8v4_v030.cache_views import bind_regions
from k8v4_v030.layout import PageLayout


def _views(hkv=4, d=128, pages=3):
    lay = PageLayout(hkv, d)
    return bind_regions(torch.zeros(pages * lay.page_bytes, dtype=torch.int8), lay)


def _variants(t):
    """The view itself, then other dtypes, ranks, shapes and strides."""
    yield t
    yield t.contiguous()
    yield t.to(torch.float16)
    yield t.reshape(-1)
    yield t[None]
    yield t[0]
    yield t.sum()
    yield t[:2]
    yield t[:, :32]
    yield t[:, :, :2]
    yield t[..., :1]
    yield t.transpose(1, 2)
    yield t.transpose(0, 1).contiguous().transpose(0, 1)
    yield torch.empty((0,) + tuple(t.shape[1:]), dtype=t.dtype)


def _refusal(call):
    try:
        call()
    except Exception as e:  # noqa: BLE001 - the kind and text of any refusal are compared
        return type(e), str(e)
    return None


@pytest.mark.parametrize("hkv,d", [(4, 128), (2, 256)])
def test_same_refusals(hkv, d):
    v = _views(hkv, d)
    accepted = refused = 0
    for name in ("k", "k_scale"):
        for t in _variants(v[name]):
            args = [t if name == x else v[x] for x in ("k", "k_scale")] + [hkv, d]
            got = _refusal(lambda: ops_api.check_paged_k(*args))
            assert got == _refusal(lambda: ops_api._reject_paged_k(*args)), (name, t.shape)
            accepted, refused = accepted + (got is None), refused + (got is not None)
    for name in ("v", "v_scale", "v_zero"):
        for t in _variants(v[name]):
            args = [t if name == x else v[x] for x in ("v", "v_scale", "v_zero")] + [hkv, d]
            got = _refusal(lambda: ops_api.check_paged_v(*args))
            assert got == _refusal(lambda: ops_api._reject_paged_v(*args)), (name, t.shape)
            accepted, refused = accepted + (got is None), refused + (got is not None)
    assert accepted >= 5 and refused >= 30
    for rows in (torch.zeros(7, hkv, d), torch.zeros(7, 8 * hkv * d)[:, : hkv * d].unflatten(1, (hkv, d))):
        for t in _variants(rows.to(torch.bfloat16)):
            assert _refusal(lambda: ops_api._src_rows(t, "k", hkv, d)) == _refusal(
                lambda: ops_api._reject_src_rows(t, "k", hkv, d)), t.shape
