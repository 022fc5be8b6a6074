"""Timed cases of the quantized paged-KV attention path.

Each case is one layer's work in a serving engine: the quantize-and-write of
new K/V rows, a decode or MTP-verify step over the cache, one sequence's
chunked prefill, or the short prefill chunks of a mixed step, through the op
table (``k8v4_v030.ops_api.ops()``).  ``listed()`` are fixed points, ``draw``
gives further ones of the same ranges: 2 or 4 KV heads (6 query heads each),
head dims 128 and 256, fp16 or bf16 activations, rows of their own or views of
a fused qkv buffer, one page or a 33-page manager block per block-table entry,
random physical pages, contexts up to 200,000 tokens in decode and 131,072 in
prefill.

``exact`` restates the ops in float64 torch: the K/V quantization rule, the
decode op's int8 query rows (part of that op's definition), bottom-right
causal softmax attention.
"""
from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "k8v4-xpu_amd"))

from k8v4_v030.cache_views import bind_regions  # noqa: E402
from k8v4_v030.layout import GQA, PAGE, PageLayout  # noqa: E402
from k8v4_v030.ops_api import ops  # noqa: E402

_REGIONS = ("k", "k_scale", "v", "v_scale", "v_zero")
_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
_CHUNK = 32768  # tokens generated and stored at a time


def listed():
    return [
        # One request decoding one token at a short context, called eagerly:
        # the store of the token's K/V and the attention, through the
        # validating calls a backend makes outside a captured graph.
        _case("step_1x2048_q1", "step", 4, 128, "fp16", False, 1, q_len=1, lens="2048", bound=False),
        # The same pair in an engine with 24 requests of uneven lengths on a
        # two-head rank at head dim 256: bf16 views of the fused qkv rows,
        # 2,112-token manager blocks.
        _case("step_24_ragged_q1_d256", "step", 2, 256, "bf16", True, 33, q_len=1, bound=True,
              lens="93 214 377 640 701 1025 1100 1333 1590 1817 2048 2300 2511 2777 3100 3501 "
                   "3999 4444 5005 5750 6144 7321 8190 9001"),
        # MTP verify of four 8K requests (six draft tokens each).
        _case("decode_4x8192_q7", "decode", 4, 128, "fp16", False, 1, q_len=7, lens="8192 8192 8192 8192", bound=True),
        # A serving batch: 40 requests of 0.3K to 16K tokens, two tokens each (one draft).
        _case("decode_40_ragged_q2", "decode", 4, 128, "bf16", True, 1, q_len=2, bound=True,
              lens=" ".join(str(300 + (i * i * 977) % 15701) for i in range(40))),
        # Long contexts: four requests of 128K tokens, MTP verify.
        _case("decode_4x131072_q7", "decode", 4, 128, "fp16", False, 1, q_len=7,
              lens="131072 131072 131072 131072", bound=False),
        # One very long request on a two-head rank at head dim 256, MTP verify.
        _case("decode_1x127853_q7_d256", "decode", 2, 256, "bf16", True, 33, q_len=7, lens="127853", bound=True),
        # Quantize-and-write of four scheduler chunks, inputs with outliers.
        _case("store_16896", "store", 4, 128, "fp16", False, 1, tokens=16896, pages=2048),
        # A whole prompt with nothing cached before it.
        _case("prefill_1999_fresh", "prefill", 4, 128, "bf16", True, 1, q_len=1999, seq_len=1999),
        # A medium chunk over a medium context at head dim 256.
        _case("prefill_512_over_7777_d256", "prefill", 4, 256, "fp16", False, 1, q_len=512, seq_len=8289),
        # The short chunks of one mixed step, one call.
        _case("prefill_8_chunks", "batch", 4, 128, "bf16", True, 1,
              q_lens="17 33 64 64 90 101 128 128", lens="800 1733 64 4164 2090 101 8128 500"),
        # A full scheduler chunk over a long cached context, both head dims
        # (head dim 256 as the two-head rank runs it).
        _case("prefill_4224_over_131072", "prefill", 4, 128, "fp16", False, 1, q_len=4224, seq_len=135296),
        _case("prefill_4224_over_59500_d256", "prefill", 2, 256, "bf16", True, 33, q_len=4224, seq_len=63724),
    ]


def draw(rng):
    kind = rng.choice(("store", "step", "decode", "prefill", "prefill", "batch"))
    hkv, d = rng.choice((2, 4)), rng.choice((128, 256))
    dtype, fused, ppb = rng.choice(("fp16", "bf16")), rng.choice((False, True)), rng.choice((1, 1, 33))
    if kind == "store":
        return _case(None, kind, hkv, d, dtype, fused, 1, tokens=_log_int(rng, 1, 16896), pages=2048)
    if kind in ("step", "decode"):
        q_len, batch = rng.choice((1, 1, 2, 4, 7, rng.randint(1, 10))), _log_int(rng, 1, 48)
        budget = 524288 * 128 // d * 4 // hkv
        top = min(200000, budget // batch)
        lens = [_log_int(rng, min(top, q_len + 64), top) for _ in range(batch)]
        return _case(None, kind, hkv, d, dtype, fused, ppb, q_len=q_len, lens=_text(lens), bound=rng.random() < 0.75)
    if kind == "prefill":
        q_len = _log_int(rng, 11, 4224)
        ctx = 0 if rng.random() < 0.25 else _log_int(rng, 64, 131072)
        # Head dim 256 takes about twice as long per operation.
        limit = (6.9e12 if d == 128 else 3.3e12) / (4.0 * d * GQA * hkv * q_len)
        ctx = max(0, min(ctx, int(limit) - q_len))
        return _case(None, kind, hkv, d, dtype, fused, ppb, q_len=q_len, seq_len=q_len + ctx)
    q_lens = [_log_int(rng, 11, 128) for _ in range(rng.randint(2, 12))]
    lens = [q + (0 if rng.random() < 0.25 else _log_int(rng, 64, 16384)) for q in q_lens]
    return _case(None, kind, hkv, d, dtype, fused, ppb, q_lens=_text(q_lens), lens=_text(lens))


def prepare(case, seed):
    dev = torch.device("cuda")
    lay = PageLayout(case["hkv"], case["head_dim"])
    o = ops()
    seqs = _sequences(case)
    table, pages = _table(case, seed, seqs)
    raw = torch.zeros(pages * lay.page_bytes, dtype=torch.int8, device=dev)
    views = bind_regions(raw, lay)
    regions = tuple(views[name] for name in _REGIONS)
    st = {"kind": case["kind"], "ops": o, "raw": raw, "regions": regions}
    if case["kind"] == "store":
        k, v = next(iter(_kv(case, seed)))[1:3]
        st.update(new=(k, v, _slots(case, seed).to(dev)))
        return st
    table = table.to(dev)
    q = _queries(case, seed)
    q_len = case.get("q_len", 0)
    for first, k, v, b in _kv(case, seed):
        # A step's own tokens are not cached yet: its run stores them.
        m = min(k.shape[0], seqs[b] - q_len - first) if case["kind"] == "step" else k.shape[0]
        if m > 0:
            o.kv_store_paged(k[:m], v[:m], _positions(case, table[b], first, m), *regions)
    # Outputs are rows of their own in the activations' type.
    out = torch.empty((q.shape[0], lay.hq, lay.head_dim), dtype=q.dtype, device=dev)
    seq_lens = torch.tensor(seqs, dtype=torch.int32, device=dev)
    scale = 1.0 / math.sqrt(lay.head_dim)
    st["out"] = out
    if case["kind"] in ("decode", "step"):
        nbytes = o.attn_workspace_bytes(len(seqs), table.shape[1], case["ppb"], q_len, lay.hkv, lay.head_dim)
        ws = torch.empty(-(-nbytes // 4), dtype=torch.float32, device=dev)
        args = (q, None, None, *regions, table, seq_lens, None, ws, None, None, None, out, q_len, case["ppb"])
        st["args"] = args
        st["call"] = o.bind_int8k_int4v_attn_batch(*args) if case["bound"] else None
        if case["kind"] == "step":
            st["new"] = _step_rows(case, seed, table)
            st["store"] = o.bind_kv_store_paged(*st["new"], *regions) if case["bound"] else None
    elif case["kind"] == "prefill":
        nbytes = o.prefill_workspace_bytes(seqs[0], q_len, lay.hkv, lay.head_dim)
        ws = torch.empty(max(4, -(-nbytes // 4)), dtype=torch.float32, device=dev)
        st["args"] = (q, *regions, table[0], seqs[0], case["ppb"], scale, out, ws)
    else:
        nbytes = o.prefill_batch_workspace_bytes(lay.hkv, lay.head_dim)
        ws = torch.empty(-(-nbytes // 4), dtype=torch.float32, device=dev)
        q_lens = _ints(case["q_lens"])
        tok0 = [sum(q_lens[:i]) for i in range(len(q_lens))]
        st["args"] = (q, *regions, table, tok0, q_lens, seqs, list(range(len(seqs))), case["ppb"], scale, out, ws)
    return st


def run(state):
    kind, o = state["kind"], state["ops"]
    if kind in ("store", "step"):
        if state.get("store") is not None:
            state["store"]()
        else:
            o.kv_store_paged(*state["new"], *state["regions"])
        if kind == "store":
            return state["raw"]
    if kind in ("decode", "step"):
        if state["call"] is not None:
            state["call"]()
        else:
            o.int8k_int4v_attn_batch(*state["args"])
        return (state["out"], state["raw"]) if kind == "step" else state["out"]
    if kind == "prefill":
        o.prefill_paged(*state["args"])
    else:
        o.prefill_paged_batch(*state["args"])
    return state["out"]


def work(case):
    hkv, d, kind = case["hkv"], case["head_dim"], case["kind"]
    slot = d + d // 2 + 12  # cache bytes of one (token, KV head)
    row = 2 * hkv * d  # activation bytes of one token's K, V or a sixth of its Q
    if kind == "store":
        n = case["tokens"]
        return {"bytes": n * (2 * row + 8 + hkv * slot), "flops": 0}
    seqs = _sequences(case)
    q_lens = _ints(case["q_lens"]) if kind == "batch" else [case["q_len"]] * len(seqs)
    tokens = sum(seqs)
    queries = sum(q_lens)
    pairs = sum(q * s - q * (q - 1) // 2 for q, s in zip(q_lens, seqs))
    nbytes = tokens * hkv * slot + 2 * queries * GQA * row + sum(4 * (-(-s // PAGE)) + 4 for s in seqs)
    if kind == "step":
        nbytes += queries * (2 * row + 8 + hkv * slot)
    return {"bytes": nbytes, "flops": 4 * d * GQA * hkv * pairs}


def tolerance(case):
    """About four times the measured distance from ``exact`` (cache bytes are whole).

    Measured: 2.6e-3 at most where a bf16 output's own rounding leads, 1.6e-3
    for a long fp16 prefill (fp16 keys and probabilities), 8e-4 for an fp16
    decode (integer scores)."""
    kind = case["kind"]
    if kind == "store":
        return "exact"
    if case["dtype"] == "bf16":
        return {"rel": 1e-2}
    return {"rel": 3e-3 if kind in ("decode", "step") else 6e-3}


def exact(case, seed):
    if case["kind"] == "store":
        return _exact_store(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    hkv, d, kind = case["hkv"], case["head_dim"], case["kind"]
    seqs = _sequences(case)
    q_lens = _ints(case["q_lens"]) if kind == "batch" else [case["q_len"]] * len(seqs)
    q = _queries(case, seed).double()
    if kind in ("decode", "step"):
        code, scale = _quant_k(q)
        q = code * scale[..., None]
    out = torch.empty((q.shape[0], GQA * hkv, d), dtype=torch.float64, device=dev)
    parts = {}
    for _, k, v, b in _kv(case, seed):
        kc, ks = _quant_k(k.double())
        vc, vs, vz = _quant_v(v.double())
        parts.setdefault(b, []).append((kc.to(torch.int8), ks.float(), vc.to(torch.int8), vs.float(), vz.float()))
    tok0 = 0
    for b, (n, ql) in enumerate(zip(seqs, q_lens)):
        kc, ks, vc, vs, vz = (torch.cat(x) for x in zip(*parts.pop(b)))
        end = n - ql + 1 + torch.arange(ql, device=dev)
        for h in range(hkv):
            kd = kc[:, h].double() * ks[:, h, None].double()
            vd = (vc[:, h].double() - vz[:, h, None].double()) * vs[:, h, None].double()
            step = max(1, (1 << 27) // (GQA * n))  # score rows of at most 1 GiB
            for j in range(0, ql, step):
                rows = q[tok0 + j : tok0 + min(ql, j + step), GQA * h : GQA * (h + 1)]
                s = torch.mm(rows.reshape(-1, d), kd.t().contiguous()) / math.sqrt(d)
                lim = end[j : j + step].repeat_interleave(GQA)
                s.masked_fill_(torch.arange(n, device=dev)[None, :] >= lim[:, None], -math.inf)
                p = torch.softmax(s, dim=1)
                out[tok0 + j : tok0 + j + rows.shape[0], GQA * h : GQA * (h + 1)] = torch.mm(p, vd).view(-1, GQA, d)
        tok0 += ql
    return (out, None) if kind == "step" else out


# ------------------------------------------------------------------ inputs
def _case(name, kind, hkv, head_dim, dtype, fused, ppb, **sizes):
    case = {"kind": kind, "hkv": hkv, "head_dim": head_dim, "dtype": dtype, "fused": fused, "ppb": ppb, **sizes}
    return case if name is None else {"name": name, **case}


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)) - 1e-9)))))


def _text(values):
    return " ".join(str(int(x)) for x in values)


def _ints(text):
    return [int(x) for x in text.split()]


def _sequences(case):
    """Cached tokens of each sequence, the call's own tokens included."""
    if case["kind"] == "store":
        return [case["tokens"]]
    return [case["seq_len"]] if case["kind"] == "prefill" else _ints(case["lens"])


def _generator(case, seed, what):
    return torch.Generator(device="cuda" if torch.cuda.is_available() else "cpu").manual_seed(1000003 * seed + what)


def _table(case, seed, seqs):
    """Random distinct block-table entries and the pages of the pool (a tenth spare)."""
    if case["kind"] == "store":
        return None, case["pages"]
    ppb = case["ppb"]
    need = [-(-n // (PAGE * ppb)) for n in seqs]
    pool = sum(need) + sum(need) // 10 + 2
    perm = torch.randperm(pool, generator=torch.Generator().manual_seed(1000003 * seed + 1)).to(torch.int32)
    table = torch.zeros((len(seqs), max(need)), dtype=torch.int32)
    at = 0
    for b, n in enumerate(need):
        table[b, :n] = perm[at : at + n]
        at += n
    return table, pool * ppb


def _positions(case, row, first, count):
    """Slots of tokens ``first .. first + count - 1`` through a block-table row."""
    t = torch.arange(first, first + count, device=row.device)
    page, ppb = t // PAGE, case["ppb"]
    return (row[page // ppb].long() * ppb + page % ppb) * PAGE + t % PAGE


def _slots(case, seed):
    """Store: runs of tokens in random pages."""
    n = case["tokens"]
    gen = torch.Generator().manual_seed(1000003 * seed + 1)
    perm = torch.randperm(case["pages"], generator=gen)[: -(-n // PAGE)]
    t = torch.arange(n)
    return perm[t // PAGE] * PAGE + t % PAGE


def _rows_of_fused(case, k, v):
    """K and V rows as views of one ``[T, (8 * hkv) * D]`` projection output."""
    hkv, d = case["hkv"], case["head_dim"]
    buf = torch.zeros((k.shape[0], (GQA + 2) * hkv * d), dtype=k.dtype, device=k.device)
    buf[:, GQA * hkv * d : (GQA + 1) * hkv * d] = k.reshape(k.shape[0], -1)
    buf[:, (GQA + 1) * hkv * d :] = v.reshape(k.shape[0], -1)
    return (buf[:, GQA * hkv * d : (GQA + 1) * hkv * d].unflatten(1, (hkv, d)),
            buf[:, (GQA + 1) * hkv * d :].unflatten(1, (hkv, d)))


def _kv(case, seed):
    """Yields (first token, K rows, V rows, sequence) in pieces.

    K has channels of uneven size, as rotary keys do; a store's rows carry 1 %
    of entries 20 times larger, the outliers a quantizer has to meet."""
    gen = _generator(case, seed, 2)
    dev, hkv, d, dtype = gen.device, case["hkv"], case["head_dim"], _DTYPES[case["dtype"]]
    channel = torch.exp(0.4 * torch.randn((hkv, d), generator=gen, device=dev))
    for b, n in enumerate(_sequences(case)):
        for first in range(0, n, _CHUNK):
            m = min(_CHUNK, n - first)
            k = torch.randn((m, hkv, d), generator=gen, device=dev) * channel
            v = torch.randn((m, hkv, d), generator=gen, device=dev)
            if case["kind"] == "store":
                k = torch.where(torch.rand(k.shape, generator=gen, device=dev) < 0.01, 20 * k, k)
                v = torch.where(torch.rand(v.shape, generator=gen, device=dev) < 0.01, 20 * v, v)
            k, v = k.to(dtype), v.to(dtype)
            if case["fused"] and case["kind"] == "store":
                k, v = _rows_of_fused(case, k, v)
            yield first, k, v, b


def _step_rows(case, seed, table):
    """K/V rows and slots of the step's own tokens (the last q_len of each sequence)."""
    seqs, ql = _sequences(case), case["q_len"]
    tails = {}
    for first, k, v, b in _kv(case, seed):
        lo = max(seqs[b] - ql, first)
        if lo < first + k.shape[0]:
            tails.setdefault(b, []).append((k[lo - first :], v[lo - first :]))
    k = torch.cat([x for b in range(len(seqs)) for x, _ in tails[b]])
    v = torch.cat([x for b in range(len(seqs)) for _, x in tails[b]])
    if case["fused"]:
        k, v = _rows_of_fused(case, k, v)
    slots = torch.cat([_positions(case, table[b], n - ql, ql) for b, n in enumerate(seqs)])
    return k, v, slots


def _queries(case, seed):
    hkv, d = case["hkv"], case["head_dim"]
    n = sum(_ints(case["q_lens"])) if case["kind"] == "batch" else case["q_len"] * len(_sequences(case))
    gen = _generator(case, seed, 3)
    q = (1.5 * torch.randn((n, GQA * hkv, d), generator=gen, device=gen.device)).to(_DTYPES[case["dtype"]])
    if not case["fused"]:
        return q
    buf = torch.zeros((n, (GQA + 2) * hkv * d), dtype=q.dtype, device=q.device)
    buf[:, : GQA * hkv * d] = q.reshape(n, -1)
    return buf[:, : GQA * hkv * d].unflatten(1, (GQA * hkv, d))


# ------------------------------------------------------- float64 restatement
def _quant_k(x):
    """Symmetric int8 codes (half away from zero) and scale of ``[..., D]`` doubles."""
    amax = x.abs().amax(-1)
    scale = amax / 127.0
    y = x * torch.where(amax == 0, torch.ones_like(scale), 1.0 / scale)[..., None]
    code = torch.where(y >= 0, torch.floor(y + 0.5), torch.ceil(y - 0.5)).clamp(-127, 127)
    return code, scale


def _quant_v(x):
    """Affine uint4 codes, scale and zero point of ``[..., D]`` doubles."""
    lo, hi = x.amin(-1), x.amax(-1)
    scale = ((hi - lo) / 15.0).clamp_min(1e-8)
    zero = torch.floor(-lo / scale + 0.5).clamp(0, 15)
    code = torch.floor(x / scale[..., None] + zero[..., None] + 0.5).clamp(0, 15)
    return code, scale, zero


def _exact_store(case, seed):
    """The cache bytes a store leaves in a zeroed pool (region-major pages)."""
    hkv, d, pages = case["hkv"], case["head_dim"], case["pages"]
    _, k, v, _ = next(iter(_kv(case, seed)))
    slots = _slots(case, seed).to(k.device)
    kc, ks = _quant_k(k.double())
    vc, vs, vz = _quant_v(v.double())
    packed = (vc[..., 0::2] + 16 * vc[..., 1::2]).to(torch.uint8)
    regions = []
    for rows in (kc.to(torch.int8), packed, ks.float(), vs.float(), vz.float()):
        rows = rows.reshape(rows.shape[0], -1).contiguous().view(torch.int8)
        region = torch.zeros((pages * PAGE, rows.shape[1]), dtype=torch.int8, device=k.device)
        region[slots] = rows
        regions.append(region.view(pages, -1))
    return torch.cat(regions, 1).reshape(-1)
