"""The calls that a program using this decoder makes, as cases whose time and outputs can be measured.

listed() gives twelve of them, draw() more of the same ranges; prepare() makes a case's inputs and plan, run() is one
pass through the public entry points, work() the bytes that a pass cannot do without and exact() the values that were
encoded. Every output is a whole number: decoded values, string offsets and bytes, selection bitmaps, encoded pages,
encoded sizes.

A case is a dict:
  op     decode (one column to values), select (a predicate on one column), stream (raw packed vectors), strings,
         rowgroup (many columns in one call), encode (values to pages), wizard (exact sizes of every candidate)
  kind   how the column's values look and which expression encodes them (KINDS)
  type   element type; vectors: 1024-value vectors of the column
  bits   width of the packed values, gaps or run values; keys: distinct dictionary values; run: mean run length
"""
from __future__ import annotations

import math

import numpy as np
import torch

import fastlanes_amd as fa
from fastlanes_amd import wizard
from fastlanes_amd import workloads as wl

# pool expression of each kind of column
KINDS = {"plain": 0, "ffor": 1, "delta": 11, "rle": 6, "dict": 17, "dict_delta": 22, "dict_rle": 27, "s_patch": 2,
         "b_patch": 4, "ll_patch": 5}
INT = {8: torch.int8, 16: torch.int16, 32: torch.int32, 64: torch.int64}
V = 1024  # values per vector


def listed() -> list[dict]:
    return [
        # One column chunk of a row-group (64 vectors): what a reader decodes when a query touches one column of one
        # row-group. Latency of a single launch.
        {"name": "delta_i64_chunk", "op": "decode", "kind": "delta", "type": "int64", "vectors": 64, "bits": 7},
        # Whole columns, at the sizes of the cascade workloads: sorted int64 timestamps (DELTA), uint32 runs (RLE),
        # int32 Zipf categories (DICT), two pages each.
        {"name": "delta_i64_column", "op": "decode", "kind": "delta", "type": "int64", "vectors": 65536, "bits": 7},
        {"name": "rle_u32_column", "op": "decode", "kind": "rle", "type": "uint32", "vectors": 65536, "bits": 20,
         "run": 16},
        {"name": "dict_i32_column", "op": "decode", "kind": "dict", "type": "int32", "vectors": 65536, "keys": 4096},
        # Narrow categorical codes of a ragged table: 16-bit values, a vector count that fills no launch evenly.
        {"name": "dict_u16_ragged", "op": "decode", "kind": "dict", "type": "uint16", "vectors": 20011, "keys": 300},
        # Measurements with 1% outliers: 64-bit values whose exceptions are patched over a narrow body.
        {"name": "patch_u64_column", "op": "decode", "kind": "s_patch", "type": "uint64", "vectors": 32768, "bits": 7},
        # The primitive alone on a large buffer: 32-bit FFOR at bit width 7, the bit-width sweep's case.
        {"name": "stream_u32_w7", "op": "stream", "kind": "ffor", "type": "uint32", "vectors": 262144, "bits": 7},
        # A text column: words of a 2000-word vocabulary, 8 to 64 bytes a string.
        {"name": "strings_text", "op": "strings", "kind": "text", "vectors": 2048, "lo": 8, "hi": 64},
        # A table: 48 columns of every kind and width and of unequal lengths, decoded by one call.
        {"name": "rowgroup_48", "op": "rowgroup", "kind": "mixed", "columns": 48, "lo": 64, "hi": 4096},
        # A scan's filter pushed into the decode: `amount < constant`, bitmaps instead of values.
        {"name": "select_i64", "op": "select", "kind": "ffor", "type": "int64", "vectors": 32768, "bits": 17,
         "pred": "<"},
        # Writing a column on the GPU: uint32 measurements to FFOR pages.
        {"name": "encode_ffor_u32", "op": "encode", "kind": "ffor", "type": "uint32", "vectors": 65536, "bits": 7},
        # Choosing the encoding of int64 columns: exact sizes of every candidate for 256 row-groups of 65536 values.
        {"name": "wizard_256", "op": "wizard", "kind": "families", "type": "int64", "vectors": 256 * 64},
    ]


def _log(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _column(rng, kinds, top: int) -> dict:
    kind = rng.choice(kinds)
    types = ["uint32", "int32", "uint64", "int64"] if kind.endswith("patch") else \
        ["uint8", "uint16", "int16", "uint32", "int32", "uint64", "int64"]
    t = rng.choice(types)
    W = np.dtype(t).itemsize * 8
    # 64-bit columns hold half the values: the same bytes
    c = {"kind": kind, "type": t, "vectors": _log(rng, 16, top // 2 if W == 64 else top) | rng.randrange(2)}
    if kind in ("dict", "dict_delta", "dict_rle"):
        c["keys"] = _log(rng, 2, 200 if W == 8 else 20000)
    elif kind in ("delta", "ffor", "s_patch", "b_patch", "ll_patch"):
        c["bits"] = rng.randrange(0 if kind == "ffor" else 1, min(W - 1, 24 if kind == "ffor" else 12))
    elif kind == "rle":
        c["bits"] = min(W, 20)
    if kind in ("rle", "dict_rle"):
        c["run"] = _log(rng, 2, 200)
    return c


def draw(rng) -> dict:
    op = rng.choice(["decode"] * 5 + ["select", "select", "stream", "strings", "strings", "rowgroup", "encode",
                                      "encode", "wizard"])
    if op == "decode":
        return {"op": op, **_column(rng, list(KINDS), 65536)}
    if op == "select":
        c = _column(rng, ["ffor", "delta", "rle", "dict", "s_patch", "dict_rle"], 65536)
        return {"op": op, **c, "pred": rng.choice(["<", ">", "==", "!=", "<=", ">="])}
    if op == "stream":
        t = rng.choice(["uint8", "uint16", "uint32", "uint64"])
        W = np.dtype(t).itemsize * 8
        return {"op": op, "kind": rng.choice(["ffor", "unpack"]), "type": t, "bits": rng.randrange(W + 1),
                "vectors": _log(rng, 16, 262144 * 32 // max(W, 32) // (2 if W == 64 else 1))}
    if op == "strings":
        lo = rng.randrange(1, 40)
        return {"op": op, "kind": "text", "vectors": _log(rng, 1, 2048), "lo": lo, "hi": lo + rng.randrange(1, 60)}
    if op == "rowgroup":
        return {"op": op, "kind": "mixed", "columns": rng.randrange(1, 49), "lo": 16, "hi": _log(rng, 64, 4096)}
    if op == "encode":
        return {"op": op, **_column(rng, ["plain", "ffor", "delta", "rle"], 65536)}
    return {"op": op, "kind": "families", "type": "int64", "vectors": 64 * _log(rng, 1, 256)}


# ---- inputs ----------------------------------------------------------------------------------------------------


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _randint(g, lo: int, hi: int, n: int) -> torch.Tensor:
    return torch.randint(lo, hi, (n,), generator=g, device="cuda", dtype=torch.int64)


def _runs(g, n: int, mean: float) -> torch.Tensor:
    """Run index of every value: runs of geometric length."""
    flags = torch.rand(n, generator=g, device="cuda") < 1.0 / mean
    return torch.cumsum(flags, 0)


def _zipf(g, n: int, n_keys: int, s: float = 1.1) -> torch.Tensor:
    p = 1.0 / torch.arange(1, n_keys + 1, device="cuda", dtype=torch.float64) ** s
    cdf = torch.cumsum(p / p.sum(), 0).float()
    r = torch.searchsorted(cdf, torch.rand(n, generator=g, device="cuda"))
    return r.clamp_(max=n_keys - 1)


def _keys(g, n_keys: int, W: int) -> torch.Tensor:
    """Distinct keys over the type's range, in random order."""
    if W <= 16:
        return torch.randperm(1 << W, generator=g, device="cuda")[:n_keys]
    step = (1 << (W - 2)) // n_keys
    k = torch.arange(n_keys, device="cuda", dtype=torch.int64) * step + _randint(g, 0, step, n_keys)
    return k[torch.randperm(n_keys, generator=g, device="cuda")]


def _values(case: dict, seed: int) -> torch.Tensor:
    """The column's values as a signed device tensor of the type's width (same bits)."""
    g, n, kind = _gen(seed), case["vectors"] * V, case["kind"]
    W = np.dtype(case["type"]).itemsize * 8
    if kind == "plain":
        x = _randint(g, -(1 << 63), (1 << 63) - 1, n)
    elif kind in ("ffor", "s_patch", "b_patch", "ll_patch"):
        bits = case["bits"]
        base = int(_randint(g, 0, max(1, (1 << (W - 2)) - (1 << bits)), 1))
        x = base + _randint(g, 0, 1 << bits, n)
        if kind != "ffor":  # 1% outliers anywhere in the type's range
            hit = torch.rand(n, generator=g, device="cuda") < 0.01
            x = torch.where(hit, _randint(g, -(1 << 63), (1 << 63) - 1, n), x)
    elif kind == "delta":
        x = 1_700_000_000_000_000_000 * (W == 64) + torch.cumsum(_randint(g, 1, 1 << case["bits"], n) if case["bits"] > 1
                                                                else _randint(g, 0, 2, n), 0)
    elif kind == "rle":
        r = _runs(g, n, case["run"])
        x = _randint(g, 0, 1 << case["bits"], n)[r]
    elif kind == "dict_rle":
        r = _runs(g, n, case["run"])
        x = _keys(g, case["keys"], W)[_zipf(g, n, case["keys"])[r]]
    elif kind in ("dict", "dict_delta"):
        x = _keys(g, case["keys"], W)[_zipf(g, n, case["keys"])]
    elif kind == "families":  # row-groups of the wizard's five families in turn
        n_rg = n // wizard.RG
        x = torch.empty(n, dtype=torch.int64, device="cuda")
        for r in range(n_rg):
            a, b = r * wizard.RG, (r + 1) * wizard.RG
            u = [int(q) for q in np.random.default_rng([seed, r]).integers(0, 1 << 30, 3)]
            m = wizard.RG
            fam = r % 5
            if fam == 0:
                x[a:b] = _randint(g, 0, 1 << (1 + u[0] % 40), m)
            elif fam == 1:
                x[a:b] = u[1] + torch.cumsum(_randint(g, 0, (1 << (u[0] % 17)) + 1, m), 0)
            elif fam == 2:
                x[a:b] = _randint(g, 0, 1 << (4 + u[0] % 29), m)[_runs(g, m, 2.0 + u[1] % 126)]
            elif fam == 3:
                nk = 16 << (u[0] % 13)
                x[a:b] = _randint(g, 0, 1 << (16 + u[1] % 32), nk)[_zipf(g, m, nk, 0.8 + (u[2] % 9) / 10)]
            else:
                y = u[1] + _randint(g, 0, 1 << (1 + u[0] % 24), m)
                hit = torch.rand(m, generator=g, device="cuda") < 0.01
                x[a:b] = torch.where(hit, _randint(g, 0, 1 << 40, m), y)
    else:
        raise ValueError(kind)
    return x.to(INT[W])


def _host(x: torch.Tensor, dtype) -> np.ndarray:
    return x.cpu().numpy().view(np.dtype(dtype))


def _packed(case: dict, seed: int):
    """A raw stream: packed bytes (any bytes are a valid packing) and one base per vector (FFOR)."""
    g, n_vec, W, bw = _gen(seed), case["vectors"], np.dtype(case["type"]).itemsize * 8, case["bits"]
    packed = torch.randint(0, 256, (n_vec * 128 * bw,), generator=g, device="cuda", dtype=torch.uint8)
    bases = None
    if case["kind"] == "ffor":
        bases = _randint(g, 0, max(1, 1 << min(W - bw, 62)), n_vec).to(INT[W])
    return packed, bases


def _text(case: dict, seed: int):
    """Strings cut from a text of vocabulary words: offsets (n + 1) and bytes, on the host."""
    g, n = _gen(seed), case["vectors"] * V
    words = [w + b" " for w in wl.vocabulary(2000)]
    ln = torch.tensor([len(w) for w in words], device="cuda")
    start = torch.cumsum(ln, 0) - ln
    chars = torch.frombuffer(bytearray(b"".join(words)), dtype=torch.uint8).cuda()
    # every length equally often, in random order: the same number of bytes for every seed
    lens = case["lo"] + torch.arange(n, device="cuda") % (case["hi"] - case["lo"] + 1)
    lens = lens[torch.randperm(n, generator=g, device="cuda")]
    offs = torch.cat([torch.zeros(1, dtype=torch.int64, device="cuda"), torch.cumsum(lens, 0)])
    total = int(offs[-1])
    idx = _randint(g, 0, len(words), total // 4 + 16)  # every word piece has at least 4 bytes
    pl = ln[idx]
    ends = torch.cumsum(pl, 0)
    idx = idx[: int(torch.searchsorted(ends, total)) + 1]
    pl, ends = ln[idx], ends[: idx.numel()]
    src = torch.repeat_interleave(start[idx] - (ends - pl), pl)[:total]
    return offs, chars[src + torch.arange(total, device="cuda")]


def _table(case: dict, seed: int):
    """Column specs of a mixed table, from the case alone: every width and kind, unequal lengths."""
    r = np.random.default_rng([case["columns"], case["lo"], case["hi"]])
    kinds = ["plain", "ffor", "ffor", "delta", "rle", "dict", "dict_delta"]
    out = []
    for c in range(case["columns"]):
        W = (8, 16, 32, 64)[c % 4]
        kind = kinds[int(r.integers(len(kinds)))]
        nv = int(np.exp(r.uniform(np.log(case["lo"]), np.log(case["hi"] + 1))))
        out.append({"kind": kind, "type": f"uint{W}", "vectors": max(1, nv), "bits": int(r.integers(1, min(W - 1, 20) + 1))
                    if kind != "rle" else min(W, 20), "keys": int(r.integers(4, 200 if W == 8 else 4097)), "run": 16})
    return [(s, seed * 101 + c) for c, s in enumerate(out)]


# ---- the interface ----------------------------------------------------------------------------------------------


def prepare(case: dict, seed: int) -> dict:
    op = case["op"]
    st = {"op": op, "case": case, "stream": fa.stream_ptr()}
    if op in ("decode", "select"):
        x = _host(_values(case, seed), case["type"])
        enc = fa.encode_from_memory(x, KINDS[case["kind"]])
        st["plan"] = fa.Plan(enc, x.dtype)
        st["in"] = torch.from_numpy(enc).cuda()
        if op == "decode":
            st["out"] = torch.empty(x.size, dtype=INT[x.itemsize * 8], device="cuda")
        else:
            at = np.random.default_rng(seed).uniform(0.05, 0.95)  # the share of values that pass `<`
            st["const"] = np.sort(x[:: max(1, x.size // 4096)])[int(at * min(4096, x.size))]
            st["bitmap"] = torch.empty(16 * case["vectors"], dtype=torch.int64, device="cuda")
            st["counts"] = torch.empty(case["vectors"], dtype=torch.int32, device="cuda")
    elif op == "stream":
        W = np.dtype(case["type"]).itemsize * 8
        st["in"], st["bases"] = _packed(case, seed)
        st["out"] = torch.empty(case["vectors"] * V, dtype=INT[W], device="cuda")
    elif op == "strings":
        offs, data = _text(case, seed)
        enc = fa.encode_strings(offs.cpu().numpy().astype(np.uint32), data.cpu().numpy())
        st["plan"] = fa.Plan(enc, "str")
        st["in"] = torch.from_numpy(enc).cuda()
        st["offsets"] = torch.empty(offs.numel(), dtype=torch.int64, device="cuda")
        st["bytes"] = torch.empty(data.numel(), dtype=torch.uint8, device="cuda")
    elif op == "rowgroup":
        encs, types, offs, at = [], [], [], 0
        for spec, s in _table(case, seed):
            x = _host(_values(spec, s), spec["type"])
            encs.append(fa.encode_from_memory(x, KINDS[spec["kind"]]))
            types.append(x.dtype)
            offs.append(at)
            at += (encs[-1].size + 255) // 256 * 256
        buf = np.zeros(at, dtype=np.uint8)
        for e, o in zip(encs, offs):
            buf[o: o + e.size] = e
        st["rg"] = fa.RowGroup(encs, types, offs)
        st["in"] = torch.from_numpy(buf).cuda()
        st["raw"] = torch.empty(st["rg"].total_bytes, dtype=torch.uint8, device="cuda")
        st["out"] = [st["raw"][o: o + spec["vectors"] * V * t.itemsize].view(INT[t.itemsize * 8])
                     for o, t, (spec, _) in zip(st["rg"].offsets, types, _table(case, seed))]
    elif op == "encode":
        st["in"] = _values(case, seed)
        st["out"] = torch.zeros(st["in"].numel() * st["in"].element_size() + case["vectors"] * 512 + 4096,
                                dtype=torch.uint8, device="cuda")
    else:
        st["in"] = _values(case, seed)
        n_rg = st["in"].numel() // wizard.RG
        st["sizes"] = torch.empty((n_rg, len(wizard.candidates())), dtype=torch.int64, device="cuda")
        st["choice"] = torch.empty(n_rg, dtype=torch.int32, device="cuda")
    return st


def run(st: dict):
    op, s = st["op"], st["stream"]
    if op == "decode":
        out = st["out"]
        st["plan"].decode(st["in"].data_ptr(), out.data_ptr(), out.numel() * out.element_size(), s)
        return out
    if op == "select":
        st["plan"].select(st["in"].data_ptr(), st["case"]["pred"], st["const"], st["bitmap"].data_ptr(),
                          st["counts"].data_ptr(), s)
        return {"bitmap": st["bitmap"], "counts": st["counts"]}
    if op == "stream":
        c = st["case"]
        fa.unffor_stream(np.dtype(c["type"]).itemsize * 8, c["bits"], st["in"].data_ptr(),
                         None if st["bases"] is None else st["bases"].data_ptr(), st["out"].data_ptr(), c["vectors"], s)
        return st["out"]
    if op == "strings":
        st["plan"].decode_strings_fused(st["in"].data_ptr(), st["offsets"].data_ptr(), st["bytes"].data_ptr(),
                                        st["bytes"].numel(), s)
        return {"bytes": st["bytes"], "offsets": st["offsets"]}
    if op == "rowgroup":
        st["rg"].decode(st["in"].data_ptr(), st["raw"].data_ptr(), 0, s)
        return st["out"]
    if op == "encode":
        c = st["case"]
        size = fa.gpu_encode(st["in"].data_ptr(), st["in"].numel(), np.dtype(c["type"]), KINDS[c["kind"]],
                             st["out"].data_ptr(), st["out"].numel(), s)
        return {"pages": st["out"], "size": size}
    n_rg = st["choice"].numel()
    wizard.exhaustive_sizes(st["in"].data_ptr(), n_rg, st["sizes"].data_ptr(), s)
    wizard.get_best(st["sizes"].data_ptr(), n_rg, st["choice"].data_ptr(), s)
    return {"sizes": st["sizes"], "choice": st["choice"]}


def _encoded_bytes(c: dict) -> float:
    """Encoded size of a column, from the page layouts: packed values and per-vector metadata."""
    nv, W, kind = c["vectors"], np.dtype(c["type"]).itemsize * 8, c["kind"]
    S = W // 8
    if kind == "plain":
        return nv * 1024 * S
    if kind == "ffor":
        return nv * (128 * c["bits"] + 1 + S)
    if kind.endswith("patch"):
        return nv * (128 * c["bits"] + 1 + S + 10 * (S + 2))
    if kind == "delta":
        return nv * (128 * min(W, c["bits"]) + 1 + S + 128)
    if kind == "rle":
        return nv * (1024 / c["run"] * S + 128 + 3 + 128)
    code = max(1, math.ceil(math.log2(c["keys"])))
    if kind == "dict_rle":
        return nv * (1024 / c["run"] * code / 8 + 128 + 3 + 128) + c["keys"] * S
    return nv * (128 * code + 5 + (128 * 2 if kind == "dict_delta" else 0)) + c["keys"] * S


def work(case: dict) -> dict:
    op, nv = case["op"], case["vectors"] if "vectors" in case else 0
    S = np.dtype(case["type"]).itemsize if "type" in case else 1
    if op in ("decode", "encode"):
        b = _encoded_bytes(case) + nv * V * S
    elif op == "select":
        b = _encoded_bytes(case) + nv * (128 + 4)
    elif op == "stream":
        b = nv * (128 * case["bits"] + V * S + (S if case["kind"] == "ffor" else 0))
    elif op == "strings":  # text compresses to about 0.7 of its bytes; a 4-byte end offset read, 8 bytes written
        b = nv * V * ((case["lo"] + case["hi"]) / 2 * 1.7 + 12)
    elif op == "rowgroup":
        b = sum(_encoded_bytes(s) + s["vectors"] * V * np.dtype(s["type"]).itemsize for s, _ in _table(case, 0))
    else:
        b = nv * V * 8 + nv / 64 * (16 * 8 + 4)
    return {"bytes": float(b), "flops": 0.0}


def exact(case: dict, seed: int):
    """What was encoded is what a decode returns; encoded bytes and sizes have no value outside this repository."""
    op = case["op"]
    if op == "decode":
        return _values(case, seed)
    if op == "strings":
        offs, data = _text(case, seed)
        return {"bytes": data, "offsets": offs}
    if op == "rowgroup":
        return [_values(s, q) for s, q in _table(case, seed)]
    if op == "stream":
        packed, bases = _packed(case, seed)
        W, bw, nv = np.dtype(case["type"]).itemsize * 8, case["bits"], case["vectors"]
        if bw == 0:
            out = torch.zeros((nv, V), dtype=INT[W], device="cuda")
        else:  # word w of lane i holds bits [w W, (w + 1) W) of the lane; value j its bits [j bw, (j + 1) bw)
            L = V // W
            words = packed.view(INT[W]).view(nv, bw, L)
            out = torch.empty((nv, W, L), dtype=INT[W], device="cuda")
            low = (1 << W) - 1
            for j in range(W):
                w, s = j * bw // W, j * bw % W
                v = (words[:, w].to(torch.int64) >> s) & (low >> s if s or W < 64 else -1)
                if s + bw > W:
                    v = v | (words[:, w + 1].to(torch.int64) << (W - s))
                out[:, j] = (v & ((1 << bw) - 1 if bw < 64 else -1)).to(INT[W])
            out = out.view(nv, V)
        if bases is not None:
            out = out + bases[:, None]
        return out.reshape(-1)
    return None
