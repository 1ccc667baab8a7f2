"""The measured workloads of the prefill -> decode cache hand-off: calls a serving engine makes through the library's
public entry points (sc_handoff.py, sc_wire.py), over the sizes, K/V formats and page tables it makes them with.

`append`   one prefill chunk's K/V written layer by layer (sc_kv_append_async / _q4), as a prompt or a few new tokens arrive
`carve`    a prefilled sequence into its decode slot, one launch (the hand-off inside one process)
`quant`    the same into int8 / q4_0 / K8V4 pools
`encode`   a slot written as a hand-off payload, with its hash
`mount`    a payload checked and mounted into a slot, through a decoder kept per slot
`handoff`  both ends of the same-GPU hand-off: encode with carries, then the carried mount
`batch`    many parked slots resumed from staging and a chunk appended to each, one launch
`park`     a slot parked to pinned host memory and resumed into another slot
"""
import ctypes as C
import sys
from pathlib import Path

import numpy as np
import torch  # before the library: the process then has one HIP runtime, torch's

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "strata-concurrent_amd"))
import sc_handoff as sc  # noqa: E402
import sc_wire  # noqa: E402

H, D, PS = 2, 256, 4
GEOKEY = [2560, 48, 4, 128, 16, 32, 4, 8192, 4096, 24, 2, 256, 128, 4, 4, 3, 1, 0]
GEOM_HASH, PACK_HASH = 0x1122334455667788, 0x0AABBCCDDEEFF001
FORMATS = {"int8": sc.SC_KV_INT8, "q4": sc.SC_KV_Q4, "k8v4": sc.SC_KV_K8V4}
ROW = {"f16": D * 2, "int8": D + 8, "q4": D // 32 * 18}


def listed():
    return [
        # the last few tokens of a prompt (or a speculated run) appended to every layer of a paged int8 slot: launches
        {"name": "append_7_int8", "kind": "append", "fmt": "int8", "layers": 48, "tokens": 7, "pos0": 4093, "paged": True},
        # one prefill chunk appended to every layer of a paged f16 slot
        {"name": "append_2048_f16", "kind": "append", "fmt": "f16", "layers": 48, "tokens": 2048, "pos0": 6141, "paged": True},
        # a short conversation's hand-off on the 16-layer configuration, its slot's plan re-pointed at the new sequence
        {"name": "carve_4096", "kind": "carve", "src": "f16", "layers": 16, "tokens": 4096, "paged": False, "retarget": True},
        # a 32K hand-off of odd length into a slot whose pages a fragmented allocator placed
        {"name": "carve_32749_paged", "kind": "carve", "src": "f16", "layers": 48, "tokens": 32749, "paged": True,
         "retarget": False},
        # the headline: the full-depth slot at 128K
        {"name": "carve_131072", "kind": "carve", "src": "f16", "layers": 48, "tokens": 131072, "paged": False,
         "retarget": False},
        # the quantizing hand-off, int8 through shuffled tables and the mixed format
        {"name": "quant_int8_30011_paged", "kind": "quant", "fmt": "int8", "layers": 48, "tokens": 30011, "paged": True},
        {"name": "quant_k8v4_98304", "kind": "quant", "fmt": "k8v4", "layers": 48, "tokens": 98304, "paged": False},
        # a paged slot leaves the process: its payload and hash
        {"name": "encode_16381_paged", "kind": "encode", "fmt": "f16", "layers": 48, "tokens": 16381, "paged": True},
        # a payload without carries (an arena's, another engine's) arrives
        {"name": "mount_131072", "kind": "mount", "fmt": "f16", "layers": 48, "tokens": 131072, "paged": False,
         "carried": False},
        # prefill and decode instances on one GPU
        {"name": "handoff_98304", "kind": "handoff", "fmt": "f16", "layers": 48, "tokens": 98304, "paged": False,
         "carried": True},
        # eight ragged slots of U[1K, 128K] tokens resumed and appended at once
        {"name": "batch_8", "kind": "batch", "slots": 8, "most": 131072, "chunk": 2048},
        # a paged 8K conversation parked and another's place taken back
        {"name": "park_8192_paged", "kind": "park", "layers": 48, "tokens": 8192, "paged": True},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["append", "carve", "carve", "quant", "encode", "mount", "handoff", "batch", "park"])
    layers, paged = rng.choice([16, 48, 48]), rng.random() < 0.5
    if kind == "append":
        return {"kind": kind, "fmt": rng.choice(["f16", "int8", "q4"]), "layers": layers, "tokens": _log(rng, 1, 4096),
                "pos0": _log(rng, 1, 16384) - 1, "paged": paged}
    if kind == "batch":
        return {"kind": kind, "slots": rng.randint(2, 8), "most": _log(rng, 2048, 65536), "chunk": _log(rng, 16, 2048)}
    if kind == "park":
        return {"kind": kind, "layers": layers, "tokens": _log(rng, 1024, 12288), "paged": paged}
    tokens = _log(rng, 1024, 131072)
    if kind == "carve":
        return {"kind": kind, "src": rng.choice(["f16", "f16", "f32"]), "layers": layers, "tokens": tokens, "paged": paged,
                "retarget": rng.random() < 0.5}
    if kind == "quant":
        return {"kind": kind, "fmt": rng.choice(["int8", "q4", "k8v4"]), "layers": layers, "tokens": tokens, "paged": paged}
    fmt = rng.choice(["f16", "f16", "int8"])   # slots in other formats than f16 have no page tables here
    return {"kind": kind, "fmt": fmt, "layers": layers, "tokens": tokens, "paged": paged and fmt == "f16",
            "carried": kind == "handoff" or (kind == "mount" and rng.random() < 0.5)}


# ---- buffers ---------------------------------------------------------------------------------------------------------

class Buf:
    """A torch tensor as the library's structures take a device buffer."""

    def __init__(self, t):
        self.t, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()

    def data_ptr(self):
        return self.ptr


def _geo(layers):
    return sc.geometry(n_layers=layers)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(shape, dtype, g):
    return Buf(torch.randn(shape, dtype=dtype, device="cuda", generator=g))


def _zeros(shape, dtype):
    return Buf(torch.zeros(shape, dtype=dtype, device="cuda"))


def _words(b):
    """A whole buffer as 64-bit words (its bits, whatever they mean)."""
    return b.t.reshape(-1).view(torch.int64)


def _prefill(geo, tokens, g, dtype=torch.float16, gdn=True):
    """A prefilled sequence: K and V rows of every attention layer, recurrence and conv rows of the others."""
    n = geo.n_gdn if gdn else 0
    S, hv, ch = geo.ssm_state_size, geo.ssm_v_heads, geo.ssm_conv_channels
    rows = min(tokens, geo.ssm_d_conv - 1)
    return sc.PrefillBuffers(geo, tokens, [_normal((tokens, H, D), dtype, g) for _ in range(geo.n_qsa)],
                             [_normal((tokens, H, D), dtype, g) for _ in range(geo.n_qsa)],
                             [_normal((hv, S, S), torch.float32, g) for _ in range(n)],
                             [_normal((rows, ch), torch.float32, g) for _ in range(n)], rows,
                             sc.SC_DTYPE_F16 if dtype == torch.float16 else sc.SC_DTYPE_F32)


def _tables(geo, pages, paged, g):
    """One shuffled page table per attention layer, or none (the identity layout)."""
    if not paged:
        return None
    return [Buf(torch.randperm(pages, device="cuda", generator=g).to(torch.int32)) for _ in range(geo.n_qsa)]


def _slot(geo, tokens, tables, g=None):
    """An f16 decode slot for `tokens` tokens: zeros, or (with a generator) a filled one."""
    pages = (tokens + PS - 1) // PS
    make = (lambda s, t: _normal(s, t, g)) if g is not None else _zeros
    k = [make((pages, H, PS, D), torch.float16) for _ in range(geo.n_qsa)]
    v = [make((pages, H, PS, D), torch.float16) for _ in range(geo.n_qsa)]
    gdn = make((geo.n_gdn, geo.gdn_row_floats), torch.float32)
    return sc.Slot(geo, pages, pages * PS, k, v, gdn, tables)


def _quant_slot(geo, fmt, tokens, tables):
    pages = (tokens + PS - 1) // PS
    rows = pages * H * PS
    k8, v8 = fmt != "q4", fmt == "int8"
    codes = lambda is8: [_zeros((rows, D if is8 else ROW["q4"]), torch.uint8) for _ in range(geo.n_qsa)]  # noqa: E731
    scales = lambda is8: [_zeros((rows, 4), torch.float16) for _ in range(geo.n_qsa)] if is8 else []  # noqa: E731
    gdn = _zeros((geo.n_gdn, geo.gdn_row_floats), torch.float32)
    return sc.QuantPools(geo, FORMATS[fmt], pages, pages * PS, codes(k8), codes(v8), scales(k8), scales(v8), gdn, tables)


def _layer_pools(geo, tokens, g=None):
    """An int8 slot with the indexer's rows (the layered slot a payload of that format comes from and goes to)."""
    def make(n):
        if g is None:
            return _zeros(n, torch.uint8)
        return Buf(torch.randint(0, 256, (n,), dtype=torch.uint8, device="cuda", generator=g))
    size = sc.layer_blob_bytes(geo, sc.SC_KV_INT8, True, tokens)
    bufs = [[make(n) for _ in range(geo.n_qsa)] if n else None for n in size]
    gdn = (geo.n_gdn, geo.gdn_row_floats)
    return sc.LayerPools(geo, sc.SC_KV_INT8, tokens, True, buffers=bufs,
                         gdn=_zeros(gdn, torch.float32) if g is None else _normal(gdn, torch.float32, g))


def _any_slot(case, geo, g):
    if case["fmt"] == "int8":
        cells = geo.cells(case["tokens"])
        return _layer_pools(geo, cells, g), _layer_pools(geo, cells)
    pages = (case["tokens"] + PS - 1) // PS
    src = _slot(geo, case["tokens"], _tables(geo, pages, case["paged"], g), g)
    return src, _slot(geo, case["tokens"], _tables(geo, pages, case["paged"], g))


# ---- a state, and one pass -------------------------------------------------------------------------------------------

def prepare(case, seed):
    g = _gen(seed)
    return {"append": _prepare_append, "carve": _prepare_carve, "quant": _prepare_quant, "encode": _prepare_wire,
            "mount": _prepare_wire, "handoff": _prepare_wire, "batch": _prepare_batch, "park": _prepare_park}[
                case["kind"]](case, g, int(seed))


def run(state):
    return state["run"](state)


def _prepare_append(case, g, seed):
    geo, T, pos0, fmt = _geo(case["layers"]), case["tokens"], case["pos0"], case["fmt"]
    pages = (pos0 + T + PS - 1) // PS
    src = _prefill(geo, T, g, torch.float32, gdn=False)
    tables = _tables(geo, pages, case["paged"], g)
    s = {"run": _run_append, "src": src, "tables": tables, "calls": [], "out": {}}
    for j in range(geo.n_qsa):
        K, V, table = src.k[j].ptr, src.v[j].ptr, tables[j].ptr if tables else None
        if fmt == "f16":
            k, v = _zeros((pages, H, PS, D), torch.float16), _zeros((pages, H, PS, D), torch.float16)
            s["calls"].append((sc.lib.sc_kv_append_async, (K, V, T, pos0, table, PS, k.ptr, v.ptr, None, None, None, None,
                                                           None, None, None)))
            s["out"][f"k{j:02d}"], s["out"][f"v{j:02d}"] = k.t, v.t
        elif fmt == "int8":
            k, v = _zeros((pages, H, PS, D), torch.int8), _zeros((pages, H, PS, D), torch.int8)
            ks, vs = _zeros((pages, H, PS, 4), torch.float16), _zeros((pages, H, PS, 4), torch.float16)
            s["calls"].append((sc.lib.sc_kv_append_async, (K, V, T, pos0, table, PS, None, None, k.ptr, v.ptr, ks.ptr,
                                                           vs.ptr, None, None, None)))
            s["out"].update({f"k{j:02d}": k.t, f"v{j:02d}": v.t, f"ks{j:02d}": ks.t, f"vs{j:02d}": vs.t})
        else:
            k, v = _zeros((pages, H, PS, ROW["q4"]), torch.uint8), _zeros((pages, H, PS, ROW["q4"]), torch.uint8)
            s["calls"].append((sc.lib.sc_kv_append_q4_async, (k.ptr, v.ptr, table, pos0, T, K, V, H, D, PS, None, None,
                                                              None)))
            s["out"][f"k{j:02d}"], s["out"][f"v{j:02d}"] = k.t, v.t
    return s


def _run_append(s):
    for fn, args in s["calls"]:
        sc.check(fn(*args), "append")
    return s["out"]


def _prepare_carve(case, g, seed):
    geo, tokens = _geo(case["layers"]), case["tokens"]
    src = _prefill(geo, tokens, g, torch.float16 if case["src"] == "f16" else torch.float32)
    slot = _slot(geo, tokens, _tables(geo, (tokens + PS - 1) // PS, case["paged"], g))
    s = {"src": src, "slot": slot, "plan": sc.plan_carve(geo, src, slot)}
    s["run"] = _run_retarget if case["retarget"] else _run_plan
    s["view"], s["keep"] = src.view()
    if case["src"] == "f16":
        s["out"] = [_words(b) for b in slot.buffers()]
    else:
        s["out"] = {**{f"k{j:02d}": b.t for j, b in enumerate(slot.k_pool)},
                    **{f"v{j:02d}": b.t for j, b in enumerate(slot.v_pool)}, "gdn": _words(slot.gdn)}
    return s


def _run_plan(s):
    s["plan"].launch()
    return s["out"]


def _run_retarget(s):
    """An engine with one plan per slot points it at the sequence that arrived."""
    sc.check(sc.lib.sc_plan_retarget(s["plan"].handle, C.byref(s["view"]), None), "sc_plan_retarget")
    s["plan"].launch()
    return s["out"]


def _prepare_quant(case, g, seed):
    geo, tokens = _geo(case["layers"]), case["tokens"]
    src = _prefill(geo, tokens, g, torch.float32)
    slot = _quant_slot(geo, case["fmt"], tokens, _tables(geo, (tokens + PS - 1) // PS, case["paged"], g))
    out = {"gdn": _words(slot.gdn)}
    for j in range(geo.n_qsa):
        out[f"k{j:02d}"], out[f"v{j:02d}"] = _words(slot.k_codes[j]), _words(slot.v_codes[j])
        if slot.k_scale:
            out[f"ks{j:02d}"] = slot.k_scale[j].t
        if slot.v_scale:
            out[f"vs{j:02d}"] = slot.v_scale[j].t
    return {"run": _run_plan, "src": src, "slot": slot, "plan": sc.plan_carve_quant(geo, src, slot), "out": out}


def _prepare_wire(case, g, seed):
    geo, tokens, kind = _geo(case["layers"]), case["tokens"], case["kind"]
    src, dst = _any_slot(case, geo, g)
    ids = ((np.arange(tokens, dtype=np.int64) * 7919 + seed) % 151_000).astype(np.int32)
    key = list(GEOKEY)
    key[1] = case["layers"]
    live, keep = sc_wire.make_live(key, ids, layer_hi=case["layers"], idx_dim=128)
    enc = sc_wire.Encoder(geo, src, tokens, live, GEOM_HASH, PACK_HASH)
    n = enc.bytes
    payload = _zeros((n + 255) // 256 * 256, torch.uint8)
    carry = _zeros((sc.carry_bytes(n) + 255) // 256 * 256, torch.uint8) if case.get("carried") else None
    s = {"src": src, "dst": dst, "keep": (live, keep), "enc": enc, "n": n, "payload": payload, "carry": carry}
    if carry is not None:
        enc.set_carry(carry.ptr)
    if kind != "encode":   # the decode side keeps one decoder per slot, opened on the first payload
        enc.encode(payload.ptr, n)
        s["hash"] = enc.hash()
        s["dec"] = sc_wire.Decoder(payload.ptr, n, geo, dst, payload_hash=s["hash"], check_hash=True,
                                   carry=carry.ptr if carry is not None else None)
        s["out"] = [_words(b) for b in dst.buffers()]
    s["run"] = {"encode": _run_encode, "mount": _run_mount, "handoff": _run_handoff}[kind]
    return s


def _signed(h):
    return h - (1 << 64) if h >= 1 << 63 else h


def _run_encode(s):
    s["enc"].encode(s["payload"].ptr, s["n"])
    return {"hash": _signed(s["enc"].hash()), "payload": _words(s["payload"])}


def _run_mount(s):
    s["dec"].reopen(s["payload"].ptr, s["n"], s["hash"], carry=s["carry"].ptr if s["carry"] is not None else None)
    s["dec"].restore()
    return s["out"]


def _run_handoff(s):
    s["enc"].encode(s["payload"].ptr, s["n"])
    s["hash"] = s["enc"].hash()
    return {"slot": _run_mount(s), "hash": _signed(s["hash"]), "payload": _words(s["payload"]), "carry": _words(s["carry"])}


def _batch_lens(case):
    """The slots' lengths: spread over [1K, most], none alike."""
    rng = np.random.default_rng(case["slots"] * 1_000_003 + case["most"])
    return [int(x) for x in rng.integers(1024, case["most"] + 1, size=case["slots"])]


def _prepare_batch(case, g, seed):
    geo, lens, chunk = _geo(48), _batch_lens(case), case["chunk"]
    n = len(lens)
    _, staging_bytes = sc.staging_layout(geo, lens)
    staging = Buf(torch.empty(staging_bytes // 8, dtype=torch.int64, device="cuda").random_(generator=g))
    chunks = [_prefill(geo, chunk, g, gdn=False) for _ in lens]
    need = [(L + chunk + PS - 1) // PS for L in lens]
    pages, arena_pages = max(need), sum(need) + 3
    order = torch.randperm(arena_pages, device="cuda", generator=g).to(torch.int32)
    tables, at = [], 0
    for k in need:
        t = torch.full((pages,), -1, dtype=torch.int32, device="cuda")
        t[:k] = order[at:at + k]
        at += k
        tables.append(Buf(t))
    arena = lambda: [_zeros((arena_pages, H, PS, D), torch.float16) for _ in range(geo.n_qsa)]  # noqa: E731
    ak, av = arena(), arena()
    gdn = [_zeros((geo.n_gdn, geo.gdn_row_floats), torch.float32) for _ in lens]
    lens_dev = Buf(torch.tensor(lens, dtype=torch.int64, device="cuda"))
    lens_out = _zeros(n, torch.int64)
    P = C.POINTER(C.c_void_p)
    arrays = [sc._ptrs([c.k[j].ptr for c in chunks for j in range(geo.n_qsa)]),
              sc._ptrs([c.v[j].ptr for c in chunks for j in range(geo.n_qsa)]),
              *(sc._ptrs([b.ptr for b in bs]) for bs in (ak, av, tables, gdn))]
    ck, cv, pk, pv, pt, pg = (C.cast(a, P) for a in arrays)
    desc = sc.BatchDesc(n_slots=n, lens=lens_dev.ptr, max_tokens=max(lens), staging=staging.ptr,
                        staging_bytes=staging_bytes, chunk_tokens=chunk, chunk_k=ck, chunk_v=cv, arena_k=pk, arena_v=pv,
                        arena_pages=arena_pages, tables=pt, table_pages=pages, gdn=pg, lens_out=lens_out.ptr)
    h = C.c_void_p()
    sc.check(sc.lib.sc_plan_resume_append(C.byref(geo), C.byref(desc), C.byref(h)), "sc_plan_resume_append")
    return {"run": _run_plan, "plan": sc.Plan(h.value, arrays), "keep": (staging, chunks, tables, lens_dev),
            "out": [_words(b) for b in ak + av + gdn] + [lens_out.t]}


def _prepare_park(case, g, seed):
    geo, tokens = _geo(case["layers"]), case["tokens"]
    pages = (tokens + PS - 1) // PS
    src = _slot(geo, tokens, _tables(geo, pages, case["paged"], g), g)
    dst = _slot(geo, tokens, _tables(geo, pages, case["paged"], g))
    _, n = sc.image_layout(geo, tokens)
    host = torch.zeros(n // 8, dtype=torch.int64, pin_memory=True)
    return {"run": _run_park, "geo": geo, "src": src, "dst": dst, "host": host, "n": n, "tokens": tokens,
            "out": [_words(b) for b in dst.buffers()]}


def _run_park(s):
    sc.park_async(s["geo"], s["src"], s["tokens"], s["host"].data_ptr(), s["n"])
    sc.resume_async(s["geo"], s["host"].data_ptr(), s["n"], s["tokens"], s["dst"])
    return {"image": s["host"], "slot": s["out"]}


# ---- what a pass cannot do without, and how results may differ ---------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "batch":
        geo, lens = _geo(48), _batch_lens(case)
        chunk = geo.n_qsa * 2 * case["chunk"] * H * D * 2
        return {"bytes": 2 * sum(sc.payload_bytes(geo, L) + chunk for L in lens), "flops": 0}
    geo, tokens = _geo(case["layers"]), case["tokens"]
    rows = geo.n_qsa * tokens * H            # K or V rows of all attention layers
    gdn = geo.n_gdn * geo.gdn_row_floats * 4
    if kind == "append":
        return {"bytes": 2 * rows * (D * 4 + ROW[case["fmt"]]), "flops": 0}
    if kind == "carve":
        return {"bytes": 2 * rows * (D * (2 if case["src"] == "f16" else 4) + D * 2) + 2 * gdn, "flops": 0}
    if kind == "quant":
        k, v = {"int8": ("int8", "int8"), "q4": ("q4", "q4"), "k8v4": ("int8", "q4")}[case["fmt"]]
        return {"bytes": rows * (2 * D * 4 + ROW[k] + ROW[v]) + 2 * gdn, "flops": 0}
    if case.get("fmt") == "int8":
        slot = geo.n_qsa * sum(sc.layer_blob_bytes(geo, sc.SC_KV_INT8, True, tokens)) + gdn
    else:
        slot = sc.payload_bytes(geo, tokens)
    # encode: the slot read, the payload written; mount: the payload read, the slot written; handoff, park: both
    return {"bytes": (4 if kind in ("handoff", "park") else 2) * slot, "flops": 0}


def tolerance(case):
    # moved bytes, rounded and quantized values and hashes are each one definite value: the reference's rounding rules
    # (nearest even to f16, the int8 and q4_0 codes) are the formats' definition
    return "exact"


def _placed(case, x, table, pages):
    """Rows x [T][H][n] at cells pos0 .. of a pool [pages][H][PS][n] through the table, zeros elsewhere."""
    T, n = x.shape[0], x.shape[2]
    cell = torch.arange(T, device="cuda") + case.get("pos0", 0)
    page = table.t.long()[cell // PS] if table is not None else cell // PS
    out = torch.zeros((pages, H, PS, n), dtype=torch.float64, device="cuda")
    out[page, :, cell % PS] = x
    return out


def exact(case, seed):
    """The computed outputs in 64 bits: f32 K/V rows placed (their f16 rounding is the pool's), and the int8 scales."""
    kind = case["kind"]
    if not (kind in ("append", "quant") or (kind == "carve" and case["src"] == "f32")):
        return None
    g, geo, tokens = _gen(seed), _geo(case["layers"]), case["tokens"]
    pages = (case.get("pos0", 0) + tokens + PS - 1) // PS
    src = _prefill(geo, tokens, g, torch.float32, gdn=kind != "append")
    tables = _tables(geo, pages, case["paged"], g)
    fmt = case.get("fmt", "f16")
    out = {}
    for j in range(geo.n_qsa):
        for name, x in (("k", src.k[j].t), ("v", src.v[j].t)):
            x, key, table = x.double(), f"{name}{j:02d}", tables[j] if tables else None
            if fmt == "f16":
                out[key] = _placed(case, x, table, pages)
                continue
            out[key] = None
            if fmt == "int8" or (fmt == "k8v4" and name == "k"):
                amax = x.reshape(tokens, H, 4, 64).abs().amax(-1)
                scales = _placed(case, amax / 127.0, table, pages)
                out[f"{name}s{j:02d}"] = scales if kind == "append" else scales.reshape(-1, 4)
    if kind != "append":
        out["gdn"] = None
    return out
