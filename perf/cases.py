"""The work that a polishing program has this library do, as measured cases.

Every case goes through the C ABI of libracon_hip.so (include/racon_hip.h), the
boundary a polisher binds to, with host buffers in and host buffers out (the
allocation-free aligner alone works on device buffers). Four kinds:

  poa     one batch of windows: upload, consensus kernels, download
  align   one batch of overlaps: upload, alignment, and either the edit
          operations (layers = False) or what a polisher takes from them: the
          breaking points and the window layers (layers = True)
  device  rh_align_run_noalloc on the caller's device buffers and stream
  serve   requests submitted together to a running server, waited for, fetched

Inputs are drawn on the GPU: random backbones, reads that are noisy copies of
a slightly different truth (substitutions, insertions and deletions at
0.4 : 0.2 : 0.4), Phred qualities of 8..30. Every output is a whole number or
a byte; buffers have the case's own size, zero past what a pass writes.
"""
import ctypes
import math

import numpy as np
import torch

import racon_amd
from racon_amd import _lib
from racon_amd.serving import PolishServer

SPLIT = (0.4, 0.2, 0.4)  # substitutions, insertions, deletions
DRAFT_ERROR = 0.03       # backbone against the truth the reads come from

LAYER = np.dtype([("sequence", "<u8"), ("quality", "<u8"), ("length", "<u4"), ("begin", "<u4"),
                  ("end", "<u4")], align=True)
WINDOW = np.dtype([("backbone", "<u8"), ("backbone_quality", "<u8"), ("backbone_length", "<u4"),
                   ("n_layers", "<u4"), ("layers", "<u8"), ("tgs", "<u4")], align=True)
PAIR = np.dtype([("query", "<u8"), ("query_length", "<u4"), ("target", "<u8"),
                 ("target_length", "<u4")], align=True)
SPAN = np.dtype([("t_begin", "<u4"), ("t_end", "<u4"), ("q_first", "<u4")])
SOURCE = np.dtype([("overlap", "<u4"), ("query_length", "<u4"), ("first_window", "<u8"),
                   ("quality", "<u8"), ("mirrored", "<u4"), ("reserved", "<u4")])


def poa(name, windows, length, depth, **more):
    """`windows` windows of `length` backbone bases (the last of each target of
    `target` windows is shorter), about `depth` layers each. read: length of
    short reads, 0 for reads longer than the window, of which `partial` begin
    or end inside it. spread: depths follow a gamma distribution in 5..200."""
    case = {"kind": "poa", "windows": windows, "length": length, "depth": depth, "error": 0.12,
            "partial": 0.12, "read": 0, "target": 20, "spread": False, "quality": True,
            "match": 3, "mismatch": -5, "gap": -4, "band": 0}
    case.update(more)
    return dict(case, name=name) if name else case


def align(name, pairs, mean, sd, **more):
    """`pairs` overlaps, target lengths lognormal(mean, sd) within 100..longest.
    error: of the query against the target's truth; target_error: of the
    target itself (reads against reads)."""
    case = {"kind": "align", "pairs": pairs, "mean": mean, "sd": sd, "longest": 40000,
            "error": 0.12, "target_error": 0.0, "layers": False, "window": 500}
    case.update(more)
    return dict(case, name=name) if name else case


def listed():
    return [
        # one window: a single correction step of an interactive caller
        poa("poa_one_window", 1, 500, 30),
        # a 50 kbp contig at 30x
        poa("poa_50kbp", 100, 500, 30),
        # a 5 Mbp contig at 50x, the throughput workload
        poa("poa_5mbp", 9980, 500, 52),
        # wider windows (-w 1000) at the uneven depth of a real assembly, two
        # read types' worth of error
        poa("poa_w1000", 1037, 1000, 28, spread=True, error=0.14),
        # fragment correction: reads as targets, no qualities, unit scores
        poa("poa_fragment", 4001, 500, 18, partial=0.35, quality=False, match=1, mismatch=-1,
            gap=-1),
        # short accurate reads over a contig (second-generation windows)
        poa("poa_short_reads", 800, 500, 110, read=150, error=0.01, match=5, mismatch=-4,
            gap=-8),
        # the banded mode (-b) on wide windows
        poa("poa_banded", 611, 1000, 30, band=256),
        # one short overlap
        align("align_one", 1, 1000, 0),
        # overlaps of a 50x contig to window layers, racon's align phase
        align("align_layers", 12000, 8000, 4000, layers=True),
        # long noisy overlaps between reads, edit operations returned
        align("align_long", 61, 30000, 9000, longest=60000, target_error=0.08),
        # device buffers to device buffers, as under graph capture
        {"name": "align_device", "kind": "device", "pairs": 48, "mean": 3000, "sd": 1500,
         "longest": 10000, "error": 0.12, "target_error": 0.0},
        # four requests of mixed size in one server
        {"name": "serve_four", "kind": "serve", "requests": 4, "windows": 40, "growth": 2.2,
         "length": 500, "depth": 30, "error": 0.12},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["poa", "poa", "poa", "align", "align", "device", "serve"])
    if kind == "poa":
        length = _log_int(rng, 150, 1200)
        depth = _log_int(rng, 3, 120)
        depth = max(3, min(depth, 40000 // length))
        most = int(0.7 * 9980 * 52 * 500 * 500 / (depth * length * length))
        windows = _log_int(rng, 1, max(2, min(8000, most)))
        scores = rng.choice([(3, -5, -4), (5, -4, -8), (1, -1, -1)])
        short = rng.random() < 0.2
        return poa(None, windows, length, depth, error=round(rng.uniform(0.01, 0.15), 3),
                   partial=round(rng.uniform(0.0, 0.4), 3),
                   read=rng.randint(100, 250) if short else 0, target=rng.randint(1, 40),
                   spread=rng.random() < 0.3 and depth >= 10 and windows >= 20,
                   quality=rng.random() < 0.7, match=scores[0], mismatch=scores[1],
                   gap=scores[2], band=256 if rng.random() < 0.15 else 0)
    if kind in ("align", "device"):
        mean = _log_int(rng, 150, 30000 if kind == "align" else 6000)
        most = int(0.7 * 12000 * 8000 / mean * min(1.0, 8000 / mean))
        pairs = _log_int(rng, 1, max(2, min(12000 if kind == "align" else 400, most)))
        case = align(None, pairs, mean, int(mean * rng.uniform(0.0, 0.6)),
                     longest=int(mean * 3) + 200, error=round(rng.uniform(0.01, 0.15), 3),
                     target_error=rng.choice([0.0, 0.0, round(rng.uniform(0.01, 0.12), 3)]),
                     layers=rng.random() < 0.5, window=rng.choice([500, 500, 1000, 200]))
        if kind == "device":
            case = dict(case, kind="device", longest=min(case["longest"], 12000))
            del case["layers"], case["window"]
        return case
    return {"kind": "serve", "requests": rng.randint(1, 6), "windows": _log_int(rng, 1, 80),
            "growth": round(rng.uniform(1.0, 2.2), 2), "length": _log_int(rng, 200, 800),
            "depth": _log_int(rng, 5, 60), "error": round(rng.uniform(0.02, 0.15), 3)}


# ---- inputs ----

def _generator(seed):
    device = "cuda" if torch.cuda.is_available() else "cpu"
    g = torch.Generator(device=device)
    g.manual_seed(int(seed))
    return g


def _spans(starts, lengths):
    """Flat indices starts[i] .. starts[i] + lengths[i] - 1 of every i."""
    ends = torch.cumsum(lengths, 0)
    total = int(ends[-1]) if len(ends) else 0
    shift = torch.repeat_interleave(starts - (ends - lengths), lengths, output_size=total)
    return shift + torch.arange(total, device=starts.device)


def _mutate(g, bases, lengths, rate):
    """Noisy copies of the segments of `bases` (codes 0..3, lengths[i] each);
    a segment's first base is never deleted. Returns (codes, lengths)."""
    n, dev = bases.numel(), bases.device
    sub, ins, dele = (rate * s for s in SPLIT)
    r = torch.rand(n, generator=g, device=dev)
    ends = torch.cumsum(lengths, 0)
    counts = torch.ones(n, dtype=torch.int32, device=dev)
    counts[(r >= sub + ins) & (r < sub + ins + dele)] = 0
    counts[ends - lengths] = 1
    is_ins = (r >= sub) & (r < sub + ins)
    counts[is_ins] = 2
    other = torch.randint(1, 4, (n,), generator=g, device=dev, dtype=torch.uint8)
    bases = torch.where(r < sub, (bases + other) & 3, bases)
    at = torch.cumsum(counts, 0, dtype=torch.int64)
    out = torch.repeat_interleave(bases, counts, output_size=int(at[-1]))
    second = at[is_ins] - 1
    out[second] = torch.randint(0, 4, (second.numel(),), generator=g, device=dev,
                                dtype=torch.uint8)
    seg_end = at[ends - 1]
    return out, torch.diff(seg_end, prepend=seg_end.new_zeros(1))


def _letters(codes):
    table = torch.tensor(list(b"ACGT"), dtype=torch.uint8, device=codes.device)
    return table[codes.int()].cpu().numpy()


def _qualities(g, n):
    q = torch.randint(41, 64, (n,), generator=g, device=g.device, dtype=torch.uint8)
    return q.cpu().numpy()


def _starts(lengths):
    """Exclusive prefix sums."""
    return torch.cumsum(lengths, 0) - lengths


def _windows(g, count, length, depth, error, partial=0.12, read=0, target=20, spread=False,
             quality=True):
    """rh_window records of `count` windows, and what they point into."""
    dev = g.device

    def rand(n):
        return torch.rand(n, generator=g, device=dev)

    n = torch.full((count,), length, dtype=torch.int64, device=dev)
    last = torch.arange(count, device=dev) % target == target - 1
    n = torch.where(last, (length * (0.2 + 0.8 * rand(count))).long(), n)
    backbone = torch.randint(0, 4, (int(n.sum()),), generator=g, device=dev, dtype=torch.uint8)
    truth, tn = _mutate(g, backbone, n, DRAFT_ERROR)
    if spread:
        d = -torch.log(rand(count).clamp_min(1e-9)) - torch.log(rand(count).clamp_min(1e-9))
        d = (d * depth / 2).long().clamp(5, 200)
    else:
        d = (depth * (0.8 + 0.4 * rand(count))).round().long().clamp_min(2)
    if read:
        d = d * math.ceil((length + read) / read)  # depth is per base
    layers = int(d.sum())
    w = torch.repeat_interleave(torch.arange(count, device=dev), d, output_size=layers)
    wl, u = n[w], rand(layers)
    least = torch.minimum(wl - 1, torch.full_like(wl, 20))
    if read:
        b = (u * (wl + read - 40)).long() - read + 20
        begin = torch.minimum(b.clamp_min(0), wl - 1 - least)
        end = torch.maximum(torch.minimum(b + read - 1, wl - 1), begin + least)
    else:
        kind = rand(layers)
        cut = least + (u * (wl - 1 - least)).long()
        zero, whole = torch.zeros_like(wl), wl - 1
        # the first and last match of a read that crosses the window lie on
        # its first and last bases or a few bases inside
        inset = [(rand(layers) < 0.12).long() + (rand(layers) < 0.02).long() for _ in range(2)]
        begin = torch.where(kind < partial / 2, whole - cut, inset[0])
        end = torch.where((kind >= partial / 2) & (kind < partial), cut, whole - inset[1])
        begin = torch.minimum(torch.maximum(begin, zero), whole - least.clamp_max(10))
        end = torch.maximum(end, begin + least.clamp_max(10))
    t0 = begin * tn[w] // wl
    t1 = torch.maximum(t0 + 1, (end + 1) * tn[w] // wl)
    codes, ln = _mutate(g, truth[_spans(_starts(tn)[w] + t0, t1 - t0)], t1 - t0, error)
    blob, back = _letters(codes), _letters(backbone)
    quals = _qualities(g, len(blob)) if quality else None
    back_quals = np.full(len(back), 33, dtype=np.uint8)  # a draft without qualities
    at = _starts(ln).cpu().numpy().astype(np.uint64)
    la = np.zeros(layers, dtype=LAYER)
    la["sequence"] = at + np.uint64(blob.ctypes.data)
    la["quality"] = at + np.uint64(quals.ctypes.data) if quality else 0
    la["length"], la["begin"], la["end"] = (x.cpu().numpy() for x in (ln, begin, end))
    bat = _starts(n).cpu().numpy().astype(np.uint64)
    arr = np.zeros(count, dtype=WINDOW)
    arr["backbone"] = bat + np.uint64(back.ctypes.data)
    arr["backbone_quality"] = bat + np.uint64(back_quals.ctypes.data)
    arr["backbone_length"], arr["n_layers"] = n.cpu().numpy(), d.cpu().numpy()
    arr["layers"] = (np.uint64(la.ctypes.data) +
                     _starts(d).cpu().numpy().astype(np.uint64) * np.uint64(LAYER.itemsize))
    arr["tgs"] = 0 if read else 1
    return arr, (la, blob, quals, back, back_quals)


def _overlap_lengths(case):
    """Lengths of the true targets: the case's own, whatever the seed."""
    mean, sd = case["mean"], case["sd"]
    sigma = math.sqrt(math.log(1 + (sd / mean) ** 2))
    z = np.random.default_rng(case["pairs"]).standard_normal(case["pairs"])
    tl = np.rint(np.exp(math.log(mean) - sigma * sigma / 2 + sigma * z)).astype(np.int64)
    return tl.clip(min(100, case["longest"]), case["longest"])


def _ops_room(case):
    """More than the query and target bytes of the case's pairs."""
    return int((2.5 * _overlap_lengths(case)).sum()) + 200 * case["pairs"]


def _pairs(g, case):
    """(query codes, query lengths, target codes, target lengths)."""
    dev = g.device
    tl = torch.from_numpy(_overlap_lengths(case)).to(dev)
    truth = torch.randint(0, 4, (int(tl.sum()),), generator=g, device=dev, dtype=torch.uint8)
    q, ql = _mutate(g, truth, tl, case["error"])
    t = truth
    if case["target_error"] > 0:
        t, tl = _mutate(g, truth, tl, case["target_error"])
    return q, ql, t, tl


def _u64(lengths):
    return _starts(lengths).cpu().numpy().astype(np.uint64)


def _check(rc, what):
    if rc != _lib.RH_OK:
        raise RuntimeError(f"{what}: {rc}: {_lib.load_library().rh_last_error().decode()}")


def _as(array, kind):
    return ctypes.cast(array.ctypes.data, ctypes.POINTER(kind))


def _result_buffers(count, length):
    room = count * (2 * length + 1040)
    return {"out": np.zeros(room, dtype=np.uint8), "offsets": np.zeros(count, dtype=np.uint64),
            "lengths": np.zeros(count, dtype=np.uint32), "status": np.zeros(count, dtype=np.uint8)}


def _bufs(b):
    """The arguments of rh_poa_download / rh_server_fetch after the handle."""
    return (ctypes.cast(b["out"].ctypes.data, ctypes.c_char_p), b["out"].nbytes,
            _as(b["offsets"], ctypes.c_uint64), _as(b["lengths"], ctypes.c_uint32),
            _as(b["status"], ctypes.c_uint8))


def _results(b):
    return {"consensus": b["out"], "lengths": b["lengths"], "status": b["status"]}


def prepare(case, seed):
    g = _generator(seed)
    return {"poa": _prepare_poa, "align": _prepare_align, "device": _prepare_device,
            "serve": _prepare_serve}[case["kind"]](case, g)


def _prepare_poa(case, g):
    keys = ("length", "depth", "error", "partial", "read", "target", "spread", "quality")
    arr, keep = _windows(g, case["windows"], **{k: case[k] for k in keys})
    batch = racon_amd.PoaBatch(case["match"], case["mismatch"], case["gap"], trim=True)
    if case["band"]:
        batch.set_band(case["band"])
    return {"run": _run_poa, "arr": arr, "keep": keep, "batch": batch,
            "out": _result_buffers(case["windows"], case["length"])}


def _run_poa(s):
    batch = s["batch"]
    batch.upload_packed(s["arr"], len(s["arr"]), s["keep"])
    batch.run()
    batch.download_into(_bufs(s["out"]))
    return _results(s["out"])


def _prepare_align(case, g):
    n = case["pairs"]
    q, ql, t, tl = _pairs(g, case)
    ql_host, tl_host = ql.cpu().numpy(), tl.cpu().numpy()
    letters = _letters(q), _letters(t)
    arr = np.zeros(n, dtype=PAIR)
    arr["query"] = _u64(ql) + np.uint64(letters[0].ctypes.data)
    arr["target"] = _u64(tl) + np.uint64(letters[1].ctypes.data)
    arr["query_length"], arr["target_length"] = ql_host, tl_host
    s = {"run": _run_align, "batch": racon_amd.AlignBatch(), "n": n, "arr": arr, "keep": letters}
    if not case["layers"]:
        s["ops"] = np.zeros(_ops_room(case), dtype=np.uint8)
        s["offsets"] = np.zeros(n, dtype=np.uint64)
        s["n_ops"] = np.zeros(n, dtype=np.uint32)
        s["distance"] = np.zeros(n, dtype=np.int32)
        return s
    # overlaps of reads with one contig, in target order, half of them on the
    # reverse strand
    contig = int(tl_host.sum()) // 40 + int(tl_host.max())
    begin = (torch.rand(n, generator=g, device=g.device) * (contig - tl)).long()
    begin = torch.sort(begin).values.cpu().numpy()
    begin = np.minimum(begin, contig - tl_host)
    spans = np.zeros(n, dtype=SPAN)
    spans["t_begin"], spans["t_end"] = begin, begin + tl_host
    quals = _qualities(g, int(ql_host.sum()))
    sources = np.zeros(n, dtype=SOURCE)
    sources["overlap"] = np.arange(n)
    sources["query_length"], sources["quality"] = ql_host, _u64(ql)
    sources["mirrored"] = np.arange(n) & 1
    room = int(_lib.load_library().rh_breaking_points_bound(
        case["window"], _as(spans, _lib.RhBreakSpan), n))
    s.update(run=_run_layers, window=case["window"], n_windows=contig // case["window"] + 1,
             spans=spans, sources=sources, quals=quals, room=room,
             points=np.zeros((room, 2), dtype=np.uint32), offsets=np.zeros(n, dtype=np.uint64),
             counts=np.zeros(n, dtype=np.uint32),
             records=np.zeros((int((2 * _overlap_lengths(case) // case["window"] + 4).sum()), 6),
                              dtype=np.uint32))
    return s


def _align(s):
    batch, lib = s["batch"], s["batch"].lib
    _check(lib.rh_align_upload(batch.handle, s["n"], _as(s["arr"], _lib.RhPair)), "upload")
    _check(lib.rh_align_run(batch.handle), "run")
    return lib, batch.handle


def _run_align(s):
    lib, handle = _align(s)
    _check(lib.rh_align_download(handle, ctypes.cast(s["ops"].ctypes.data, ctypes.c_char_p),
                                 s["ops"].nbytes, _as(s["offsets"], ctypes.c_uint64),
                                 _as(s["n_ops"], ctypes.c_uint32),
                                 _as(s["distance"], ctypes.c_int32)), "download")
    return {"ops": s["ops"], "n_ops": s["n_ops"], "distance": s["distance"]}


def _run_layers(s):
    lib, handle = _align(s)
    _check(lib.rh_align_breaking_points(handle, s["window"], _as(s["spans"], _lib.RhBreakSpan),
                                        _as(s["offsets"], ctypes.c_uint64),
                                        _as(s["counts"], ctypes.c_uint32),
                                        _as(s["points"], ctypes.c_uint32), s["room"]), "points")
    layers = ctypes.c_void_p()
    _check(lib.rh_layers_create(0, s["window"], 10.0, s["n_windows"], s["room"] // 2,
                                ctypes.cast(s["quals"].ctypes.data, ctypes.c_char_p),
                                s["quals"].nbytes, ctypes.byref(layers)), "layer set")
    try:
        _check(lib.rh_layers_add(layers, handle, _as(s["sources"], _lib.RhLayerSource), s["n"]),
               "layers")
        n = ctypes.c_uint64()
        _check(lib.rh_layers_finish(layers, ctypes.byref(n)), "grouping")
        _check(lib.rh_layers_download(layers, _as(s["records"], _lib.RhLayerRecord),
                                      len(s["records"])), "records")
    finally:
        lib.rh_layers_destroy(layers)
    return {"records": s["records"], "counts": s["counts"]}


def _prepare_device(case, g):
    n = case["pairs"]
    q, ql, t, tl = _pairs(g, case)
    table = torch.tensor(list(b"ACGT"), dtype=torch.uint8, device=g.device)
    arena = torch.cat([table[q.int()], table[t.int()]])
    pairs = np.zeros(n, dtype=np.dtype(_lib.DEV_PAIR_FIELDS))
    pairs["query_offset"] = _u64(ql)
    pairs["target_offset"] = _u64(tl) + np.uint64(int(ql.sum()))
    pairs["ops_offset"] = _u64(ql + tl)
    pairs["query_length"], pairs["target_length"] = ql.cpu().numpy(), tl.cpu().numpy()
    return {"run": _run_device, "n": n, "arena": arena,
            "pairs": torch.from_numpy(pairs.view(np.uint8).copy()).to(g.device),
            "longest": (int(ql.max()), int(tl.max())),
            "ops": torch.zeros(_ops_room(case), dtype=torch.uint8, device=g.device),
            "results": torch.zeros((n, 4), dtype=torch.int32, device=g.device)}


def _run_device(s):
    lib = _lib.load_library()
    stream = torch.cuda.current_stream().cuda_stream
    _check(lib.rh_align_run_noalloc(0, stream, s["n"], s["pairs"].data_ptr(),
                                    s["arena"].data_ptr(), *s["longest"], s["ops"].data_ptr(),
                                    s["results"].data_ptr()), "rh_align_run_noalloc")
    # op count, distance, status (the last word of a result is reserved)
    return {"ops": s["ops"], "results": s["results"][:, :3]}


def _request_sizes(case):
    return [max(1, int(case["windows"] * case["growth"] ** k)) for k in range(case["requests"])]


def _prepare_serve(case, g):
    server = PolishServer(1 << 30, executors=4, launch_windows=2048)
    requests = []
    for count in _request_sizes(case):
        arr, keep = _windows(g, count, case["length"], case["depth"], case["error"])
        requests.append((arr, keep, _result_buffers(count, case["length"])))
    arr = requests[-1][0]
    _check(server.lib.rh_server_warm(server.handle, len(arr), _as(arr, _lib.RhWindow)), "warm")
    return {"run": _run_serve, "server": server, "requests": requests}


def _run_serve(s):
    lib, handle = s["server"].lib, s["server"].handle
    ids = []
    for arr, _, _ in s["requests"]:
        rid = ctypes.c_uint64()
        _check(lib.rh_server_submit(handle, len(arr), _as(arr, _lib.RhWindow), ctypes.byref(rid)),
               "submit")
        ids.append(rid.value)
    for rid, (_, _, out) in zip(ids, s["requests"]):
        _check(lib.rh_server_wait(handle, rid, -1), "wait")
        _check(lib.rh_server_fetch(handle, rid, *_bufs(out)), "fetch")
    return [_results(out) for _, _, out in s["requests"]]


def run(state):
    return state["run"](state)


# ---- the work a pass cannot do without ----

def _poa_work(windows, length, depth, read, quality):
    layers = windows * depth * (math.ceil((length + read) / read) if read else 1)
    span = min(read, length) if read else length
    each = 2 if quality else 1
    # 6 integer operations for each cell of a layer against the backbone span
    # it covers (the graph only grows from there)
    return {"bytes": 3.0 * windows * length + each * layers * span,
            "flops": 6.0 * layers * span * span}


def work(case):
    if case["kind"] == "poa":
        return _poa_work(case["windows"], case["length"], case["depth"], case["read"],
                         case["quality"])
    if case["kind"] == "serve":
        parts = [_poa_work(n, case["length"], case["depth"], 0, True)
                 for n in _request_sizes(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    n, length = case["pairs"], case["mean"]
    distance = length * min(0.5, case["error"] + case["target_error"])
    # 20 operations on 32-bit words for 32 cells of the diagonal band that the
    # distance needs
    bases = 2.0 * n * length
    return {"bytes": 2 * bases if case.get("layers") else 1.5 * bases,
            "flops": 20.0 / 32 * n * length * max(32.0, distance)}


def exact(case, seed):
    """Every output is a whole number or a byte: there is no rounding."""
    return None
