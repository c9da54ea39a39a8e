"""What this library's speed is measured on: the calls that its users make.

A user of the library searches a Graph500 Kronecker graph (edgefactor 16, up
to scale 26 on one GPU) in one of these ways, and each listed case is one:

  batch     64 searches together, the headline of bench.py: g5_msbfs_run, the
            final maps where they lie in HBM, the TEPS numerators
  single    one search of the direction-optimised plug-in: g5_bfs_run, its
            predecessor and level maps, its TEPS numerator; with the codec on
            every level's queue (bench.py's c2) or without
  grid      the level loop of an R x C grid over the plug-in's hooks, ranks in
            turn on one GPU, frontiers left in HBM (host/g5_grid.cpp)
  combine   the column step's combines of one 4 x 4 rank: the frontier OR and
            the predecessor minimum (bench.py's c3)
  codec     one queue encoded at the sender and decoded at the receiver
  validate  Graph500 validation of one predecessor map on the device
  serve     the serving engine's loop (host/g5_serve.cpp): roots join and
            leave the batched search between levels

Every output is whole numbers, which have one right value.
"""
import ctypes
import math
import random

import numpy as np
import torch

import gpugraph500_amd as g5


def listed():
    return [
        # the smallest graph that bench.py knows (its c1): launches and host
        # round trips count
        {"name": "batch_s16", "path": "batch", "scale": 16, "edgefactor": 16, "roots": 64, "shapes": "default"},
        {"name": "single_s16", "path": "single", "scale": 16, "edgefactor": 16, "codec": False},
        # the ordinary sizes
        {"name": "batch_s24", "path": "batch", "scale": 24, "edgefactor": 16, "roots": 64, "shapes": "default"},
        {"name": "single_s22_codec", "path": "single", "scale": 22, "edgefactor": 16, "codec": True},
        {"name": "grid2x2_s22", "path": "grid", "scale": 22, "edgefactor": 16, "parts": 2, "codec": True},
        # a server's engine under load, on a graph of middle size
        {"name": "serve_s20", "path": "serve", "scale": 20, "edgefactor": 16, "roots": 96, "arrivals": 12},
        # one rank of a 4 x 4 grid at scale 26: 2^24 columns
        {"name": "combine_4x4_s26", "path": "combine", "k": 4, "words": 262144, "preds": 1 << 24},
        # a sparse level's queue, and the longest queue of a rank at scale 26
        {"name": "codec_short", "path": "codec", "values": 3001, "ids": 1 << 22},
        {"name": "codec_long", "path": "codec", "values": 7000003, "ids": 1 << 24},
        # Graph500 validates every search
        {"name": "validate_s24", "path": "validate", "scale": 24, "edgefactor": 16, "depth": False, "broken": False},
        # the largest: the headline's graph, with the shapes the benchmark runs
        {"name": "single_s26", "path": "single", "scale": 26, "edgefactor": 16, "codec": False},
        {"name": "batch_s26", "path": "batch", "scale": 26, "edgefactor": 16, "roots": 64, "shapes": "tuned"},
    ]


def draw(rng):
    path = rng.choice(["batch", "single", "grid", "combine", "codec", "validate", "serve"])
    ef = rng.randint(7, 18)

    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if path == "batch":
        return {"path": path, "scale": rng.randint(14, 25), "edgefactor": ef, "roots": spread(1, 64),
                "shapes": "default"}
    if path == "single":
        return {"path": path, "scale": rng.randint(14, 25), "edgefactor": ef, "codec": rng.random() < 0.4}
    if path == "grid":
        return {"path": path, "scale": rng.randint(14, 22), "edgefactor": ef, "parts": rng.randint(1, 3),
                "codec": rng.random() < 0.6}
    if path == "combine":
        k = rng.randint(2, 9)
        return {"path": path, "k": k, "words": spread(100, 1 << 20), "preds": spread(5000, (1 << 26) // k)}
    if path == "codec":
        n = spread(1, 8 << 20)
        return {"path": path, "values": n, "ids": min(1 << 30, spread(2 * n, 4000 * n))}
    if path == "validate":
        return {"path": path, "scale": rng.randint(14, 24), "edgefactor": ef, "depth": rng.random() < 0.3,
                "broken": rng.random() < 0.25}
    return {"path": path, "scale": rng.randint(14, 21), "edgefactor": ef, "roots": spread(8, 128),
            "arrivals": rng.randint(1, 32)}


# the shapes that the benchmark's autotune chose for the headline's graph
# (gpugraph500_amd/tuned_shapes.json)
TUNED = {"thread_max": 256, "wave_max": 2048, "push_ratio": 4, "active_ratio": 2, "lane_ratio": 128, "split_max": 32}


class _Dev:
    """A torch tensor as the bindings' methods take a device buffer."""

    def __init__(self, t):
        self.t = t
        self.ptr = ctypes.c_void_p(t.data_ptr())


class _Borrowed:
    """Device memory that `owner` holds, for torch to view in place."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr, "strides": None,
                                         "version": 2}


def _empty(n, dtype):
    return torch.empty(n, dtype=dtype, device="cuda")


def _graph(case, seed):
    return g5.Graph.kronecker(case["scale"], case["edgefactor"], seed1=1 + seed, seed2=2)


def _roots(g, seed, n):
    """n search keys: a seeded choice among the benchmark's draws."""
    keys = g.select_roots(g.nglobal, 4 * max(n, 16)).tolist()
    return random.Random(seed).sample(keys, n)


def _queue(gen, n, ids):
    """n ascending distinct ids, spread over about `ids` as a level's are."""
    mean = max(ids / n, 1.0)
    gaps = 1 + (torch.empty(n, device="cuda", dtype=torch.float64).exponential_(1.0, generator=gen) * (mean - 1))
    return (torch.cumsum(gaps.to(torch.int64), 0) - 1).to(torch.int32)


def _maps(gen, k, n):
    """k frontier bitmaps of n words, a quarter of the bits set."""
    r = [torch.randint(-(1 << 62), 1 << 62, (k, n), generator=gen, device="cuda") for _ in range(2)]
    return r[0] & r[1]


def _preds(gen, k, n):
    """k predecessor arrays of n global ids, absent (-1) in six of ten places."""
    p = torch.randint(0, 1 << 26, (k, n), generator=gen, device="cuda")
    gone = torch.rand((k, n), generator=gen, device="cuda") < 0.6
    return p.masked_fill_(gone, -1)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _inputs(case, seed):
    """The device inputs of the paths that take no graph."""
    gen = _generator(seed)
    if case["path"] == "codec":
        return {"queue": _queue(gen, case["values"], case["ids"])}
    return {"maps": _maps(gen, case["k"], case["words"]), "preds": _preds(gen, case["k"], case["preds"])}


def prepare(case, seed):
    g5.init(0)
    path = case["path"]
    st = {"path": path, "case": case}
    if path in ("combine", "codec"):
        st.update(_inputs(case, seed))
        if path == "codec":
            cap = g5.s4_max_words(case["values"])
            st.update(words=torch.zeros(cap, dtype=torch.int32, device="cuda"), back=_empty(case["values"], torch.int32))
        else:
            st.update(any=_empty(case["words"], torch.int64), least=_empty(case["preds"], torch.int64))
        torch.cuda.synchronize()
        return st
    if path == "grid":
        k = case["parts"]
        blocks = g5.Graph.kronecker_2d(case["scale"], k, k, case["edgefactor"], seed1=1 + seed, seed2=2)
        n = [b.n_cols for b in blocks[:k]]
        # keys: vertices of the first rank that have a neighbour there
        st.update(blocks=blocks, n=n, ranks=[g5.BFS(b) for b in blocks],
                  root=_roots(blocks[0], seed, 1)[0], wide=max(n),
                  red=[_empty(m // 64, torch.int64) for m in n], fold=_empty(max(n) // 64, torch.int64),
                  queue=_empty(max(n), torch.int32), back=_empty(max(n), torch.int32),
                  words=_empty(g5.s4_max_words(max(n)), torch.int32), preds=_empty(k * max(n), torch.int64),
                  pred=[_empty(m, torch.int64) for m in n], level=[_empty(m, torch.int32) for m in n])
        torch.cuda.synchronize()
        return st
    g = _graph(case, seed)
    st["graph"] = g
    if path == "batch":
        m = g5.MSBFS(g)
        roots = _roots(g, seed, case["roots"])
        if case["shapes"] == "tuned":
            m.tune(**TUNED)
            # as bench.py does before it times anything
            m.place(_roots(g, seed + 1, case["roots"]), 4)
        st.update(search=m, roots=np.array(roots, np.int64))
    elif path == "serve":
        m = g5.MSBFS(g)
        m.open()
        keys = _roots(g, seed, min(case["roots"], 64))
        pick = random.Random(seed + 1)
        st.update(search=m, roots=[pick.choice(keys) for _ in range(case["roots"])])
    else:
        b = g5.BFS(g)
        st.update(root=_roots(g, seed, 1)[0], pred=_empty(g.n_cols, torch.int64))
        if path == "validate":
            b.run(st["root"])
            b.pred_device(_Dev(st["pred"]))
            b.free()
            if case["broken"]:  # a reached vertex that names itself
                reached = (st["pred"] >= 0).nonzero()
                v = int(reached[random.Random(seed).randrange(reached.numel())])
                st["pred"][v] = v
            st.update(check=g5.Validator(g))
        else:
            st.update(search=b, level=_empty(g.n_cols, torch.int32))
    torch.cuda.synchronize()
    return st


def _run_batch(st):
    m = st["search"]
    levels, _ = m.run(st["roots"])
    pred, level, lane_of, _ = m.maps()
    n, k = st["graph"].n_rows, len(st["roots"])
    pred = torch.as_tensor(_Borrowed(m, pred, (n, 64), "<i4"), device="cuda")
    level = torch.as_tensor(_Borrowed(m, level, (n, 64), "|u1"), device="cuda")
    # the slots of lanes that hold no root are undefined
    return {"pred": pred[:, :k], "level": level[:, :k], "lane_of": lane_of, "nedge": m.nedge(), "levels": levels}


def _run_single(st):
    b = st["search"]
    levels, _ = b.run(st["root"], codec=st["case"]["codec"])
    b.pred_device(_Dev(st["pred"]))
    b.level_device(_Dev(st["level"]))
    return {"pred": st["pred"], "level": st["level"], "nedge": b.nedge(), "levels": levels}


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _run_grid(st):
    lib, k, blocks, ranks = g5.lib(), st["case"]["parts"], st["blocks"], st["ranks"]
    n_total, bottom_up, levels = sum(st["n"]), False, 0
    for b in ranks:
        b.start(st["root"])
    while True:
        found = False
        for r in range(k):
            for c in range(k):
                b = ranks[r * k + c]
                found |= b.expand_bottom_up(blocks[c * k + r]) if bottom_up else b.expand()
        if not found:
            break
        levels += 1
        new = 0
        for c in range(k):  # the column step: the OR of the column's out-bitmaps
            words = st["n"][c] // 64
            maps, nw = (ctypes.c_void_p * k)(), ctypes.c_int64()
            for r in range(k):
                p = ctypes.c_void_p()
                g5.check(lib.g5_bfs_out_bitmap(ranks[r * k + c].h, ctypes.byref(p), ctypes.byref(nw)))
                maps[r] = p.value
            g5.check(lib.g5_vreduce_or_list(maps, k, words, _p(st["red"][c])))
            new += g5.bitmap_count(_Dev(st["red"][c]), words)
            for r in range(k):
                g5.check(lib.g5_bfs_set_out_bitmap(ranks[r * k + c].h, _p(st["red"][c])))
        for r in range(k):  # the row step: the diagonal rank's bitmap to its row
            words, src = st["n"][r] // 64, st["red"][r]
            if st["case"]["codec"]:
                n, nw = ctypes.c_int64(), ctypes.c_size_t()
                g5.check(lib.g5_bitmap_to_queue(_p(src), words, _p(st["queue"]), ctypes.byref(n)))
                g5.check(lib.g5_s4_roundtrip(_p(st["queue"]), n.value, _p(st["words"]), st["words"].numel(),
                                             _p(st["back"]), ctypes.byref(nw)))
                g5.check(lib.g5_queue_to_bitmap(_p(st["back"]), n.value, _p(st["fold"]), words))
                src = st["fold"]
            for c in range(k):
                g5.check(lib.g5_bfs_set_in_bitmap(ranks[r * k + c].h, _p(src)))
        if not bottom_up and new > n_total // 64:
            bottom_up = True
        elif bottom_up and new < n_total // 24:
            bottom_up = False
    for c in range(k):
        n = st["n"][c]
        for r in range(k):
            ranks[r * k + c].pred_device(_Dev(st["preds"][r * n:(r + 1) * n]))
        g5.check(lib.g5_vreduce_min_pred(_p(st["preds"]), k, n, _p(st["pred"][c])))
        ranks[c].level_device(_Dev(st["level"][c]))
    return {"pred": st["pred"], "level": st["level"], "levels": levels}


def _run_combine(st):
    lib, k = g5.lib(), st["case"]["k"]
    maps = (ctypes.c_void_p * k)(*[m.data_ptr() for m in st["maps"]]) if st["case"]["words"] % 2 == 0 else None
    if maps is not None:  # the ranks' bitmaps where they lie
        g5.check(lib.g5_vreduce_or_list(maps, k, st["case"]["words"], _p(st["any"])))
    else:  # one gathered buffer
        g5.check(lib.g5_vreduce_or(_p(st["maps"]), k, st["case"]["words"], _p(st["any"])))
    g5.check(lib.g5_vreduce_min_pred(_p(st["preds"]), k, st["case"]["preds"], _p(st["least"])))
    return {"any": st["any"], "least": st["least"]}


def _run_codec(st):
    lib, n = g5.lib(), st["case"]["values"]
    nw, back = ctypes.c_size_t(), ctypes.c_size_t()
    g5.check(lib.g5_s4_encode(_p(st["queue"]), n, _p(st["words"]), st["words"].numel(), ctypes.byref(nw)))
    g5.check(lib.g5_s4_decode(_p(st["words"]), nw.value, _p(st["back"]), n, ctypes.byref(back)))
    # the stream is the first nw words; the rest of its buffer stays as it was
    return {"words": st["words"], "nw": nw.value, "back": st["back"], "n": back.value}


def _run_validate(st):
    bad, nedge, depth, _ = st["check"].validate_device(st["root"], _Dev(st["pred"]), want_depth=st["case"]["depth"])
    out = {"bad": bad, "nedge": nedge}
    if depth is not None:
        out["depth"] = depth
    return out


def _run_serve(st):
    """The engine's loop: `arrivals` roots come with every level, and join
    while the running cohort's lanes are all in their first level."""
    m, roots = st["search"], st["roots"]
    nedge, checksum = np.zeros(len(roots), np.int64), np.zeros(len(roots), np.int64)
    holds, joined, level, come, taken = {}, {}, 0, 0, 0
    while taken < len(roots) or holds:
        come = min(len(roots), come + st["case"]["arrivals"])
        if all(level - joined[lane] <= 1 for lane in holds):
            free = [lane for lane in range(64) if lane not in holds][:come - taken]
            for i, lane in enumerate(free):
                holds[lane], joined[lane] = taken + i, level
            if free:
                m.join(roots[taken:taken + len(free)], free)
                taken += len(free)
        live, _ = m.step()
        level += 1
        gone = [lane for lane in holds if not live >> lane & 1]
        if gone:
            ne, ck = m.leave(sum(1 << lane for lane in gone))
            for lane in gone:
                i = holds.pop(lane)
                nedge[i], checksum[i] = ne[lane], ck[lane].astype(np.int64)
    return {"nedge": nedge, "checksum": checksum}


def run(st):
    return _RUN[st["path"]](st)


_RUN = {"batch": _run_batch, "single": _run_single, "grid": _run_grid, "combine": _run_combine, "codec": _run_codec,
        "validate": _run_validate, "serve": _run_serve}


def work(case):
    """Whole-number work on memory: bytes only.  About half of a Kronecker
    graph's vertices have edges."""
    path = case["path"]
    if path == "combine":
        return {"bytes": 8.0 * (case["k"] + 1) * (case["words"] + case["preds"]), "flops": 0}
    if path == "codec":
        # the coded id takes the bits of a gap and one or two for its spread
        bits = min(32.0, 2 + math.log2(max(4.0 * case["ids"] / case["values"], 2)))
        return {"bytes": case["values"] * (8 + 2 * bits / 8) + 16, "flops": 0}
    n = 1 << case["scale"]
    graph = 8.0 * n + 4 * 2 * case["edgefactor"] * n
    if path == "batch":  # the graph once; 5 bytes per root and vertex
        return {"bytes": graph + 5.0 * case["roots"] * n / 2, "flops": 0}
    if path == "serve":
        # the graph once per 64 roots; the maps written, then read when a root leaves
        return {"bytes": graph * math.ceil(case["roots"] / 64) + 9.0 * case["roots"] * n / 2, "flops": 0}
    if path == "validate":
        return {"bytes": graph + 8.0 * n, "flops": 0}
    # a search that knows where to look reads at least one neighbour of every
    # vertex with edges, and writes every vertex's predecessor and level
    return {"bytes": 8.0 * n + 4.0 * n / 2 + 12.0 * n, "flops": 0}


def exact(case, seed):
    """The combines and the codec in plain torch; the searches' answers are
    whole numbers of the graph, which only the library generates."""
    if case["path"] == "combine":
        x = _inputs(case, seed)
        any_ = x["maps"][0].clone()
        for m in x["maps"][1:]:
            any_ |= m
        far = torch.iinfo(torch.int64).max
        least = torch.where(x["preds"] < 0, far, x["preds"]).amin(0)
        return {"any": any_, "least": torch.where(least == far, -1, least)}
    if case["path"] == "codec":
        return {"words": None, "nw": None, "back": _inputs(case, seed)["queue"], "n": case["values"]}
    return None
