"""The work a program hands this engine, as measurable cases.

Every case is one pass through the package's public calls (`pcx.PIR`,
`pcx.BitsPIR`, `pcx.Batch`, `pcx.Server`), over the sizes the benchmark and the
tests use: networks of 1,000 to 4,000,000 propagators with a quarter as many
variables, batches of up to 4,096 search nodes.  A case says which path it
takes:

  single    one store in host memory to its fixpoint (PIR.fixpoint): what a
            caller of the reference's Gauss-Seidel fixpoint switches to
  noalloc   one store in device memory to its fixpoint without an allocation
            (PIR.fixpoint_noalloc): a tight serving loop
  nodes     a batch of search nodes from host memory to their fixpoints and
            back (Batch.load, run, read): a search that lives on the host
  fresh     new search nodes already in device memory (Batch.load_device,
            run): a search that lives on the device; its stores stay there
            and the program reads which nodes failed (`read`: a small batch,
            whose stores it reads too)
  step      the step after a fixpoint: every node split in two on the device
            and the children propagated (Batch.branch, run; `read` as above)
  ask       which propagators of which nodes are still open (Batch.ask): the
            subsets of the next batch
  formulas  PC's is_extractable over formula trees (Batch.ask_formulas)
  serve     requests over several resident networks (Server.submit, step,
            poll)

`domain` is "itv" (int32 intervals) or "bits" (64-value words).  `start` says
whether a batch's nodes are splits of the network's root fixpoint (a search)
or of its told store (nothing propagated yet).  Networks are the planted ones
of `pcx.gen_network` (they cannot fail; their nodes can), seeded, so another
seed is another network with other nodes.  The bounds of a failed node depend
on the order of propagation and mean nothing to a program, which drops them:
they come back as zeros.
"""
import functools
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lala-pc_amd"))

import pcx  # noqa: E402

MODES = {"batched": pcx.MODE_BATCHED, "persistent": pcx.MODE_PERSISTENT, "plain": pcx.MODE_PLAIN}


def listed():
    return [
        # The smallest network of the serving traces: one call's latency.
        {"name": "single_1k", "path": "single", "domain": "itv", "nvars": 250, "nprops": 1000},
        # The root fixpoint a search computes before its first batch.
        {"name": "single_200k", "path": "single", "domain": "itv", "nvars": 50000, "nprops": 200000},
        # The largest network: one model of a million variables.
        {"name": "single_4m", "path": "single", "domain": "itv", "nvars": 1000000, "nprops": 4000000},
        # A serving loop that keeps its stores on the device (odd sizes).
        {"name": "noalloc_120k", "path": "noalloc", "domain": "itv", "nvars": 30011, "nprops": 120019},
        # A host search over a small model: stores that fit in a compute
        # unit's local memory, one launch for the whole batch.
        {"name": "nodes_persistent", "path": "nodes", "domain": "itv", "inst": 256, "nvars": 4001,
         "nprops": 16003, "mode": "persistent", "start": "told"},
        # The same kind of batch, unpropagated and larger, in the default mode.
        {"name": "nodes_told", "path": "nodes", "domain": "itv", "inst": 1000, "nvars": 3001,
         "nprops": 12007, "mode": "batched", "start": "told"},
        # The benchmark's step: 4,096 new nodes with their own active subsets.
        {"name": "fresh_4096", "path": "fresh", "domain": "itv", "inst": 4096, "nvars": 50000,
         "nprops": 200000, "mode": "batched", "subsets": True, "read": False},
        # 1,024 nodes branched into 2,048 children, which are propagated.
        {"name": "step_1024", "path": "step", "domain": "itv", "inst": 1024, "nvars": 50000,
         "nprops": 200000, "read": False},
        # The open propagators of 128 nodes.
        {"name": "ask_128", "path": "ask", "domain": "itv", "inst": 128, "nvars": 12500, "nprops": 50000},
        # Candidate solutions tested against the model's own formulas.
        {"name": "formulas_512", "path": "formulas", "domain": "itv", "inst": 512, "nvars": 12500,
         "nprops": 50000},
        # Bitset nodes of a host search (bitset batches load from the host).
        {"name": "bits_nodes", "path": "nodes", "domain": "bits", "inst": 64, "nvars": 50000,
         "nprops": 200000, "mode": "batched", "start": "root"},
        # A burst of requests over twelve resident networks of mixed sizes.
        {"name": "serve_48", "path": "serve", "domain": "itv", "requests": 48, "networks": 12,
         "pmin": 1000, "pmax": 128000},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over the logarithm."""
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    path = rng.choice(["single", "single", "noalloc", "nodes", "nodes", "fresh", "step", "ask", "formulas",
                       "serve"])
    if path == "serve":
        nets = rng.randint(2, 12)
        return {"path": path, "domain": "itv", "requests": rng.randint(8, 48), "networks": nets, "pmin": 1000,
                "pmax": _log(rng, 2000, 128000)}
    top = {"single": 4000000, "noalloc": 400000, "nodes": 32000, "fresh": 200000, "step": 200000,
           "ask": 100000, "formulas": 50000}[path]
    p = _log(rng, {"single": 1000, "noalloc": 1000, "nodes": 2000}.get(path, 8000), top)
    v = max(200, p // 4 + rng.randint(-3, 3))
    case = {"path": path, "domain": "itv", "nvars": v, "nprops": p}
    if path == "single" and p <= 800000 and rng.random() < 0.3:
        case["domain"] = "bits"
    if path == "nodes":
        case.update(inst=max(3, min(_log(rng, 16, 1000), 3000000 // v)), mode=rng.choice(["batched", "persistent"]),
                    start=rng.choice(["told", "root"]))
        if rng.random() < 0.3:
            case.update(domain="bits", mode="batched", start="root")
    elif path == "fresh":
        case.update(inst=_log(rng, 64, 4096), mode="batched", subsets=rng.random() < 0.5)
        case["read"] = case["inst"] * v <= 2000000
    elif path == "step":
        case.update(inst=_log(rng, 32, 1024))
        case["read"] = 2 * case["inst"] * v <= 2000000
    elif path == "ask":
        case.update(inst=max(3, min(_log(rng, 16, 512), 6400000 // p)))
    elif path == "formulas":
        case.update(inst=_log(rng, 16, 512))
    return case


# ---- what a program has in hand before the call ----------------------------


@functools.lru_cache(maxsize=1)
def _subsets(nprops, inst):
    """Active subsets of 1 to 100% of the propagators, as the benchmark draws
    them (the same for every seed: drawing them takes seconds)."""
    return pcx.gen_subsets(7, nprops, inst, max(1, nprops // 100), nprops)


def _network(case, seed):
    """(op, x, y, z, lb, ub, hidden solution) of the case's network, told order."""
    return pcx.gen_network(pcx.gen_params(seed=seed, nvars=case["nvars"], nprops=case["nprops"]))


def _told(case, seed):
    """A told engine and its told store."""
    op, x, y, z, lb, ub, _ = _network(case, seed)
    pir = pcx.PIR()
    pir.tell(op, x, y, z, lb, ub)
    return pir, lb, ub


def _told_bits(case, seed):
    op, x, y, z, words = pcx.gen_bits_network(seed, case["nvars"], case["nprops"])
    pir = pcx.BitsPIR()
    pir.tell(op, x, y, z, words)
    return pir, words


def _nodes(case, seed, lb, ub):
    """Search nodes: each the store lb/ub with 1 to 20 random splits."""
    return pcx.gen_splits(seed + 1, lb, ub, case["inst"], 1, 20)


def _cuda(a):
    return torch.from_numpy(a).cuda()


def prepare(case, seed):
    seed = int(seed) % (1 << 30) + 1
    return globals()["_prepare_" + case["path"]](case, seed)


def _prepare_single(case, seed):
    if case["domain"] == "bits":
        pir, words = _told_bits(case, seed)
        return {"case": case, "pir": pir, "words": words}
    pir, lb, ub = _told(case, seed)
    return {"case": case, "pir": pir, "lb": lb, "ub": ub}


def _prepare_noalloc(case, seed):
    pir, lb, ub = _told(case, seed)
    pir.fixpoint(lb.copy(), ub.copy())          # sizes the engine's device table
    lb, ub = _cuda(lb), _cuda(ub)
    return {"case": case, "pir": pir, "lb": lb, "ub": ub, "d_lb": lb.clone(), "d_ub": ub.clone()}


def _prepare_nodes(case, seed):
    inst, nvars = case["inst"], case["nvars"]
    if case["domain"] == "bits":
        pir, words = _told_bits(case, seed)
        if case["start"] == "root":
            pir.fixpoint(words)
        return {"case": case, "batch": pcx.Batch(pir, inst, nvars),
                "words": pcx.gen_bits_splits(seed + 1, words, inst, 1, 20)}
    pir, lb, ub = _told(case, seed)
    if case["start"] == "root":
        pir.fixpoint(lb, ub)
    lo, hi = _nodes(case, seed, lb, ub)
    return {"case": case, "batch": pcx.Batch(pir, inst, nvars), "lb": lo, "ub": hi}


def _prepare_fresh(case, seed):
    pir, lb, ub = _told(case, seed)
    pir.fixpoint(lb, ub)
    lo, hi = _nodes(case, seed, lb, ub)
    off, idx = _subsets(case["nprops"], case["inst"]) if case["subsets"] else (None, None)
    return {"case": case, "batch": pcx.Batch(pir, case["inst"], case["nvars"], off, idx),
            "lb": _cuda(lo), "ub": _cuda(hi)}


def _fixpoints(case, seed):
    """A batch that holds the fixpoints of the case's nodes; in the place of
    those that fail, which a search drops, the root's."""
    pir, lb, ub = _told(case, seed)
    pir.fixpoint(lb, ub)
    lo, hi = _nodes(case, seed, lb, ub)
    batch = pcx.Batch(pir, case["inst"], case["nvars"])
    batch.load(lo, hi)
    failed = batch.run(pcx.MODE_BATCHED)[0].failed != 0
    lo.reshape(case["inst"], -1)[failed] = lb
    hi.reshape(case["inst"], -1)[failed] = ub
    batch.load(lo, hi)
    batch.run(pcx.MODE_BATCHED)
    return batch


def _prepare_step(case, seed):
    parent = _fixpoints(case, seed)
    return {"case": case, "parent": parent,
            "child": pcx.Batch(parent.pir, 2 * case["inst"], case["nvars"])}


def _prepare_ask(case, seed):
    return {"case": case, "batch": _fixpoints(case, seed),
            "open": np.full(case["inst"] * case["nprops"], -1, np.int32)}


def _prepare_formulas(case, seed):
    """Half of the stores are the hidden solution, half are it with one to
    three values moved by one (a local search's neighbours)."""
    inst, nvars = case["inst"], case["nvars"]
    op, x, y, z, lb, ub, w = _network(case, seed)
    model = pcx.Model(pcx.flatzinc(op, x, y, z, lb, ub))
    nodes, off = model.formulas()
    pir = pcx.PIR()
    pir.tell(op, x, y, z)
    rng = np.random.default_rng(seed)
    stores = np.tile(w.astype(np.int32), (inst, 1))
    for k in range(0, inst, 2):
        at = rng.integers(0, nvars, rng.integers(1, 4))
        stores[k, at] += rng.choice(np.array([-1, 1], np.int32), len(at))
    stores = stores[rng.permutation(inst)].reshape(-1)
    batch = pcx.Batch(pir, inst, nvars)
    batch.load(stores, stores)
    return {"case": case, "batch": batch, "nodes": nodes, "off": off}


def _network_sizes(case):
    """Propagators of each resident network: even over the logarithm."""
    n = case["networks"]
    return [int(case["pmin"] * (case["pmax"] / case["pmin"]) ** (j / (n - 1))) for j in range(n)]


def _prepare_serve(case, seed):
    server = pcx.Server()
    pirs, stores = [], []
    for j, p in enumerate(_network_sizes(case)):
        pir, lb, ub = _told({"nvars": p // 4, "nprops": p}, seed + 1000 * j)
        pirs.append(pir)
        server.set_root(server.add_network(pir), lb, ub)
        stores.append((lb, ub))
    reqs = []
    for i in range(case["requests"]):
        net = i % len(pirs)
        lo, hi = pcx.gen_splits(seed + 7 * i, *stores[net], 1, 1, 10)
        reqs.append((net, lo, hi))
    work = [(lo.copy(), hi.copy()) for _, lo, hi in reqs]
    return {"case": case, "server": server, "requests": reqs, "work": work}


# ---- one pass ---------------------------------------------------------------


def run(state):
    return globals()["_run_" + state["case"]["path"]](state)


def _run_single(s):
    if s["case"]["domain"] == "bits":
        words = s["words"].copy()
        r = s["pir"].fixpoint(words)
        return {"words": words.view(np.int64), "failed": int(r.failed)}
    lb, ub = s["lb"].copy(), s["ub"].copy()
    r = s["pir"].fixpoint(lb, ub)
    return {"lb": lb, "ub": ub, "failed": int(r.failed)}


def _run_noalloc(s):
    s["d_lb"].copy_(s["lb"])
    s["d_ub"].copy_(s["ub"])
    torch.cuda.current_stream().synchronize()   # the engine works on a stream of its own
    r = s["pir"].fixpoint_noalloc(s["d_lb"].data_ptr(), s["d_ub"].data_ptr(), s["case"]["nvars"])
    return {"lb": s["d_lb"], "ub": s["d_ub"], "failed": int(r.failed)}


def _read(case, batch, failed):
    """The batch's stores, failed ones as zeros."""
    stores = (batch.read_words(),) if case["domain"] == "bits" else batch.read()
    stores = [a.reshape(batch.n_inst, batch.nvars) for a in stores]
    for a in stores:
        a[failed != 0] = 0
    return [a.view(np.int64) if a.dtype == np.uint64 else a for a in stores]


def _run_nodes(s):
    c, batch = s["case"], s["batch"]
    if c["domain"] == "bits":
        batch.load_words(s["words"])
    else:
        batch.load(s["lb"], s["ub"])
    res, _ = batch.run(MODES[c["mode"]])
    return {"stores": _read(c, batch, res.failed), "failed": res.failed.copy()}


def _run_fresh(s):
    c, batch = s["case"], s["batch"]
    batch.load_device(s["lb"].data_ptr(), s["ub"].data_ptr())
    res, _ = batch.run(MODES[c["mode"]])
    out = {"failed": res.failed.copy(), "changed": res.has_changed.copy()}
    return dict(out, stores=_read(c, batch, res.failed)) if c["read"] else out


def _run_step(s):
    c, child = s["case"], s["child"]
    var = s["parent"].branch(child, from_fixpoint=True)
    res, _ = child.run(pcx.MODE_BATCHED)
    out = {"var": var, "failed": res.failed.copy(), "changed": res.has_changed.copy()}
    return dict(out, stores=_read(c, child, res.failed)) if c["read"] else out


def _run_ask(s):
    extractable, off, idx = s["batch"].ask()
    s["open"][:len(idx)] = idx                  # the program's own list, sized for every propagator
    return {"extractable": extractable, "off": off, "open": s["open"]}


def _run_formulas(s):
    return {"extractable": s["batch"].ask_formulas(s["nodes"], s["off"])}


def _run_serve(s):
    server, left = s["server"], len(s["requests"])
    for tag, ((net, lo, hi), (lb, ub)) in enumerate(zip(s["requests"], s["work"])):
        np.copyto(lb, lo)
        np.copyto(ub, hi)
        server.submit(net, lb, ub, tag)
    failed = np.zeros(left, np.int32)
    while left:
        server.step()
        for tag, res, _ in server.poll():
            failed[tag] = res.failed
            left -= 1
    for k in np.nonzero(failed)[0]:
        s["work"][k][0][:] = 0
        s["work"][k][1][:] = 0
    return {"lb": np.concatenate([lb for lb, _ in s["work"]]), "ub": np.concatenate([ub for _, ub in s["work"]]),
            "failed": failed}


def work(case):
    """Bytes no pass can do without: the propagator table (12 B each) and the
    stores (8 B a variable) read once, the fixpoints or answers written once.
    The engine does integer work only."""
    path = case["path"]
    if path == "serve":
        sizes = _network_sizes(case)
        got = [sizes[i % len(sizes)] for i in range(case["requests"])]
        return {"bytes": float(sum(12 * p + 16 * (p // 4) for p in got)), "flops": 0.0}
    v, p, n = case["nvars"], case["nprops"], case.get("inst", 1)
    table, stores = 12 * p, 8 * v * n
    moved = {"single": table + 2 * stores, "noalloc": table + 2 * stores, "nodes": table + 2 * stores,
             "fresh": table + stores + 8 * n,           # the fixpoints differ from the nodes in few values
             "step": table + 3 * stores + 20 * n,       # parents read, two children each written
             "ask": table + stores + 12 * n,            # and 4 B for each open propagator
             "formulas": 16 * 5 * p + stores + n}[path]  # about five nodes a formula
    return {"bytes": float(moved), "flops": 0.0}


# ---- the same answers from plain numpy --------------------------------------

_LO, _HI = -(2**31), 2**31 - 1


def _meet(lb, ub, v, lo, hi):
    np.maximum.at(lb, v, np.clip(lo, _LO, _HI))
    np.minimum.at(ub, v, np.clip(hi, _LO, _HI))


def _sweep(op, x, y, z, lb, ub):
    """Every given propagator once, on the bounds before the sweep (finite
    and not negative, as the generated networks' are)."""
    old_l, old_u = lb.copy(), ub.copy()
    for o in np.unique(op):
        at = op == o
        X, Y, Z = x[at], y[at], z[at]
        xl, xu, yl, yu, zl, zu = old_l[X], old_u[X], old_l[Y], old_u[Y], old_l[Z], old_u[Z]
        if o == pcx.ADD:
            xl, xu = np.maximum(xl, yl + zl), np.minimum(xu, yu + zu)
            yl, yu = np.maximum(yl, xl - zu), np.minimum(yu, xu - zl)
            zl, zu = np.maximum(zl, xl - yu), np.minimum(zu, xu - yl)
        elif o == pcx.MUL:
            xl, xu = np.maximum(xl, np.minimum(yl * zl, _HI)), np.minimum(xu, np.minimum(yu * zu, _HI))
            zl = np.where((xl > 0) & (zl == 0), 1, zl)
            can = (zl > 0) & (zl <= zu)
            d, e = np.maximum(zu, 1), np.maximum(zl, 1)
            yl, yu = np.where(can, np.maximum(yl, -(-xl // d)), yl), np.where(can, np.minimum(yu, xu // e), yu)
            yl = np.where((xl > 0) & (yl == 0), 1, yl)
            can = (yl > 0) & (yl <= yu)
            d, e = np.maximum(yu, 1), np.maximum(yl, 1)
            zl, zu = np.where(can, np.maximum(zl, -(-xl // d)), zl), np.where(can, np.minimum(zu, xu // e), zu)
        elif o == pcx.MIN:
            xl, xu = np.maximum(xl, np.minimum(yl, zl)), np.minimum(xu, np.minimum(yu, zu))
            yl, zl2 = np.maximum(yl, xl), np.maximum(zl, xl)
            yu, zu, zl = np.where(xu < zl, np.minimum(yu, xu), yu), np.where(xu < yl, np.minimum(zu, xu), zu), zl2
        elif o == pcx.MAX:
            xl, xu = np.maximum(xl, np.maximum(yl, zl)), np.minimum(xu, np.maximum(yu, zu))
            yu, zu2 = np.minimum(yu, xu), np.minimum(zu, xu)
            yl, zl, zu = np.where(xl > zu, np.maximum(yl, xl), yl), np.where(xl > yu, np.maximum(zl, xl), zl), zu2
        else:                                           # x <=> (y = z), x <=> (y <= z)
            t, f = (xl == 1) & (xu == 1), (xl == 0) & (xu == 0)
            if o == pcx.EQ:
                fy, fz = f & (zl == zu), f & (yl == yu) & (zl != zu)
                low, high = yl == zl, yu == zu
                true, false = (yl == yu) & (zl == zu) & (yl == zl), (yl > zu) | (yu < zl)
                ny = np.where(t, zl, np.where(fy & low, yl + 1, yl)), np.where(t, zu, np.where(fy & high, yu - 1, yu))
                nz = np.where(t, yl, np.where(fz & low, zl + 1, zl)), np.where(t, yu, np.where(fz & high, zu - 1, zu))
            else:
                true, false = yu <= zl, yl > zu
                ny = np.where(f, zl + 1, yl), np.where(t, zu, yu)
                nz = np.where(t, yl, zl), np.where(f, yu - 1, zu)
            xl = np.where(~t & ~f & true, 1, xl)
            xu = np.where(~t & ~f & ~true & false, 0, xu)
            (yl, yu), (zl, zu) = ny, nz
        _meet(lb, ub, X, xl, xu)
        _meet(lb, ub, Y, yl, yu)
        _meet(lb, ub, Z, zl, zu)
    return (lb != old_l) | (ub != old_u)


def exact(case, seed):
    """The greatest common fixpoint of one interval store, by sweeps of numpy
    in 64 bits over the propagators whose operands changed.  None for batches,
    servers and bitsets (minutes of numpy) and for the largest networks."""
    if case["path"] not in ("single", "noalloc") or case["domain"] != "itv" or case["nprops"] > 500000:
        return None
    op, x, y, z, lb, ub, _ = _network(case, int(seed) % (1 << 30) + 1)
    lb, ub = lb.astype(np.int64), ub.astype(np.int64)
    out = x[(op == pcx.EQ) | (op == pcx.LEQ)]           # reified outputs are told in [0, 1]
    lb[out], ub[out] = np.maximum(lb[out], 0), np.minimum(ub[out], 1)
    on = np.ones(len(op), bool)
    while on.any():
        changed = _sweep(op[on], x[on], y[on], z[on], lb, ub)
        on = changed[x] | changed[y] | changed[z]
    return {"lb": lb.astype(np.int32), "ub": ub.astype(np.int32), "failed": int((lb > ub).any())}
