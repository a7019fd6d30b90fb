"""The framework's performance cases: whole annealing runs, population steps and scoring of start trees through
treesa_gpu_amd.capi, at the sizes its configurations, tests and benchmark use.

A case names a network family (random 3-SAT, random 3-regular graph, open square lattice), the way a program drives
the library and the run's size:

* anneal: independent chains, the whole beta schedule through tsa_track_begin / tsa_anneal / tsa_track_end, then the
  energies of every chain;
* population: population annealing, the level loop on the host: tsa_sweeps, tsa_energy, systematic resampling;
* buffers: tsa_sweeps_noalloc on device buffers that the caller owns, energies included;
* score: a population of trees uploaded and evaluated, as before every run.

A pass starts from the population as the previous pass left it (a first pass from the start trees) and goes through
the schedule again from its hottest level, with random numbers of its own.
"""
import math

import numpy as np
import torch

from treesa_gpu_amd import capi, host, instances

# Populations of up to this size come back whole; of larger ones a program takes the best tree, the trace and
# every chain's energies, and leaves the records on the device.
RECORDS_MAX = 128 << 20


def listed():
    return [
        # one short call on buffers a serving loop owns: launches and latency count
        dict(name="buffers_sat60", kind="buffers", family="sat", size=60, order="par", mode="tc", slicing=False,
             chains=64, levels=1, niters=2, beta0=4.0, beta1=4.0, sc_target=20.0),
        # the pre-order sweep with one chain per compute unit: random 3-SAT n=100, 256 chains x 100 sweeps
        dict(name="preorder_sat100", kind="anneal", family="sat", size=100, order="preorder", mode="tc", slicing=False,
             chains=256, levels=100, niters=1, beta0=0.01, beta1=15.0, sc_target=20.0),
        # best-of-N over a population that fills the device: the benchmark's default workload
        dict(name="best_of_n_sat100", kind="anneal", family="sat", size=100, order="par", mode="tc", slicing=False,
             chains=8192, levels=100, niters=1, beta0=1.0, beta1=15.0, sc_target=20.0),
        # few chains and several sweeps per level, the usual shape of one user's run: 72 trials on a 14 x 14 lattice
        dict(name="trials_sq14", kind="anneal", family="sq", size=14, order="par", mode="tc", slicing=False, chains=72,
             levels=20, niters=10, beta0=0.01, beta1=15.0, sc_target=12.0),
        # population annealing with slice moves: random 3-SAT n=70, 2048 chains x 200 sweeps
        dict(name="sliced_population_sat70", kind="population", family="sat", size=70, order="par", mode="tc",
             slicing=True, chains=2048, levels=20, niters=10, beta0=0.01, beta1=15.0, sc_target=24.0),
        # the modeled GPU time as the energy, as in the second stage of a two-stage run
        dict(name="gpu_time_sat100", kind="anneal", family="sat", size=100, order="par", mode="gpu", slicing=False,
             chains=576, levels=10, niters=10, beta0=1.0, beta1=15.0, sc_target=30.0),
        # the measured-time model, pre-order, on a 3-regular graph of 375 labels
        dict(name="h100_time_reg250", kind="anneal", family="reg3", size=250, order="preorder", mode="h100",
             slicing=False, chains=144, levels=10, niters=5, beta0=1.0, beta1=15.0, sc_target=30.0),
        # label sets of 47 words in HBM, a population of two chains per compute unit: 3-regular graph n=2000
        dict(name="wide_reg2000", kind="anneal", family="reg3", size=2000, order="par", mode="tc", slicing=False,
             chains=512, levels=40, niters=1, beta0=1.0, beta1=15.0, sc_target=40.0),
        # the 64 x 64 lattice, 8064 labels, few chains
        dict(name="wide_sq64", kind="anneal", family="sq", size=64, order="par", mode="tc", slicing=False, chains=72,
             levels=40, niters=2, beta0=0.01, beta1=15.0, sc_target=70.0),
        # the pre-order sweep on label sets in HBM: 32 x 32 lattice, 1984 labels
        dict(name="wide_preorder_sq32", kind="anneal", family="sq", size=32, order="preorder", mode="tc",
             slicing=False, chains=64, levels=3, niters=2, beta0=0.01, beta1=15.0, sc_target=25.0),
        # slicing where it is needed most, on a network whose tensors outgrow one device: 24 x 24 lattice
        dict(name="wide_sliced_sq24", kind="anneal", family="sq", size=24, order="par", mode="tc", slicing=True,
             chains=128, levels=5, niters=4, beta0=0.01, beta1=15.0, sc_target=18.0),
        # the start of every run: a population of trees uploaded, checked and evaluated
        dict(name="score_sat100", kind="score", family="sat", size=100, order="par", mode="tc", slicing=False,
             chains=1024, levels=0, niters=0, beta0=0.0, beta1=0.0, sc_target=20.0),
    ]


# What draw() takes its cases from: kind, family, sizes, chains, orders, modes, slicing, and the most visits (internal
# nodes x chains x sweeps) that a drawn case has, as many as the listed case of that sort.
SORTS = (
    ("buffers", "sat", (20, 100), (16, 512), ("par", "preorder"), ("tc",), False, 4e6),
    ("anneal", "sat", (20, 120), (16, 4096), ("par", "preorder"), ("tc", "tc", "gpu", "h100"), False, 2e7),
    ("anneal", "sat", (60, 100), (3072, 8192), ("par",), ("tc",), False, 3.4e8),
    ("anneal", "reg3", (40, 320), (16, 576), ("par", "preorder"), ("tc", "tc", "gpu", "h100"), False, 5e6),
    ("anneal", "sq", (6, 16), (16, 576), ("par", "preorder"), ("tc", "tc", "gpu"), False, 5e6),
    ("population", "sat", (30, 100), (128, 2048), ("par",), ("tc",), True, 1e8),
    ("population", "reg3", (60, 300), (64, 1024), ("par", "preorder"), ("tc",), False, 1e7),
    ("anneal", "reg3", (400, 2000), (64, 512), ("par",), ("tc", "tc", "gpu"), False, 2e7),
    ("anneal", "sq", (18, 64), (24, 192), ("par",), ("tc",), False, 1e7),
    ("anneal", "sq", (18, 46), (16, 96), ("preorder",), ("tc",), False, 5e5),
    ("anneal", "sq", (18, 32), (16, 192), ("par",), ("tc",), True, 7e5),
    ("score", "sat", (40, 120), (64, 2048), ("par",), ("tc",), False, 0),
)


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind, family, sizes, chains, orders, modes, slicing, most = rng.choice(SORTS)
    size = spread(*sizes)
    if family == "reg3":
        size += size & 1  # a 3-regular graph has an even number of vertices
    c = dict(kind=kind, family=family, size=size, order=rng.choice(orders), mode=rng.choice(modes), slicing=slicing,
             chains=spread(*chains), levels=0, niters=0, beta0=rng.choice((0.01, 1.0)), beta1=rng.choice((8.0, 15.0)),
             sc_target=float(rng.randint(10, 40)))
    if kind == "score":
        return c
    nodes = {"sat": round(4.26 * size), "reg3": size, "sq": size * size}[family] - 1
    if c["mode"] != "tc":
        most /= 4
    sweeps = max(2, int(most * rng.uniform(0.2, 1.0) / (nodes * c["chains"])))
    if kind == "buffers":
        c["levels"], c["niters"] = 1, min(sweeps, 8)
        return c
    c["niters"] = rng.choice([k for k in (1, 2, 5, 10, 25, 50) if 2 * k <= sweeps])
    c["levels"] = max(2, min(100, sweeps // c["niters"]))
    c["chains"] = max(2, min(c["chains"], int(most / (nodes * c["levels"] * c["niters"])) or 2))
    return c


def _network(case, seed):
    """(tensors' labels, host instance, layout) of the case's network; random families draw it from the seed."""
    if case["family"] == "sq":
        ixs, iy = instances.sq(case["size"])
    elif case["family"] == "sat":
        ixs, iy = instances.sat(case["size"], seed=seed)
    else:
        ixs, iy = instances.reg3(case["size"], seed=seed)
    names = instances.label_map(ixs, iy)
    ixs = [[names[x] for x in ix] for ix in ixs]
    inst = host.Instance(m=len(ixs), nlab=len(names), ixs=ixs, iy=[])
    return ixs, inst, capi.layout(inst.m, inst.nlab)


def _trees(case, inst, seed):
    """Start trees: the greedy method's, or on lattices the row by row path; eight random ones to score."""
    if case["kind"] == "score":
        return np.stack([host.random_tree(inst.m, host.splitmix64(seed * 8 + k)) for k in range(8)])
    if case["family"] == "sq":
        return host.path_tree(np.arange(inst.m))[None]
    return np.stack([inst.greedy_tree(1, seed + k)[0] for k in range(2)])


def prepare(case, seed):
    ixs, inst, lay = _network(case, seed)
    chains = case["chains"]
    cfg = capi.make_config(mode=case["mode"], sc_target=case["sc_target"], seed=seed, slicing=case["slicing"],
                           fused_energy=True)
    pop = inst.population(lay, _trees(case, inst, seed), chains, seed=seed)
    leaf = inst.leaf(lay.W)
    order = capi.ORDER_PAR if case["order"] == "par" else capi.ORDER_PREORDER
    levels = case["levels"]
    st = dict(case=case, lay=lay, cfg=cfg, order=order, sweep=0, leaf_sc=inst.leaf_sc)
    st["betas"] = np.linspace(case["beta0"], case["beta1"], levels, dtype=np.float32) if levels else None
    st["niters"] = np.full(levels, case["niters"], np.int32)
    st["every"] = np.ones(levels, np.uint8)
    if case["kind"] == "buffers":
        st["leaf"] = torch.from_numpy(leaf.view(np.int64)).cuda()
        st["pop"] = torch.from_numpy(pop.view(np.int64)).cuda()
        st["lc"] = torch.empty(chains, dtype=torch.float32, device="cuda")
        st["sc"], st["ns"] = (torch.empty(chains, dtype=torch.int32, device="cuda") for _ in range(2))
        st["stats"] = torch.empty(7, dtype=torch.int64, device="cuda")
        return st
    st["ctx"] = capi.Context(lay, leaf, inst.leaf_sc, cfg, chains)
    st["rng"] = np.random.RandomState(seed % (1 << 31))
    if case["kind"] == "score":
        # a program that scores trees holds them in page-locked memory, like every buffer it copies from
        st["trees"] = torch.from_numpy(pop.view(np.int64)).pin_memory()
        return st
    st["ctx"].upload(pop)
    if pop.nbytes <= RECORDS_MAX:
        st["records"] = torch.empty(pop.shape, dtype=torch.int64, pin_memory=True)
    return st


def _finish(st, out):
    """What a program takes after a run: every chain's energies, the counters and, where they fit, the records."""
    ctx = st["ctx"]
    out["lc"], out["sc"], out["ns"] = ctx.energy()
    now = np.array(ctx.stats(), np.int64)
    out["counters"] = now - st.get("counted", 0)
    st["counted"] = now
    if "records" in st:
        ctx._check(ctx.lib.tsa_download(ctx.h, 0, ctx.nchains, st["records"].data_ptr()))
        out["records"] = st["records"]
    return out


def _advance(st, sweeps):
    """The sweep counter (the random numbers' second key) goes on from pass to pass."""
    s = st["sweep"]
    st["sweep"] = (s + sweeps) % (1 << 30)
    return s


def _anneal(st):
    case, ctx = st["case"], st["ctx"]
    ctx.track_begin(case["mode"], case["slicing"], sc_target=case["sc_target"], max_levels=case["levels"])
    ctx.anneal(st["order"], st["betas"], st["niters"], st["every"], sweep0=_advance(st, int(st["niters"].sum())))
    chain, level, score, record, rows, _, _ = ctx.track_end()
    lay = st["lay"]
    out = dict(chain=chain, level=level, score=score, tree=record[lay.ch_off:lay.s_off + lay.W].view(np.int64))
    for field in ("lc", "sc", "ns", "chain", "score", "meanE", "meanNs"):
        out["trace_" + field] = np.ascontiguousarray(rows[field])
    return _finish(st, out)


def _population(st):
    case, ctx, betas, n = st["case"], st["ctx"], st["betas"], st["case"]["chains"]
    sweep = _advance(st, int(st["niters"].sum()))
    energies, ancestors = [], []
    for k in range(case["levels"]):
        ctx.sweeps(st["order"], betas[k], sweep, case["niters"])
        sweep += case["niters"]
        if k + 1 == case["levels"]:
            break
        lc, sc, ns = ctx.energy()
        energies.append(lc)
        over = np.maximum(sc - case["sc_target"], 0.0)
        e = lc.astype(np.float64) + ns + over
        w = np.cumsum(np.exp(-float(betas[k + 1] - betas[k]) * (e - e.min())))
        u = (np.arange(n) + st["rng"].random_sample()) / n * w[-1]
        anc = np.minimum(np.searchsorted(w, u, side="right"), n - 1).astype(np.int32)
        ancestors.append(anc)
        ctx.resample(anc)
    return _finish(st, dict(energies=np.stack(energies), ancestors=np.stack(ancestors)))


def _buffers(st):
    case = st["case"]
    s = _advance(st, case["niters"])
    capi.sweeps_noalloc(st["lay"], st["cfg"], st["leaf_sc"], st["leaf"].data_ptr(), st["pop"].data_ptr(),
                        case["chains"], st["order"], case["beta1"], s, case["niters"], st["lc"].data_ptr(),
                        st["sc"].data_ptr(), st["ns"].data_ptr(), st["stats"].data_ptr(),
                        torch.cuda.current_stream().cuda_stream)
    return dict(records=st["pop"], lc=st["lc"], sc=st["sc"], ns=st["ns"], counters=st["stats"])


def _score(st):
    ctx = st["ctx"]
    ctx._check(ctx.lib.tsa_upload(ctx.h, st["trees"].data_ptr()))
    lc, sc, ns = ctx.energy()
    return dict(lc=lc, sc=sc, ns=ns)


def run(state):
    return {"anneal": _anneal, "population": _population, "buffers": _buffers,
            "score": _score}[state["case"]["kind"]](state)


def _shape(case):
    """(tensors, labels at most) of the case's network, without making it."""
    n = case["size"]
    if case["family"] == "sat":
        return round(4.26 * n), n
    if case["family"] == "reg3":
        return n, 3 * n // 2
    return n * n, 2 * n * (n - 1)


def work(case):
    """Bytes: the records and the leaf sets read once, the records written once (an evaluation: read only).  Flops:
    32-bit integer operations of the visits' set arithmetic (four label sets per proposal: the pivot's new set, two
    sizes and two intersections, a logic operation and a population count each) and of one evaluation per level."""
    m, labels = _shape(case)
    lay = capi.layout(m, labels)
    records = 8 * lay.chain_words * case["chains"]
    words = -(-labels // 32)
    visits = (m - 1) * case["chains"] * case["levels"] * case["niters"]
    evaluated = (m - 1) * case["chains"] * max(1, case["levels"])
    model = 1 if case["mode"] == "tc" else 3
    return {"bytes": records * (1 if case["kind"] == "score" else 2) + 8 * m * lay.W,
            "flops": float(visits * (10 * words * model + 60) + evaluated * (4 * words + 40))}


def tolerance(case):
    # Trees and counters are whole numbers, and an energy is a fold of its nodes' costs in a fixed order of 32-bit
    # operations: the library promises the same bits from every kernel and every plan, and selection and slice moves
    # decide on them.
    return "exact"


def exact(case, seed):
    """Energies of scored trees: log2 of the sum of 2^cost over the contractions, cost = the number of labels in the
    two operands.  What a run returns follows from a chain of accept decisions on 32-bit energies and has no 64-bit
    value of its own."""
    if case["kind"] != "score":
        return None
    ixs, inst, _ = _network(case, seed)
    lc = []
    for tree in _trees(case, inst, seed):
        m = inst.m
        left = {}
        for ix in ixs:
            for x in ix:
                left[x] = left.get(x, 0) + 1
        child = [(int(w) & 0xFFFF, int(w) >> 16) for w in tree]
        depth, todo = [], [2 * m - 2]
        while todo:  # parents before children
            v = todo.pop()
            if v >= m:
                depth.append(v)
                todo.extend(child[v - m])
        inside = {i: _count(ixs[i]) for i in range(m)}
        costs = []
        for v in reversed(depth):
            a, b = inside.pop(child[v - m][0]), inside.pop(child[v - m][1])
            costs.append(float(len(a.keys() | b.keys())))
            for x, k in b.items():
                a[x] = a.get(x, 0) + k
            inside[v] = {x: k for x, k in a.items() if k < left[x]}
        costs = np.array(costs)
        lc.append(costs.max() + np.log2(np.sum(np.exp2(costs - costs.max()))))
    lc = np.array(lc, np.float64)
    return dict(lc=lc[np.arange(case["chains"]) % len(lc)], sc=None, ns=None)


def _count(labels):
    n = {}
    for x in labels:
        n[x] = n.get(x, 0) + 1
    return n
