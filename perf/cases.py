"""The work that users of this package have it do, as measurable cases.

The sizes are those of the served model and its tensor-parallel shares
(16 / 8 / 4 q/k heads, 32 / 16 / 8 v heads of width 128, up to 24 GDN layers,
8192 / tp conv channels) and of the draft trees it verifies (1 to 64 nodes,
chains, bushy and random trees), at batch 1 (the serving plugin) up to 128.

The kinds of case, each one a part of a speculative decoding step:

plugin     what the serving hooks drive at batch 1, per draft tree: the
           ancestry pack, conv + verify of every GDN layer, then the snapshot
           commit of the accepted path.  Captured in a HIP graph, as the
           serving engine runs its verify forward.
pipelined  the batched step: per layer one launch that commits the previous
           step's accepted path into the state pool and verifies this step's
           trees on it.  In a HIP graph.
separate   the batched step in two passes: the verify of every layer, saving
           keys, values and gains, then one in-place commit over all layers.
           In a HIP graph.
conv       the batched front end: the tree conv of every layer, with each
           node's window.  In a HIP graph.
plan       the attention plan's packed mask of one request, from the boolean
           mask the worker hands over (eager, once per step).
mask       the packed masks of a whole batch from the ancestry bits (eager,
           once per step).
trees      the structure of a batch of fresh draft trees (eager, once per
           step).
invert     the standalone block inverse, in place (eager).

A graph is captured once in prepare() and replayed by run(), so a pass is the
launches themselves; it is captured from the same entry points that the eager
kinds call.
"""
from __future__ import annotations

import math
import types

import torch

D = 128
HK, HV, CHANNELS = 16, 32, 8192  # the whole model's; a tp share has 1 / tp of each
PATH_COLS = 16                   # columns of an accepted path (-1 padded)
SIZES = (16, 32, 64)             # tree sizes the plugin dispatches on


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the serving plugin at batch 1: small and default draft trees
        dict(name="plugin_b1_n32", kind="plugin", nodes=32, layers=24, tp=1, tree="random"),
        dict(name="plugin_b1_n64", kind="plugin", nodes=64, layers=24, tp=1, tree="random"),
        # the batched step: a full server, a quiet one, and one with trees of every size
        dict(name="pipelined_b64_n32", kind="pipelined", batch=64, lo=32, hi=32, layers=24, tp=1, gates="bf16", shape=1),
        dict(name="pipelined_b4_n27", kind="pipelined", batch=4, lo=27, hi=27, layers=24, tp=1, gates="bf16", shape=2),
        dict(name="pipelined_b48_ragged", kind="pipelined", batch=48, lo=8, hi=64, layers=8, tp=1, gates="f32", shape=3),
        # verify and commit as two passes: a large ragged batch, and a middling one at tp 2
        dict(name="separate_b128_ragged", kind="separate", batch=128, lo=8, hi=64, layers=4, tp=1, gates="bf16", shape=4),
        dict(name="separate_b12_n48_tp2", kind="separate", batch=12, lo=48, hi=48, layers=12, tp=2, gates="f32", shape=5),
        # the front end of a full server's step
        dict(name="conv_b64_n32", kind="conv", batch=64, nodes=32, layers=6, tp=1, tree="random"),
        # the attention masks: one request with a long context; a full batch with middling ones
        dict(name="plan_n64_ctx32k", kind="plan", nodes=64, prefix=32731),
        dict(name="mask_b64_ctx6k", kind="mask", batch=64, lo=16, hi=64, prefix=6000, shape=6),
        # a batch of fresh draft trees
        dict(name="trees_b128", kind="trees", batch=128, lo=8, hi=64, shape=7),
        # one 64-node inverse per (request, head) of a full batch
        dict(name="invert_n64_x2048", kind="invert", nodes=64, mats=2048),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def _tree_range(rng):
    """Nodes per tree: one size for the batch, or a range of sizes."""
    if rng.random() < 0.5:
        n = rng.randint(4, 64)
        return n, n
    lo = rng.randint(1, 32)
    return lo, rng.randint(lo + 8, 64)


def draw(rng):
    kind = rng.choice(["plugin", "pipelined", "pipelined", "separate", "separate", "conv", "plan", "mask", "trees",
                       "invert"])
    tp = rng.choice([1, 1, 2, 4])
    shape = rng.randrange(1 << 20)
    tree = rng.choice(["random", "random", "chain", "bushy"])
    gates = rng.choice(["bf16", "f32"])
    if kind == "plugin":
        return dict(kind=kind, nodes=rng.choice(SIZES), layers=rng.randint(6, 24), tp=tp, tree=tree)
    if kind in ("pipelined", "separate"):
        batch = _log_int(rng, 1, 96)
        lo, hi = _tree_range(rng)
        layers = max(1, min(rng.randint(4, 24), 480 * tp // batch))
        return dict(kind=kind, batch=batch, lo=lo, hi=hi, layers=layers, tp=tp, gates=gates, shape=shape)
    if kind == "conv":
        batch = _log_int(rng, 1, 64)
        return dict(kind=kind, batch=batch, nodes=rng.randint(4, 64), layers=rng.randint(2, 6), tp=tp, tree=tree)
    if kind == "plan":
        return dict(kind=kind, nodes=rng.choice(SIZES), prefix=_log_int(rng, 100, 131072))
    if kind == "mask":
        lo, hi = _tree_range(rng)
        return dict(kind=kind, batch=_log_int(rng, 1, 128), lo=lo, hi=hi, prefix=_log_int(rng, 100, 32768), shape=shape)
    if kind == "trees":
        lo, hi = _tree_range(rng)
        return dict(kind=kind, batch=_log_int(rng, 1, 256), lo=lo, hi=hi, shape=shape)
    return dict(kind="invert", nodes=rng.choice(SIZES), mats=_log_int(rng, 16, 4096))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _device():
    return torch.device("cuda:0")


class _Source:
    """Seeded device tensors."""

    def __init__(self, seed):
        self.g = torch.Generator(device=_device()).manual_seed(int(seed) * 7919 + 17)

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        return torch.empty(shape, device=_device(), dtype=dtype).normal_(0.0, std, generator=self.g)


def _sizes(case):
    """Nodes of every request (from the case alone: they are its shape)."""
    if "lo" not in case:
        return [case["nodes"]] * case.get("batch", 1)
    if case["lo"] == case["hi"]:
        return [case["lo"]] * case["batch"]
    g = torch.Generator().manual_seed(case["shape"])
    return torch.randint(case["lo"], case["hi"] + 1, (case["batch"],), generator=g).tolist()


def _prefixes(case):
    """Committed tokens of every request, about the case's prefix (from the case alone)."""
    g = torch.Generator().manual_seed(case["shape"] + 1)
    return (case["prefix"] * (0.5 + torch.rand(case["batch"], generator=g))).int().tolist()


def _parents(sizes, seed, kind=None):
    """int32 parents (-1 for the root) of one tree per request; a batch mixes
    random, chain and bushy trees unless it is of one kind."""
    g = torch.Generator().manual_seed(int(seed) * 31 + 5)
    u = torch.rand(sum(sizes), generator=g).tolist()
    out, at = [], 0
    for r, n in enumerate(sizes):
        k = kind or ("random", "random", "chain", "bushy")[r % 4]
        wide = max(1, int(math.sqrt(max(n - 1, 1))))  # depth-1 nodes of a bushy tree
        for i in range(n):
            x = u[at + i]
            if i == 0:
                p = -1
            elif k == "chain":
                p = i - 1
            elif k == "bushy":
                p = 0 if i <= wide else 1 + int(x * wide)
            else:
                p = min(int(x * i), i - 1)
            out.append(p)
        at += n
    return out


def _paths(parents, sizes, seed):
    """One accepted root-to-node walk per request, at most PATH_COLS long."""
    g = torch.Generator().manual_seed(int(seed) * 131 + 3)
    u = torch.rand(len(sizes), PATH_COLS + 1, generator=g).tolist()
    out, at = [], 0
    for r, n in enumerate(sizes):
        children = [[] for _ in range(n)]
        for i in range(1, n):
            children[parents[at + i]].append(i)
        path, most = [0], 1 + int(u[r][PATH_COLS] * PATH_COLS)
        while len(path) < min(most, PATH_COLS) and children[path[-1]]:
            ch = children[path[-1]]
            path.append(ch[min(int(u[r][len(path)] * len(ch)), len(ch) - 1)])
        out.append(path)
        at += n
    return out


def _padded(paths, cols=PATH_COLS):
    t = torch.full((len(paths), cols), -1, dtype=torch.int32)
    for i, p in enumerate(paths):
        t[i, :len(p)] = torch.tensor(p, dtype=torch.int32)
    return t.to(_device())


def _captured(fn):
    """fn's launches as a HIP graph, and what fn returned while captured."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


def _heads(case):
    return HK // case["tp"], HV // case["tp"]


def _gate_dtype(case):
    return torch.bfloat16 if case.get("gates", "bf16") == "bf16" else torch.float32


def _inputs(case, seed):
    """The tensors of a case, before anything of the package is called."""
    dev, src, kind = _device(), _Source(seed), case["kind"]
    s = types.SimpleNamespace(case=case)
    s.sizes = _sizes(case)
    if kind == "invert":
        n = case["nodes"]
        a = src.normal(case["mats"], n, n, std=0.2)
        on = torch.rand(case["mats"], n, n, device=dev, generator=src.g) < 0.25
        s.a = torch.tril(a * on, -1).contiguous()
        return s
    if kind == "plan":
        n, plen = case["nodes"], case["prefix"]
        s.parents = _parents([n], seed, "random")
        s.mask = torch.cat((torch.ones(n, plen, device=dev, dtype=torch.bool), _anc64(s.parents, [n])[0] > 0), 1)
        return s
    s.parents = _parents(s.sizes, seed, case.get("tree"))
    s.parent = torch.tensor(s.parents, dtype=torch.int32, device=dev)
    rows, batch = sum(s.sizes), len(s.sizes)
    s.n = max(s.sizes)
    s.cu = None
    if min(s.sizes) != s.n:
        s.cu = torch.tensor([0] + torch.tensor(s.sizes).cumsum(0).tolist(), dtype=torch.int32, device=dev)
    if kind == "trees":
        return s
    if kind == "mask":
        s.plens = _prefixes(case)
        s.prefix = torch.tensor(s.plens, dtype=torch.int32, device=dev)
        return s
    L, tp = case["layers"], case["tp"]
    hk, hv = _heads(case)
    chan = CHANNELS // tp
    bf16 = torch.bfloat16
    if kind in ("plugin", "conv"):
        s.x = src.normal(L, batch, s.n, chan, dtype=bf16)
        s.conv_state = src.normal(L, batch, chan, 3, dtype=bf16)
        s.weight = src.normal(L, chan, 4, std=0.5, dtype=bf16)
        if kind == "conv":
            s.y = torch.empty(L, batch, s.n, chan, device=dev, dtype=bf16)
            s.window = torch.empty(L, batch, s.n, chan, 3, device=dev, dtype=bf16)
            return s
    else:
        s.y = src.normal(L, rows, chan, dtype=bf16)
    s.a = src.normal(L, rows, hv, dtype=_gate_dtype(case))
    s.b = src.normal(L, rows, hv, dtype=_gate_dtype(case))
    s.A_log = torch.empty(L, hv, device=dev).uniform_(-1.5, 0.5, generator=src.g)
    s.dt_bias = src.normal(L, hv, std=0.3)
    s.state = src.normal(L, batch, hv, D, D, std=0.02)  # [layer, slot, head, V, K]
    s.slots = torch.randperm(batch, generator=src.g, device=dev).to(torch.int32)
    s.o = None if kind == "plugin" else torch.empty(L, rows, hv, D, device=dev, dtype=bf16)
    s.gains = torch.empty(L, hv, rows, device=dev)
    paths = _paths(s.parents, s.sizes, seed)
    if kind == "plugin":
        s.paths = paths
        s.track = paths[0][len(paths[0]) // 2]
        s.keys = torch.empty(L, hv, rows, D, device=dev)
        s.values = torch.empty(L, hv, rows, D, device=dev)
        s.window = torch.empty(L, 1, s.n, chan, 3, device=dev, dtype=bf16)
        s.snapshots = torch.zeros(L, 1, s.n, hv, D, D, device=dev)
    elif kind == "separate":
        s.paths = paths
        s.keys = torch.empty(L, hk, rows, D, device=dev)
        s.values = torch.empty(L, hv, rows, D, device=dev)
    else:  # the previous step's: trees of the same sizes, rows, gates, decays and accepted walk
        s.prev_parents = _parents(s.sizes, seed + 101)
        s.paths = _paths(s.prev_parents, s.sizes, seed)
        s.prev_parent = torch.tensor(s.prev_parents, dtype=torch.int32, device=dev)
        s.prev_y = src.normal(L, rows, chan, dtype=bf16)
        s.prev_b = src.normal(L, rows, hv, dtype=_gate_dtype(case))
        prev_a = src.normal(L, rows, hv, dtype=_gate_dtype(case))
        anc = _anc64(s.prev_parents, s.sizes)
        g = _decay64(prev_a, s.A_log, s.dt_bias)  # [L, rows, hv]
        s.prev_gains = _unpad(torch.matmul(anc, _pad(g, s.sizes)), s.sizes).permute(0, 2, 1).float().contiguous()
    return s


def prepare(case, seed):
    from dforktree_amd import ops

    s = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("invert", "trees"):
        return s
    if kind == "plan":
        # the attention wrapper's own buffers, sized for its longest context
        s.wrapper = types.SimpleNamespace(
            _custom_mask_buf=torch.zeros((s.mask.numel() + 7) // 8, device=_device(), dtype=torch.uint8),
            _mask_indptr_buf=torch.zeros(2, device=_device(), dtype=torch.int32))
        return s
    packed = {} if s.cu is None else dict(cu_seqlens=s.cu)
    tree = ops.tree_struct(s.parent, 4, batch=len(s.sizes), n_nodes=s.n, want=("anc", "anc_bits", "cidx"),
                           index_dtype=torch.int32, **packed)
    s.anc_bits = tree["anc_bits"]
    if kind == "mask":
        s.out = torch.zeros(_mask_bytes(s.sizes, s.plens), device=_device(), dtype=torch.uint8)
        s.indptr = torch.zeros(len(s.sizes) + 1, device=_device(), dtype=torch.int32)
        return s
    if kind == "conv":
        s.cidx = tree["cidx"].view(len(s.sizes), s.n, 4)
        s.graph, _ = _captured(lambda: _conv_layers(s))
        return s
    if kind == "plugin":
        s.anc, s.cidx = tree["anc"][0].contiguous(), tree["cidx"]
        s.neg = [-s.A_log[l].exp() for l in range(case["layers"])]
        s.accept = _padded(s.paths)
        s.ends = torch.tensor([[s.paths[0][-1], s.track]], device=_device(), dtype=torch.int32)
        s.islot = torch.zeros(1, device=_device(), dtype=torch.int32)
        s.graph, s.out = _captured(lambda: _plugin_step(s))
        return s
    # the capture's own warm-up pass commits nothing: every path is empty until it is done
    accept = _padded(s.paths)
    s.accept = torch.full_like(accept, -1)
    s.order = None if s.cu is None else ops.size_order(s.cu, s.n)
    if kind == "pipelined":
        s.prev_anc_bits = ops.tree_struct(s.prev_parent, 4, batch=len(s.sizes), n_nodes=s.n, want=("anc_bits",),
                                          **packed)["anc_bits"]
        s.graph, _ = _captured(lambda: _pipelined_step(s))
    else:
        s.graph, _ = _captured(lambda: _separate_step(s))
    s.accept.copy_(accept)
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _conv_layers(s):
    from dforktree_amd import ops
    for l in range(s.case["layers"]):
        ops.tree_conv(s.x[l], s.conv_state[l], s.weight[l], None, s.cidx, y=s.y[l], iw=s.window[l])


def _plugin_step(s):
    from dforktree_amd import ops
    from dforktree_amd.plugin import fc1_conv, fc1_fused, tree_kernels
    hk, hv = _heads(s.case)
    bits = torch.empty(s.n, device=_device(), dtype=torch.int64)
    ys, os = [], []
    for l in range(s.case["layers"]):
        y = torch.empty(1, s.n, s.x.shape[-1], device=_device(), dtype=s.x.dtype)
        fc1_conv.conv(s.x[l].transpose(1, 2), s.conv_state[l], s.weight[l], None, s.cidx, s.slots, s.islot,
                      s.window[l], y)
        if l == 0:
            ops.anc_pack(s.anc, out=bits)
        pool = s.state[l]
        o = tree_kernels.tree_gdn_split(y[0], s.a[l], s.b[l], s.A_log[l], s.dt_bias[l], pool[0].transpose(-1, -2),
                                        s.anc, hk, hv, D, D, aux=(s.keys[l], s.values[l], s.gains[l]),
                                        neg_exp_A=s.neg[l], state_indices=s.slots, state_slot_stride=pool.stride(0),
                                        anc_bits=bits)
        ys.append(y)
        os.append(o)
    fc1_fused.snapshot_commit(s.state, s.keys, s.values, s.gains, s.anc, s.accept, s.ends, s.slots, s.islot,
                              s.snapshots, anc_bits=bits)
    return ys, os


def _pipelined_step(s):
    from dforktree_amd import ops
    hk, hv = _heads(s.case)
    for l in range(s.case["layers"]):
        prev = s.prev_y[l]
        ops.tree_commit_verify(
            s.y[l], s.a[l], s.b[l], s.A_log[l], s.dt_bias[l], s.state[l].transpose(-1, -2), hk=hk, hv=hv,
            anc_bits=s.anc_bits, batch=len(s.sizes), n_nodes=s.n, cu_seqlens=s.cu, state_indices=s.slots, o=s.o[l],
            aux_g=s.gains[l], size_order=s.order, pending_path=s.accept, pending_keys=None, pending_values=None,
            pending_key_rows=prev[:, hk * D:2 * hk * D].unflatten(1, (hk, D)),
            pending_value_rows=prev[:, 2 * hk * D:].unflatten(1, (hv, D)), pending_b=s.prev_b[l],
            pending_gains=s.prev_gains[l], prev_cu_seqlens=s.cu, prev_n_nodes=s.n, pending_k_head_div=hv // hk,
            pending_anc_bits=s.prev_anc_bits)


def _separate_step(s):
    from dforktree_amd import ops
    hk, hv = _heads(s.case)
    for l in range(s.case["layers"]):
        ops.tree_verify(s.y[l], s.a[l], s.b[l], s.A_log[l], s.dt_bias[l], s.state[l].transpose(-1, -2), hk=hk, hv=hv,
                        anc_bits=s.anc_bits, batch=len(s.sizes), n_nodes=s.n, cu_seqlens=s.cu, state_indices=s.slots,
                        o=s.o[l], aux_k=s.keys[l], aux_v=s.values[l], aux_g=s.gains[l], aux_k_per_khead=True,
                        size_order=s.order)
    ops.tree_commit(s.state, s.keys, s.values, s.gains, s.accept, n_nodes=s.n, cu_seqlens=s.cu, src_slots=s.slots,
                    k_head_div=hv // hk)


def run(s):
    from dforktree_amd import ops
    from dforktree_amd.plugin import fc1_block_inverse, fc1_plan
    kind = s.case["kind"]
    if kind == "invert":
        n = s.case["nodes"]
        x = s.a.clone()  # the inverse overwrites its matrix
        getattr(fc1_block_inverse, f"invert{n}")[(s.case["mats"],)](x, n)
        return x
    if kind == "plan":
        kv = s.case["prefix"] + s.case["nodes"]
        fc1_plan.pack_mask_into(s.wrapper, s.mask, s.case["nodes"], kv)
        return [s.wrapper._custom_mask_buf, s.wrapper._mask_indptr_buf]
    if kind == "mask":
        packed = {} if s.cu is None else dict(cu_seqlens=s.cu)
        ops.tree_mask_pack(s.anc_bits, s.prefix, batch=len(s.sizes), n_nodes=s.n, out=s.out, out_indptr=s.indptr,
                           **packed)
        return [s.out, s.indptr]
    if kind == "trees":
        packed = {} if s.cu is None else dict(cu_seqlens=s.cu)
        return ops.tree_struct(s.parent, 4, batch=len(s.sizes), n_nodes=s.n, **packed)
    s.graph.replay()
    if kind == "conv":
        return [s.y, s.window]
    if kind == "plugin":
        return dict(y=s.out[0], o=s.out[1], keys=s.keys, values=s.values, gains=s.gains, window=s.window,
                    snapshots=s.snapshots)
    if kind == "pipelined":
        return dict(o=s.o, gains=s.gains, state=s.state)
    return dict(o=s.o, keys=s.keys, values=s.values, gains=s.gains, state=s.state)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _mask_bytes(sizes, plens):
    return sum((n * (p + n) + 7) // 8 for n, p in zip(sizes, plens))


def work(case):
    """Every input read once, every output written once.  An accepted path's
    own rows (under 1% of a state tile) are left out."""
    kind = case["kind"]
    if kind == "invert":
        n, m = case["nodes"], case["mats"]
        # read, the copy that keeps the input, and the inverse; n^3 / 3 multiply-adds
        return dict(bytes=4 * 4 * m * n * n, flops=m * 2 * n ** 3 / 3)
    if kind == "plan":
        bits = case["nodes"] * (case["prefix"] + case["nodes"])
        return dict(bytes=bits + bits / 8, flops=0)
    sizes = _sizes(case)
    rows = sum(sizes)
    if kind == "mask":
        return dict(bytes=_mask_bytes(sizes, _prefixes(case)) + 8 * rows, flops=0)
    if kind == "trees":
        # parents; bits, depth, four gather columns, two links; the dense matrix
        return dict(bytes=rows * (4 + 8 + 8 + 32 + 16) + 4 * len(sizes) * max(sizes) ** 2, flops=0)
    L, chan = case["layers"], CHANNELS // case["tp"]
    hk, hv = _heads(case)
    conv = rows * chan * 2 * 5 + len(sizes) * chan * 3 * 2 + chan * 8
    conv_flops = rows * chan * 2 * 4
    if kind == "conv":
        return dict(bytes=L * conv, flops=L * conv_flops)
    gate = 2 if case.get("gates", "bf16") == "bf16" else 4
    tile = hv * D * D * 4
    verify = rows * (chan * 2 + 2 * hv * gate + 8 + hv * D * 2 + hv * 4) + len(sizes) * tile
    saves = rows * (hv * D * 4 + (hv if kind == "plugin" else hk) * D * 4)
    flops = sum(hv * (2 * 2 * n * D * D + 2 * n * n * D + 2 * n * n * D) for n in sizes)
    if kind == "plugin":
        return dict(bytes=L * (conv + verify + saves + 3 * tile), flops=L * (conv_flops + flops))
    if kind == "pipelined":
        return dict(bytes=L * (verify + len(sizes) * tile), flops=L * flops)
    return dict(bytes=L * (verify + saves + 2 * len(sizes) * tile), flops=L * flops)


def tolerance(case):
    """Whole numbers and copies are exact.  The inverse is a 32-bit sum of up
    to 64 terms, a few of them large.  The layers return bf16 rows beside
    32-bit states: half a bf16 unit in the last place is 2e-3 relative, and
    a value that rounds the other way is one unit (8e-3) off."""
    kind = case["kind"]
    if kind in ("plan", "mask", "trees"):
        return "exact"
    if kind == "invert":
        return dict(rel=1e-5, max=1e-3)
    return dict(rel=8e-3, max=0.1)


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _pad(x, sizes):
    """[L, rows, ..] -> [L, requests, most nodes, ..], zeros past a tree."""
    out = x.new_zeros(x.shape[0], len(sizes), max(sizes), *x.shape[2:])
    at = 0
    for r, n in enumerate(sizes):
        out[:, r, :n] = x[:, at:at + n]
        at += n
    return out


def _unpad(x, sizes):
    return torch.cat([x[:, r, :n] for r, n in enumerate(sizes)], 1)


def _anc64(parents, sizes):
    """Ancestor-or-self, [requests, most nodes, most nodes] of 0 / 1."""
    m = max(sizes)
    anc = torch.zeros(len(sizes), m, m, dtype=torch.float64)
    at = 0
    for r, n in enumerate(sizes):
        for i in range(n):
            p = parents[at + i]
            if i:
                anc[r, i] = anc[r, p]
            anc[r, i, i] = 1
        at += n
    return anc.to(_device())


def _decay64(a, A_log, dt_bias):
    """log decay of every row and head, [L, rows, hv]."""
    x = a.double() + dt_bias.double()[:, None]
    return -A_log.double().exp()[:, None] * torch.nn.functional.softplus(x, threshold=1e9)


def _solve64(A, W):
    """(I + A)^-1 W for strictly lower A, row by row."""
    X = W.clone()
    for i in range(1, A.shape[-1]):
        X[..., i, :] -= torch.matmul(A[..., i:i + 1, :i], X[..., :i, :])[..., 0, :]
    return X


def _decays64(G, anc, strict=False):
    """e^{G_i - G_j} where j is an ancestor (or self) of i, else 0; G [B, H, N], anc [B, N, N]."""
    on = anc[:, None] > 0
    if strict:
        on = on & ~torch.eye(anc.shape[-1], dtype=torch.bool, device=anc.device)
    d = (G[..., :, None] - G[..., None, :]).masked_fill(~on, -math.inf)
    return d.exp()


def _verify64(y, b, G, S, anc, hk, hv):
    """One layer: y [B, N, C], b [B, N, hv] (-inf past a tree), G [B, hv, N],
    S [B, hv, V, K]; returns o [B, hv, N, V], k, vn."""
    B, N, _ = y.shape

    def heads(x, h):
        x = x.double().reshape(B, N, h, D).transpose(1, 2)
        return x.repeat_interleave(hv // h, 1)
    q, k, v = heads(y[..., :hk * D], hk), heads(y[..., hk * D:2 * hk * D], hk), heads(y[..., 2 * hk * D:], hv)
    q = q * (q.square().sum(-1, keepdim=True) + 1e-6).rsqrt() * D ** -0.5
    k = k * (k.square().sum(-1, keepdim=True) + 1e-6).rsqrt()
    beta = torch.sigmoid(b.double()).transpose(1, 2)[..., None]
    e = G.exp()[..., None]
    kt, St = k.transpose(-1, -2).contiguous(), S.transpose(-1, -2).contiguous()
    A = beta * torch.matmul(k, kt) * _decays64(G, anc, strict=True)
    vn = _solve64(A, beta * (v - e * torch.matmul(k, St)))
    o = e * torch.matmul(q, St) + torch.matmul(torch.matmul(q, kt) * _decays64(G, anc), vn)
    return o, k, vn


def _commit64(S, k, vn, G, path, end=None):
    """S [hv, V, K] after the nodes of `path` (ending at `end`)."""
    u = path[-1] if end is None else end
    p = torch.tensor(path, device=S.device)
    w = (G[:, u, None] - G[:, p]).exp()[..., None]
    return G[:, u].exp()[:, None, None] * S + torch.matmul((w * vn[:, p]).transpose(-1, -2).contiguous(), k[:, p])


def _conv64(x, state, weight, parents):
    """x [B, N, C], state [B, C, 3], weight [C, 4], parents of every request's
    nodes; returns y [B, N, C] in bf16, as it is handed on, and the window."""
    B, N, C = x.shape
    xt = torch.cat((state.transpose(1, 2), x), 1)
    cols = torch.zeros(B, N, 4, dtype=torch.int64)
    for r in range(B):
        for i in range(N):
            c = i + 3
            for j in (3, 2, 1, 0):
                cols[r, i, j] = c
                c = c - 1 if c <= 3 else max(parents[r * N + c - 3], 0) + 3
    at = cols.to(x.device).reshape(B, N * 4, 1).expand(B, N * 4, C)
    taps = torch.gather(xt, 1, at).reshape(B, N, 4, C)
    acc = (taps.double() * weight.double().t()).sum(2)
    y = (acc * torch.sigmoid(acc)).to(x.dtype)
    return y, taps[:, :, 1:].transpose(2, 3)


def exact(case, seed):
    kind = case["kind"]
    s = _inputs(case, seed)
    if kind == "invert":
        eye = torch.eye(case["nodes"], device=_device(), dtype=torch.float64)
        return _solve64(s.a.double(), eye.expand(case["mats"], -1, -1).contiguous())
    if kind in ("plan", "mask", "trees"):
        return None  # whole numbers
    L = case["layers"]
    if kind == "conv":
        both = [_conv64(s.x[l], s.conv_state[l], s.weight[l], s.parents) for l in range(L)]
        return [torch.stack([y for y, _ in both]).double(), torch.stack([w for _, w in both]).double()]
    hk, hv = _heads(case)
    batch, slots = len(s.sizes), s.slots.tolist()
    anc = _anc64(s.parents, s.sizes)
    past = torch.zeros(1, sum(s.sizes), 1, device=_device())
    past = _pad(past + 1, s.sizes)[0] == 0  # [B, N, 1]: past the tree
    G = torch.matmul(anc, _pad(_decay64(s.a, s.A_log, s.dt_bias), s.sizes)).transpose(-1, -2)  # [L, B, hv, N]
    state = s.state.double()
    os, ks, vs = [], [], []
    ys, windows = [], []
    if kind == "pipelined":
        prev_anc = _anc64(s.prev_parents, s.sizes)
        prev_G = _pad(s.prev_gains.double().transpose(1, 2), s.sizes).transpose(-1, -2)
    snapshots = torch.zeros_like(s.snapshots, dtype=torch.float64) if kind == "plugin" else None
    for l in range(L):
        if kind == "plugin":
            y, w = _conv64(s.x[l], s.conv_state[l], s.weight[l], s.parents)
            ys.append(y.double())
            windows.append(w)
        else:
            y = _pad(s.y[l:l + 1], s.sizes)[0]
        b = _pad(s.b[l:l + 1].double(), s.sizes)[0].masked_fill(past, -math.inf)
        S = state[l, s.slots.long()]
        if kind == "pipelined":
            pb = _pad(s.prev_b[l:l + 1].double(), s.sizes)[0].masked_fill(past, -math.inf)
            _, k, vn = _verify64(_pad(s.prev_y[l:l + 1], s.sizes)[0], pb, prev_G[l], S, prev_anc, hk, hv)
            S = torch.stack([_commit64(S[r], k[r], vn[r], prev_G[l, r], s.paths[r]) for r in range(batch)])
            state[l, s.slots.long()] = S
        o, k, vn = _verify64(y, b, G[l], S, anc, hk, hv)
        os.append(_unpad(o.transpose(1, 2)[None], s.sizes)[0])
        if kind == "pipelined":
            continue
        kv = k if kind == "plugin" else k[:, ::hv // hk]
        ks.append(_unpad(kv.transpose(1, 2)[None], s.sizes)[0].transpose(0, 1))
        vs.append(_unpad(vn.transpose(1, 2)[None], s.sizes)[0].transpose(0, 1))
        if kind == "separate":
            for r in range(batch):
                state[l, slots[r]] = _commit64(S[r], k[r], vn[r], G[l, r], s.paths[r])
        else:
            path = s.paths[0]
            for end in {path[-1], s.track}:
                snapshots[l, 0, end] = _commit64(S[0], k[0], vn[0], G[l, 0], path[:path.index(end) + 1], end)
    gains = _unpad(G.transpose(-1, -2), s.sizes).transpose(1, 2)
    if kind == "plugin":
        return dict(y=ys, o=os, keys=torch.stack(ks), values=torch.stack(vs), gains=gains,
                    window=torch.stack(windows).double(), snapshots=snapshots)
    if kind == "pipelined":
        return dict(o=torch.stack(os), gains=gains, state=state)
    return dict(o=torch.stack(os), keys=torch.stack(ks), values=torch.stack(vs), gains=gains, state=state)
