"""What this framework is timed on: the calls that a user's program makes, over the sizes that they are made with.

Four kinds of case:

* ``gemm``    one local contraction on gathered slices (``gemm_os`` / ``gemm_ls`` / ``gemm_rs``): the forward, backward-data and
              backward-weight products of a mesh device, bf16 or fp32, plain or with the fused GELU + residual epilogue;
* ``device``  one mesh device's body as ``SPMD(mesh, algorithm).OS/LS/RS(K).device(i, j)`` runs it: the slices are gathered from
              the peers' shards, then multiplied;
* ``layer``   one training step of a ``ShardedFFLayer``: forward, backward-data and backward-weight on the whole mesh;
* ``reshard`` the layout steps alone: a shard cut into its block-cyclic slices, and a shard made from its peers' partial chunks.

Sizes are per device for ``gemm`` and ``reshard`` and of the whole mesh for ``device`` and ``layer``.  ``m`` and ``n`` are the rows and
columns of the whole product, ``k`` its whole contraction, ``S`` the slice count; which of them is cut into slices is the
dataflow's choice (OS: k, LS: n, RS: m).
"""
import math

import torch

from meshslice_amd import gemm_ls, gemm_os, gemm_rs
from meshslice_amd.ShardedLayers import ShardedFFLayer
from meshslice_amd.TensorParallel import SPMD
from meshslice_amd.mesh import Mesh, create_device_mesh
from meshslice_amd.slice_layout import pack_slices, unpack_chunks

BLOCK = 8                              # the block size of the block-cyclic slices, the builders' default
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
MAX_FLOPS = {"bf16": 1.23e12, "fp32": 1.0e11}     # of a drawn product
MAX_LAYER_FLOPS = 4.6e11               # of a drawn training step
MAX_RESHARD_ELEMENTS = 4096 * 12288    # of a drawn shard


def gemm(name, flow, m, n, k, S, dtype="bf16", out="bf16", gelu=False, residual=False):
    return {"name": name, "kind": "gemm", "flow": flow, "m": m, "n": n, "k": k, "S": S, "dtype": dtype, "out": out, "gelu": gelu, "residual": residual}


def listed():
    return [
        # the plumbing product of the benchmark's first configuration: fp32, four slices; launch and latency
        gemm("os_fp32_512", "os", 512, 512, 1024, 4, "fp32", "fp32"),
        # a feed-forward up-projection's forward pass on one device of a 4x4 mesh (the benchmark's main product)
        gemm("os_ff_up", "os", 4096, 12288, 12288, 4),
        # the down-projection's forward pass there: eight fp32 partial chunks for the reduce-scatter
        gemm("ls_ff_down", "ls", 4096, 12288, 12288, 8, out="fp32"),
        # the up-projection's weight gradient there: four fp32 partial chunks
        gemm("rs_ff_up_dw", "rs", 3072, 12288, 4096, 4, out="fp32"),
        # an attention output projection's backward-data pass on one device of an 8x8 mesh: few output tiles, long contraction
        gemm("os_8x8_dx", "os", 2048, 1536, 12288, 4),
        # the same layer's forward pass there: short contraction, bf16 chunks
        gemm("ls_8x8_fwd", "ls", 2048, 12288, 1536, 8),
        # a layer with GELU and residual on the last, ragged batch of a data set: no extent a multiple of a tile
        gemm("os_ragged_gelu", "os", 1499, 4104, 3096, 3, gelu=True, residual=True),
        # a weight gradient in full precision with ragged extents
        gemm("rs_fp32_ragged", "rs", 1040, 2056, 1023, 4, "fp32", "fp32"),
        # one device's forward body on a 2x4 mesh, gathers included
        {"name": "device_ls_2x4", "kind": "device", "algorithm": "meshflow", "flow": "ls", "rows": 2, "cols": 4, "m": 4096, "n": 4096, "k": 8192, "S": 8, "dtype": "bf16"},
        # a training step of a layer of the walkthrough's size (512 tokens, 256 in, 1024 out) on its 4x2 mesh: many small calls
        {"name": "layer_small_4x2", "kind": "layer", "algorithm": "meshflow", "flow": "os", "rows": 4, "cols": 2, "tokens": 512, "inner": 256, "outer": 1024, "S": 4},
        # a training step of an up-projection on a 2x4 mesh
        {"name": "layer_2x4", "kind": "layer", "algorithm": "meshflow", "flow": "os", "rows": 2, "cols": 4, "tokens": 2048, "inner": 3072, "outer": 12288, "S": 8},
        # a large shard sliced for its all-gathers, and a shard made from the fp32 chunks of four peers
        {"name": "reshard_4096", "kind": "reshard", "rows": 4096, "cols": 12288, "S": 8, "axis": 1, "peers": 4, "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _up(v, q):
    """v as the nearest multiple of q, at least q"""
    return max(q, int(round(v / q)) * q)


def _draw_gemm(rng):
    dtype = "bf16" if rng.random() < 0.75 else "fp32"
    flow = rng.choice(["os", "ls", "rs"])
    S = rng.choice([1, 2, 3, 4, 6, 8, 16])
    m, n, k = _log(rng, 64, 8192), _log(rng, 256, 12288), _log(rng, 256, 12288)
    while 2 * m * n * k > MAX_FLOPS[dtype]:
        m, n, k = m * 0.9, n * 0.9, k * 0.9
    fused = flow == "os" and dtype == "bf16" and rng.random() < 0.25
    # contiguous extents are whole blocks, per slice where they are sliced; the others take any length
    m = _up(m, S * BLOCK) if flow == "rs" else int(m)
    n = _up(n, S * BLOCK) if flow == "ls" else _up(n, BLOCK)
    k = _up(k, S * BLOCK) if flow == "os" else int(k) if flow == "rs" else _up(k, BLOCK)
    out = "bf16" if dtype == "bf16" and (flow == "os" or rng.random() < 0.5) else "fp32"
    case = gemm("", flow, m, n, k, S, dtype, out, gelu=fused, residual=fused and rng.random() < 0.5)
    del case["name"]
    return case


def _mesh_case(rng):
    rows, cols = rng.choice([(1, 2), (2, 2), (2, 4), (4, 2)])
    return rng.choice(["meshflow", "meshflow", "collective", "wang"]), rng.choice(["os", "ls", "rs"]), rows, cols, rng.choice([2, 4, 8])


def _draw_device(rng):
    algorithm, flow, rows, cols, S = _mesh_case(rng)
    q = rows * cols * S * BLOCK            # whole slices of whole shards on either mesh axis
    m, n, k = _log(rng, 256, 8192), _log(rng, 256, 12288), _log(rng, 256, 12288)
    m = _up(m, q) if flow == "rs" else _up(m, rows)
    n = _up(n, q) if flow == "ls" else _up(n, cols * BLOCK)
    k = _up(k, q) if flow == "os" else _up(k, cols * BLOCK) if flow == "ls" else _up(k, rows)
    return {"kind": "device", "algorithm": algorithm, "flow": flow, "rows": rows, "cols": cols, "m": m, "n": n, "k": k, "S": S,
            "dtype": "bf16" if rng.random() < 0.75 else "fp32"}


def _draw_layer(rng):
    algorithm, flow, rows, cols, S = _mesh_case(rng)
    t, i, o = _log(rng, 256, 4096), _log(rng, 256, 8192), _log(rng, 256, 12288)
    while 6 * t * i * o > MAX_LAYER_FLOPS:
        t, i, o = t * 0.9, i * 0.9, o * 0.9
    q, edge = rows * cols * S * BLOCK, rows * cols * BLOCK
    sliced = {"os": (edge, q, edge), "ls": (edge, edge, q), "rs": (q, edge, edge)}[flow]
    t, i, o = (_up(v, e) for v, e in zip((t, i, o), sliced))
    return {"kind": "layer", "algorithm": algorithm, "flow": flow, "rows": rows, "cols": cols, "tokens": t, "inner": i, "outer": o, "S": S}


def _draw_reshard(rng):
    S, axis, peers = rng.choice([2, 3, 4, 8]), rng.choice([0, 1]), rng.choice([1, 2, 4])
    rows, cols = _log(rng, 64, 8192), _log(rng, 128, 12288)
    while rows * cols > MAX_RESHARD_ELEMENTS:
        rows, cols = rows * 0.9, cols * 0.9
    rows, cols = (_up(rows, S * BLOCK * peers), _up(cols, BLOCK)) if axis == 0 else (int(rows), _up(cols, S * BLOCK * peers))
    return {"kind": "reshard", "rows": rows, "cols": cols, "S": S, "axis": axis, "peers": peers, "dtype": rng.choice(["bf16", "bf16", "fp32"])}


def draw(rng):
    pick = rng.random()
    return (_draw_gemm if pick < 0.5 else _draw_device if pick < 0.7 else _draw_layer if pick < 0.85 else _draw_reshard)(rng)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(rows, cols, scale=1.0, dtype=torch.bfloat16):
        return torch.randn(rows, cols, generator=gen, device="cuda").mul_(scale).to(dtype)

    st = dict(case)
    if case["kind"] == "gemm":
        flow, m, n, k, S, dt = (case[x] for x in ("flow", "m", "n", "k", "S", "dtype"))
        dt = DTYPES[dt]
        if flow == "os":
            st["a"] = [normal(m, k // S, 1.0, dt) for _ in range(S)]
            st["b"] = [normal(k // S, n, 0.02, dt) for _ in range(S)]
            st["res"] = normal(m, n, 1.0, DTYPES[case["out"]]) if case["residual"] else None
        elif flow == "ls":
            st["a"], st["b"] = normal(m, k, 1.0, dt), [normal(n // S, k, 0.02, dt) for _ in range(S)]
        else:
            st["a"], st["b"] = [normal(k, m // S, 1.0, dt) for _ in range(S)], normal(k, n, 0.02, dt)
    elif case["kind"] in ("device", "layer"):
        mesh = Mesh(create_device_mesh((case["rows"], case["cols"])), ("row", "col"))
        flow = case["flow"]
        if case["kind"] == "device":
            dt = DTYPES[case["dtype"]]
            m, n, k = case["m"], case["n"], case["k"]
            builder = SPMD(mesh, case["algorithm"], BLOCK)
            build = {"os": builder.OS, "ls": builder.LS, "rs": builder.RS}[flow]
            st["body"] = build(case["S"]).device(case["rows"] - 1, case["cols"] - 1)
            st["x"] = normal(k, m, 1.0, dt) if flow == "rs" else normal(m, k, 1.0, dt)
            st["w"] = normal(n, k, 0.02, dt) if flow == "ls" else normal(k, n, 0.02, dt)
        else:
            t, i, o = case["tokens"], case["inner"], case["outer"]
            layer = ShardedFFLayer(mesh, case["algorithm"], flow, case["S"], i, o, BLOCK, seed=seed)
            layer.weight.mul_(0.02).requires_grad_()
            st["layer"] = layer
            st["x"] = (normal(i, t) if flow == "rs" else normal(t, i)).requires_grad_()
            st["dy"] = normal(t, o, 0.01)
    else:
        rows, cols, S, axis, peers = (case[x] for x in ("rows", "cols", "S", "axis", "peers"))
        st["x"] = normal(rows, cols, 1.0, DTYPES[case["dtype"]])
        shape = (rows, cols // S) if axis == 1 else (rows // S, cols)
        st["chunks"] = [[normal(*shape, 1.0, torch.float32) for _ in range(S)] for _ in range(peers)]
    return st


def run(state):
    kind = state["kind"]
    if kind == "gemm":
        if state["flow"] == "os":
            return gemm_os(state["a"], state["b"], out_dtype=DTYPES[state["out"]], activation="gelu" if state["gelu"] else None, residual=state["res"])
        return (gemm_ls if state["flow"] == "ls" else gemm_rs)(state["a"], state["b"], out_dtype=DTYPES[state["out"]])
    if kind == "device":
        return state["body"](state["x"], state["w"])
    if kind == "layer":
        y = state["layer"].forward(state["x"])
        dx, dw = torch.autograd.grad(y, (state["x"], state["layer"].weight), state["dy"])
        return y.detach(), dx, dw
    slices = pack_slices(state["x"], state["S"], BLOCK, state["axis"])
    shard = unpack_chunks(state["chunks"], BLOCK, state["axis"], window=state["peers"] - 1, parts=state["peers"], out_dtype=DTYPES[state["dtype"]])
    return slices, shard


def work(case):
    es = 2 if case.get("dtype", "bf16") == "bf16" else 4
    if case["kind"] == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        eo = 2 if case["out"] == "bf16" else 4
        return {"bytes": es * (m * k + k * n) + eo * m * n * (2 if case["residual"] else 1), "flops": 2 * m * n * k}
    if case["kind"] == "device":
        m, n, k, R, C = (case[x] for x in ("m", "n", "k", "rows", "cols"))
        # the operands that the device multiplies (its own shard, and what it is sent), and its output block or fp32 chunks
        m, n, k = {"os": (m // R, n // C, k), "ls": (m // R, n, k // C), "rs": (m, n // C, k // R)}[case["flow"]]
        return {"bytes": es * (m * k + k * n) + (es if case["flow"] == "os" else 4) * m * n, "flops": 2 * m * n * k}
    if case["kind"] == "layer":
        t, i, o = case["tokens"], case["inner"], case["outer"]
        # x, w and dy in; y, dx and dw out
        return {"bytes": 4 * (t * i + i * o + t * o), "flops": 6 * t * i * o}
    elements = case["rows"] * case["cols"]
    # the shard in and out, and of each peer's chunks the window that this device keeps
    return {"bytes": elements * (2 * es + 4) + elements // case["peers"] * es, "flops": 0}


def tolerance(case):
    if case["kind"] == "reshard":
        return "exact"             # moved bytes, and fp32 sums in peer order
    # against float64: at most 7e-7 for fp32 results (contractions up to 12288), 1.7e-3 for ones rounded to bf16; four times that
    fp32_out = case["kind"] == "gemm" and case["out"] == "fp32" or case["kind"] == "device" and (case["dtype"] == "fp32" or (case["flow"] != "os"))
    return {"rel": 3e-6 if fp32_out else 7e-3}


def _cut(t, S, axis):
    """The S block-cyclic slices of a matrix: slice s holds its blocks b with b % S == s"""
    shape = t.shape
    if axis == 1:
        return [s.reshape(shape[0], -1) for s in t.reshape(shape[0], -1, S, BLOCK).unbind(2)]
    return [s.reshape(-1, shape[1]) for s in t.reshape(-1, S, BLOCK, shape[1]).unbind(1)]


def _exact_device(case, x, w):
    """The last device's output block, or its partial chunks, in the order that its algorithm hands them out"""
    flow, R, C, S = (case[v] for v in ("flow", "rows", "cols", "S"))
    m, n, k = case["m"], case["n"], case["k"]
    i, j = R - 1, C - 1
    x, w = x.double(), w.double()
    if flow == "os":
        return x[i * (m // R):] @ w[:, j * (n // C):]
    if flow == "ls":
        own, axis, peers = x[i * (m // R):, j * (k // C):], 0, w[:, j * (k // C):].chunk(R, 0)
    else:
        own, axis, peers = w[i * (k // R):, j * (n // C):], 1, x[i * (k // R):].chunk(C, 1)
    parts = [_cut(p, S, axis) for p in peers] if case["algorithm"] == "meshflow" else [[p] for p in peers]
    gathered = [torch.cat([p[s] for p in parts], axis) for s in range(len(parts[0]))]
    return [own @ g.t() if flow == "ls" else g.t() @ own for g in gathered]


def exact(case, seed):
    st = prepare(case, seed)
    if case["kind"] == "gemm":
        if case["flow"] == "os":
            c = sum(a.double() @ b.double() for a, b in zip(st["a"], st["b"]))
            if case["gelu"]:
                c = torch.nn.functional.gelu(c, approximate="tanh")
            return c if st["res"] is None else c + st["res"].double()
        if case["flow"] == "ls":
            a = st["a"].double()
            return [a @ w.double().t() for w in st["b"]]
        b = st["b"].double()
        return [x.double().t() @ b for x in st["a"]]
    if case["kind"] == "device":
        return _exact_device(case, st["x"], st["w"])
    if case["kind"] == "layer":
        x, w, dy = st["x"].detach().double(), st["layer"].weight.detach().double(), st["dy"].double()
        if case["flow"] == "os":
            return x @ w, dy @ w.t(), x.t() @ dy
        if case["flow"] == "ls":
            return x @ w.t(), dy @ w, dy.t() @ x
        return x.t() @ w, w @ dy.t(), x @ dy
    S, axis, peers = (case[v] for v in ("S", "axis", "peers"))
    mine = [sum(c[s].double().chunk(peers, axis)[peers - 1] for c in st["chunks"]) for s in range(S)]
    if axis == 1:
        shard = torch.stack([c.reshape(c.shape[0], -1, BLOCK) for c in mine], 2).reshape(case["rows"], -1)
    else:
        shard = torch.stack([c.reshape(-1, BLOCK, c.shape[1]) for c in mine], 1).reshape(-1, case["cols"])
    return [s.double() for s in _cut(st["x"], S, axis)], shard
