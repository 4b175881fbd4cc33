"""Small product functions for the GPU tests: C[m, n] = Σ_k f(A)·g(B) + bias[n] over the operand
layouts, at sizes where a tile, a chunk of k or a row's alignment ends. build() compiles them ahead."""
from anvil import ir
from anvil.hip_function import Lowered

# (layout, M, N, K, operand function): layout "NT" = x[m, k]·w[n, k], "NN" = x[m, k]·w[k, n],
# "TN" = x[k, m]·w[k, n], "GT" = x[pick[m], k]·w[n, k]
RAGGED = [
    ("NT", 95, 70, 17, ""), ("NT", 33, 64, 71, "exp"), ("NN", 64, 45, 24, ""), ("NN", 197, 513, 1001, ""),
    ("NN", 65, 97, 262, "exp"), ("TN", 77, 50, 333, ""), ("TN", 129, 131, 8197, ""), ("NT", 333, 257, 701, "relu"),
    ("GT", 90, 100, 75, ""), ("NN", 1040, 1031, 67, ""), ("NN", 1500, 1490, 33, "exp"), ("NT", 2111, 1999, 65, "relu"),
    ("TT", 1470, 1481, 64, ""), ("GT", 1600, 1500, 41, ""), ("NN", 4090, 2950, 37, ""), ("TN", 600, 999, 701, "exp"),
    ("TN", 128, 129, 527, ""), ("NN", 1480, 1470, 24, "relu"), ("NT", 2111, 999, 531, ""), ("NN", 72, 64, 16, "exp"),
    ("NN", 4090, 2950, 69, "exp"), ("NT", 2950, 4090, 96, ""), ("TN", 1030, 520, 2065, ""), ("TN", 1024, 520, 2064, "relu"),
    ("TN", 1030, 520, 528, ""),
]


# products with infinities and nans: shared tiles of 64 x 64 (K below 64 included) and 128 x 128, the
# split K split, and the float32 K split
SPECIAL = [("NT", 1500, 1500, 70), ("NN", 4096, 2944, 40), ("NN", 4096, 2944, 72), ("TN", 1030, 520, 777), ("NT", 64, 96, 64)]

# K that leaves a short last chunk: one and two tiles to a wavefront, one dimension below a tile, the
# split K split
TAILS = [("NT", 1409, 308, 2114), ("NN", 1000, 999, 1001), ("TN", 268, 60, 2489), ("TN", 129, 140, 777), ("TN", 1000, 600, 1323)]

# shared 64 x 64 tiles with a short K
SHORT = [("NT", 2048, 1024, 64), ("NN", 1531, 2003, 72), ("NT", 2112, 1100, 65)]

# one size of each bf16 schedule, for operands of any magnitude
SMALL = [("NT", 1500, 1500, 70), ("NN", 4096, 2944, 72), ("TN", 1030, 520, 777)]


def product(layout, M, N, K, op=""):
    """The lowered function (inputs x, w, bias[, pick]) of one product."""
    rows = M + 9 if layout[0] == "G" else M
    x = ir.Buffer("input0", (K, M) if layout[0] == "T" else (rows, K), "f32", "input")
    w = ir.Buffer("input1", (N, K) if layout[1] == "T" else (K, N), "f32", "input")
    bias = ir.Buffer("input2", (N,), "f32", "input")
    y = ir.Buffer("output0", (M, N), "f32", "output")
    m, n, k = ir.Var("m", M), ir.Var("n", N), ir.Var("k", K)
    bufs = [x, w, bias, y]
    row = m
    if layout[0] == "G":
        pick = ir.Buffer("input3", (M,), "i32", "input")
        bufs.append(pick)
        for i, obj in enumerate(bufs + [m, n, k], 1):    # a gather hashes by its ids
            obj.id = i
        row = ir.Gather(ir.Load(pick, ir.Affine(0, {m: 1})), rows)
    a = ir.Load(x, ir.Affine(0, {m: 1, k: M} if layout[0] == "T" else {row: K, k: 1}))
    b = ir.Load(w, ir.Affine(0, {n: K, k: 1} if layout[1] == "T" else {n: 1, k: N}))
    if op == "relu":
        a = ir.Binary("max", a, ir.Const(0.0))
    elif op:
        a, b = ir.Unary(op, a), ir.Unary(op, b)
    kern = ir.Kernel([m, n], [ir.Store(y, ir.Affine(0, {m: N, n: 1}),
                                       ir.Binary("add", ir.Acc(), ir.Load(bias, ir.Affine(0, {n: 1}))))],
                     red=ir.Reduction([k], "sum", ir.Binary("mul", a, b)), name="y", label="y")
    return lowered([ir.KernelStmt(kern)], bufs, name="product")


def lowered(stmts, bufs, name):
    """A Lowered with ids in program order (the same source, so the same library, in every process)."""
    seen = {}
    for s in stmts:
        for v in s.kernel.all_vars() + [s.kernel]:
            seen.setdefault(id(v), v)
    for i, obj in enumerate(bufs + list(seen.values()), 1):
        obj.id = i
    ins = sorted((b for b in bufs if b.kind == "input"), key=lambda b: b.name)
    outs = sorted((b for b in bufs if b.kind == "output"), key=lambda b: b.name)
    return Lowered(ir.Program(ir.Block(list(stmts)), bufs), ins, outs, tuple_result=len(outs) > 1, name=name)


def convolution(n, c, side, o, win=3):
    """A win x win convolution's forward and weight gradient as the front end lowers them (the patches
    copy, then products over it): K = win^2 c read through a table, and K over images and positions."""
    full, P, K = side + win - 1, side * side, win * win * c
    x = ir.Buffer("input0", (n, c, full, full), "f32", "input")
    w = ir.Buffer("input1", (o, c, win, win), "f32", "input")
    dy = ir.Buffer("input2", (n, o, side, side), "f32", "input")
    y = ir.Buffer("output0", (n, o, side, side), "f32", "output")
    dw = ir.Buffer("output1", (o, c, win, win), "f32", "output")
    p = ir.Buffer("patches", (n, side, side, c, win, win), "f32", "temp")
    vs = [ir.Var(a, e) for a, e in zip("nijcuv", p.shape)]
    nn, i, j, ch, u, v = vs
    src = ir.Affine(0, {nn: c * full * full, ch: full * full, i: full, u: full, j: 1, v: 1})
    copy = ir.Kernel(vs, [ir.Store(p, ir.Affine(0, dict(zip(vs, p.strides))), ir.Load(x, src))], name="p", label="p")

    def load(buf, **terms):
        return ir.Load(buf, ir.Affine(0, {names[k]: s for k, s in terms.items()}))
    names = {a: ir.Var(a, e) for a, e in (("n", n), ("o", o), ("t", P), ("k", K))}
    fwd = ir.Kernel([names[a] for a in "not"],
                    [ir.Store(y, ir.Affine(0, {names["n"]: o * P, names["o"]: P, names["t"]: 1}), ir.Acc())],
                    red=ir.Reduction([names["k"]], "sum", ir.Binary("mul", load(p, n=P * K, t=K, k=1), load(w, o=K, k=1))),
                    name="y", label="y")
    names = {a: ir.Var(a, e) for a, e in (("n", n), ("o", o), ("t", P), ("k", K))}
    grad = ir.Kernel([names["o"], names["k"]],
                     [ir.Store(dw, ir.Affine(0, {names["o"]: K, names["k"]: 1}), ir.Acc())],
                     red=ir.Reduction([names["n"], names["t"]], "sum",
                                      ir.Binary("mul", load(dy, n=o * P, o=P, t=1), load(p, n=P * K, t=K, k=1))),
                     name="dw", label="dw")
    return lowered([ir.KernelStmt(k) for k in (copy, fwd, grad)], [x, w, dy, y, dw, p], name="convolution")


def attention(B, Lq, Lk, D):
    """softmax(q kᵀ / sqrt(D)) v as the front end lowers it (six kernels)."""
    def kern(domain, buf, off, value, red=None):
        return ir.KernelStmt(ir.Kernel(domain, [ir.Store(buf, ir.Affine(0, off), value)], red=red, name=buf.name, label=buf.name))

    def load(buf, **off):
        return ir.Load(buf, ir.Affine(0, {v[k]: c for k, c in off.items()}))
    q, k, w = (ir.Buffer(f"input{i}", (B, n, D), "f32", "input") for i, n in enumerate((Lq, Lk, Lk)))
    o = ir.Buffer("output0", (B, Lq, D), "f32", "output")
    s, e, p = (ir.Buffer(n, (B, Lq, Lk), "f32", "temp") for n in "sep")
    m, t = (ir.Buffer(n, (B, Lq), "f32", "temp") for n in "mt")
    var = lambda **ext: {a: ir.Var(a, n) for a, n in ext.items()}                          # noqa: E731
    R, mul = B * Lq, lambda a, b: ir.Binary("mul", a, b)                                   # noqa: E731
    stmts = []
    v = var(n=B, i=Lq, j=Lk, c=D)
    stmts.append(kern([v["n"], v["i"], v["j"]], s, {v["n"]: Lq * Lk, v["i"]: Lk, v["j"]: 1}, ir.Acc(),
                      ir.Reduction([v["c"]], "sum", mul(ir.Const(D ** -0.5), mul(load(q, n=Lq * D, i=D, c=1), load(k, n=Lk * D, j=D, c=1))))))
    v = var(r=R, j=Lk)
    stmts.append(kern([v["r"]], m, {v["r"]: 1}, ir.Unary("detach", ir.Acc()), ir.Reduction([v["j"]], "max", load(s, r=Lk, j=1))))
    v = var(r=R, j=Lk)
    stmts.append(kern([v["r"], v["j"]], e, {v["r"]: Lk, v["j"]: 1},
                      ir.Unary("exp", ir.Binary("sub", load(s, r=Lk, j=1), load(m, r=1)))))
    v = var(r=R, j=Lk)
    stmts.append(kern([v["r"]], t, {v["r"]: 1}, ir.Acc(), ir.Reduction([v["j"]], "sum", load(e, r=Lk, j=1))))
    v = var(r=R, j=Lk)
    stmts.append(kern([v["r"], v["j"]], p, {v["r"]: Lk, v["j"]: 1}, ir.Binary("div", load(e, r=Lk, j=1), load(t, r=1))))
    v = var(n=B, i=Lq, l=Lk, c=D)
    stmts.append(kern([v["n"], v["i"], v["c"]], o, {v["n"]: Lq * D, v["i"]: D, v["c"]: 1}, ir.Acc(),
                      ir.Reduction([v["l"]], "sum", mul(load(p, n=Lq * Lk, i=Lk, l=1), load(w, n=Lk * D, l=D, c=1)))))
    return lowered(stmts, [q, k, w, o, s, m, e, t, p], name="attention")


# (heads, queries, keys, width): ragged tails of both, every width class, keys for one wavefront only,
# and (many keys, few queries) eight wavefronts
ATTENTIONS = [(2, 40, 65, 32), (3, 33, 70, 16), (1, 77, 31, 48), (2, 64, 128, 64), (1, 100, 257, 80), (8, 61, 300, 96),
              (45, 45, 130, 112), (36, 96, 640, 128), (4, 513, 1025, 64), (1, 33, 1030, 64), (72, 33, 1030, 128),
              (2, 513, 1025, 96), (5, 1100, 600, 48)]
# two key tiles, the second nearly empty, over many heads
TWO_TILES = [(60, 36, 36, 48)]
# (of ATTENTIONS) for operands of any magnitude
MAGNITUDES = [(2, 40, 65, 32), (2, 64, 128, 64), (1, 100, 257, 80), (36, 96, 640, 128)]
# few queries for their keys and width: products and rows in launches of their own
SEPARATE = [(1, 96, 640, 128), (1, 33, 1030, 128), (1, 513, 1001, 80)]

CONVOLUTIONS = [(5, 5, 10, 40), (3, 21, 18, 37), (7, 8, 6, 33)]
# other windows than 3 x 3
WINDOWS = [(64, 2, 20, 32, 2), (9, 6, 10, 35, 3)]


def programs():
    """Every lowered function the GPU tests call, for the build."""
    for args in RAGGED + SPECIAL + TAILS + SHORT + SMALL:
        yield product(*args)
    for args in ATTENTIONS + SEPARATE + TWO_TILES:
        yield attention(*args)
    for args in CONVOLUTIONS + WINDOWS:
        yield convolution(*args)
