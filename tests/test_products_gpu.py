"""Products at the edges of the matrix-core schedules: every K tail, row length and tile remainder
against float64, within the forward error bound of a K-term float32 sum in any order (K + 8 rounding
errors of 2^-24 of Σ|a b|; the operand functions' own errors, a few units in the last place, are in
the 8)."""
import re

import numpy as np
import pytest

import product_programs as PP

from anvil.backend import hip
from anvil.hip_function import Compiled

U = 2.0 ** -24


def _run(low, args):
    return Compiled(low.name, low).call(args)


def _operand(layout, M, N, K, op, seed=4):
    rng = np.random.default_rng(seed)
    rows = M + 9 if layout[0] == "G" else M
    x = rng.standard_normal((K, M) if layout[0] == "T" else (rows, K)).astype(np.float32)
    w = rng.standard_normal((N, K) if layout[1] == "T" else (K, N)).astype(np.float32)
    b = rng.standard_normal(N).astype(np.float32)
    args = [x, w, b]
    a64, w64 = x.astype(np.float64), w.astype(np.float64)
    if layout[0] == "G":
        pick = rng.permutation(rows)[:M].astype(np.int32)
        args.append(pick)
        a64 = a64[pick]
    a64 = a64.T if layout[0] == "T" else a64
    w64 = w64.T if layout[1] == "T" else w64
    if op == "relu":
        a64 = np.maximum(a64, 0)
    elif op:
        a64, w64 = np.exp(a64), np.exp(w64)
    return args, a64, w64, b.astype(np.float64)


@pytest.mark.gpu
@pytest.mark.parametrize("layout,M,N,K,op", PP.RAGGED)
def test_gpu_ragged_product(layout, M, N, K, op):
    print(f"gpu product {layout} {M}x{N}x{K} {op}", flush=True)
    args, a, w, b = _operand(layout, M, N, K, op)
    got = _run(PP.product(layout, M, N, K, op), args)
    want = a @ w + b
    bound = (K + 8) * U * (np.abs(a) @ np.abs(w) + np.abs(b))
    assert np.all(np.abs(got - want) <= bound)
    assert np.linalg.norm(got - want) <= _usual(K) * np.linalg.norm(want)


def _usual(K):
    """The 2-norm error, over the result's, of a float32 sum of K products: its roundings are independent,
    the k-th of a partial sum of k terms, together at most 2^-24 sqrt(K / 2); no sum runs over more than
    512 k before it is added to another. Two more for the last addition and the operands' functions. (Two
    bf16 to an operand instead of three: 2.4e-6 or more at every size without exp, 2.2 times this bound.)"""
    return U * (2 + (min(K, 512) / 2) ** 0.5)


@pytest.mark.gpu
@pytest.mark.parametrize("layout,M,N,K", PP.TAILS)
def test_gpu_short_last_chunk_keeps_sixteen_runs(layout, M, N, K):
    """The 2-norm error is that of sixteen sums of K / 16 products added up: a rounding for each product,
    0.41 x 2^-24 of a partial sum whose square grows evenly to the sum's (so half of them count), then
    sixteen additions likewise: 0.41 sqrt(K / 32 + 8), a tenth allowed, and half a unit for the result and
    the bias. (Four runs, 0.41 sqrt(K / 8 + 2), are past the bound at each of these sizes.)"""
    print(f"gpu product {layout} {M}x{N}x{K}", flush=True)
    args, a, w, b = _operand(layout, M, N, K, "")
    got, want = _run(PP.product(layout, M, N, K), args), a @ w + b
    assert np.linalg.norm(got - want) <= U * (0.5 + 0.45 * (K / 32 + 8) ** 0.5) * np.linalg.norm(want)


@pytest.mark.gpu
@pytest.mark.parametrize("layout,M,N,K", PP.SHORT)
def test_gpu_short_sums_on_bf16_keep_the_float32_error(layout, M, N, K):
    """The 2-norm error is at most that of the float32 K split over four wavefronts: runs of K / 4
    roundings, then four additions (as above), and 0.29 units for the bias's."""
    print(f"gpu product {layout} {M}x{N}x{K}", flush=True)
    args, a, w, b = _operand(layout, M, N, K, "")
    got, want = _run(PP.product(layout, M, N, K), args), a @ w + b
    assert np.linalg.norm(got - want) <= U * (0.29 + 0.41 * (K / 8 + 2) ** 0.5) * np.linalg.norm(want)


@pytest.mark.gpu
@pytest.mark.parametrize("ea,eb", [(-118, 90), (90, -118), (-60, -60), (0, -124)])
@pytest.mark.parametrize("layout,M,N,K", PP.SMALL)
def test_gpu_small_operands_keep_their_bits(layout, M, N, K, ea, eb):
    """Operands around 2^ea and 2^eb: the bounds are those of operands around 1, since every bit of a float32
    is in its bf16 parts (a part below the smallest bf16 would cost 2^-16 at 2^-118)."""
    print(f"gpu product {layout} {M}x{N}x{K} at 2^{ea}, 2^{eb}", flush=True)
    args, a, w, b = _operand(layout, M, N, K, "")
    args[0], args[1], args[2] = args[0] * np.float32(2.0 ** ea), args[1] * np.float32(2.0 ** eb), args[2] * np.float32(2.0 ** (ea + eb))
    a, w = args[0].astype(np.float64), args[1].astype(np.float64)      # (as rounded: some are subnormal)
    a, w = a.T if layout[0] == "T" else a, w.T if layout[1] == "T" else w
    got, want = _run(PP.product(layout, M, N, K), args), a @ w + args[2].astype(np.float64)
    print("error", np.linalg.norm(got - want) / np.linalg.norm(want))
    assert np.all(np.abs(got - want) <= (K + 8) * U * (np.abs(a) @ np.abs(w) + np.abs(args[2])))
    assert np.linalg.norm(got - want) <= _usual(K) * np.linalg.norm(want)


def test_convolution_with_eight_terms_reads_its_window():
    """K = 8 (two channels, a 2 x 2 window) goes through a table like any multiple of 8, short as it is: the
    window is read in place of a copy of it, for the sums and their weight gradient."""
    src = hip.generate(PP.convolution(64, 2, 20, 32, 2).prog, library=True)
    assert "// map: p " not in src and "32x25600x8 · outer" in src


@pytest.mark.parametrize("n,c,side,o,copied", [(128, 6, 26, 32, True), (128, 22, 10, 64, True), (128, 6, 28, 32, False),
                                               (128, 8, 26, 32, False), (128, 4, 26, 32, False), (128, 7, 13, 33, False)])
def test_convolution_keeps_its_copy_where_the_weight_gradient_needs_it(n, c, side, o, copied):
    """Rows of positions that are no multiple of 4 long leave the weight gradient without the copy no four
    adjacent k; with 13 x 13 positions the copy does not give it any either."""
    src = hip.generate(PP.convolution(n, c, side, o).prog, library=True)
    assert ("// map: p " in src) == copied


@pytest.mark.gpu
@pytest.mark.parametrize("n,c,side,o,win", [a + (3,) for a in PP.CONVOLUTIONS] + PP.WINDOWS)
def test_gpu_ragged_convolution(n, c, side, o, win):
    """Forward and weight gradient; with 7 images of 6 x 6 positions, K = 252 is no multiple of 8."""
    print(f"gpu convolution {n} x {c} x {side} x {side} -> {o}, window {win}", flush=True)
    rng, full = np.random.default_rng(8), side + win - 1
    x = rng.standard_normal((n, c, full, full)).astype(np.float32)
    w = rng.standard_normal((o, c, win, win)).astype(np.float32)
    dy = rng.standard_normal((n, o, side, side)).astype(np.float32)
    y, dw = Compiled("convolution", PP.convolution(n, c, side, o, win)).call([x, w, dy])
    win = np.lib.stride_tricks.sliding_window_view(x.astype(np.float64), (win, win), axis=(2, 3))
    for got, spec, other, terms in ((y, "ncijuv,ocuv->noij", w, w[0].size), (dw, "ncijuv,noij->ocuv", dy, n * side * side)):
        want = np.einsum(spec, win, other.astype(np.float64))
        bound = (terms + 8) * U * np.einsum(spec, np.abs(win), np.abs(other.astype(np.float64)))
        assert got.shape == want.shape and np.all(np.abs(got - want) <= bound)


def _kernel(args):
    src = hip.generate(PP.product(*args).prog, library=True)
    kern = src[src.index("// gemm: "):]
    return kern[:kern.index("\n}\n")]


def test_ragged_products_take_the_pipelined_split():
    """No product of these sizes is left to per-element loads: each is a matrix-core schedule, with
    the guarded last chunk exactly where K is no multiple of the chunk."""
    for args in PP.RAGGED:
        kern, K = _kernel(args), args[3]
        assert "ANVIL_LD_ANY" not in kern, args
        (name, params), = re.findall(r"(anvil_mm_tile_\w+)<(.*)>\(\w", kern)
        chunk = {"anvil_mm_tile_kpipe": 8, "anvil_mm_tile_split": 16, "anvil_mm_tile_shared": 32}[name]
        assert params.endswith("true") == (K % chunk != 0), (args, params)


def test_ragged_and_special_products_take_every_split_template():
    """Between them: each shared tile and the split K split with and without a short last slice, the
    latter also with a run long enough (32 chunks) for its second accumulators; and the shared tiles and
    the split K split among the products with infinities."""
    seen, special = set(), set()
    for args in PP.RAGGED + [a + ("",) for a in PP.SPECIAL]:
        (name, params), = re.findall(r"anvil_mm_tile_(\w+)<(.*)>\(\w", _kernel(args))
        v = [x.strip() for x in params.split(",")]
        if name == "shared":
            variant = (name, int(v[0]), v[-1] == "true")
        elif name == "split":
            variant = (name, int(v[5]) >= 32, v[-1] == "true")
        else:
            continue
        seen.add(variant)
        if args[:4] in PP.SPECIAL:
            special.add(variant[:2])
    assert seen == {("shared", b, t) for b in (64, 128) for t in (False, True)} | {
        ("split", f, t) for f in (False, True) for t in (False, True)}
    assert special == {("shared", 64), ("shared", 128), ("split", False)}


SCHEDULES = [("NT", 1500, 1500, 70, "tile 64x64"), ("NN", 4096, 2944, 40, "tile 64x64"), ("NN", 4096, 2944, 64, "tile 128x128"), ("TN", 600, 1000, 777, "ksplit 64x64"),
             ("TN", 600, 1000, 500, "ksplit 32x32"), ("NT", 4096, 256, 1024, "ksplit 64x64"), ("NT", 256, 1024, 1024, "ksplit 32x32")]


@pytest.mark.parametrize("layout,M,N,K,sched", SCHEDULES)
def test_schedule_by_tile_count_and_layout(layout, M, N, K, sched):
    """Shared tiles from two per CU on, 128 x 128 where there are two of those and K is at least 64;
    weight-gradient layouts with a long K split it over four wavefronts of 2 x 2 bf16 tiles; the rest in float32."""
    kern = _kernel((layout, M, N, K, ""))
    assert f"· {sched}," in kern
    assert ("bf16 x 3" in kern) == (sched.startswith("tile") or (layout == "TN" and K >= 512))


@pytest.mark.parametrize("M,N,K,split,slices", [
    (1000, 600, 777, True, 1), (1000, 512, 3000, True, 1), (1000, 448, 3000, False, 1), (256, 512, 2048, False, 1),
    (512, 512, 4095, False, 1), (512, 512, 4096, True, 8), (256, 768, 4096, True, 8), (256, 256, 4096, True, 8),
    (128, 128, 4096, False, 8), (1000, 600, 511, False, 1)])
def test_weight_gradients_split_into_bf16_where_workgroups_fill_half_the_chip(M, N, K, split, slices):
    """From 128 workgroups on, those of the K split across workgroups counted; below, float32 tiles."""
    kern = _kernel(("TN", M, N, K, ""))
    assert ("anvil_mm_tile_split<" in kern) == split
    assert re.findall(r"K in (\d+) slices", kern) == ([] if slices == 1 else [str(slices)])


def _special(args, layout):
    """A row of A with an infinity, one with a nan, one whose products pass the float32 range, and a
    column of B with an infinity; returns the affected rows and column."""
    x, w = args[0], args[1]
    xm = x.T if layout[0] == "T" else x                     # views: row m, k
    wn = w if layout[1] == "T" else w.T                     # row n, k
    xm[3, 5], xm[40, 1], wn[7, 9] = np.inf, np.nan, -np.inf
    xm[50, :] = 2e37
    return args


@pytest.mark.gpu
@pytest.mark.parametrize("layout,M,N,K", PP.SPECIAL)
def test_gpu_split_product_keeps_infinities_and_nans(layout, M, N, K):
    """Non-finite results are those of the float32 product (an operand split into bf16 parts would
    turn an infinity into a nan), and every other result keeps the bound."""
    print(f"gpu product with infinities {layout} {M}x{N}x{K}", flush=True)
    args, _, _, b = _operand(layout, M, N, K, "")
    args = _special(args, layout)
    a = (args[0].T if layout[0] == "T" else args[0]).astype(np.float64)
    w = (args[1].T if layout[1] == "T" else args[1]).astype(np.float64)
    got = _run(PP.product(layout, M, N, K, ""), args)
    with np.errstate(all="ignore"):
        want, mag = a @ w + b, np.abs(a) @ np.abs(w) + np.abs(b)
    rows = [i for i in range(M) if i != 50]
    assert np.array_equal(np.isnan(got[rows]), np.isnan(want[rows]))
    assert np.array_equal(np.isinf(got[rows]), np.isinf(want[rows]))
    fin = np.isfinite(want) & (mag < 1e38)
    fin[50] = False
    assert np.all(np.abs(got[fin] - want[fin]) <= (K + 8) * U * mag[fin])
    # row 50: finite where no partial sum can pass the range, and within the bound where finite
    ok = np.isfinite(got[50])
    assert ok[mag[50] < 3e38].all()
    assert np.all(np.abs(got[50][ok] - want[50][ok]) <= (K + 8) * U * mag[50][ok])
