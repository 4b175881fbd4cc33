"""The one-kernel attention at ragged numbers of queries and keys and every head width it takes."""
import re

import numpy as np
import pytest

import product_programs as PP

from anvil.backend import hip
from anvil.hip_function import Compiled

U = 2.0 ** -24


def _args(B, Lq, Lk, D, seed=3):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal((B, n, D)).astype(np.float32) for n in (Lq, Lk, Lk)]


def _exact(q, k, v):
    s = np.matmul(q.astype(np.float64), k.astype(np.float64).transpose(0, 2, 1)) / np.sqrt(q.shape[-1])
    p = np.exp(s - s.max(axis=2, keepdims=True))
    p /= p.sum(axis=2, keepdims=True)
    return p, np.matmul(p, v.astype(np.float64))


@pytest.mark.parametrize("B,Lq,Lk,D", PP.ATTENTIONS)
def test_attention_is_one_kernel_at_any_length(B, Lq, Lk, D):
    src = hip.generate(PP.attention(B, Lq, Lk, D).prog, library=True)
    assert "// attention: " in src and "// rows: " not in src and "// gemm: " not in src


@pytest.mark.parametrize("B,Lq,Lk,D", PP.SEPARATE + [(1, 2048, 2048, 128), (1, 2048, 2048, 80), (1, 64, 4096, 32)])
def test_attention_of_few_queries_is_three_launches(B, Lq, Lk, D):
    """Where one kernel's chain of key tiles takes longer than the products and rows on their own."""
    src = hip.generate(PP.attention(B, Lq, Lk, D).prog, library=True)
    assert "// attention: " not in src and src.count("// gemm: ") == 2


def test_eight_wavefronts_only_where_their_registers_hold():
    for args in PP.ATTENTIONS + [(2, 1500, 1500, 96), (4, 700, 700, 128), (4, 2048, 2048, 64)]:
        src = hip.generate(PP.attention(*args).prog, library=True)
        D, W = map(int, re.search(r"anvil_attention_tile<(\d+), (\d+)[,>]", src).groups())
        B, Lq, Lk, _ = args
        assert W == (8 if D <= 96 and -(-Lq // 32) * B <= 128 and Lk > 480 else 4), args


@pytest.mark.gpu
@pytest.mark.parametrize("B,Lq,Lk,D", PP.ATTENTIONS + PP.SEPARATE)
def test_gpu_attention_matches_float64(B, Lq, Lk, D):
    """Each output is a weighted mean of V: its error is within that of its scores (a D-term sum of
    |q k| each, in the exponent, and the scale's rounding), an exponential's few units, and the two
    Lk-term sums, times the weighted mean of |V|."""
    print(f"gpu attention {B} x ({Lq} x {Lk}, D = {D})", flush=True)
    q, k, v = _args(B, Lq, Lk, D)
    got = Compiled("attention", PP.attention(B, Lq, Lk, D)).call([q, k, v])
    p, want = _exact(q, k, v)
    s = np.matmul(q.astype(np.float64), k.astype(np.float64).transpose(0, 2, 1)) / np.sqrt(D)
    smax = np.matmul(np.abs(q).astype(np.float64), np.abs(k).astype(np.float64).transpose(0, 2, 1)).max() / np.sqrt(D)
    rel = U * (2 * (D + 8) * smax + 2 * (Lk + 16))
    assert np.all(np.abs(got - want) <= rel * np.matmul(p, np.abs(v).astype(np.float64)))
    # and the 2-norm error is that of float32: roundings of a D-term score (2^-24 sqrt(D / 2) of it, in the
    # exponent) and of the weighted sum, run by run of at most 512 keys, independent of one another. Two
    # bf16 in place of three for any of q, k, p and v: 2e-6 or more at each of these sizes.
    usual = U * (4 + (D / 2) ** 0.5 * np.std(s) + (min(Lk, 512) / 2) ** 0.5)
    assert np.linalg.norm(got - want) <= min(usual, 1e-6) * np.linalg.norm(want)


@pytest.mark.gpu
@pytest.mark.parametrize("B,Lq,Lk,D", PP.TWO_TILES)
def test_gpu_attention_of_two_key_tiles_keeps_the_float32_error(B, Lq, Lk, D):
    """The 2-norm error over many heads is that measured with the chain's three launches on float32 products,
    1.24e-7, and a fortieth (Vᵀ p with all its terms in one truncated sum: 1.33e-7)."""
    print(f"gpu attention {B} x ({Lq} x {Lk}, D = {D})", flush=True)
    q, k, v = _args(B, Lq, Lk, D)
    got, (_, want) = Compiled("attention", PP.attention(B, Lq, Lk, D)).call([q, k, v]), _exact(q, k, v)
    print("error", np.linalg.norm(got - want) / np.linalg.norm(want))
    assert np.linalg.norm(got - want) <= 1.27e-7 * np.linalg.norm(want)


@pytest.mark.gpu
@pytest.mark.parametrize("eq,ek,ev", [(0, 0, -118), (-118, 118, 0), (118, -118, 0), (60, -60, -60), (-70, 70, 100), (0, 0, 110)])
@pytest.mark.parametrize("B,Lq,Lk,D", PP.MAGNITUDES)
def test_gpu_attention_keeps_small_and_large_values(B, Lq, Lk, D, eq, ek, ev):
    """q, k and v around 2^eq, 2^ek and 2^ev, whose result is that around 1 times 2^ev: the 2-norm error too
    (a bf16 part lost at 2^-118 costs 2^-16 of a value, 1e-6 or more here)."""
    print(f"gpu attention {B} x ({Lq} x {Lk}, D = {D}) at 2^{eq}, 2^{ek}, 2^{ev}", flush=True)
    q, k, v = (x * np.float32(2.0 ** e) for x, e in zip(_args(B, Lq, Lk, D), (eq, ek, ev)))
    got, (_, want) = Compiled("attention", PP.attention(B, Lq, Lk, D)).call([q, k, v]), _exact(q, k, v)
    print("error", np.linalg.norm(got / 2.0 ** ev - want / 2.0 ** ev) / np.linalg.norm(want / 2.0 ** ev))
    assert np.linalg.norm((got - want) / 2.0 ** ev) <= 5e-7 * np.linalg.norm(want / 2.0 ** ev)


@pytest.mark.gpu
@pytest.mark.parametrize("B,Lq,Lk,D", PP.MAGNITUDES)
def test_gpu_attention_keeps_small_weights(B, Lq, Lk, D):
    """Every 32nd key has a score 122 (base 2) above the others' and a value of 0, so that the result is made
    of weights around 2^-122. A score of 122 is rounded at 2^-18, in the exponent; three bf16 of a weight
    without their low bits would be 2^-12 off."""
    print(f"gpu attention {B} x ({Lq} x {Lk}, D = {D}), small weights", flush=True)
    q, k, v = _args(B, Lq, Lk, D)
    q *= 0.1
    q[:, :, 0], k[:, :, 0], v[:, ::32] = D ** 0.5, 0, 0
    k[:, ::32] = 0
    k[:, ::32, 0] = 122 * np.log(2)
    got, (_, want) = Compiled("attention", PP.attention(B, Lq, Lk, D)).call([q, k, v]), _exact(q, k, v)
    up = 2.0 ** 120
    print("error", np.linalg.norm(got * up - want * up) / np.linalg.norm(want * up))
    assert np.linalg.norm(got * up - want * up) <= 1e-5 * np.linalg.norm(want * up)


@pytest.mark.gpu
@pytest.mark.parametrize("B,Lq,Lk,D", [(2, 40, 65, 32), (1, 100, 257, 80), (1, 96, 640, 128), (36, 96, 640, 128)])
def test_gpu_attention_keeps_infinities_and_nans(B, Lq, Lk, D):
    """An infinity in V reaches its column of every query, a nan in Q its own row only; the other results
    keep their tolerance."""
    print(f"gpu attention with infinities {B} x ({Lq} x {Lk}, D = {D})", flush=True)
    q, k, v = _args(B, Lq, Lk, D)
    v[0, Lk - 1, 3] = np.inf
    v[0, 2, 5] = -np.inf
    q[0, 7, 0] = np.nan
    got = Compiled("attention", PP.attention(B, Lq, Lk, D)).call([q, k, v])
    rest = [i for i in range(Lq) if i != 7]
    assert np.isnan(got[0, 7]).all()
    assert np.isposinf(got[0, rest, 3]).all() and np.isneginf(got[0, rest, 5]).all()
    v[0, Lk - 1, 3], v[0, 2, 5], q[0, 7, 0] = 0, 0, 0
    _, want = _exact(q, k, v)
    cols = [c for c in range(D) if c not in (3, 5)]
    np.testing.assert_allclose(got[0][np.ix_(rest, cols)], want[0][np.ix_(rest, cols)], rtol=1e-4, atol=1e-5)
    if B > 1:
        np.testing.assert_allclose(got[1:], want[1:], rtol=1e-4, atol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("B,Lq,Lk,D", [(2, 40, 65, 32), (1, 100, 257, 80), (1, 96, 640, 128), (36, 96, 640, 128)])
def test_gpu_attention_keys_of_minus_infinity_weigh_nothing(B, Lq, Lk, D):
    """Scores of -inf over a wavefront's whole share of the keys (and its first tile) leave the softmax
    of the others; a row of nothing else is nan."""
    print(f"gpu attention with -inf scores {B} x ({Lq} x {Lk}, D = {D})", flush=True)
    q, k, v = _args(B, Lq, Lk, D)
    q[0, :, 0] = np.abs(q[0, :, 0]) + 0.5
    gone = max(40, Lk // 2)
    k[0, :gone, 0] = -np.inf
    fn = Compiled("attention", PP.attention(B, Lq, Lk, D))
    got = fn.call([q, k, v])
    _, want = _exact(q[:1], k[:1, gone:], v[:1, gone:])
    np.testing.assert_allclose(got[:1], want, rtol=1e-4, atol=1e-5)
    k[0, :, 0] = -np.inf
    assert np.isnan(fn.call([q, k, v])[0]).all()
