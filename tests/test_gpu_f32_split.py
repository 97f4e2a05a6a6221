"""f32 attention whose products go through bf16 matrix instructions, every value as three bf16 parts (f32_split.h): the edges of its tiles
of 64 keys and blocks of 64 rows, values at the ends of f32's range, infinities, and its error against 64 bits."""
import numpy as np
import pytest

from incin_amd import capi, host
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def inputs(seed, B, H, Sq, Skv, D):
    r = np.random.Generator(np.random.PCG64(seed))
    return [r.standard_normal((B, H, n, D), dtype=np.float32) for n in (Sq, Skv, Skv)]


@pytest.mark.parametrize("D", [4, 64, 72, 96, 100, 128])
@pytest.mark.parametrize("Sq,Skv", [(1, 1), (33, 31), (64, 64), (63, 65), (65, 33), (127, 129), (130, 200)])
@pytest.mark.parametrize("causal", [False, True])
def test_tile_edges(gpu, D, Sq, Skv, causal):
    """One key, blocks and tiles with one row or key more or less than full, a tile whose second block is empty; the causal edge in each."""
    if causal and Skv < Sq:
        pytest.skip("rows without keys: test_gpu_parity has those")
    q, k, v = inputs(Sq * 7 + Skv + D, 2, 3, Sq, Skv, D)
    got, info = host.sdpa(q, k, v, capi.F32, causal=causal, impl=capi.IMPL_MFMA, return_info=True)
    assert info["impl"] == capi.IMPL_MFMA
    assert np.max(np.abs(got - O.sdpa(q, k, v, causal=causal))) <= 1e-5


@pytest.mark.parametrize("D", [64, 96, 128])
def test_values_that_are_not_finite(gpu, D):
    """What an infinity or a NaN reaches is what the IEEE products give: against the generic kernel (f32 multiply-adds), for an infinite
    value of V (its column), of K (rows whose score is +inf are NaN, those of -inf do without the key) and a NaN in Q (its row)."""
    q, k, v = inputs(5, 1, 2, 70, 90, D)
    for what, t, at, x in (("v", v, (0, 0, 40, 3), np.inf), ("v", v, (0, 1, 89, D - 1), -np.inf), ("k", k, (0, 0, 11, 5), np.inf), ("q", q, (0, 1, 69, 0), np.nan)):
        was = t[at]
        t[at] = x
        with np.errstate(invalid="ignore"):
            got = host.sdpa(q, k, v, capi.F32, impl=capi.IMPL_MFMA)
            ref = host.sdpa(q, k, v, capi.F32, impl=capi.IMPL_GENERIC)
        t[at] = was
        assert np.array_equal(np.isnan(got), np.isnan(ref)), what
        assert np.array_equal(np.isposinf(got), np.isposinf(ref)) and np.array_equal(np.isneginf(got), np.isneginf(ref)), what
        fin = np.isfinite(ref)
        assert fin.any() and not fin.all() and np.max(np.abs(got[fin] - ref[fin])) <= 1e-5, what


@pytest.mark.parametrize("exponent", [-60, -20, 20, 60, 120])
def test_values_of_any_size(gpu, exponent):
    """Values far from 1 keep their 24 bits: Q large where K is small, V of any size; and values that round to infinity in bf16."""
    q, k, v = inputs(9, 1, 2, 100, 100, 64)
    s = np.float32(2.0 ** (exponent / 2))
    ref = O.sdpa(q, k, v)
    got = host.sdpa(q * s, k / s, v * np.float32(2.0 ** exponent), capi.F32, impl=capi.IMPL_MFMA)
    assert np.max(np.abs(got.astype(np.float64) * 2.0 ** -exponent - ref)) <= 1e-5
    if exponent == 120:      # (the largest finite value: its first bf16 part would be infinite)
        v[0, 0, 7, 5] = np.finfo(np.float32).max
        got, gen = (host.sdpa(q, k, v, capi.F32, impl=i) for i in (capi.IMPL_MFMA, capi.IMPL_GENERIC))
        assert np.isfinite(got).all() and np.max(np.abs(got - gen) / np.maximum(np.abs(gen), 1)) <= 1e-5


@pytest.mark.parametrize("S,D,causal", [(1024, 64, False), (512, 96, True), (700, 128, False)])
def test_error_against_64_bits(gpu, S, D, causal):
    """No larger than that of IEEE-f32 products: those leave 2.2e-7 - 3.5e-7 of the 2-norm here, this kernel 1.2e-7 - 2.0e-7.  The bound is the
    rounding of P and O in f32 (2^-24 each) and of a sum of S / 32 steps (2^-25 sqrt(S / 32) at most), together below 2.5e-7."""
    q, k, v = inputs(S + D, 1, 4, S, S, D)
    q64, k64, v64 = (x.astype(np.float64) for x in (q, k, v))
    s = q64 @ k64.transpose(0, 1, 3, 2) / np.sqrt(D)
    if causal:
        s += np.triu(np.full((S, S), -np.inf), 1)
    p = np.exp(s - s.max(-1, keepdims=True))
    ref = (p / p.sum(-1, keepdims=True)) @ v64
    got = host.sdpa(q, k, v, capi.F32, causal=causal, impl=capi.IMPL_MFMA)
    assert np.linalg.norm(got - ref) / np.linalg.norm(ref) < 2.5e-7
