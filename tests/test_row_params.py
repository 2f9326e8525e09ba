"""A row's scale and zero point without divisions (litert_amd/csrc/row_params.h): on the host against the
reference's sequence of divisions, bit for bit, and through the row quantizers against the oracle."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import oracle

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CODE = r"""
#include <string.h>
#include "litert_amd/csrc/row_params.h"
using namespace lrtfc;
template <bool P> static int one(float mn, float mx, double eps) {
  RowQuantParams q;
  if (!AsymmetricParamsFast<P>(mn, mx, [&](double x) { return (1.0 / x) * (1.0 + eps); }, &q)) return 1;
  const RowQuantParams r = AsymmetricParamsDivided<P>(mn, mx);
  return !memcmp(&q.scale, &r.scale, 4) && !memcmp(&q.inv, &r.inv, 4) && q.zero_point == r.zero_point ? 0 : 2;
}
static int one127(float d, double eps) {
  const float over = Over127(d), r = static_cast<float>(static_cast<double>(d) / 127.0);
  if (memcmp(&over, &r, 4)) return 2;
  float q;
  if (!Quotient127Fast(d, [&](double x) { return (1.0 / x) * (1.0 + eps); }, &q)) return 1;
  const float want = static_cast<float>(127.0 / static_cast<double>(d));
  return memcmp(&q, &want, 4) ? 2 : 0;
}
extern "C" void asymmetric(int portable, long n, const float* mn, const float* mx, const double* eps, unsigned char* out) {
  for (long i = 0; i < n; ++i) out[i] = portable ? one<true>(mn[i], mx[i], eps[i]) : one<false>(mn[i], mx[i], eps[i]);
}
extern "C" int refused(int portable, float mn, float mx) {
  RowQuantParams q;
  const auto reciprocal = [](double x) { return 1.0 / x; };
  return portable ? !AsymmetricParamsFast<true>(mn, mx, reciprocal, &q) : !AsymmetricParamsFast<false>(mn, mx, reciprocal, &q);
}
extern "C" void quotient127(long n, const float* d, const double* eps, unsigned char* out) {
  for (long i = 0; i < n; ++i) out[i] = one127(d[i], eps[i]);
}
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    d = tmp_path_factory.mktemp("row_params")
    (d / "t.cc").write_text(CODE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared", "-I", ROOT,
                    str(d / "t.cc"), "-o", str(d / "t.so")], check=True)
    return C.CDLL(str(d / "t.so"))


def _p(a):
    return a.ctypes.data_as(C.c_void_p)


def _ranges(n, rng):
    """Rows' (min, max): exponents over the whole range and around one, one side zero, and ranges
    whose zero point or choice of its end is a tie or next to one."""
    def floats(lo, hi):
        return np.ldexp(1 + rng.random(n), rng.integers(lo, hi, n)).astype(np.float32)
    s = np.ldexp(1.0, rng.integers(-40, 40, n))
    half = rng.integers(0, 511, n) * 0.5
    tie = (-half * s).astype(np.float32), ((255 - half) * s).astype(np.float32)
    beside = np.nextafter(tie[0], np.float32(1e30) * (1 - 2 * rng.integers(0, 2, n))).astype(np.float32)
    zero = np.zeros(n, np.float32)
    pairs = [(-floats(-148, 127), floats(-148, 127)), (-floats(-6, 3), floats(-6, 3)),
             (zero, floats(-148, 127)), (-floats(-148, 127), zero), tie,
             (np.minimum(beside, 0), np.maximum(tie[1], np.float32(1e-30)))]
    mn, mx = (np.concatenate(v).astype(np.float32) for v in zip(*pairs))
    keep = mn < mx
    return np.ascontiguousarray(mn[keep]), np.ascontiguousarray(mx[keep])


@pytest.mark.parametrize("portable", [1, 0])
def test_short_form_gives_the_divided_forms_bits(host, portable):
    rng = np.random.default_rng(5 + portable)
    with np.errstate(over="ignore", under="ignore"):
        mn, mx = _ranges(300000, rng)
    out = np.empty(mn.size, np.uint8)
    eps = rng.uniform(-2.0 ** -20, 2.0 ** -20, mn.size)  # a start four bits worse than the hardware's
    host.asymmetric(portable, C.c_long(mn.size), _p(mn), _p(mx), _p(eps), _p(out))
    assert not (out == 2).any(), (mn[out == 2][:4], mx[out == 2][:4])
    # ordinary ranges that are no ties are vouched for
    ordinary = rng.normal(size=(2, 100000)).astype(np.float32)
    mn, mx = np.minimum(ordinary.min(0), 0), np.maximum(ordinary.max(0), np.float32(0.1))
    out = np.empty(mn.size, np.uint8)
    host.asymmetric(portable, C.c_long(mn.size), _p(mn), _p(mx), _p(eps[:mn.size].copy()), _p(out))
    assert (out == 0).mean() > 0.999


@pytest.mark.parametrize("portable", [1, 0])
def test_short_form_leaves_spans_beyond_its_limits(host, portable):
    """Infinities and NaN, spans of 1e30 and more (3e38 to each side overflows the float span) or of 1e-30 and
    less: the caller divides."""
    host.refused.argtypes = [C.c_int, C.c_float, C.c_float]
    inf, nan = np.inf, np.nan
    for mn, mx in ((-inf, 1.0), (-1.0, inf), (-inf, inf), (nan, 1.0), (-1.0, nan), (nan, nan), (-3e38, 3e38),
                   (0.0, 1.01e30), (-0.6e30, 0.6e30), (0.0, 0.99e-30), (-1e-45, 0.0)):
        assert host.refused(portable, mn, mx), (mn, mx)
    for mn, mx in ((0.0, 0.99e30), (0.0, 1.01e-30), (-1.0, 3.0)):
        assert not host.refused(portable, mn, mx), (mn, mx)


def test_quotients_with_127(host):
    # every exponent, subnormals, the largest value and infinity
    bits = np.append(np.arange(1, 0x7F800000, 1511), [0x7F7FFFFF, 0x7F800000]).astype(np.uint32)
    d = bits.view(np.float32)
    out = np.empty(d.size, np.uint8)
    eps = np.random.default_rng(3).uniform(-2.0 ** -20, 2.0 ** -20, d.size)
    host.quotient127(C.c_long(d.size), _p(d), _p(eps), _p(out))
    assert not (out == 2).any()
    assert (out[(d > 1e-29) & (d < 1e29)] == 0).all()


def _rows(depth):
    """Rows at the edges of the short form: ties of the zero point and of its end, one-sided, all
    zero, spans at and beyond its limits. (Below 1e-36 the reference multiplies by infinity and what the
    conversion of that gives is not fixed; the host test goes there, and to infinities and NaN.)"""
    f = np.float32
    ends = [(-k - 0.5, 254.5 - k) for k in (0, 1, 60, 126, 127, 200, 254)] + [(-127.0, 128.0), (-128.0, 127.0)]
    ends += [(-126.5, 128.5), (-127.5, 127.5), (-1.0, 1.0), (0.0, 1.0), (-1.0, 0.0), (0.0, 0.0)]
    ends += [(-s * 0.3, s * 0.7) for s in (1e-35, 0.99e-30, 1.01e-30, 0.99e30, 1.01e30, 1.5e30, 1e33, 3e38)]
    rng = np.random.default_rng(depth)
    x = np.zeros((len(ends), depth), f)
    for i, (lo, hi) in enumerate(ends):
        x[i] = (lo + (hi - lo) * rng.random(depth)).astype(f)
        x[i, 0], x[i, -1] = lo, hi
    return x


@pytest.mark.gpu
@pytest.mark.parametrize("variant", [0, 1, 2])
@pytest.mark.parametrize("asym", [True, False])
@pytest.mark.parametrize("depth", [7, 96, 4100])
def test_row_quantizer_at_the_short_forms_edges(variant, asym, depth):
    import torch
    from litert_amd import fully_connected as fc
    x = _rows(depth)
    q, sf, zp = (t.cpu().numpy() for t in fc.batch_quantize_floats(torch.from_numpy(x).cuda(), asym, variant))
    wq, wsf, wzp = oracle.batch_quantize_floats(x, asym, variant)
    assert np.array_equal(sf.view(np.uint32), wsf.view(np.uint32))
    assert np.array_equal(zp, wzp)
    assert np.array_equal(q, wq)


@pytest.mark.gpu
def test_symmetric_4bit_quantizer_at_the_short_forms_edges():
    """Whole-row products show scale and multiplier: per-channel int4 rows of 1 (fused) and of all
    (the quantizer's own launch) at once."""
    import torch
    from litert_amd import fully_connected as fc
    K, N = 96, 40
    rng = np.random.default_rng(1)
    w = rng.integers(0, 256, (N, K // 2), dtype=np.uint8)
    scales = rng.uniform(0.01, 0.02, N).astype(np.float32)
    x = _rows(K)
    x = x[(np.abs(x).max(axis=1) > 4e-37) | (x == 0).all(axis=1)]
    assert (np.abs(x).max(axis=1) > 1e30).sum() >= 3  # beyond the short form's limit
    op = fc.FullyConnectedHybridInt4PerChannel(torch.from_numpy(w).cuda(), K, scales)
    xs = torch.from_numpy(x).cuda()
    want = oracle.fc_hybrid_int4_per_channel(x, w, N, scales)
    assert np.array_equal(op(xs).cpu().numpy().view(np.uint32), want.view(np.uint32))
    for i in range(len(x)):
        assert np.array_equal(op(xs[i:i + 1]).cpu().numpy().view(np.uint32), want[i:i + 1].view(np.uint32))


@pytest.mark.gpu
def test_infinite_rows_of_the_4bit_path_are_the_same_fused_and_not():
    """A row whose largest magnitude is infinite: scale infinite, every product a zero or no number. What that
    is depends on no rounding, and is the same from the product's own quantizer and the one of its own."""
    import torch
    from litert_amd import fully_connected as fc
    K, N = 96, 40
    rng = np.random.default_rng(2)
    w = rng.integers(0, 256, (N, K // 2), dtype=np.uint8)
    scales = rng.uniform(0.01, 0.02, N).astype(np.float32)
    x = rng.standard_normal((20, K)).astype(np.float32)
    x[::3, 5], x[1::3, 7] = np.inf, -np.inf
    op = fc.FullyConnectedHybridInt4PerChannel(torch.from_numpy(w).cuda(), K, scales)
    xs = torch.from_numpy(x).cuda()
    split = op(xs).cpu().numpy()
    fused = np.concatenate([op(xs[i:i + 1]).cpu().numpy() for i in range(len(x))])
    ordinary = np.isfinite(x).all(axis=1)
    assert np.array_equal(split[ordinary].view(np.uint32), fused[ordinary].view(np.uint32))
    assert np.array_equal(np.isnan(split), np.isnan(fused))
    assert np.array_equal(split[~np.isnan(split)], fused[~np.isnan(fused)])
