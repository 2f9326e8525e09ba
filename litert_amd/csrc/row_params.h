// Scale and zero point of an activation row from its range, in two forms that give the same bits:
// the reference's own sequence of double divisions (tflite/kernels/internal/reference/
// portable_tensor_utils.cc:74-119, optimized/neon_tensor_utils.cc:2470-2552), and a short one
// that replaces them by one reciprocal and says when it cannot vouch for the result. Arithmetic
// only, so that the two can be compared on the host (g++) as well.
//
// Every row quantizer waits for these few numbers between its two passes, on one chain of dependent
// instructions: three divisions in sequence, two of them double, are some 100 of them at 8 cycles
// and more each (0.36-0.40 us by the clock read before and after, the short form 0.1). Most of that
// hides behind the weights on their way: the launch itself goes from 3.88 to 3.82 us (blockwise int4,
// 2048 -> 2048 at one row; four rows 4.77 -> 4.66). The per-channel int4 row quantizer's launch of its own
// gains nothing (362 x 4764 -> 899 with its product: divided 14.8, short 15.0) and keeps the divisions.
#ifndef LITERT_AMD_CSRC_ROW_PARAMS_H_
#define LITERT_AMD_CSRC_ROW_PARAMS_H_

#include <math.h>
#include <stdint.h>

#if defined(__HIPCC__)
#define LRTFC_ROW_PARAMS __host__ __device__ __forceinline__
#else
#define LRTFC_ROW_PARAMS inline
#endif

namespace lrtfc {

struct RowQuantParams {
  float scale;     // scaling factor stored for the row
  float inv;       // multiplier applied to each element
  int32_t zero_point;
  bool all_zero;   // the row quantizes to zeros with scale 1 / zero point 0
};

// max - min of a row as the two builds of the reference form it: portable widens to double before
// subtracting (portable_tensor_utils.cc:81-87), the NEON build subtracts in float
// (neon_tensor_utils.cc:2486).
template <bool kPortable>
LRTFC_ROW_PARAMS double RowSpan(float mn, float mx) {
  return kPortable ? static_cast<double>(mx) - static_cast<double>(mn) : static_cast<double>(mx - mn);
}

// The reference's sequence. mn < mx.
template <bool kPortable>
LRTFC_ROW_PARAMS RowQuantParams AsymmetricParamsDivided(float mn, float mx) {
  RowQuantParams p;
  p.all_zero = false;
  const double qmin = -128.0, qmax = 127.0;
  const double rmin = static_cast<double>(mn);
  const double rmax = static_cast<double>(mx);
  const double scale = RowSpan<kPortable>(mn, mx) / (qmax - qmin);
  const double zp_from_min = qmin - rmin / scale;
  const double zp_from_max = qmax - rmax / scale;
  const double err_from_min = fabs(qmin) + fabs(rmin / scale);
  const double err_from_max = fabs(qmax) + fabs(rmax / scale);
  const double zp_double = err_from_min < err_from_max ? zp_from_min : zp_from_max;
  if (zp_double <= qmin) {
    p.zero_point = -128;
  } else if (zp_double >= qmax) {
    p.zero_point = 127;
  } else {
    p.zero_point = static_cast<int8_t>(round(zp_double));
  }
  p.scale = static_cast<float>(scale);
  if (kPortable) {
    p.inv = 1.0f / p.scale;
  } else {
    p.inv = p.scale == 0.0f ? 0.0f : static_cast<float>(1.0 / static_cast<double>(p.scale));
  }
  return p;
}

// num / den, correctly rounded, from the correctly rounded reciprocal of den (Markstein's
// correction step: the remainder of the rounded product is exact in one fma). For numerators that
// are widened floats or differences of two, so nothing under- or overflows.
LRTFC_ROW_PARAMS double DivideByConstant(double num, double den, double reciprocal) {
  const double q = num * reciprocal;
  return fma(fma(-q, den, num), reciprocal, q);
}

// One Newton step of y = 1 / x.
LRTFC_ROW_PARAMS double RefineReciprocal(double x, double y) { return fma(fma(-x, y, 1.0), y, y); }

// The same numbers; false: the caller takes AsymmetricParamsDivided. `reciprocal(x)` is 1 / x to
// 2^-20 or better; two steps make it good to a few units in the last place of a double.
//   scale  Correctly rounded, see above.
//   inv    The float nearest to 1 / (float)scale. The quotient of two floats is never within 2^-49
//          (relative) of the midpoint of two floats, so a double that is wrong in its last places
//          rounds to the same float as the exact quotient (and as the double quotient of the NEON
//          form).
//   zero_point  The two candidates are off by less than 1e-12 (at most 255 in magnitude), so the
//          choice between them and the rounding are certain unless either is closer to its tie
//          than 1e-6. Values beyond [-128, 127] round to its ends, like the reference's clamp.
// Rows whose span leaves [1e-30, 1e30] (infinities and NaN among them) are the caller's.
template <bool kPortable, typename Reciprocal>
LRTFC_ROW_PARAMS bool AsymmetricParamsFast(float mn, float mx, Reciprocal reciprocal,
                                           RowQuantParams* p) {
  const double span = RowSpan<kPortable>(mn, mx);
  const double scale = DivideByConstant(span, 255.0, 1.0 / 255.0);
  const float scale_f = static_cast<float>(scale);
  const double start = reciprocal(scale);
  const double per_unit = RefineReciprocal(scale, RefineReciprocal(scale, start));
  const double rounded = static_cast<double>(scale_f);
  const double inv = RefineReciprocal(rounded, RefineReciprocal(rounded, start));
  const double from_min = static_cast<double>(mn) * per_unit;
  const double from_max = static_cast<double>(mx) * per_unit;
  const double margin = (128.0 + fabs(from_min)) - (127.0 + fabs(from_max));
  const double zp = margin < 0.0 ? -128.0 - from_min : 127.0 - from_max;
  const double nearest = rint(zp);
  p->scale = scale_f;
  p->inv = static_cast<float>(inv);
  const int32_t whole = static_cast<int32_t>(nearest);
  p->zero_point = whole < -128 ? -128 : (whole > 127 ? 127 : whole);
  p->all_zero = false;
  return span > 1e-30 && span < 1e30 && fabs(margin) > 1e-6 && fabs(zp - nearest) < 0.499999;
}

// 127.0 / d and d / 127.0 as floats, divided in double as the reference does; d > 0. The first is
// certain for the reason given at `inv`, in the same range.
template <typename Reciprocal>
LRTFC_ROW_PARAMS bool Quotient127Fast(float d, Reciprocal reciprocal, float* quotient) {
  const double x = static_cast<double>(d);
  *quotient = static_cast<float>(127.0 * RefineReciprocal(x, RefineReciprocal(x, reciprocal(x))));
  return d > 1e-30f && d < 1e30f;
}
LRTFC_ROW_PARAMS float Over127(float d) {
  const float q = static_cast<float>(DivideByConstant(static_cast<double>(d), 127.0, 1.0 / 127.0));
  return d > 3.402823466e38f ? d : q;  // infinity has no remainder to correct by
}

}  // namespace lrtfc

#endif  // LITERT_AMD_CSRC_ROW_PARAMS_H_
