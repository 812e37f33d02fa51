/* The oracle's correctly rounded leaves where the reference's CORE-MATH
 * source is not at hand: the same chelis_crmath_ffi_* symbols and results
 * (correct rounding has one answer), from wider arithmetic and Ziv's test. A
 * binary32 result is the C library's binary64 value rounded once, a binary64
 * result its x87 extended one, unless the rounding falls inside the wider
 * value's error bound; then libquadmath's binary128 value (113 bits) decides.
 * NaN is the canonical quiet NaN. tests/test_oracle_pins.py checks these
 * against the MPFR fixtures bit for bit, as it does CORE-MATH. */
#include <math.h>
#include <quadmath.h>
#include <stdint.h>
#include <string.h>

/* 2^-45 and 2^-57: far above the few ulps (2^-52, 2^-63) of the C library's
 * functions, so the test never accepts a wrong rounding; the wider value is
 * recomputed for about one result in 2^20 (binary32) or 2^4 (binary64). */
static float cr32(double y, float x, __float128 (*wide)(__float128)) {
    if (y != y) {
        const uint32_t q = 0x7fc00000u;
        float r;
        memcpy(&r, &q, 4);
        return r;
    }
    const float lo = (float)(y - fabs(y) * 0x1p-45), hi = (float)(y + fabs(y) * 0x1p-45);
    return lo == hi ? lo : (float)wide((__float128)x);
}
static double cr64(long double y, double x, __float128 (*wide)(__float128)) {
    if (y != y) {
        const uint64_t q = 0x7ff8000000000000ull;
        double r;
        memcpy(&r, &q, 8);
        return r;
    }
    const double lo = (double)(y - fabsl(y) * 0x1p-57L), hi = (double)(y + fabsl(y) * 0x1p-57L);
    return lo == hi ? lo : (double)wide((__float128)x);
}

float chelis_crmath_ffi_expf(float x) { return cr32(exp((double)x), x, expq); }
float chelis_crmath_ffi_logf(float x) { return cr32(log((double)x), x, logq); }
float chelis_crmath_ffi_erfcf(float x) { return cr32(erfc((double)x), x, erfcq); }
float chelis_crmath_ffi_tanhf(float x) { return cr32(tanh((double)x), x, tanhq); }
double chelis_crmath_ffi_exp(double x) { return cr64(expl((long double)x), x, expq); }
double chelis_crmath_ffi_log(double x) { return cr64(logl((long double)x), x, logq); }
double chelis_crmath_ffi_erfc(double x) { return cr64(erfcl((long double)x), x, erfcq); }
double chelis_crmath_ffi_tanh(double x) { return cr64(tanhl((long double)x), x, tanhq); }
