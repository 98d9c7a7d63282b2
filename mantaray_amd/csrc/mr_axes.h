// mr_axes.h -- what the records hold of an axis: the exact cell thresholds of
// the reference's index rules, and the fast regions of its cells.  Host code
// without the HIP runtime.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <vector>

namespace mr {

// ---- cell thresholds -------------------------------------------------------
// The reference's cell along an axis is a monotone step function of the
// coordinate: the fractional index RN(RN(p - a0) / sp) is non-decreasing in
// p (each rounding is monotone), and the cell is its floor, clamped to n-2 on
// the last node.  T[i] = min{p : index(p) >= i} for i < n-1 and T[n-1] =
// min{p : index(p) > n-1} make cell i exactly [T[i], T[i+1]) and the valid
// range [T[0], T[n-1]).  Each T is found by bisection over the totally
// ordered floating-point values, evaluating the index with the reference's
// own operations (cartesian_netcdf3.rs:285, cartesian_current.rs:244).
// T[i] is within a few roundings of a0 + i sp, so the search widens from there
// (first_true) before it bisects: from the whole range an axis of 1500 nodes
// takes 0.54 ms (f64) or 0.31 ms (f32) of the first trace of its field, from
// the guess 0.012 and 0.008 ms.

inline uint32_t key32(float f)
{
    uint32_t b;
    std::memcpy(&b, &f, 4);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
inline float unkey32(uint32_t k)
{
    uint32_t b = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
    float f;
    std::memcpy(&f, &b, 4);
    return f;
}
inline uint64_t key64(double f)
{
    uint64_t b;
    std::memcpy(&b, &f, 8);
    return (b >> 63) ? ~b : (b | (uint64_t(1) << 63));
}
inline double unkey64(uint64_t k)
{
    uint64_t b = (k >> 63) ? (k & ~(uint64_t(1) << 63)) : ~k;
    double f;
    std::memcpy(&f, &b, 8);
    return f;
}

// The first key of (lo, hi] whose pred is true; pred does not decrease, is
// taken as false at lo and as true at hi, and is evaluated at neither.
template <class Key, class Pred>
Key first_true(Key lo, Key hi, Key guess, Pred pred)
{
    if (guess > lo && guess < hi) {
        // (hi - lo bounds the step, so doubling it cannot wrap)
        if (pred(guess)) {
            hi = guess;
            for (Key step = 1; hi - lo > step; step *= 2) {
                if (!pred(hi - step)) {
                    lo = hi - step;
                    break;
                }
                hi -= step;
            }
        } else {
            lo = guess;
            for (Key step = 1; hi - lo > step; step *= 2) {
                if (pred(lo + step)) {
                    hi = lo + step;
                    break;
                }
                lo += step;
            }
        }
    }
    while (hi - lo > 1) {
        const Key mid = lo + (hi - lo) / 2;
        if (pred(mid)) hi = mid; else lo = mid;
    }
    return hi;
}

// f32 axis (bathymetry): thresholds T[0..n-1]
inline std::vector<float> thresholds32(const std::vector<float> &a)
{
    const size_t n = a.size();
    const float a0 = a[0], sp = std::fabs(a[1] - a[0]);
    auto index = [&](float p) { return (p - a0) / sp; };        // :285
    std::vector<float> t(n);
    for (size_t i = 0; i < n; i++) {
        const float lim = (float)i;
        const bool upper = i == n - 1;                         // index > n-1 errs
        auto pred = [&](uint32_t k) {
            const float x = index(unkey32(k));
            return upper ? x > lim : x >= lim;
        };
        const uint32_t lo = key32(-INFINITY), hi = key32(INFINITY);
        // (a spacing that overflows leaves no order to widen in: lo, no guess)
        const uint32_t guess =
            std::isfinite(sp) ? key32((float)((double)a0 + (double)i * (double)sp)) : lo;
        t[i] = unkey32(first_true(lo, hi, guess, pred));
    }
    return t;
}

// f64 axis (current): thresholds T[0..n-1]
inline std::vector<double> thresholds64(const std::vector<double> &a)
{
    const size_t n = a.size();
    const double a0 = a[0], sp = std::fabs(a[1] - a[0]);
    auto index = [&](double p) { return (p - a0) / sp; };       // :244
    std::vector<double> t(n);
    for (size_t i = 0; i < n; i++) {
        const double lim = (double)i;
        const bool upper = i == n - 1;
        auto pred = [&](uint64_t k) {
            const double x = index(unkey64(k));
            return upper ? x > lim : x >= lim;
        };
        const uint64_t lo = key64(-INFINITY), hi = key64(INFINITY);
        const uint64_t guess = std::isfinite(sp) ? key64(a0 + (double)i * sp) : lo;
        t[i] = unkey64(first_true(lo, hi, guess, pred));
    }
    return t;
}

// The fast region of each cell along one axis (SCell, DCell, UCell): the f32
// targets p in [lo, hi] lie in cell i for the depth's f32 index rule (T32[i]
// <= p < T32[i+1]; t32 null: no depth on this axis), for every f64 coordinate
// that rounds to p lie in cell i for the current's f64 index rule (T64[i] <=
// x < T64[i+1]; t64 null: no current), and are strictly between the cell's
// node coordinates a[i] and a[i+1] (no corner).  If RN32(x) >= lo >
// ceil32(T64[i]) then x > T64[i]; if RN32(x) <= hi < floor32(T64[i+1]) then
// x < T64[i+1] (rounding is monotone).  The intervals need not meet (on axes
// whose spacing varies, the index rules, which use the first spacing, can map
// a cell's targets outside its nodes): an empty interval is stored as
// (-inf, -inf), the one form of an empty region that the device's region
// test (med3(p, lo, hi) - p) reads as empty; lo > hi would read as [hi, lo].
// (Pair: a struct of two floats x, y.)
template <class Pair>
std::vector<Pair> fast_bounds(const std::vector<float> &a, const std::vector<float> *t32,
                              const std::vector<double> *t64)
{
    auto up = [](float f) { return std::nextafter(f, INFINITY); };
    auto down = [](float f) { return std::nextafter(f, -INFINITY); };
    auto ceil32 = [&](double d) {
        float f = (float)d;
        return (double)f < d ? up(f) : f;
    };
    auto floor32 = [&](double d) {
        float f = (float)d;
        return (double)f > d ? down(f) : f;
    };
    std::vector<Pair> b(a.size() - 1);
    for (size_t i = 0; i + 1 < a.size(); i++) {
        float lo = up(a[i]), hi = down(a[i + 1]);
        if (t32) {
            lo = std::max(lo, (*t32)[i]);
            hi = std::min(hi, down((*t32)[i + 1]));
        }
        if (t64) {
            lo = std::max(lo, up(ceil32((*t64)[i])));
            hi = std::min(hi, down(floor32((*t64)[i + 1])));
        }
        b[i] = lo <= hi ? Pair{lo, hi} : Pair{-INFINITY, -INFINITY};
    }
    return b;
}

// The largest share of a cell's coordinates along the axis, over its cells,
// that lie outside the cell's fast region: a bound [lo, hi] stands for the
// coordinates that round to it, cell i for [t[i], t[i+1]), of the last cell
// without the last node.
template <class Pair, class T>
double worst_outside(const std::vector<Pair> &bounds, const std::vector<T> &t)
{
    double worst = 0.0;
    for (size_t i = 0; i < bounds.size(); i++) {
        const double lo = bounds[i].x, hi = bounds[i].y;
        const double in = std::isfinite(lo)
                              ? hi - lo + ((double)std::nextafter(bounds[i].y, INFINITY) - hi)
                              : 0.0;
        const T end = i + 1 < bounds.size() ? t[i + 1] : std::nextafter(t[i + 1], (T)-INFINITY);
        worst = std::max(worst, 1.0 - in / ((double)end - (double)t[i]));
    }
    return worst;
}

}  // namespace mr
