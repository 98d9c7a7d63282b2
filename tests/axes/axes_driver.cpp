// Reads axes (records of: int64 kind 32 or 64, int64 n, n doubles) from the
// file argv[1] and checks what mr_axes.h makes of each: the thresholds against
// a bisection over every floating-point value, the fast regions against the
// index rules themselves.  Prints "<wrong thresholds> <wrong regions>
// <worst_outside>" a line.
#include "mr_axes.h"

#include <cstdio>

struct Pair {
    float x, y;
};

// the axis index rules, as the reference rounds them
template <class T>
T index_of(const std::vector<T> &a, T p)
{
    return (T)(p - a[0]) / std::fabs(a[1] - a[0]);
}

template <class T, class Key>
std::vector<T> plain(const std::vector<T> &a, Key (*key)(T), T (*unkey)(Key))
{
    std::vector<T> t(a.size());
    for (size_t i = 0; i < a.size(); i++) {
        Key lo = key(-INFINITY), hi = key(INFINITY);
        while (hi - lo > 1) {
            const Key mid = lo + (hi - lo) / 2;
            const T x = index_of(a, unkey(mid));
            if (i + 1 == a.size() ? x > (T)i : x >= (T)i) hi = mid;
            else lo = mid;
        }
        t[i] = unkey(hi);
    }
    return t;
}

template <class T>
bool in_cell(const std::vector<T> &a, T p, size_t i)
{
    const T x = index_of(a, p);
    return x >= (T)i && (i + 2 == a.size() ? x <= (T)(i + 1) : x < (T)(i + 1));
}

template <class T>
size_t wrong(const std::vector<T> &got, const std::vector<T> &want)
{
    size_t n = 0;
    for (size_t i = 0; i < got.size(); i++)
        n += std::memcmp(&got[i], &want[i], sizeof(T)) != 0;
    return n;
}

int main(int argc, char **argv)
{
    std::FILE *f = argc > 1 ? std::fopen(argv[1], "rb") : nullptr;
    if (!f) return 2;
    int64_t head[2];
    while (std::fread(head, 8, 2, f) == 2) {
        std::vector<double> d((size_t)head[1]);
        if (std::fread(d.data(), 8, d.size(), f) != d.size()) return 2;
        const std::vector<float> a(d.begin(), d.end());
        std::vector<Pair> r;
        size_t bad_t, bad_r = 0;
        double out;
        if (head[0] == 32) {
            const std::vector<float> t = mr::thresholds32(a);
            bad_t = wrong(t, plain<float, uint32_t>(a, mr::key32, mr::unkey32));
            r = mr::fast_bounds<Pair>(a, &t, nullptr);
            out = mr::worst_outside(r, t);
        } else {
            const std::vector<double> t = mr::thresholds64(d);
            bad_t = wrong(t, plain<double, uint64_t>(d, mr::key64, mr::unkey64));
            r = mr::fast_bounds<Pair>(a, nullptr, &t);
            out = mr::worst_outside(r, t);
        }
        // (a spacing that overflows gives indexes without an order: nothing
        // runs on that one cell's region, whose share outside is 1)
        const bool order = std::isfinite(head[0] == 32 ? std::fabs(a[1] - a[0])
                                                       : std::fabs(d[1] - d[0]));
        for (size_t i = 0; order && i < r.size(); i++) {
            const float lo = r[i].x, hi = r[i].y;
            if (lo == -INFINITY && hi == -INFINITY) continue;
            bool ok = lo <= hi && !(a[i] >= lo && a[i] <= hi) && !(a[i + 1] >= lo && a[i + 1] <= hi);
            if (head[0] == 32) {
                ok = ok && in_cell(a, lo, i) && in_cell(a, hi, i);
            } else {
                // every f64 value that rounds to the bounds: the halfway points
                const double below = 0.5 * ((double)lo + (double)std::nextafter(lo, -INFINITY));
                const double above = 0.5 * ((double)hi + (double)std::nextafter(hi, INFINITY));
                ok = ok && in_cell(d, below, i) && in_cell(d, above, i);
            }
            bad_r += !ok;
        }
        std::printf("%zu %zu %.17g\n", bad_t, bad_r, out);
    }
    std::fclose(f);
    return 0;
}
