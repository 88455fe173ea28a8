// Host-side cache of requantisation threshold tables (see epilogue.h): one table per
// (activation, src scale, filter scale, dst scale), built on first use with the reference's
// literal float sequence evaluated by the host CPU - the same IEEE single-precision multiply,
// multiply, divide, roundf the generated C kernels execute - and kept for later calls (at most 4096 of them).
#include <math.h>

#include <algorithm>
#include <cstring>
#include <map>
#include <mutex>
#include <tuple>

#include "common.h"
#include "epilogue.h"

namespace mg {

// what has been worked out for (activation, scales): emptied when it is full, so that a process that meets ever new
// scales does not grow
template <typename T>
class ScaleCache {
public:
    static constexpr size_t MOST = 4096;
    typedef std::tuple<int, uint32_t, uint32_t, uint32_t> Key;
    static Key key(int act, float s_src, float s_flt, float s_dst) {
        auto bits = [](float f) {
            uint32_t u;
            memcpy(&u, &f, 4);
            return u;
        };
        return std::make_tuple(act, bits(s_src), bits(s_flt), bits(s_dst));
    }
    bool find(const Key& k, T* out) {
        std::lock_guard<std::mutex> guard(lock_);
        auto it = map_.find(k);
        if (it == map_.end())
            return false;
        *out = it->second;
        return true;
    }
    void put(const Key& k, const T& v) {
        std::lock_guard<std::mutex> guard(lock_);
        if (map_.size() >= MOST)
            map_.clear();
        map_[k] = v;
    }

private:
    std::mutex lock_;
    std::map<Key, T> map_;
};

// Entry by entry the largest accumulator whose output is still below j: a gallop and a bisection from the estimate,
// with the literal sequence up to the activation. Its rounding is a comparison here: roundf(x) < j iff x < j - 0.5,
// or x = j - 0.5 where the half goes away from zero to j - 1 (a NaN is below everything, as the conversion has it).
// 3 or 4 evaluations an entry. (A first launch with new scales waits for this and for the search below: over 60000
// scales 13 us -> 3.6 for the table and 8.6 -> 4.6 for the multiply-add's constants on one host core, against
// a call of the rounding function and a bisection from +-8 for each entry.)
template <int ACT>
static void requant_thresholds(float s_src, float s_flt, float s_dst, float c, int* t) {
    for (int i = 0; i < REQUANT_TABLE_ENTRIES - 1; ++i) {
        const int j = i - 127;
        const float edge = (float)j - 0.5f;
        auto below = [&](long long a) {
            const float x = act_apply<ACT>((float)(int)a * s_src * s_flt / s_dst);
            return j > 0 ? !(x >= edge) : !(x > edge);
        };
        if (!below(INT32_MIN)) {
            t[i] = INT32_MIN;  // F never drops below j: entry not used (j <= lowest output)
            continue;
        }
        float v = edge;
        if (ACT == MEGCC_NONLINE_H_SWISH && v > 0.f && v < 3.f)
            v = 0.5f * (sqrtf(9.f + 24.f * v) - 3.f);
        const float est = v / c;
        long long lo = INT32_MIN, hi = (long long)INT32_MAX + 1;  // F(lo) < j, F(hi) >= j (beyond the last: taken as such)
        if (est > -2.0e9f && est < 2.0e9f) {
            const long long e = (long long)est;
            long long step = 1;
            if (below(e)) {
                lo = e;
                while (lo + step < hi && below(lo + step)) {
                    lo += step;
                    step *= 2;
                }
                hi = std::min(hi, lo + step);
            } else {
                hi = e;
                while (hi - step > lo && !below(hi - step)) {
                    hi -= step;
                    step *= 2;
                }
                lo = std::max(lo, hi - step);
            }
        }
        while (hi - lo > 1) {
            const long long mid = lo + (hi - lo) / 2;
            if (below(mid))
                lo = mid;
            else
                hi = mid;
        }
        t[i] = (int)lo;
    }
    t[REQUANT_TABLE_ENTRIES - 1] = 0;
}

std::shared_ptr<const RequantTable> requant_table_for(int act, float s_src, float s_flt, float s_dst) {
    static ScaleCache<std::shared_ptr<const RequantTable>> cache;
    const auto key = cache.key(act, s_src, s_flt, s_dst);
    std::shared_ptr<const RequantTable> found;
    if (cache.find(key, &found))
        return found;
    const std::shared_ptr<RequantTable> t = std::make_shared<RequantTable>();
    const float c = make_requant_fast(s_src, s_flt, s_dst).c;
    if (act == MEGCC_NONLINE_RELU)
        requant_thresholds<MEGCC_NONLINE_RELU>(s_src, s_flt, s_dst, c, t->t);
    else if (act == MEGCC_NONLINE_H_SWISH)
        requant_thresholds<MEGCC_NONLINE_H_SWISH>(s_src, s_flt, s_dst, c, t->t);
    else
        requant_thresholds<MEGCC_NONLINE_IDENTITY>(s_src, s_flt, s_dst, c, t->t);
    cache.put(key, t);
    return t;
}

// Both sides of every step of F and the ends of the accumulator range, with the outputs there: F(T) is one less than the
// first level whose threshold is T, F(T + 1) the last such level.
struct RequantSteps {
    int n = 0;
    int a[2 * REQUANT_TABLE_ENTRIES + 2], y[2 * REQUANT_TABLE_ENTRIES + 2];
    void add(int acc, int out) {
        a[n] = acc;
        y[n++] = out;
    }
};
// (from the third point on) the first accumulator with its output, which bounds d from below - the last one with an output
// bounds it from above, and for no slope that is positive does the other bound of either count
static inline bool above_step(int i) {
    return i & 1;
}
static RequantSteps requant_steps(int act, float s_src, float s_flt, float s_dst) {
    const std::shared_ptr<const RequantTable> table = requant_table_for(act, s_src, s_flt, s_dst);
    const RequantTable& T = *table;
    const int lo = act == MEGCC_NONLINE_IDENTITY ? -128 : 0;
    RequantSteps s;
    int first = lo + 128;  // (levels up to the lowest output have no step)
    int low = lo, high = lo;  // outputs of the smallest and the largest accumulator
    while (first < REQUANT_TABLE_ENTRIES - 1 && T.t[first] == INT32_MIN)
        low = high = first++ - 127;
    for (int i = first; i < REQUANT_TABLE_ENTRIES - 1; ++i)
        if (T.t[i] < INT32_MAX)
            high = i - 127;
    s.add(INT32_MIN, low);
    s.add(INT32_MAX, high);
    for (int i = first; i < REQUANT_TABLE_ENTRIES - 1;) {
        int k = i;
        while (k + 1 < REQUANT_TABLE_ENTRIES - 1 && T.t[k + 1] == T.t[i])
            ++k;
        s.add(T.t[i], i - 128);
        if (T.t[i] < INT32_MAX)
            s.add(T.t[i] + 1, k - 127);
        i = k + 1;
    }
    return s;
}

// A search for constants, F, for processors with a fused multiply-add, where fmaf, rintf and floorf are an instruction each, and for
// the others, where they are calls of the library. All are exact: the results are the same.
// (us on one core for a launch's constants, table and all, scales of calibrated layers with 64 / 1152 / 4096 products to a sum: IDENTITY 9.5 /
// 12.8 / 13.8, RELU 4.9 / 12.2 / 13.8, H_SWISH 3.1 / 3.5 / 3.7; with both sides of a step in both hulls and the points one by one 11.2 / 16.1 /
// 16.7, 5.8 / 14.6 / 15.9 and 4.0 / 4.1 / 4.5.)
#define MG_INLINE __attribute__((always_inline))
#if defined(__HIP_DEVICE_COMPILE__)
#define MG_FMA
#else
#define MG_FMA __attribute__((target("avx2,fma")))
#endif
template <auto F>
MG_FMA static auto search_fma(int act, float s_src, float s_flt, float s_dst, const RequantSteps& pts) {
    return F(act, s_src, s_flt, s_dst, pts);
}
template <auto F>
static auto search(int act, float s_src, float s_flt, float s_dst, const RequantSteps& pts) {
#if !defined(__HIP_DEVICE_COMPILE__)
    static const bool fma = __builtin_cpu_supports("fma") && __builtin_cpu_supports("avx2");
    if (fma)
        return search_fma<F>(act, s_src, s_flt, s_dst, pts);
#endif
    return F(act, s_src, s_flt, s_dst, pts);
}

// Lower (or upper) bounds for d: at[i] - x[i] c <= d (>=), of which the largest (smallest) counts for a given c. Bounds come in
// the order of x, and those that are the tightest for no c at all are dropped as they come: what stays is one side of the
// points' convex hull, a dozen of 255, and a slope costs as many products. (All 255 kept, the searches below took 40 us.)
template <bool LOWER>
struct RequantBounds {
    int n = 0;
    double x[REQUANT_TABLE_ENTRIES], at[REQUANT_TABLE_ENTRIES];
    int point[REQUANT_TABLE_ENTRIES];  // which step's
    static bool tighter(double a, double b) { return LOWER ? a > b : a < b; }
    MG_INLINE void add(double v, double bound, int p) {
        if (n && x[n - 1] == v) {
            if (!tighter(bound, at[n - 1]))
                return;
            --n;
        }
        // (the last one is not beyond the line from the one before it to this one)
        while (n >= 2 && !tighter((at[n - 1] - at[n - 2]) * (v - x[n - 2]), (bound - at[n - 2]) * (x[n - 1] - x[n - 2])))
            --n;
        x[n] = v;
        at[n] = bound;
        point[n++] = p;
    }
    // (a hull: from the bound that was the tightest for another slope, downhill)
    MG_INLINE double tightest(double c) {
        if (!n)
            return LOWER ? -1e30 : 1e30;
        double m = at[best] - x[best] * c, v;
        for (; best + 1 < n && tighter(v = at[best + 1] - x[best + 1] * c, m); ++best)
            m = v;
        for (; best > 0 && tighter(v = at[best - 1] - x[best - 1] * c, m); --best)
            m = v;
        return m;
    }
    int best = 0;
};

// the float `n` floats above (a positive, normal) v
static float by_ulps(float v, int n) {
    uint32_t u;
    memcpy(&u, &v, 4);
    u += (uint32_t)n;
    memcpy(&v, &u, 4);
    return v;
}

// whether `eval` gives the outputs of every step: first where the bounds are tightest, where a wrong candidate shows
template <typename F>
MG_INLINE static bool requant_verified(const RequantSteps& pts, const RequantBounds<true>& from, const RequantBounds<false>& to, F eval) {
    for (int i = 0; i < from.n; ++i)
        if (eval(pts.a[from.point[i]]) != pts.y[from.point[i]])
            return false;
    for (int i = 0; i < to.n; ++i)
        if (eval(pts.a[to.point[i]]) != pts.y[to.point[i]])
            return false;
    int wrong = 0;  // (no way out of this loop: eight points at a time)
    for (int i = 0; i < pts.n; ++i)
        wrong |= eval(pts.a[i]) ^ pts.y[i];
    return !wrong;
}

// host evaluation of requant_conv_affine (fmaf is the correctly rounded single fused multiply-add,
// floorf + saturation what v_cvt_flr_i32_f32 does)
MG_INLINE static int affine_eval(int a, float c, float d, int lo) {
    const float g = floorf(fmaf((float)a, c, d));
    const float r = g < (float)lo ? (float)lo : (g > 127.f ? 127.f : g);
    return (int)r;
}

// from, to: y + up <= a c + d < y + 1 + up for an output y (another `up` moves the hulls as they are)
MG_INLINE static RequantAffine affine_within(
        const RequantSteps& pts, RequantBounds<true>& from, RequantBounds<false>& to, double up, int lo, float c0) {
    RequantAffine found = {0.f, 0.f};
    for (int k = 0; k <= 16 && found.d == 0.f; ++k) {
        // c' = c0 moved (k + 1) / 2 ulps up (k odd) or down (k even)
        const float c = by_ulps(c0, (k & 1) ? (k + 1) / 2 : -(k / 2));
        const double dlo = from.tightest((double)c) - up, dhi = to.tightest((double)c) - up;
        if (!(dlo < dhi))
            continue;
        // the middle of the interval first (the most room for the rounding of the fused multiply-add),
        // then points nearer its ends
        static const double kPos[] = {0.5, 0.375, 0.625, 0.25, 0.75};
        for (double pos : kPos) {
            const float d = (float)(dlo + (dhi - dlo) * pos);
            if (!(d > 0.f && d < 1.f))
                continue;
            if (requant_verified(pts, from, to, [&](int a) MG_INLINE { return affine_eval(a, c, d, lo); })) {
                found = {c, d};
                break;
            }
        }
    }
    return found;
}
MG_INLINE static RequantAffine affine_constants(int act, float s_src, float s_flt, float s_dst, const RequantSteps& pts) {
    const int lo = act == MEGCC_NONLINE_RELU ? 0 : -128;
    RequantBounds<true> from;  // floor(a c + d) == y  <=>  y <= a c + d < y + 1
    RequantBounds<false> to;
    for (int i = 2; i < pts.n; ++i) {  // (the ends of the range bound nothing)
        if (above_step(i))
            from.add((double)(float)pts.a[i], (double)pts.y[i], i);
        else
            to.add((double)(float)pts.a[i], (double)pts.y[i] + 1, i);
    }
    return affine_within(pts, from, to, 0., lo, make_requant_fast(s_src, s_flt, s_dst).c);
}

RequantAffine requant_affine_for(int act, float s_src, float s_flt, float s_dst) {
    static ScaleCache<RequantAffine> cache;
    const RequantAffine none = {0.f, 0.f};
    if ((act != MEGCC_NONLINE_IDENTITY && act != MEGCC_NONLINE_RELU) || !requant_table_ok(s_src, s_flt, s_dst))
        return none;
    const auto key = cache.key(act, s_src, s_flt, s_dst);
    RequantAffine found = none;
    if (cache.find(key, &found))
        return found;
    found = search<affine_constants>(act, s_src, s_flt, s_dst, requant_steps(act, s_src, s_flt, s_dst));
    cache.put(key, found);
    return found;
}

// host evaluation of requant_pack4 for one output
MG_INLINE static int pack_eval(int a, int act, const RequantPack& q) {
    float x = (float)a;
    if (q.mode == 5) {
        uint32_t u;
        memcpy(&u, &q.s1, 4);
        u += (uint32_t)a;
        memcpy(&x, &u, 4);
    }
    if (q.mode == 2 || q.mode == 3 || q.mode == 6)
        x = x * q.s1 * q.s2;
    float y;
    if (q.mode == 6) {
        const float t = truncf(fmaf(x, q.c, copysignf(q.d, x)));  // (v_cvt_i32_f32 truncates and saturates)
        return (int)std::min(std::max(t, -128.f), 127.f);
    }
    if (q.mode == 3) {
        float v = fmaf(x, q.c, x * q.d);
        if (act == MEGCC_NONLINE_IDENTITY) {
            const float t = truncf(v + copysignf(0x1.fffffep-2f, v));
            return (int)(t < -128.f ? -128.f : t > 127.f ? 127.f : t);
        }
        if (act == MEGCC_NONLINE_H_SWISH) {
            const float t = v + 3;
            v = v * std::min(std::max(t, 0.f), 6.f) * (2.f * (1.f / 6.f));
        }
        y = v + 0x1.fffffep-2f;
    } else {
        y = fmaf(x, q.c, q.d);
    }
    const float r = rintf(y);  // (round to nearest even: the host's default mode)
    const int u = r < 0.f ? 0 : r > 255.f ? 255 : (int)r;
    return act == MEGCC_NONLINE_IDENTITY ? u - 128 : u >> 1;
}

// Mode 6, or mode 0 where it has no constants. Of IDENTITY's steps those above zero and the one to -128: the others are their
// mirror images, here as in the reference (which is checked like the rest).
MG_INLINE static RequantPack pack_symmetric(const RequantSteps& pts, float s_src, float s_flt, float s_dst) {
    RequantBounds<true> from;  // trunc(x c + d) == y  <=>  y <= x c + d < y + 1
    RequantBounds<false> to;
    auto value = [&](int a) MG_INLINE { return std::fabs((double)((float)a * s_src * s_flt)); };
    for (int i = 2; i < pts.n; ++i) {
        if (above_step(i) && pts.y[i] > 0)
            from.add(value(pts.a[i]), (double)pts.y[i], i);
        if (!above_step(i) && pts.y[i] >= 0 && pts.a[i] >= 0)
            to.add(value(pts.a[i]), (double)pts.y[i] + 1, i);
    }
    for (int i = 2; i < pts.n; ++i) {
        if (pts.y[i] == -128)
            from.add(value(pts.a[i]), 128., i);
        if (pts.y[i] == -127 && pts.a[i - 1] == pts.a[i] - 1)
            to.add(value(pts.a[i]), 128., i);
    }
    const float c0 = 1.f / s_dst;
    for (int k = 0; k <= 8; ++k) {  // (up to 48: one scale in a hundred more)
        const float c = by_ulps(c0, (k & 1) ? (k + 1) / 2 : -(k / 2));
        const double dlo = from.tightest((double)c), dhi = to.tightest((double)c);
        if (!(dlo <= dhi))
            continue;
        static const double kPos[] = {0.5, 0.375, 0.625, 0.25, 0.75, 0.125, 0.875};
        for (double pos : kPos) {
            const RequantPack q = {s_src, s_flt, c, (float)(dlo + (dhi - dlo) * pos), 6};
            if (q.d >= 0.f && q.d < 1.f &&
                requant_verified(pts, from, to, [&](int a) MG_INLINE { return pack_eval(a, MEGCC_NONLINE_IDENTITY, q); }))
                return q;
        }
    }
    return {s_src, s_flt, s_dst, 0.f, 0};
}

// Mode 1, 2, 4 or 6, or mode 0 where none has constants.
MG_INLINE static RequantPack pack_affine(int act, float s_src, float s_flt, float s_dst, const RequantSteps& pts) {
    RequantPack found = {s_src, s_flt, s_dst, 0.f, 0};
    const bool relu = act == MEGCC_NONLINE_RELU;
    const int lowest = relu ? 0 : -128;
    // the forms in order of cost: no product in front, one, two (IDENTITY, whose outputs are rounded 128 away from zero, hardly
    // ever has constants for those where it has none without)
    struct Form {
        int mode;
        float s1, s2, c0;
    };
    const float unit = relu ? 2.f : 1.f;
    const Form forms[] = {{1, 1.f, 1.f, make_requant_fast(s_src, s_flt, s_dst).c * unit},
                          {2, s_src, 1.f, s_flt / s_dst * unit},
                          {2, s_src, s_flt, 1.f / s_dst * unit}};
    for (const Form& f : forms) {
        RequantBounds<true> from;  // RELU: 2 y <= rint <= 2 y + 1; IDENTITY: rint == y + 128
        RequantBounds<false> to;
        for (int i = 2; i < pts.n; ++i) {
            const double x = f.mode == 2 ? (float)pts.a[i] * f.s1 * f.s2 : (float)pts.a[i];
            const int y = pts.y[i];
            if (above_step(i))
                from.add(x, relu ? 2.0 * y - 0.5 : y + 127.5, i);
            else
                to.add(x, relu ? 2.0 * y + 1.5 : y + 128.5, i);
        }
        for (int k = 0; k <= 48 && !found.mode; ++k) {
            // c = c0 moved (k + 1) / 2 ulps up (k odd) or down (k even)
            const float c = by_ulps(f.c0, (k & 1) ? (k + 1) / 2 : -(k / 2));
            const double dlo = from.tightest((double)c), dhi = to.tightest((double)c);
            if (!(dlo <= dhi))
                continue;
            static const double kPos[] = {0.5, 0.375, 0.625, 0.25, 0.75, 0.125, 0.875};
            for (double pos : kPos) {
                const RequantPack q = {f.s1, f.s2, c, (float)(dlo + (dhi - dlo) * pos), f.mode};
                if (requant_verified(pts, from, to, [&](int a) MG_INLINE { return pack_eval(a, act, q); })) {
                    found = q;
                    break;
                }
            }
        }
        if (found.mode)
            break;
        if (!relu) {
            const RequantAffine a = affine_within(pts, from, to, 127.5, lowest, f.c0);
            if (a.d != 0.f)
                found = {0.f, 0.f, a.c, a.d, 4};
            else
                found = pack_symmetric(pts, s_src, s_flt, s_dst);
            break;
        }
    }
    return found;
}

// Mode 3, or mode 0 where it is not proven. The quotient it works with is at most one float from the reference's, so
// outputs can only differ where the reference's own value is within two of its floats of a step, 2 * 2^-17 for outputs up
// to 128: accumulators on both sides of each step are compared, and as many beyond them as lie within 1e-4 of it (with
// H_SWISH the output changes by half to one and a half of what the quotient does): 215 a step at the smallest ratios.
MG_INLINE static RequantPack pack_exact(int act, float s_src, float s_flt, float s_dst, const RequantSteps& pts) {
    const RequantPack none = {s_src, s_flt, s_dst, 0.f, 0};
    auto mid = [](float s) { return s >= 1e-12f && s <= 1e12f; };  // (nothing overflows or loses bits on the way)
    const float c = make_requant_fast(s_src, s_flt, s_dst).c;
    if (!mid(s_src) || !mid(s_flt) || !mid(s_dst) || !(c <= 1e12f))
        return none;
    const double inv = (act == MEGCC_NONLINE_RELU ? 2.0 : 1.0) / (double)s_dst;
    RequantPack q = {s_src, s_flt, (float)inv, 0.f, 3};
    q.d = (float)(inv - (double)q.c);
    const long long near = (long long)(1e-4f / c);
    if (near == 0) {  // (no other accumulator is that near to a step: the points alone, eight at a time)
        int wrong = 0;
        for (int i = 0; i < pts.n; ++i)
            wrong |= pack_eval(pts.a[i], act, q) ^ pts.y[i];
        return wrong ? none : q;
    }
    // (pts: the ends of the range, then each step's last accumulator below and first one above)
    for (int i = 0; i < pts.n; ++i) {
        const bool above = i >= 2 && pts.y[i] > pts.y[i - 1] && pts.a[i] == pts.a[i - 1] + 1;
        const long long from = i < 2 || above ? pts.a[i] : std::max<long long>(pts.a[i] - near, i > 2 ? pts.a[i - 1] : INT32_MIN);
        const long long to = i < 2 || !above ? pts.a[i] : std::min<long long>(pts.a[i] + near, i + 1 < pts.n ? pts.a[i + 1] : INT32_MAX);
        for (long long a = from; a <= to; ++a)
            if (pack_eval((int)a, act, q) != pts.y[i])
                return none;
    }
    return q;
}

// Mode 5: for each slope near the quotient the interval that mode 1's d may lie in, moved to where the sums' floats are; of the
// shifts m up to 1023 those whose d comes closest to its middle are verified.
MG_INLINE static RequantPack pack_shifted(int act, float s_src, float s_flt, float s_dst, const RequantSteps& pts) {
    const RequantPack none = {s_src, s_flt, s_dst, 0.f, 0};
    const bool relu = act == MEGCC_NONLINE_RELU;
    RequantBounds<true> from;
    RequantBounds<false> to;
    for (int i = 2; i < pts.n; ++i) {
        if (std::abs((long long)pts.a[i]) >= (1 << 22) - 1024)
            return none;
        const double x = pts.a[i];
        if (above_step(i))
            from.add(x, relu ? 2.0 * pts.y[i] - 0.5 : pts.y[i] + 127.5, i);
        else
            to.add(x, relu ? 2.0 * pts.y[i] + 1.5 : pts.y[i] + 128.5, i);
    }
    // (the outputs at the ends of the range are then those beyond the first and the last step; the ends themselves have no float)
    RequantSteps inner;
    for (int i = 2; i < pts.n; ++i)
        inner.add(pts.a[i], pts.y[i]);
    for (int i = 0; i < from.n; ++i)
        from.point[i] -= 2;
    for (int i = 0; i < to.n; ++i)
        to.point[i] -= 2;
    const float c0 = make_requant_fast(s_src, s_flt, s_dst).c * (relu ? 2.f : 1.f);
    for (int k = 0; k <= 48; ++k) {
        const float c = by_ulps(c0, (k & 1) ? (k + 1) / 2 : -(k / 2));
        const double dlo = from.tightest((double)c), dhi = to.tightest((double)c);
        if (!(dlo <= dhi))
            continue;
        const double middle = (dlo + dhi) / 2 - 12582912.0 * (double)c;
        struct {
            double off;
            int m;
        } best[2] = {{1e30, 0}, {1e30, 0}};
        for (int m = 0; m < 1024; ++m) {
            const double d = middle - (double)c * m;
            const double off = std::fabs((double)(float)d - d);
            if (off < best[1].off) {
                best[1] = {off, m};
                if (off < best[0].off)
                    std::swap(best[0], best[1]);
            }
        }
        for (const auto& b : best) {
            const int bits = 0x4b400000 + b.m;
            RequantPack q = {0.f, 0.f, c, (float)(middle - (double)c * b.m), 5};
            memcpy(&q.s1, &bits, 4);
            if (b.off <= (dhi - dlo) / 2 && requant_verified(inner, from, to, [&](int a) MG_INLINE { return pack_eval(a, act, q); }))
                return q;
        }
    }
    return none;
}

RequantPack requant_shifted_for(int act, float s_src, float s_flt, float s_dst) {
    static ScaleCache<RequantPack> cache;
    RequantPack found = {s_src, s_flt, s_dst, 0.f, 0};
    if ((act != MEGCC_NONLINE_IDENTITY && act != MEGCC_NONLINE_RELU) || !requant_table_ok(s_src, s_flt, s_dst))
        return found;
    const auto key = cache.key(act, s_src, s_flt, s_dst);
    if (!cache.find(key, &found)) {
        found = search<pack_shifted>(act, s_src, s_flt, s_dst, requant_steps(act, s_src, s_flt, s_dst));
        cache.put(key, found);
    }
    return found;
}

RequantPack requant_pack_for(int act, float s_src, float s_flt, float s_dst, bool affine) {
    static ScaleCache<RequantPack> multiply_adds, exact;
    if (!requant_table_act(act) || !requant_table_ok(s_src, s_flt, s_dst))
        return {s_src, s_flt, s_dst, 0.f, 0};
    const auto key = multiply_adds.key(act, s_src, s_flt, s_dst);
    RequantPack found;
    RequantSteps pts;
    if (affine && act != MEGCC_NONLINE_H_SWISH) {
        if (!multiply_adds.find(key, &found)) {
            pts = requant_steps(act, s_src, s_flt, s_dst);
            found = search<pack_affine>(act, s_src, s_flt, s_dst, pts);
            multiply_adds.put(key, found);
        }
        if (found.mode)
            return found;
    }
    if (!exact.find(key, &found)) {
        if (!pts.n)
            pts = requant_steps(act, s_src, s_flt, s_dst);
        found = search<pack_exact>(act, s_src, s_flt, s_dst, pts);
        exact.put(key, found);
    }
    return found;
}

RequantPack requant_started_for(int act, float s_src, float s_flt, float s_dst, bool affine) {
    if (affine) {
        RequantPack q = requant_shifted_for(act, s_src, s_flt, s_dst);
        if (q.mode)
            return q;
        q = requant_pack_for(act, s_src, s_flt, s_dst, true);
        if (q.mode != 1)
            return q;
        if (act == MEGCC_NONLINE_RELU)
            return {1.f, 1.f, q.c, q.d, 2};
        const RequantAffine a = requant_affine_for(act, s_src, s_flt, s_dst);
        if (a.d != 0.f)
            return {0.f, 0.f, a.c, a.d, 4};
    }
    return requant_pack_for(act, s_src, s_flt, s_dst, false);
}

RequantPack requant_pack_pick(int act, float s_src, float s_flt, float s_dst) {
    return requant_pack_for(act, s_src, s_flt, s_dst, !options().no_affine);
}

RequantAffine requant_affine_pick(bool table, int act, float s_src, float s_flt, float s_dst) {
    RequantAffine a = {0.f, 0.f};
    if (table && !options().no_affine)
        a = requant_affine_for(act, s_src, s_flt, s_dst);
    note_requant_affine(a.d != 0.f);
    return a;
}

}  // namespace mg
