// Host-side cache of requantisation threshold tables (see epilogue.h): one table per
// (activation, src scale, filter scale, dst scale), built on first use with the reference's
// literal float sequence evaluated by the host CPU - the same IEEE single-precision multiply,
// multiply, divide, roundf the generated C kernels execute - and kept for later calls (at most 4096 of them).
#include <math.h>

#include <cstring>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

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

RequantTable requant_table_for(int act, float s_src, float s_flt, float s_dst) {
    static ScaleCache<RequantTable> cache;
    const auto key = cache.key(act, s_src, s_flt, s_dst);
    RequantTable t;
    if (cache.find(key, &t))
        return t;
    const float c = make_requant_fast(s_src, s_flt, s_dst).c;
    for (int i = 0; i < REQUANT_TABLE_ENTRIES; ++i) {
        if (i == REQUANT_TABLE_ENTRIES - 1)
            t.t[i] = 0;
        else if (act == MEGCC_NONLINE_RELU)
            t.t[i] = requant_threshold<MEGCC_NONLINE_RELU>(i, s_src, s_flt, s_dst, c);
        else if (act == MEGCC_NONLINE_H_SWISH)
            t.t[i] = requant_threshold<MEGCC_NONLINE_H_SWISH>(i, s_src, s_flt, s_dst, c);
        else
            t.t[i] = requant_threshold<MEGCC_NONLINE_IDENTITY>(i, s_src, s_flt, s_dst, c);
    }
    cache.put(key, t);
    return t;
}

// host evaluation of requant_conv_affine (fmaf is the correctly rounded single fused multiply-add,
// floorf + saturation what v_cvt_flr_i32_f32 does)
static int affine_eval(int a, float c, float d, int lo) {
    const float g = floorf(fmaf((float)a, c, d));
    const float r = g < (float)lo ? (float)lo : (g > 127.f ? 127.f : g);
    return (int)r;
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
    const RequantTable T = requant_table_for(act, s_src, s_flt, s_dst);
    const int lo = act == MEGCC_NONLINE_RELU ? 0 : -128;
    auto literal = [&](int a) {
        return act == MEGCC_NONLINE_RELU ? requant_conv<MEGCC_NONLINE_RELU>(a, s_src, s_flt, s_dst)
                                         : requant_conv<MEGCC_NONLINE_IDENTITY>(a, s_src, s_flt, s_dst);
    };
    // both sides of every step of F, and the ends of the accumulator range
    struct Point {
        int a, y;
    };
    std::vector<Point> pts;
    pts.push_back({INT32_MIN, literal(INT32_MIN)});
    pts.push_back({INT32_MAX, literal(INT32_MAX)});
    for (int i = 0; i < REQUANT_TABLE_ENTRIES - 1; ++i) {
        const int t = T.t[i];
        if (t == INT32_MIN)
            continue;  // F never drops below this level
        pts.push_back({t, literal(t)});
        if (t < INT32_MAX)
            pts.push_back({t + 1, literal(t + 1)});
    }
    const float c0 = make_requant_fast(s_src, s_flt, s_dst).c;
    for (int k = 0; k <= 16 && found.d == 0.f; ++k) {
        // c' = c0 moved (k + 1) / 2 ulps up (k odd) or down (k even)
        float c = c0;
        for (int s = 0; s < (k + 1) / 2; ++s)
            c = nextafterf(c, (k & 1) ? INFINITY : 0.f);
        double dlo = -1e30, dhi = 1e30;  // floor(a c + d) == y  <=>  y <= a c + d < y + 1
        for (const Point& p : pts) {
            const double prod = (double)(float)p.a * (double)c;
            if (p.y > lo && (double)p.y - prod > dlo)
                dlo = (double)p.y - prod;
            if (p.y < 127 && (double)p.y + 1 - prod < dhi)
                dhi = (double)p.y + 1 - prod;
        }
        if (!(dlo < dhi))
            continue;
        // the middle of the interval first (the most room for the rounding of the fused multiply-add),
        // then points nearer its ends
        static const double kPos[] = {0.5, 0.375, 0.625, 0.25, 0.75};
        for (double pos : kPos) {
            const float d = (float)(dlo + (dhi - dlo) * pos);
            if (!(d > 0.f && d < 1.f))
                continue;
            bool ok = true;
            for (const Point& p : pts)
                if (affine_eval(p.a, c, d, lo) != p.y) {
                    ok = false;
                    break;
                }
            if (ok) {
                found = {c, d};
                break;
            }
        }
    }
    cache.put(key, found);
    return found;
}

// host evaluation of requant_pack4 for one output
static int pack_eval(int a, int act, const RequantPack& q) {
    float x = (float)a;
    if (q.mode == 2)
        x = x * q.s1 * q.s2;
    const float r = rintf(fmaf(x, q.c, q.d));  // (round to nearest even: the host's default mode)
    const int u = r < 0.f ? 0 : r > 255.f ? 255 : (int)r;
    return act == MEGCC_NONLINE_RELU ? u >> 1 : u - 128;
}

RequantPack requant_pack_for(int act, float s_src, float s_flt, float s_dst) {
    static ScaleCache<RequantPack> cache;
    const RequantPack none = {0.f, 0.f, 0.f, 0.f, 0};
    if ((act != MEGCC_NONLINE_IDENTITY && act != MEGCC_NONLINE_RELU) || !requant_table_ok(s_src, s_flt, s_dst) ||
        options().no_affine)
        return none;
    const auto key = cache.key(act, s_src, s_flt, s_dst);
    RequantPack found = none;
    if (cache.find(key, &found))
        return found;
    const RequantTable T = requant_table_for(act, s_src, s_flt, s_dst);
    const bool relu = act == MEGCC_NONLINE_RELU;
    auto literal = [&](int a) {
        return relu ? requant_conv<MEGCC_NONLINE_RELU>(a, s_src, s_flt, s_dst)
                    : requant_conv<MEGCC_NONLINE_IDENTITY>(a, s_src, s_flt, s_dst);
    };
    // both sides of every step of F, and the ends of the accumulator range
    struct Point {
        int a, y;
    };
    std::vector<Point> pts;
    pts.push_back({INT32_MIN, literal(INT32_MIN)});
    pts.push_back({INT32_MAX, literal(INT32_MAX)});
    for (int i = 0; i < REQUANT_TABLE_ENTRIES - 1; ++i) {
        const int t = T.t[i];
        if (t == INT32_MIN)
            continue;  // F never drops below this level
        pts.push_back({t, literal(t)});
        if (t < INT32_MAX)
            pts.push_back({t + 1, literal(t + 1)});
    }
    // the forms in order of cost: no product in front, one, two
    struct Form {
        int mode;
        float s1, s2, c0;
    };
    const float unit = relu ? 2.f : 1.f;
    const Form forms[] = {{1, 1.f, 1.f, make_requant_fast(s_src, s_flt, s_dst).c * unit},
                          {2, s_src, 1.f, s_flt / s_dst * unit},
                          {2, s_src, s_flt, 1.f / s_dst * unit}};
    std::vector<float> x(pts.size());
    for (const Form& f : forms) {
        for (size_t i = 0; i < pts.size(); ++i)
            x[i] = f.mode == 2 ? (float)pts[i].a * f.s1 * f.s2 : (float)pts[i].a;
        for (int k = 0; k <= 48 && !found.mode; ++k) {
            // c = c0 moved (k + 1) / 2 ulps up (k odd) or down (k even)
            float c = f.c0;
            for (int s = 0; s < (k + 1) / 2; ++s)
                c = nextafterf(c, (k & 1) ? INFINITY : 0.f);
            double dlo = -1e30, dhi = 1e30;
            for (size_t i = 0; i < pts.size(); ++i) {
                const double prod = (double)x[i] * (double)c;
                const int y = pts[i].y;
                // RELU: 2 y <= rint <= 2 y + 1; IDENTITY: rint == y + 128
                const double lo = relu ? 2.0 * y - 0.5 : y + 127.5, hi = relu ? 2.0 * y + 1.5 : y + 128.5;
                if (y > (relu ? 0 : -128) && lo - prod > dlo)
                    dlo = lo - prod;
                if (y < 127 && hi - prod < dhi)
                    dhi = hi - prod;
            }
            if (!(dlo <= dhi))
                continue;
            static const double kPos[] = {0.5, 0.375, 0.625, 0.25, 0.75, 0.125, 0.875};
            for (double pos : kPos) {
                const RequantPack q = {f.s1, f.s2, c, (float)(dlo + (dhi - dlo) * pos), f.mode};
                bool ok = true;
                for (size_t i = 0; i < pts.size() && ok; ++i)
                    ok = pack_eval(pts[i].a, act, q) == pts[i].y;
                if (ok) {
                    found = q;
                    break;
                }
            }
        }
        if (found.mode)
            break;
    }
    cache.put(key, found);
    return found;
}

RequantAffine requant_affine_pick(bool table, int act, float s_src, float s_flt, float s_dst) {
    RequantAffine a = {0.f, 0.f};
    if (table && !options().no_affine)
        a = requant_affine_for(act, s_src, s_flt, s_dst);
    note_requant_affine(a.d != 0.f);
    return a;
}

}  // namespace mg
