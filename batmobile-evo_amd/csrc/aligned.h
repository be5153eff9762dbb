// The per-path product of one edge in the frame whose polar axis y is the edge.
//
// T_p is equivariant, T_p(x, Y(u)) = D^T T_p(D x, Y(y)) with D the rotation that takes the
// edge's unit vector u to y, and Y(y) has only its m = 0 components, sqrt(2l + 1).  There a
// path (l1, l2, l3) joins component m of x to component m (l1 + l2 + l3 even) or -m (odd)
// of the result, with a coefficient of |m| alone up to the odd paths' sign: the 611
// coefficient terms, 256 products and 156 weightings of a pair become 85 + 72 multiply-adds
// and two rotations of 66 (Passaro and Zitnick, "Reducing SO(3) convolutions to SO(2) for
// efficient equivariant GNNs", ICML 2023).
//
// The rotations mix the components of a degree: an infinite weight of l3 > 0, or an infinite
// component of x, comes out NaN in every component of its degree.
//
// D = (tilt about x) (turn about y): with u = (s sin f, c, s cos f) the turn by f mixes
// components m and -m, the tilt by the angle of (c, s) the components m >= 0 and those
// m < 0 among themselves (kTilt).
#pragma once

#include "common.h"

namespace bmhip {

// Coefficient of path p in the aligned frame from component ma of l1 to mo of l_out.
constexpr float aligned_coef(int p, int mo, int ma) {
    constexpr float norm[4] = {1.0f, 1.7320508075688772f, 2.23606797749979f, 2.6457513110645907f};
    const int l1 = kPathL[p][0], l2 = kPathL[p][1], l3 = kPathL[p][2];
    for (int i = kPathEntry[p]; i < kPathEntry[p + 1]; ++i)
        if (kCG[i].b == l2 * l2 + l2 && kCG[i].a == l1 * l1 + l1 + ma &&
            kCG[i].o == l3 * l3 + l3 + mo)
            return kCG[i].c * norm[l2];
    return 0.0f;
}
constexpr bool aligned_even(int p) { return (kPathL[p][0] + kPathL[p][1] + kPathL[p][2]) % 2 == 0; }
constexpr int aligned_min(int a, int b) { return a < b ? a : b; }
constexpr bool aligned_near(float a, float b) { return a - b < 1e-5f && b - a < 1e-5f; }
constexpr bool aligned_structure() {
    for (int p = 0; p < kNumPaths; ++p)
        for (int mo = -kPathL[p][2]; mo <= kPathL[p][2]; ++mo)
            for (int ma = -kPathL[p][0]; ma <= kPathL[p][0]; ++ma) {
                const float c = aligned_coef(p, mo, ma);
                const bool joined = aligned_even(p) ? mo == ma : (mo == -ma && mo != 0);
                if (!joined && c != 0.0f) return false;
                if (joined && !aligned_near(c, (aligned_even(p) ? 1.0f : -1.0f) *
                                                   aligned_coef(p, -mo, -ma)))
                    return false;
            }
    return true;
}
static_assert(aligned_structure(), "a path joins m to m (even) or antisymmetrically to -m (odd)");

constexpr bool tilt_zero(int l, int i, int j) {
    for (int k = 0; k < 4; ++k)
        if (kTilt[l][i][j][k] != 0.0f) return false;
    return true;
}
// sign of entry (i, j) against (j, i)
constexpr float tilt_sign(int l, int i, int j) {
    for (int k = 0; k < 4; ++k)
        if (!aligned_near(kTilt[l][i][j][k], kTilt[l][j][i][k])) return -1.0f;
    return 1.0f;
}

// q = (cos f, sin f, c, s) of an edge: cos and sin of 1, 2, 3 f and the tilt's entries i <= j.
struct AlignedFrame {
    float cp[4], sp[4];
    float t[4][28];
};

__device__ __forceinline__ void aligned_frame(float cf, float sf, float c, float s,
                                              AlignedFrame& f) {
    f.cp[1] = cf;
    f.sp[1] = sf;
    f.cp[2] = cf * cf - sf * sf;
    f.sp[2] = 2.0f * cf * sf;
    f.cp[3] = f.cp[2] * cf - f.sp[2] * sf;
    f.sp[3] = f.sp[2] * cf + f.cp[2] * sf;
    const float cc = c * c, cs = c * s, ss = s * s;
    const float mono[4][4] = {{1.0f, 0, 0, 0}, {c, s, 0, 0}, {cc, cs, ss, 0},
                              {cc * c, cc * s, c * ss, ss * s}};
    static_for<4>([&](auto lc) {
        constexpr int l = decltype(lc)::value;
        static_for<2 * l + 1>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            static_for<j + 1>([&](auto ic) {
                constexpr int i = decltype(ic)::value, d = i >= l ? l : l - 1;
                float v = 0.0f;
                static_for<4>([&](auto kc) {
                    constexpr int k = decltype(kc)::value;
                    constexpr float w = kTilt[l][i][j][k];
                    if constexpr (w != 0.0f) v = fmaf(w, mono[d < 0 ? 0 : d][k], v);
                });
                f.t[l][j * (j + 1) / 2 + i] = v;
            });
        });
    });
}

// entry (i, j) of degree l times x, added to acc
template <int l, int i, int j>
__device__ __forceinline__ float tilt_fma(const AlignedFrame& f, float x, float acc) {
    if constexpr (i <= j) return fmaf(f.t[l][j * (j + 1) / 2 + i], x, acc);
    else if constexpr (tilt_sign(l, i, j) > 0.0f) return fmaf(f.t[l][i * (i + 1) / 2 + j], x, acc);
    else return fmaf(-f.t[l][i * (i + 1) / 2 + j], x, acc);
}

// o = D v
__device__ __forceinline__ void to_aligned(const AlignedFrame& f, const float* v, float* o) {
    o[0] = v[0];
    static_for<3>([&](auto lc) {
        constexpr int l = decltype(lc)::value + 1, a0 = l * l;
        float w[2 * l + 1];
        w[l] = v[a0 + l];
        static_for<l>([&](auto mc) {
            constexpr int m = decltype(mc)::value + 1;
            const float c = v[a0 + l + m], s = v[a0 + l - m];
            w[l + m] = fmaf(s, f.sp[m], c * f.cp[m]);
            w[l - m] = fmaf(-c, f.sp[m], s * f.cp[m]);
        });
        static_for<2 * l + 1>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            float acc = 0.0f;
            static_for<2 * l + 1>([&](auto jc) {
                constexpr int j = decltype(jc)::value;
                if constexpr (!tilt_zero(l, i, j)) acc = tilt_fma<l, i, j>(f, w[j], acc);
            });
            o[a0 + i] = acc;
        });
    });
}

// o = D^T v
__device__ __forceinline__ void from_aligned(const AlignedFrame& f, const float* v, float* o) {
    o[0] = v[0];
    static_for<3>([&](auto lc) {
        constexpr int l = decltype(lc)::value + 1, a0 = l * l;
        float w[2 * l + 1];
        static_for<2 * l + 1>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            float acc = 0.0f;
            static_for<2 * l + 1>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                if constexpr (!tilt_zero(l, i, j)) acc = tilt_fma<l, i, j>(f, v[a0 + i], acc);
            });
            w[j] = acc;
        });
        o[a0 + l] = w[l];
        static_for<l>([&](auto mc) {
            constexpr int m = decltype(mc)::value + 1;
            o[a0 + l + m] = fmaf(-w[l - m], f.sp[m], w[l + m] * f.cp[m]);
            o[a0 + l - m] = fmaf(w[l + m], f.sp[m], w[l - m] * f.cp[m]);
        });
    });
}

// The weights r_p of the paths between degrees l1 and l3, joined per |m|: e[m] couples m to
// m, d[m] couples -m of l1 to m of l3 (and m to -m with the other sign).
template <int l1, int l3>
__device__ __forceinline__ void aligned_weights(const float* r, float* e, float* d) {
    constexpr int M = aligned_min(l1, l3);
    static_for<M + 1>([&](auto mc) {
        constexpr int m = decltype(mc)::value;
        float ve = 0.0f, vd = 0.0f;
        static_for<kNumPaths>([&](auto pc) {
            constexpr int p = decltype(pc)::value;
            if constexpr (kPathL[p][0] == l1 && kPathL[p][2] == l3) {
                // (the coefficients named: as arguments they are looked up at run time)
                constexpr float ce = aligned_coef(p, m, m), cd = aligned_coef(p, m, -m);
                if constexpr (aligned_even(p)) ve = fmaf(ce, r[p], ve);
                else if constexpr (m > 0) vd = fmaf(cd, r[p], vd);
            }
        });
        e[m] = ve;
        d[m] = vd;
    });
}
constexpr bool aligned_has_odd(int l1, int l3) {
    for (int p = 0; p < kNumPaths; ++p)
        if (kPathL[p][0] == l1 && kPathL[p][2] == l3 && !aligned_even(p)) return true;
    return false;
}

// o (degree l3, at o[0]) += K x, K the weighted sum of the paths from degree l1
template <int l1, int l3>
__device__ __forceinline__ void aligned_apply(const float* e, const float* d, const float* x,
                                              float* o) {
    constexpr int M = aligned_min(l1, l3), a = l1 * l1 + l1;
    o[l3] = fmaf(e[0], x[a], o[l3]);
    static_for<M>([&](auto mc) {
        constexpr int m = decltype(mc)::value + 1;
        o[l3 + m] = fmaf(e[m], x[a + m], o[l3 + m]);
        o[l3 - m] = fmaf(e[m], x[a - m], o[l3 - m]);
        if constexpr (aligned_has_odd(l1, l3)) {
            o[l3 + m] = fmaf(d[m], x[a - m], o[l3 + m]);
            o[l3 - m] = fmaf(-d[m], x[a + m], o[l3 - m]);
        }
    });
}
// y (degree l1, in place) += K^T g (degree l3)
template <int l1, int l3>
__device__ __forceinline__ void aligned_apply_t(const float* e, const float* d, const float* g,
                                                float* y) {
    constexpr int M = aligned_min(l1, l3), a = l1 * l1 + l1, o = l3 * l3 + l3;
    y[a] = fmaf(e[0], g[o], y[a]);
    static_for<M>([&](auto mc) {
        constexpr int m = decltype(mc)::value + 1;
        y[a + m] = fmaf(e[m], g[o + m], y[a + m]);
        y[a - m] = fmaf(e[m], g[o - m], y[a - m]);
        if constexpr (aligned_has_odd(l1, l3)) {
            y[a - m] = fmaf(d[m], g[o + m], y[a - m]);
            y[a + m] = fmaf(-d[m], g[o - m], y[a + m]);
        }
    });
}

// Message of the pair: m[o] = sum_p r_p T_p(x, Y(u)).
__device__ __forceinline__ void aligned_message(const AlignedFrame& f, const float* x,
                                                const float* r, float* m) {
    float xt[16], mt[16];
    to_aligned(f, x, xt);
#pragma unroll
    for (int i = 0; i < 16; ++i) mt[i] = 0.0f;
    static_for<4>([&](auto l3c) {
        constexpr int l3 = decltype(l3c)::value;
        static_for<4>([&](auto l1c) {
            constexpr int l1 = decltype(l1c)::value;
            float e[4], d[4];
            aligned_weights<l1, l3>(r, e, d);
            aligned_apply<l1, l3>(e, d, xt, mt + l3 * l3);
        });
    });
    from_aligned(f, mt, m);
}

// With g the gradient of the message: the torques tx, tz about the aligned x and z (the
// derivative under a rotation of the edge, with K of the weights r), and gs = <g, K(s) x>.
//   t_k = <g, J_k K x> - <K^T g, J_k x>   (x and g in the aligned frame)
__device__ __forceinline__ void aligned_gradient(const AlignedFrame& f, const float* x,
                                                 const float* g, const float* r, const float* s,
                                                 float& tx, float& tz, float& gs) {
    float xt[16], gt[16], yt[16], t[2] = {0.0f, 0.0f};
    to_aligned(f, x, xt);
    to_aligned(f, g, gt);
#pragma unroll
    for (int i = 0; i < 16; ++i) yt[i] = 0.0f;
    gs = 0.0f;
    static_for<4>([&](auto l3c) {
        constexpr int l3 = decltype(l3c)::value, o0 = l3 * l3;
        float mt[2 * l3 + 1], st[2 * l3 + 1];
#pragma unroll
        for (int i = 0; i < 2 * l3 + 1; ++i) mt[i] = st[i] = 0.0f;
        static_for<4>([&](auto l1c) {
            constexpr int l1 = decltype(l1c)::value;
            float e[4], d[4];
            aligned_weights<l1, l3>(r, e, d);
            aligned_apply<l1, l3>(e, d, xt, mt);
            aligned_apply_t<l1, l3>(e, d, gt, yt);
            aligned_weights<l1, l3>(s, e, d);
            aligned_apply<l1, l3>(e, d, xt, st);
        });
#pragma unroll
        for (int i = 0; i < 2 * l3 + 1; ++i) gs = fmaf(gt[o0 + i], st[i], gs);
        static_for<kNumGen>([&](auto nc) {
            constexpr GenTerm J = kGen[decltype(nc)::value];
            if constexpr (J.i >= o0 && J.i < o0 + 2 * l3 + 1)
                t[J.axis] = fmaf(J.v, fmaf(gt[J.i], mt[J.j - o0], -gt[J.j] * mt[J.i - o0]), t[J.axis]);
        });
    });
    static_for<kNumGen>([&](auto nc) {
        constexpr GenTerm J = kGen[decltype(nc)::value];
        t[J.axis] = fmaf(-J.v, fmaf(yt[J.i], xt[J.j], -yt[J.j] * xt[J.i]), t[J.axis]);
    });
    tx = t[0];
    tz = t[1];
}

}  // namespace bmhip
