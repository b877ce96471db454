// shade.h -- pixel_shader_light_and_texture<pixel_shader_lights_phong,
// pixel_shader_texture_bilinear> for gfx950 (swegl/render/pixel_shaders.hpp,
// src/render/pixel_shaders.cpp), same float operation order as the CPU.
#pragma once
#include "core.h"

namespace sw {

// (float)pow((double)s, 32) (pixel_shaders.cpp:193): glibc's pow rounds
// s^32 to double, the store rounds that to float.  Five plain double
// squarings give s^32 within 31 double-rounding errors (relative 2^-48);
// when every value within 2^-46 of it rounds to the same float, that float
// is the answer.  Otherwise (values near a float rounding boundary) s^32 is
// recomputed in double-double by exact squarings (two-product through fma)
// and rounded once to double and then to float.
SW_HD float pow32(float s)
{
    double p = (double)s;
    p *= p;
    p *= p;
    p *= p;
    p *= p;
    p *= p;
    const float lo = (float)(p * (1.0 - 0x1p-46)), hi = (float)(p * (1.0 + 0x1p-46));
    if (lo == hi)
        return lo;
    double h = (double)s, l = 0.0;
    for (int i = 0; i < 5; i++) {
        double q = h * h;
        double e = fma(h, h, -q);
        e += 2.0 * h * l;
        double h2 = q + e;
        l = e - (h2 - q);
        h = h2;
    }
    return (float)(h + l);
}

struct Light4 { float x, y, z, I; };

// pixel_shader_lights_phong::shade (pixel_shaders.cpp:159-205).  The two
// quotients over a light's squared distance d2 share its reciprocal where
// div_rn holds: d2 and the intensity within [2^-40, 2^40], and the second
// numerator, which may be tiny, scaled by 2^64 (exact) and the quotient
// scaled back: exact again unless it is below the normal range, a band of
// s^32 that takes the plain division.
SW_D int32_t phong(f3 center, f3 normal, f3 cam, float ambient, f3 sun, float sun_I,
                   const Light4 *lights, int n_lights)
{
    f3 camv = normalize(cam - center);
    float fs = -dot(normal, sun);
    if (fs < 0.0f)
        fs = 0.0f;
    else
        fs *= sun_I;
    float acc = 0.0f;
    for (int i = 0; i < n_lights; i++) {
        const Light4 l = ro(lights)[i];
        f3 L = center - f3{l.x, l.y, l.z};
        const float d2 = L.x * L.x + L.y * L.y + L.z * L.z;
        const bool fast = d2 >= 0x1p-40f && d2 <= 0x1p40f && fabsf(l.I) >= 0x1p-40f && fabsf(l.I) <= 0x1p40f;
        float r2 = 0.0f, diffuse;
        if (fast) {
            r2 = rcp_rn(d2);
            diffuse = div_rn(l.I, d2, r2);
        } else {
            diffuse = l.I / d2;
        }
        if (diffuse < SW_DIFFUSE_CUT)
            continue;
        L = normalize_s(L, d2);
        float a = -dot(normal, L);
        if (a < 0.0f)
            continue;
        diffuse *= a;
        f3 R = L + normal * (a * 2.0f);
        float s = dot(R, camv);
        if (s > 0) {
            s = pow32(s);
            s = s * 32.0f / 2.0f;
            const float q = div_rn(s * 0x1p64f, d2, r2);
            if (fast && s <= 0x1p10f && (q >= 0x1p-62f || s == 0.0f))
                s = q * 0x1p-64f;
            else
                s = s / d2;
            acc += diffuse + s;
        } else {
            acc += diffuse;
        }
    }
    return cvtt(65536.0f * (ambient + fs + acc));
}

// pixel_shader_texture_bilinear::shade (pixel_shaders.cpp:348-384).  The
// reference reads outside the bitmap for coordinates that wrap to a negative
// index (UB); here such a tap is clamped and counted.
// (x + m) % m with the reference's wrapping add and C remainder: x itself
// when it lies in [0, m) already (no division: the common case of
// coordinates inside the texture), a mask when m is a power of two.
SW_D int wrap_mod(int x, int m)
{
    if ((uint32_t)x < (uint32_t)m)
        return x;
    const int s = wrap_add(x, m);
    if (s >= 0 && (m & (m - 1)) == 0)
        return s & (m - 1);
    return s % m;
}

// A texture as the shaders read it: w x h texels at p, or, with p null, the
// 1x1 texture holding the material colour (pixel_shaders.cpp:288-302).
// Keeping that colour by value (not behind a pointer to a local) keeps the
// kernels free of private memory.
struct TexView {
    const uint32_t *p;
    uint32_t one;
    int w, h;
};
SW_D uint32_t texel(const TexView &X, int64_t i) { return X.p ? ro(X.p)[i] : X.one; }

struct Texel2 { uint32_t x, y; };   // two neighbours, aligned as one

// The four texels and weights of one bilinear sample.
struct BilTaps {
    uint32_t p[4];
    float w[4];
};

SW_D BilTaps bilinear_taps(const TexView &X, f2 t, uint32_t &oob)
{
    const int tw = X.w, th = X.h;
    float v = t.x;
    float u = t.y;
    // (float)((double)u - 0.5), float minus double literal stored to float,
    // equals the float operation u - 0.5f: the double difference is exact
    // whenever |u| >= 2^-30, and below that both round to -0.5 (or +0.5).
    float u1 = u - 0.5f;
    float u2 = u + 0.5f;
    float v1 = v - 0.5f;
    float v2 = v + 0.5f;
    u = floorf(u2);
    v = floorf(v2);
    int v1m = wrap_mod(cvtt(v1), th);
    int v2m = v1m + 1;
    if (v2m == th)
        v2m = 0;
    const int u1m = wrap_mod(cvtt(u1), tw);
    int u2m = u1m + 1;
    if (u2m == tw)
        u2m = 0;
    BilTaps T;
    if ((v1m | u1m) >= 0 && (tw | th) < 32768) {
        // both taps of either axis inside the bitmap, and products of 30
        // bits at most: 24-bit multiplies and 32-bit indices
        const uint32_t r1 = __umul24((uint32_t)v1m, (uint32_t)tw), r2 = __umul24((uint32_t)v2m, (uint32_t)tw);
        T.p[0] = T.p[1] = T.p[2] = T.p[3] = X.one;
        if (X.p) {
            // the taps of a row are neighbours unless the second wraps
            const uint32_t i0 = r1 + (uint32_t)u1m, i1 = r2 + (uint32_t)u1m;
            if (u2m) {
                const Texel2 a = *(const SW_RO Texel2 *)(ro(X.p) + i0), b = *(const SW_RO Texel2 *)(ro(X.p) + i1);
                T.p[0] = a.x;
                T.p[2] = a.y;
                T.p[1] = b.x;
                T.p[3] = b.y;
            } else {
                T.p[0] = ro(X.p)[i0];
                T.p[1] = ro(X.p)[i1];
                T.p[2] = ro(X.p)[r1];
                T.p[3] = ro(X.p)[r2];
            }
        }
    } else {
        const int64_t lim = (int64_t)tw * th;
        v1m *= tw;
        v2m *= tw;
        int64_t idx[4] = {(int64_t)v1m + u1m, (int64_t)v2m + u1m, (int64_t)v1m + u2m,
                          (int64_t)v2m + u2m};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            int64_t i = idx[k];
            if (i < 0 || i >= lim) {
                oob++;
                i = i < 0 ? 0 : lim - 1;
            }
            T.p[k] = texel(X, i);
        }
    }
    T.w[0] = (u - u1) * (v - v1);
    T.w[1] = (u - u1) * (v2 - v);
    T.w[2] = (u2 - u) * (v - v1);
    T.w[3] = (u2 - u) * (v2 - v);
    return T;
}

// Channel c (0 b, 1 g, 2 r, 3 alpha) of a bilinear sample.
SW_D uint32_t bilinear_channel(const BilTaps &T, int c)
{
    float a = (float)((T.p[0] >> (8 * c)) & 0xFF) * T.w[0];
    float b = (float)((T.p[1] >> (8 * c)) & 0xFF) * T.w[1];
    float d = (float)((T.p[2] >> (8 * c)) & 0xFF) * T.w[2];
    float e = (float)((T.p[3] >> (8 * c)) & 0xFF) * T.w[3];
    const float s = ((a + b) + d) + e;
    // roundf (halves away from zero) and the conversion to a byte through a
    // 32-bit int: s is never negative (the weights are not), so it is the
    // integer part, plus one when the fraction, exact, reaches a half; NaN
    // gives 0 as the conversion does
    const float f = floorf(s);
    return ((uint32_t)(int32_t)f + (s - f >= 0.5f ? 1u : 0u)) & 0xFFu;
}

SW_D uint32_t bilinear(const TexView &X, f2 t, uint32_t &oob)
{
    const BilTaps T = bilinear_taps(X, t, oob);
    uint32_t out = 0;
#pragma unroll
    for (int c = 0; c < 4; c++)
        out |= bilinear_channel(T, c) << (8 * c);
    return out;
}

// pixel_shader_texture::shade (pixel_shaders.cpp:275-281): twidth and
// theight are unsigned there, so (int)t % twidth is the unsigned remainder
// of the int's bits, always inside the bitmap; column from t.x, row from t.y.
SW_D uint32_t nearest(const TexView &X, f2 t)
{
    const uint32_t tw = (uint32_t)X.w, th = (uint32_t)X.h;
    const uint32_t x = (uint32_t)cvtt(t.x), y = (uint32_t)cvtt(t.y);
    const uint32_t u = (tw & (tw - 1)) == 0 ? x & (tw - 1) : x % tw;
    const uint32_t v = (th & (th - 1)) == 0 ? y & (th - 1) : y % th;
    return texel(X, v * tw + u);
}

// pixel_shader_lights_flat::prepare_for_triangle (pixel_shaders.cpp:33-84),
// returned by shade as int: the face normal normal_t(cross(e1, e2)) is
// normalised once, and again when negated for an inverted triangle (unary
// minus builds a normal_t, points.hpp:171-174); the light is evaluated at
// the centroid ((v0 + v1) + v2) / 3 exactly as Phong evaluates a pixel.
SW_D int32_t flat_light(f3 w0, f3 w1, f3 w2, bool inverted, f3 cam, float ambient, f3 sun, float sun_I,
                        const Light4 *lights, int n_lights)
{
    const f3 e1 = w1 - w0, e2 = w2 - w0;
    f3 nrm = normalize({e1.y * e2.z - e1.z * e2.y, e1.z * e2.x - e1.x * e2.z, e1.x * e2.y - e1.y * e2.x});
    if (inverted)
        nrm = normalize(neg(nrm));
    const f3 s = (w0 + w1) + w2;
    const f3 center = {s.x / 3.0f, s.y / 3.0f, s.z / 3.0f};
    return phong(center, nrm, cam, ambient, sun, sun_I, lights, n_lights);
}

// pixel_shader_light_and_texture::shade combine (pixel_shaders.hpp:159-178)
SW_D uint32_t combine(uint32_t color, int32_t light_i)
{
    // (float)((double)light_i / 65536.0): the double quotient is exact (a
    // power-of-two scale of an int), so this is the int rounded to float and
    // scaled by 2^-16, which the float operations below reproduce exactly.
    float light = (float)light_i * 0x1p-16f;
    uint32_t out = color & 0xFF000000u;
    // Conversions to int need no range check here: |c * light| < 2^24 (light
    // is an int32 over 2^16), and the quotients below lie in [0, 255].
    if (light < 1) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            uint32_t c = (color >> (8 * k)) & 0xFF;
            out |= ((uint32_t)(int32_t)((float)c * light) & 0xFFu) << (8 * k);
        }
    } else {
        light = sqrt_rn(light);   // 1 <= light <= 32768
        light = sqrt_rn(light);
        const FDiv by_light(light);
#pragma unroll
        for (int k = 0; k < 3; k++) {
            uint32_t c = (color >> (8 * k)) & 0xFF;
            out |= (255u - (uint32_t)(int32_t)by_light((float)(255 - (int)c))) << (8 * k);
        }
    }
    return out;
}

// One quantity over a scanline (prepare_for_triangle / _upper / _lower /
// _scanline, pixel_shaders.cpp:88-158 and :304-346): a0, a1, a2 at the
// y-sorted vertices.  The long side runs from vertex 0 to 2, the short one
// from 0 to 1 in the upper half and 1 to 2 in the lower; the left end lies on
// the short side when the long one is on the right (lr).  The reference's
// left + (right - left) * u is `base` + `d` * (lr ? -u : u) here: d is the
// short end minus the long one, and negation is exact.
struct RowEnds {
    bool lower, lr;
    float ps, pL;   // progresses along the short and the long side
    SW_D RowEnds(bool lower_, bool lr_, float pl, float pr)
        : lower(lower_), lr(lr_), ps(lr_ ? pl : pr), pL(lr_ ? pr : pl)
    {
    }
    SW_D float along(float u) const { return lr ? -u : u; }
};
struct RowVal {
    float base, d;
    SW_D RowVal() {}
    SW_D RowVal(const RowEnds &E, float a0, float a1, float a2)
    {
        const float s0 = E.lower ? a1 : a0, s1 = E.lower ? a2 : a1;
        const float s = s0 + (s1 - s0) * E.ps, l = a0 + (a2 - a0) * E.pL;
        base = E.lr ? s : l;
        d = s - l;
    }
    SW_D float at(float su) const { return base + d * su; }
};

}  // namespace sw
