// eval3d compositing kernels (reference csrc/rasterization/eval3d_{fwd,bwd}.cu, eval3d_dynamic_*.cu).
//
// One workgroup per (camera, tile). The tile's pixels form strips of 64 consecutive ones (row-major); a
// wavefront owns one or more whole strips, one pixel of each per lane. Gaussians of the tile's depth-sorted
// list are staged in LDS in batches. Where all rays of a tile start at one origin and run within 84 degrees of the
// middle one, the tile is swept in a turned frame and affine ray coordinates (below; a block vote decides, and the
// tiles of a static pinhole, fisheye or spherical camera pass unless they span half the sphere); else with the rows
// of M = S^-1 R^T, as the reference does per pair. Pixels without such a ray (masked ones, say) do not hold the
// others back: they are swept by themselves, a second time through the list, in the second form.
#pragma once
#include "xsg_common.h"

namespace xsg {

constexpr int kTileThreads = 256;
constexpr int kMaxTilePixels = 1024;  // largest tile: the reference's 1024-thread workgroup limit
constexpr int kBwdNoRayCdim = 16;    // backward: channels up to which per-pixel ray gradients can be left out
constexpr int kBwdColorLdsMax = 33;  // backward: channels staged in LDS; larger CDIM read from HBM

// The backward's variants of one group are compiled in one translation unit (eval3d_bwd_g<k>.hip).
#define XSG_CDIM_GROUP0(X) X(0) X(1) X(2) X(3) X(4) X(5)
#define XSG_CDIM_GROUP1(X) X(8) X(9) X(16) X(17)
#define XSG_CDIM_GROUP2(X) X(32) X(33)
#define XSG_CDIM_GROUP3(X) X(64) X(65)
#define XSG_CDIM_GROUP4(X) X(128) X(129)
#define XSG_CDIM_GROUP5(X) X(256) X(257)
#define XSG_CDIM_GROUP6(X) X(512)
#define XSG_CDIM_GROUP7(X) X(513)
#define XSG_CDIM_LIST(X)                                                                                \
    XSG_CDIM_GROUP0(X) XSG_CDIM_GROUP1(X) XSG_CDIM_GROUP2(X) XSG_CDIM_GROUP3(X) XSG_CDIM_GROUP4(X) \
    XSG_CDIM_GROUP5(X) XSG_CDIM_GROUP6(X) XSG_CDIM_GROUP7(X)

struct TileGrid {
    int width, height, tile_w, tile_h, n_tiles_w, n_tiles_h, n_cams;
    int64_t n;          // Gaussians (flatten id = cam * n + gaussian)
    int64_t n_isects;
};

// A tile of a grid larger than the image that has no pixel: its first one, from which a tile's set-up reads
// rays and times, is past the image (the whole workgroup agrees).
XSG_DEV bool past_image(const TileGrid& g, int trow, int tcol) {
    return (int64_t)trow * g.tile_h >= g.height || (int64_t)tcol * g.tile_w >= g.width;
}

// Rows of M = S^-1 R^T from the raw quaternion (w, x, y, z) and activated scales: row i is column i
// of R / s_i (utils.h:61-83 and eval3d_fwd.cu:92-107). Explicit roundings: see Turn.
XSG_DEV void iscl_rot_rows(float4 q, f3 s, f3& r0, f3& r1, f3& r2) {
    float w = q.x, x = q.y, y = q.z, z = q.w;
    const float inv = rsqrtf(fmaf(w, w, fmaf(z, z, fmaf(y, y, x * x))));
    x *= inv; y *= inv; z *= inv; w *= inv;
    const float yz2 = fmaf(y, y, z * z), xz2 = fmaf(x, x, z * z), xy2 = fmaf(x, x, y * y), wx = w * x, wy = w * y, wz = w * z;
    const float i0 = 1.0f / s.x, i1 = 1.0f / s.y, i2 = 1.0f / s.z;
    r0 = mk3(i0 * fmaf(-2.f, yz2, 1.f), i0 * (2.f * fmaf(x, y, wz)), i0 * (2.f * fmaf(x, z, -wy)));
    r1 = mk3(i1 * (2.f * fmaf(x, y, -wz)), i1 * fmaf(-2.f, xz2, 1.f), i1 * (2.f * fmaf(y, z, wx)));
    r2 = mk3(i2 * (2.f * fmaf(x, z, wy)), i2 * (2.f * fmaf(y, z, -wx)), i2 * fmaf(-2.f, xy2, 1.f));
}

XSG_DEV f3 sel3(bool c, f3 a, f3 b) { return mk3(c ? a.x : b.x, c ? a.y : b.y, c ? a.z : b.z); }
XSG_DEV f3 rows_mul(f3 r0, f3 r1, f3 r2, f3 v) { return mk3(dot(r0, v), dot(r1, v), dot(r2, v)); }
XSG_DEV f3 rows_tmul(f3 r0, f3 r1, f3 r2, f3 v) {  // M^T v
    return mk3(r0.x * v.x + r1.x * v.y + r2.x * v.z, r0.y * v.x + r1.y * v.y + r2.y * v.z,
               r0.z * v.x + r1.z * v.y + r2.z * v.z);
}

// Hides a value's origin from the optimiser (which would turn sign masks back into compares and selects,
// at twice the issue cycles of the integer operations).
XSG_DEV int32_t opaque(int32_t v) {
    asm("" : "+v"(v));
    return v;
}

// Reductions over a full wavefront by DPP moves (rows of 16 lanes, then row 0's and rows 0-1's last lanes
// broadcast up), whose result lane 63 holds and every lane returns: a lane exchange through the LDS unit
// (__shfl_xor) takes some twenty times a DPP move's latency, and a tile's set-up is a chain of nine
// reductions.
template <class F>
XSG_DEV float wave_reduce_f(float v, float identity, F&& f) {
#define XSG_STEP(CTRL, ROWS)                                                                            \
    v = f(v, __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(identity), __float_as_int(v), CTRL, ROWS, 0xF, false)))
    XSG_STEP(0x111, 0xF);  // row_shr:1
    XSG_STEP(0x112, 0xF);  // row_shr:2
    XSG_STEP(0x114, 0xF);  // row_shr:4
    XSG_STEP(0x118, 0xF);  // row_shr:8
    XSG_STEP(0x142, 0xA);  // row_bcast:15 into rows 1 and 3
    XSG_STEP(0x143, 0xC);  // row_bcast:31 into rows 2 and 3
#undef XSG_STEP
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
XSG_DEV float wave_max_f(float v) {
    return wave_reduce_f(v, -__builtin_inff(), [](float a, float b) { return fmaxf(a, b); });
}
XSG_DEV float wave_min_f(float v) {
    return wave_reduce_f(v, __builtin_inff(), [](float a, float b) { return fminf(a, b); });
}
// A wave-uniform 64-bit value read from LDS, moved to scalar registers (readfirstlane is signed:
// each half goes through uint32_t so that the low half is not sign-extended).
XSG_DEV uint64_t uniform_u64(uint64_t v) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}
XSG_DEV float uniform_f(float v) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))); }
XSG_DEV bool finite3(f3 v) { return isfinite(v.x) && isfinite(v.y) && isfinite(v.z); }

// ---------------------------------------------------------------------------------------------
// Tiles whose rays share one origin and run within 84 degrees of an axis (every tile of a camera without a
// rolling shutter): two changes of variables make a pair cheap.
//
// 1. The frame of a Gaussian is turned until gro = M (o - mu) is (0, 0, D). Everything a pair computes
//    depends on the normalised Gaussian only up to a rotation of its frame, and with t1, t2, u the turned
//    rows of M and d the ray,
//      grd = (t1.d, t2.d, u.d),  |grd x gro|^2 = D^2 ((t1.d)^2 + (t2.d)^2),  gro.grd = D u.d,
//    and the Gaussian's offset from the ray, gro + hit_t grd, is (hit_t t1.d, hit_t t2.d, D tt / |grd|^2).
//    The turn is the Householder reflection that sends gro to the axis of its largest component (so that
//    nothing cancels).
// 2. The tile's rays are d = k (A + x X + y Y) in an orthonormal basis whose A is the tile's middle ray
//    (basis_pixel), so that t1.d / k and the others are affine in the pixel's (x, y): two FMAs each. Power and
//    alpha do not depend on k; hit_t is 1 / k times what A + x X + y Y gives.
// A pair's alpha then takes 14 FMA-rate instructions instead of 27, its backward 8 fewer again.
//
// What float32 would lose is the small difference t.A of a Gaussian near the tile's middle ray, an error of
// the ray's distance from the Gaussian of about an ulp of |gro|, as with the cross product: t.A, the pixel's
// (x, y) and D are therefore summed in float64 (once per Gaussian and tile, or pixel), t.A with the
// residual of t.(o - mu), which the turn leaves at rounding, taken out. Measured over Gaussians of
// exp(-3 +- 0.7) at 2 to 80 from the origin, the root mean square error of exp(-d^2 / 2) is 1.0e-7,
// against 9.7e-6 with the cross product in float32.
struct d3 {
    double x, y, z;
};
XSG_DEV double dot64(d3 a, d3 b) { return fma(a.x, b.x, fma(a.y, b.y, a.z * b.z)); }
XSG_DEV d3 to64(f3 a) { return d3{(double)a.x, (double)a.y, (double)a.z}; }
XSG_DEV f3 to32(d3 a) { return mk3((float)a.x, (float)a.y, (float)a.z); }
XSG_DEV d3 mul64(d3 a, double s) { return d3{a.x * s, a.y * s, a.z * s}; }
// 1 / sqrt and 1 / of ordinary float64 numbers: the float32 instruction and two Newton steps
XSG_DEV double rsqrt64(double v) {
    double r = (double)__builtin_amdgcn_rsqf((float)v);
    r = r * fma(-0.5 * v * r, r, 1.5);
    return r * fma(-0.5 * v * r, r, 1.5);
}
XSG_DEV double rcp64(double v) {
    double r = (double)__builtin_amdgcn_rcpf((float)v);
    r = r * fma(-v, r, 2.0);
    return r * fma(-v, r, 2.0);
}
XSG_DEV bool regular_ray(f3 d) {
    const float l = dot(d, d);
    return l >= 1e-12f && l <= 1e12f;
}

struct TileBasis {
    d3 a, x, y;
};
// mid: the tile's middle ray, side: the ray at the left end of its row
XSG_DEV TileBasis tile_basis(f3 mid, f3 side) {
    TileBasis b;
    const d3 m = to64(mid), s = to64(side);
    b.a = mul64(m, rsqrt64(dot64(m, m)));
    const double sa = dot64(s, b.a);
    d3 e = d3{fma(-sa, b.a.x, s.x), fma(-sa, b.a.y, s.y), fma(-sa, b.a.z, s.z)};
    if (!(dot64(e, e) > 1e-10 * dot64(s, s))) {  // no direction of its own: any perpendicular one
        const bool fx = fabs(b.a.x) < 0.6;
        e = d3{fx ? 1.0 - b.a.x * b.a.x : -b.a.x * b.a.y, fx ? -b.a.x * b.a.y : 1.0 - b.a.y * b.a.y,
               fx ? -b.a.x * b.a.z : -b.a.y * b.a.z};
    }
    b.x = mul64(e, rsqrt64(dot64(e, e)));
    b.y = d3{fma(b.a.y, b.x.z, -b.a.z * b.x.y), fma(b.a.z, b.x.x, -b.a.x * b.x.z), fma(b.a.x, b.x.y, -b.a.y * b.x.x)};
    return b;
}

XSG_DEV double uniform_d(double v) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)), __builtin_amdgcn_readfirstlane(__double2loint(v)));
}
XSG_DEV d3 uniform_d3(d3 v) { return d3{uniform_d(v.x), uniform_d(v.y), uniform_d(v.z)}; }
XSG_DEV TileBasis uniform_basis(TileBasis b) { return TileBasis{uniform_d3(b.a), uniform_d3(b.x), uniform_d3(b.y)}; }

// What staging a Gaussian needs of the tile, kept in LDS between batches (as scalars it would cost the pair
// loops eighteen registers and their spills).
struct TileFrame {
    double basis[9];
    float hx, hy, slack_o, slack_t;
};
XSG_DEV void put_basis(TileFrame& f, const TileBasis& b) {
    f.basis[0] = b.a.x; f.basis[1] = b.a.y; f.basis[2] = b.a.z;
    f.basis[3] = b.x.x; f.basis[4] = b.x.y; f.basis[5] = b.x.z;
    f.basis[6] = b.y.x; f.basis[7] = b.y.y; f.basis[8] = b.y.z;
}
XSG_DEV TileBasis get_basis(const TileFrame& f) {
    const double* b = f.basis + opaque(0);
    return TileBasis{d3{b[0], b[1], b[2]}, d3{b[3], b[4], b[5]}, d3{b[6], b[7], b[8]}};
}
XSG_DEV f3 uniform3(f3 v) { return mk3(uniform_f(v.x), uniform_f(v.y), uniform_f(v.z)); }

// The pixel a tile's basis is built on, and whose origin and time its pixels count theirs from: the middle one
// (pix) or, where that has no ray (a masked pixel), the tile's first one that has. pixel_at(q) is the image index
// of the tile's q-th pixel, -1 outside; every wavefront looks for itself, with all of its lanes. A tile without
// any such pixel counts from 0 (what is no number must not reach the other pixels).
struct BasisPixel {
    int64_t pix;
    f3 o, d;
    float t;
};
template <bool DYN, class PixelAt>
XSG_DEV BasisPixel basis_pixel(const float* ray_o, const float* ray_d, const float* rtd, int64_t pix, int n_pixels,
                               PixelAt&& pixel_at) {
    BasisPixel b;
    auto load = [&](int64_t at) {
        b.pix = at;
        b.o = ld3(ray_o + 3 * at);
        b.d = ld3(ray_d + 3 * at);
        b.t = 0.f;
        if constexpr (DYN) b.t = rtd ? rtd[at] : 0.f;
        return regular_ray(b.d) && finite3(b.o) && isfinite(b.t);
    };
    if (!load(pix)) {
        for (int q = 0; q < n_pixels; q += 64) {
            const int64_t at = pixel_at(q + (int)__lane_id());
            const uint64_t m = __ballot(at >= 0 && load(at));
            if (m == 0) continue;
            pix = (int64_t)__shfl((long long)at, (int)__builtin_ctzll(m), 64);
            break;
        }
        load(pix);
    }
    b.o = uniform3(finite3(b.o) ? b.o : mk3(0.f, 0.f, 0.f));
    b.t = uniform_f(isfinite(b.t) ? b.t : 0.f);
    return b;
}

// A pixel's (x, y) and 1 / k; false where the ray does not run within 84 degrees of the axis.
XSG_DEV bool ray_xy(const TileBasis& b, f3 d, float& x, float& y, float& inv_k) {
    const d3 v = to64(d);
    const double k = dot64(v, b.a), r = rcp64(k);
    x = (float)(dot64(v, b.x) * r);
    y = (float)(dot64(v, b.y) * r);
    inv_k = (float)r;
    return regular_ray(d) && k > 0.0 && k * k > 0.01 * dot64(v, v);
}

// The box of (x, y) that the rays of a strip's 64 pixels fill: centre and half extents (hx < 0: no pixel has a
// ray). A pixel whose ray gives no (x, y), or is none at all, is a bare one: it is in no box, any Gaussian may reach
// it, and its strip is kept whole where it is evaluated.
XSG_DEV float4 strip_box(bool ray, float x, float y) {
    const float big = __builtin_inff();
    const float x0 = wave_min_f(ray ? x : big), x1 = wave_max_f(ray ? x : -big);
    const float y0 = wave_min_f(ray ? y : big), y1 = wave_max_f(ray ? y : -big);
    if (__ballot(ray) == 0) return make_float4(0.f, 0.f, -1.f, -1.f);
    return make_float4(0.5f * (x0 + x1), 0.5f * (y0 + y1), 0.500001f * (x1 - x0) + 1.2e-7f * (1.f + fabsf(x0) + fabsf(x1)),
                       0.500001f * (y1 - y0) + 1.2e-7f * (1.f + fabsf(y0) + fabsf(y1)));
}

// A wavefront's vote on its tile (the tile's is their conjunction): the pixels that have a ray share the basis
// pixel's origin; no pixel has one. And in the complement (so that the conjunction is their union), from bit 8 on,
// the strips with bare pixels.
constexpr int kVoteOneOrigin = 1, kVoteNoRay = 2;
XSG_DEV int tile_vote(bool one_origin, bool has_ray, int bare_strips) {
    return (one_origin ? kVoteOneOrigin : 0) | (has_ray ? 0 : kVoteNoRay) | (~bare_strips << 8);
}
XSG_DEV int bare_strips(int vote) { return (~vote >> 8) & 0xffff; }

// The tile's largest |x| and |y| and its slack (strip_cull), from its strips' and wavefronts'.
XSG_DEV void tile_bounds(TileFrame& f, const float4* boxes, int n_boxes, const float* far2, const float* late, int nw) {
    float hx = 0.f, hy = 0.f, o = 0.f, t = 0.f;
    for (int k = 0; k < n_boxes; ++k) {
        hx = fmaxf(hx, fabsf(boxes[k].x) + boxes[k].z);
        hy = fmaxf(hy, fabsf(boxes[k].y) + boxes[k].w);
    }
    for (int k = 0; k < nw; ++k) {
        o = fmaxf(o, far2[k]);
        t = fmaxf(t, late[k]);
    }
    f.hx = hx; f.hy = hy; f.slack_o = __builtin_amdgcn_sqrtf(o); f.slack_t = t;
}

// The turn: the largest component of gro (kx: x, ky: y, else z), the components with that one (k) apart, and the
// reflection I - beta n n^T, n = (ga, gb, vk), that sends gro to axis k. The backward derives it a second time, to
// turn back: every rounding here and in the rows is therefore explicit (no sum that a compiler may contract one way
// in one copy and another in the other), so that both copies take the same axis where components nearly tie.
struct Turn {
    bool kx, ky;
    float gk, ga, gb, D, vk, beta;
};
XSG_DEV Turn turn_of(f3 r0, f3 r1, f3 r2, f3 v) {
    auto dot1 = [](f3 a, f3 b) { return fmaf(a.z, b.z, fmaf(a.y, b.y, a.x * b.x)); };
    const f3 g = mk3(dot1(r0, v), dot1(r1, v), dot1(r2, v));
    const float ax = fabsf(g.x), ay = fabsf(g.y), az = fabsf(g.z);
    Turn t;
    t.kx = ax >= ay && ax >= az;
    t.ky = !t.kx && ay >= az;
    t.gk = t.kx ? g.x : t.ky ? g.y : g.z;
    t.ga = t.kx ? g.y : g.x;
    t.gb = (t.kx || t.ky) ? g.z : g.y;
    t.D = __builtin_amdgcn_sqrtf(dot1(g, g));
    t.vk = t.gk + copysignf(t.D, t.gk);
    const float den = t.D * (t.D + fabsf(t.gk));
    // at the Gaussian's centre any frame will do (and the reciprocals of smaller numbers are infinite)
    t.beta = den > 1e-36f ? __builtin_amdgcn_rcpf(den) : 0.f;
    return t;
}

// One Gaussian's turned frame (rows in world space) and its affine rows (value, d/dx, d/dy).
struct RayFrame {
    f3 t1, t2, u;
    f3 a1, a2, au;
    float D;
};

XSG_DEV RayFrame ray_frame(f3 r0, f3 r1, f3 r2, f3 mu, f3 o, const TileBasis& bas) {
    const f3 v = o - mu;
    const Turn t = turn_of(r0, r1, r2, v);
    const f3 rk = sel3(t.kx, r0, sel3(t.ky, r1, r2)), ra = sel3(t.kx, r1, r0), rb = sel3(t.kx || t.ky, r2, r1);
    const f3 w = t.ga * ra + t.gb * rb + t.vk * rk;
    RayFrame f;
    f.t1 = ra - (t.beta * t.ga) * w;
    f.t2 = rb - (t.beta * t.gb) * w;
    f.u = copysignf(1.0f, t.gk) * ((t.beta * t.vk) * w - rk);
    const d3 v64 = d3{(double)o.x - (double)mu.x, (double)o.y - (double)mu.y, (double)o.z - (double)mu.z};
    const d3 q1 = to64(f.t1), q2 = to64(f.t2);
    const f3 bx = to32(bas.x), by = to32(bas.y), ba = to32(bas.a);
    const float vv = dot(v, v);
    const float va = vv > 1e-37f && t.beta > 0.f ? dot(v, ba) * __builtin_amdgcn_rcpf(vv) : 0.f;
    f.a1 = mk3((float)(dot64(q1, bas.a) - (double)((float)dot64(q1, v64) * va)), dot(f.t1, bx), dot(f.t1, by));
    f.a2 = mk3((float)(dot64(q2, bas.a) - (double)((float)dot64(q2, v64) * va)), dot(f.t2, bx), dot(f.t2, by));
    f.au = mk3(dot(f.u, ba), dot(f.u, bx), dot(f.u, by));
    f.D = (float)dot64(to64(f.u), v64);
    return f;
}

// A vector and a symmetric matrix (upper triangle, row-major) of the turned frame, turned back into the
// Gaussian's own normalised frame; the rows, mean and origin are those ray_frame was given.
XSG_DEV void turn_back(f3 r0, f3 r1, f3 r2, f3 mu, f3 o, f3& v, float (&Q)[6]) {
    const Turn t = turn_of(r0, r1, r2, o - mu);
    const bool kx = t.kx, ky = t.ky;
    const float beta = t.beta, s = -copysignf(1.0f, t.gk);  // u is s times the reflected row k
    const f3 n = mk3(t.ga, t.gb, t.vk);
    f3 w = mk3(v.x, v.y, s * v.z);
    w = w - (beta * dot(n, w)) * n;  // in the order (a, b, k)
    v = mk3(kx ? w.z : w.x, kx ? w.x : ky ? w.z : w.y, (kx || ky) ? w.y : w.z);
    const float aa = Q[0], ab = Q[1], ak = s * Q[2], bb = Q[3], bk = s * Q[4], kk = Q[5];
    const f3 y = beta * mk3(aa * n.x + ab * n.y + ak * n.z, ab * n.x + bb * n.y + bk * n.z, ak * n.x + bk * n.y + kk * n.z);
    // n z^T + z n^T with z = y - beta (n . y) / 2 n
    const f3 z = y - (0.5f * beta * dot(n, y)) * n;
    const float raa = aa - 2.f * n.x * z.x, rab = ab - n.x * z.y - n.y * z.x, rak = ak - n.x * z.z - n.z * z.x;
    const float rbb = bb - 2.f * n.y * z.y, rbk = bk - n.y * z.z - n.z * z.y, rkk = kk - 2.f * n.z * z.z;
    Q[0] = kx ? rkk : raa;
    Q[1] = kx || ky ? rak : rab;
    Q[2] = kx ? rbk : ky ? rab : rak;
    Q[3] = kx ? raa : ky ? rkk : rbb;
    Q[4] = kx ? rab : rbk;
    Q[5] = kx || ky ? rbb : rkk;
}

// alpha / opacity of one pair; a.w = -log2(e) / 2 D^2. |grd|^2 is at least 1e-36, so that a Gaussian without
// any extent (M = 0) gives power 0 as safe_normalize does.
struct RayEval {
    float x, y, u, tt, inv_dd, e;
};
XSG_DEV RayEval ray_eval(float4 a, float4 b, float4 c, float x, float y) {
    RayEval v;
    v.x = fmaf(y, a.z, fmaf(x, a.y, a.x));
    v.y = fmaf(y, b.z, fmaf(x, b.y, b.x));
    v.u = fmaf(y, c.z, fmaf(x, c.y, c.x));
    v.tt = fmaf(v.y, v.y, fmaf(v.x, v.x, 1e-36f));
    v.inv_dd = __builtin_amdgcn_rcpf(fmaf(v.u, v.u, v.tt));
    v.e = __builtin_amdgcn_exp2f(v.tt * a.w * v.inv_dd);
    return v;
}

// Conservative culling of the same tiles. A pixel takes a Gaussian only where d = D |t| / |grd| <= d_lim =
// sqrt(2 ln(255 op)), that is |t| <= rho |u|, rho = d_lim / sqrt(D^2 - d_lim^2). Over a box of (x, y), |t1|,
// |t2| and |u| are bounded by their affine forms' values at its centre and their slopes (three separating
// axes), and over the tile the region lies in the ellipse |t| <= rho max|u|, whose bounding box gives the
// other two. The 64 pixels of a strip keep 3 % more Gaussians than some pixel of it takes (Gaussians of
// exp(-3 +- 0.7) over 2 to 80, 1080p), where a cone about the strip's rays keeps 33 % more. Margins: 1e-6 of
// the terms for the rounding of these forms and of the pairs', 1e-4 and 3e-3 in d_lim for that of exp2 and
// the logarithm. Non-finite or degenerate Gaussians are kept, so that they reach the alpha test as in the
// reference.
struct StripCull {
    f3 a1, a2, au;
    float rho2, m1, m2;       // rho^2; margins of t1 and t2
    float xg, yg, ex, ey;     // the ellipse's box
    bool keep_all;
};

// What of a Gaussian the test needs beside its frame, taken before it (its inputs then end there).
struct CullInput {
    float lim;       // d_lim
    bool ok, low;    // finite and not degenerate; below the alpha threshold everywhere
};
XSG_DEV CullInput cull_input(f3 mu, f3 s, float4 q, float op) {
    const float s_max = fmaxf(s.x, fmaxf(s.y, s.z)), s_min = fminf(s.x, fminf(s.y, s.z));
    const float q2 = q.x * q.x + q.y * q.y + q.z * q.z + q.w * q.w;
    CullInput c;
    c.ok = finite3(mu) && s_min >= 1e-12f && s_max <= 1e9f && q2 >= 1e-30f && q2 <= 1e30f && isfinite(op);
    c.low = op < 1.f / 255.f;
    // 2 ln(255 op) through log2; + 3e-3 covers the rounding of log, exp, the product and the compare
    const float l2 = 2.f * 0.69314718f * __builtin_amdgcn_logf(fmaxf(255.f * op, 1.f));
    c.lim = __builtin_amdgcn_sqrtf(l2) * 1.0001f + 3e-3f;
    return c;
}

// hx, hy: the tile's largest |x| and |y|.
XSG_DEV StripCull strip_cull(const RayFrame& f, const CullInput& in, float hx, float hy) {
    StripCull c;
    c.a1 = f.a1; c.a2 = f.a2; c.au = f.au;
    const float lim = in.lim;
    const bool ok = in.ok && fabsf(f.D) < 1e15f;
    const float room = f.D * f.D - lim * lim;
    const bool drop_all = ok && in.low;
    c.keep_all = !drop_all && (!ok || !(room > 1e-3f * lim * lim));
    c.rho2 = lim * lim * __builtin_amdgcn_rcpf(room) * 1.0001f;
    const float u_max = fabsf(f.au.x) + fabsf(f.au.y) * hx + fabsf(f.au.z) * hy;
    c.m1 = 1e-6f * (fabsf(f.a1.x) + fabsf(f.a1.y) * hx + fabsf(f.a1.z) * hy);
    c.m2 = 1e-6f * (fabsf(f.a2.x) + fabsf(f.a2.y) * hx + fabsf(f.a2.z) * hy);
    // the centre solves t1 = t2 = 0; what rounding can move it by is added to the half extents
    const float p0 = f.a1.y * f.a2.z, p1 = f.a1.z * f.a2.y;
    const float id = __builtin_amdgcn_rcpf(p0 - p1);
    const float nx0 = f.a1.z * f.a2.x, nx1 = f.a1.x * f.a2.z, ny0 = f.a1.x * f.a2.y, ny1 = f.a1.y * f.a2.x;
    c.xg = (nx0 - nx1) * id;
    c.yg = (ny0 - ny1) * id;
    const float reach = __builtin_amdgcn_sqrtf(c.rho2) * u_max + c.m1 + c.m2;
    const float aid = fabsf(id), det_err = 4e-6f * (fabsf(p0) + fabsf(p1));
    c.ex = aid * (reach * __builtin_amdgcn_sqrtf(f.a1.z * f.a1.z + f.a2.z * f.a2.z) + 4e-6f * (fabsf(nx0) + fabsf(nx1)) +
                  det_err * fabsf(c.xg)) * 1.0002f;
    c.ey = aid * (reach * __builtin_amdgcn_sqrtf(f.a1.y * f.a1.y + f.a2.y * f.a2.y) + 4e-6f * (fabsf(ny0) + fabsf(ny1)) +
                  det_err * fabsf(c.yg)) * 1.0002f;
    c.ex = drop_all ? -__builtin_inff() : c.ex;  // out of every box
    return c;
}

// The same where the rays do not share one origin, or the Gaussian moves. The frame belongs to the tile's basis
// pixel (origin o0, the Gaussian then at `at`), and slack bounds how far any pixel's origin or time takes
// (o - mu) from there: the ellipsoid of semi-axes d_lim s_i that such a ray must meet, widened by a ball of that
// radius, lies in the one of semi-axes sqrt((1 + 1 / p) (d_lim s_i)^2 + (1 + p) slack^2) for every p > 0. p is
// d_lim s_min / slack, for which the thinnest axis grows by slack alone, but at least 3: the axes of a flat Gaussian
// then grow by 15 %, or to twice the slack. (Widening by slack / s_min instead, which is exact for a ball, kept
// nearly everything of a flat one.) The pairs' float32 error, about 17 ulp of |gro|, adds to d_lim (2e-5 of it here).
XSG_DEV StripCull strip_cull_moving(f3 r0, f3 r1, f3 r2, f3 at, f3 s, CullInput in, f3 o0, float slack,
                                    const TileFrame& tile) {
    const f3 away = at - o0;
    const float far = __builtin_amdgcn_sqrtf(dot(away, away)) + slack, s_min = fminf(s.x, fminf(s.y, s.z));
    in.ok = in.ok && s_min * s_min * 1e12f >= far;  // the pairs' products stay finite
    in.lim += 2.00001e-5f * far * __builtin_amdgcn_rcpf(s_min);
    const float ball = fmaxf(slack * 1.00001f, 1e-20f);
    const float p = fmaxf(3.f, in.lim * s_min * __builtin_amdgcn_rcpf(ball)), a = 1.f + __builtin_amdgcn_rcpf(p);
    const float w = ball * __builtin_amdgcn_rcpf(in.lim), b = (1.f + p) * w * w;
    const RayFrame f = ray_frame(s.x * __builtin_amdgcn_rsqf(a * s.x * s.x + b) * r0, s.y * __builtin_amdgcn_rsqf(a * s.y * s.y + b) * r1,
                                 s.z * __builtin_amdgcn_rsqf(a * s.z * s.z + b) * r2, at, o0, get_basis(tile));
    return strip_cull(f, in, tile.hx, tile.hy);
}

// True unless no pixel in the strip's box can take the Gaussian (every comparison fails on a NaN).
XSG_DEV bool strip_keep(float4 box, const StripCull& c) {
    const float b1 = fabsf(fmaf(box.y, c.a1.z, fmaf(box.x, c.a1.y, c.a1.x))) - fabsf(c.a1.y) * box.z - fabsf(c.a1.z) * box.w;
    const float b2 = fabsf(fmaf(box.y, c.a2.z, fmaf(box.x, c.a2.y, c.a2.x))) - fabsf(c.a2.y) * box.z - fabsf(c.a2.z) * box.w;
    const float bu = fabsf(fmaf(box.y, c.au.z, fmaf(box.x, c.au.y, c.au.x))) + fabsf(c.au.y) * box.z + fabsf(c.au.z) * box.w;
    const float n1 = fmaxf(0.f, b1 - c.m1), n2 = fmaxf(0.f, b2 - c.m2);
    const bool out = n1 * n1 + n2 * n2 > c.rho2 * bu * bu || fabsf(box.x - c.xg) > box.z + c.ex ||
                     fabsf(box.y - c.yg) > box.w + c.ey;
    return box.z >= 0.f && (c.keep_all || !out);
}

// Lane-to-lane moves inside rows of 16 lanes (DPP). `update_dpp` with all rows/banks enabled and
// in-bounds patterns returns the source lane's value for every lane.
template <int CTRL>
XSG_DEV float dpp_mov(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, false));
}
constexpr int kDppQuadSwap1 = 0xB1;    // quad_perm [1,0,3,2]: lane ^ 1
constexpr int kDppQuadSwap2 = 0x4E;    // quad_perm [2,3,0,1]: lane ^ 2

struct Eval3dParams {
    TileGrid g;
    const float* means;
    const float4* quats;
    const float* scales;
    const float* colors;
    const float* opac;
    const float* velocity;
    const float* rtd;
    const float* ray_o;
    const float* ray_d;
    const int32_t* offsets;
    const int32_t* flatten;
    float* out_rgb;
    float* out_depth;
    float* out_alpha;
    int32_t* out_last;
    const float* render_alpha;
    const int32_t* last_ids;
    const float* v_rgb;
    const float* v_depth;
    const float* v_alpha;
    float* v_means;
    float* v_opac;
    float* v_colors;
    float* v_ray_o;
    float* v_ray_d;
    float* v_velocity;
    float* v_time;
    float* v_mt;         // workspace [n, 6]: upper triangle of the symmetric Q = sum of v_grd (x) grd + v_gro (x) gro
    // colours of flatten id fid in camera cam sit at fid * CDIM - cam * col_shift: 0 for per-camera
    // colours [n_cams, n, CDIM], n * CDIM for one colour set [n, CDIM] that every camera shares
    int64_t col_shift;
    unsigned long long* pair_counts;  // optional: += [evaluated, composited] pixel-pairs
    // optional (backward): logical (camera, tile) block launched at each position of xcd_tile's order
    const int32_t* tile_order;
    int px_hint;  // backward pixels per lane for 129..256-pixel tiles: 0 (by grid size), 2 or 4
    // optional (forward): per (camera, tile) the backward's work estimate, the tile's intersections up
    // to its pixels' largest last id (what tile_work_kernel derives from the last ids)
    int32_t* tile_work;
};

int eval3d_fwd_launch(int cdim, bool dyn, const Eval3dParams& p, hipStream_t s);
int eval3d_bwd_launch(int cdim, bool dyn, const Eval3dParams& p, hipStream_t s);
// per-CDIM backward launcher, instantiated for each supported CDIM by eval3d_bwd_g<k>.hip
template <int CDIM>
int eval3d_bwd_cdim(bool dyn, bool ray_grads, const Eval3dParams& p, hipStream_t s);

}  // namespace xsg
