// Backward eval3d compositing: rasterize_eval3d_[dynamic_]bwd_kernel (eval3d_bwd.cu:66-294,
// eval3d_dynamic_bwd.cu kernel before :312).
//
// Differences in structure (not in what is computed):
//  * batches start at the largest last_id of the tile instead of the end of the tile's list; the
//    reference loads and skips those trailing batches (every index there exceeds every pixel's
//    last_id, eval3d_bwd.cu:155-159);
//  * the gradient of M = S^-1 R^T is accumulated per Gaussian, as the symmetric Q = sum of
//    v_grd (x) grd + v_gro (x) gro (dL/dM = Q S R^T, six entries), and turned into quaternion /
//    scale gradients once per Gaussian by the epilogue: quat_scale_to_preci_half_vjp
//    (utils.h:232-263) is linear in dL/dM, so the sum of per-pair vjps equals the vjp of the sum,
//    and the scale gradient is -Q_ii / s_i;
//  * tiles whose rays share one origin work in the forward's turned frame and affine form (xsg_eval3d.h); Q and
//    the mean's gradient are turned back once per Gaussian and batch;
//  * per-pair gradients are summed over the 64 lanes of a wavefront through LDS and the totals left in the
//    Gaussian's own staging slot; after a batch one lane per Gaussian finishes them (the turn, M^T, the
//    opacity) and the atomics add 16 components of four Gaussians per instruction;
//  * a thread owns PX pixels, one in each of PX strips of 64 consecutive pixels of the tile, so the staged
//    Gaussian's LDS reads and the reduction serve all of them, and a strip that no pixel of can take the
//    Gaussian is skipped unevaluated (strip_keep; it would add exact zeros);
//  * divisions in the per-pair math are reciprocal-multiplies (v_rcp_f32, 1 ulp).
//
// Bound by VALU issue. The whole op against per-pair M^T products and atomics per Gaussian and wavefront, in the
// unturned frame: 1920x1080, 1 M Gaussians 422 -> 333-352 us; six cameras of 1600x900 1675 -> 1240; moving origins
// 459 -> 312; 32 channels at 640x480 445 -> 316; 2048x128 lidar 189 -> 172.
//
// This header holds the kernel template and its per-CDIM launcher; eval3d_bwd_g*.hip instantiate the
// launcher for groups of colour dimensions in separate translation units (the variants compile in
// parallel) and eval3d_bwd.hip dispatches on the dimension.
#pragma once
#include <type_traits>

#include "xsg_eval3d.h"

namespace xsg {
namespace {

constexpr float kMaxAlpha = 0.99f;  // eval3d_bwd.cu:38

XSG_DEV int wave_max(int v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v = max(v, __shfl_xor(v, off, 64));
    return v;
}

XSG_DEV void wave_lds_order() {  // LDS instructions of one wavefront complete in order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Reduce-scatter of the first nv (<= 16) of 16 per-lane values over the 64 lanes of a wavefront through a
// wavefront-private LDS buffer: lane l stores value k at row k (rows of kRedRow floats, padded so that
// the four lanes reading one quarter-row each fall in different banks), then lane 4k + q adds lanes
// 16q .. 16q + 15 of row k with four 16-byte reads and the quad adds its four sums (DPP). Every lane of
// quad k ends with the wave total of value k. The reads see the stores and the next call's stores follow
// these reads without a barrier. All 64 lanes active.
constexpr int kRedRow = 68;
XSG_DEV float wave_reduce_scatter16_lds(const float (&v)[16], int nv, float* __restrict__ buf) {
    const int lane = __lane_id();
#pragma unroll
    for (int k = 0; k < 16; ++k)
        if (k < nv) buf[k * kRedRow + lane] = v[k];
    wave_lds_order();
    const int k = lane >> 2, q = lane & 3;
    float s = 0.0f;
    if (k < nv) {
        const float4* row = reinterpret_cast<const float4*>(buf + k * kRedRow + 16 * q);
        const float4 a = row[0], b = row[1], c = row[2], d = row[3];
        s = (((a.x + a.y) + (a.z + a.w)) + ((b.x + b.y) + (b.z + b.w))) +
            (((c.x + c.y) + (c.z + c.w)) + ((d.x + d.y) + (d.z + d.w)));
    }
    s += dpp_mov<kDppQuadSwap2>(s);
    s += dpp_mov<kDppQuadSwap1>(s);
    wave_lds_order();
    return s;
}

// Per-pixel state of the backward sweep.
template <int CS>
struct BwdPixel {
    float x, y;    // one origin: the affine form's coordinates
    float T;
    float buf;     // sum over composited pairs of fac (rgb . v_rgb + hit_t v_depth), minus T_final v_alpha
    float v_c[CS];
    float v_d;     // dL/ddepth; one origin: of -k hit_t (times -1 / k)
    int32_t bin_final;
    float v_t;
    f3 v_ro, v_rd;
};

// The staged Gaussian of one loop step. One origin: affine rows a, b, c (with -log2(e) / 2 D^2, D and the
// opacity). Any origins: rows of M with the mean in the fourth components, vel and M vel.
struct BwdGauss {
    float4 a, b, c;
    f3 vel, mv;
    float op;
};

// One pair's evaluation (eval3d_bwd.cu:172-205) in the forward kernel's arithmetic, so that the
// transmittance this sweep divides out is the one the forward pass multiplied in.
struct BwdEval {
    f3 grd, p;    // M d (one origin: divided by k) and the Gaussian's offset from the ray
    f3 gro;
    float inv_dd, hit;  // 1 / |grd|^2; hit_t (one origin: -k hit_t)
    float vis, araw;    // exp(-d^2 / 2); opacity times it, 0 if the pair is not valid
    bool valid;
};

// Gradient contribution of one pair into acc (eval3d_bwd.cu:206-271). A pair that is not valid
// adds exact zeros (its alpha is 0, so fac = 0 and T / (1 - 0) = T; every other gradient is a multiple of
// araw or fac) and leaves the pixel's transmittance and buffer unchanged.
//
// The reference's dL/dalpha sums, per channel, rgb T - buffer / (1 - alpha) and the depth and
// alpha terms; here one running buffer carries all of them, so dL/dalpha = T u - buf / (1 - alpha)
// with u = rgb . v_rgb + hit_t v_depth. Its chain through gcrod = n x gro, n = grd / |grd|, and
// safe_normalize_bwd collapses to the offset p of the Gaussian from the ray (perpendicular to it, in the
// normalised frame): dL/dgro = -araw dL/dalpha p - k1 grd with k1 = dL/dhit_t / |grd|^2, and
// dL/dgrd = hit_t (dL/dgro - k1 grd) - k1 gro.
//
// Q: with gro = p - hit_t grd the hit_t terms of Q = dL/dgrd (x) grd + dL/dgro (x) gro cancel exactly and
//   Q = dL/dgro (x) p - p (x) k1 grd = A p (x) p - k1 (grd (x) p + p (x) grd),
// which is symmetric (the loss depends on M only through rotation invariants of gro and grd).
// Accumulating it in this form skips the two products of size |hit_t| |grd| that cancel (the
// far-from-the-Gaussian part of the ray), which in float32 lose the scale gradient of thin
// Gaussians seen from far away. The mean's gradient -M^T dL/dgro (and the velocity's, with the pixel's
// time) is applied once to the sum over the pixels, and the opacity's, the sum of exp(-d^2 / 2) dL/dalpha,
// is that of araw dL/dalpha over the opacity.
//
// acc: colours, sum of dL/dgro, Q (upper triangle, row-major), araw dL/dalpha, sum of time dL/dgro.
//
// HIGH: the pair's alpha can exceed kMaxAlpha, or be no number (decided per Gaussian: exp(-d^2 / 2) <= 1).
template <int CDIM, int CS, int K, bool DYN, bool RG, bool FIXED, bool HIGH>
XSG_DEV void bwd_pair(BwdPixel<CS>& px, float rt, const BwdGauss& gs, const BwdEval& e, const float (&rgb)[CS],
                      float (&acc)[K]) {
    float alpha = e.araw;
    if constexpr (HIGH) alpha = e.valid ? fminf(kMaxAlpha, e.araw) : 0.f;
    // 1 / max(1e-6, 1 - alpha) (eval3d_bwd.cu:221): alpha <= kMaxAlpha, so the max never applies
    const float ra = __builtin_amdgcn_rcpf(1.0f - alpha);
    px.T = px.T * ra;
    const float T = px.T;
    const float fac = alpha * T;
    float rv = 0.0f;
#pragma unroll
    for (int k = 0; k < CDIM; ++k) {
        acc[k] += px.v_c[k] * fac;
        rv = (k == 0) ? rgb[0] * px.v_c[0] : fmaf(rgb[k], px.v_c[k], rv);
    }
    const float u = (CDIM > 0) ? fmaf(e.hit, px.v_d, rv) : e.hit * px.v_d;
    float A = -e.araw * (T * u - ra * px.buf);
    px.buf = fmaf(fac, u, px.buf);
    float k1 = px.v_d * fac * e.inv_dd;
    if constexpr (HIGH) {  // geometry and opacity only below the clamp (eval3d_bwd.cu:243)
        const bool geo = e.valid && e.araw <= kMaxAlpha;
        A = geo ? A : 0.f;
        k1 = geo ? k1 : 0.f;
    }
    if constexpr (FIXED) k1 = -k1;  // v_d is that of -k hit_t: this is k times k1, and grd is grd / k
    const f3 kg = k1 * e.grd;
    const f3 v_gro = A * e.p - kg;
    acc[CDIM + 0] += v_gro.x;
    acc[CDIM + 1] += v_gro.y;
    acc[CDIM + 2] += v_gro.z;
    // Q_ij = dL/dgro_i p_j - p_i k1 grd_j
    acc[CDIM + 3] = fmaf(e.p.x, v_gro.x - kg.x, acc[CDIM + 3]);
    acc[CDIM + 4] = fmaf(-e.p.x, kg.y, fmaf(v_gro.x, e.p.y, acc[CDIM + 4]));
    acc[CDIM + 5] = fmaf(-e.p.x, kg.z, fmaf(v_gro.x, e.p.z, acc[CDIM + 5]));
    acc[CDIM + 6] = fmaf(e.p.y, v_gro.y - kg.y, acc[CDIM + 6]);
    acc[CDIM + 7] = fmaf(-e.p.y, kg.z, fmaf(v_gro.y, e.p.z, acc[CDIM + 7]));
    acc[CDIM + 8] = fmaf(e.p.z, v_gro.z - kg.z, acc[CDIM + 8]);
    acc[CDIM + 9] -= A;
    if constexpr (DYN) {
        acc[CDIM + 10] += v_gro.x * rt;
        acc[CDIM + 11] += v_gro.y * rt;
        acc[CDIM + 12] += v_gro.z * rt;
        px.v_t -= dot(v_gro, gs.mv);
    }
    if constexpr (RG) {
        f3 v_grd;
        if constexpr (FIXED) {  // times k
            v_grd = -e.hit * (v_gro - kg);
            v_grd.z -= k1 * gs.b.w;
        } else {
            v_grd = e.hit * (v_gro - kg) - k1 * e.gro;
        }
        // one origin: in the basis (A, X, Y), whose rows of M the affine ones are
        const f3 r0 = mk3(gs.a.x, gs.a.y, gs.a.z), r1 = mk3(gs.b.x, gs.b.y, gs.b.z), r2 = mk3(gs.c.x, gs.c.y, gs.c.z);
        px.v_ro = px.v_ro + rows_tmul(r0, r1, r2, v_gro);
        px.v_rd = px.v_rd + rows_tmul(r0, r1, r2, v_grd);
    }
}

// The four-pixel variants of up to four channels without per-pixel ray or time gradients have a loop body of
// their own for Gaussians whose alpha cannot reach the clamp, and four waves per SIMD (128 registers; the few
// that do not fit are set-up values spilled outside the pair loop). The ray-gradient variants fit three (168
// registers), the many-channel ones two (256); the others take what registers they need.
template <int CDIM, bool DYN, bool RG, int PX>
constexpr bool kBwdSplit = PX == 4 && !RG && !DYN && CDIM <= 4;
template <int CDIM, bool DYN, bool RG, int PX, int NT>
constexpr int kBwdWaves = kBwdSplit<CDIM, DYN, RG, PX> && NT == 64 ? 4 : NT > 128 || CDIM > 33 ? 1 : CDIM > 16 ? 2 : CDIM <= 4 && RG ? 3 : 1;

// Motion with four pixels per lane runs faster with two waves than with the three it would fit (1280x800,
// 400 k moving Gaussians: 310 us against 327).
template <bool DYN, bool RG, int PX>
constexpr int kBwdMaxWaves = DYN && !RG && PX == 4 ? 2 : 8;

// PX pixels per thread: a workgroup of one wavefront per PX strips of 64 pixels. The batch is one Gaussian
// per thread.
template <int CDIM, bool DYN, bool RG, int PX, int NT, bool COUNT>
__global__ __launch_bounds__(NT)
    __attribute__((amdgpu_waves_per_eu(kBwdWaves<CDIM, DYN, RG, PX, NT>, kBwdMaxWaves<DYN, RG, PX>))) void eval3d_bwd_kernel(
        Eval3dParams p) {
    constexpr int CL = (CDIM > 0 && CDIM <= kBwdColorLdsMax) ? CDIM : 0;
    constexpr int C4 = (CL + 3) / 4;
    constexpr int CS = CDIM > 0 ? CDIM : 1;
    constexpr int K = CDIM + 3 + 6 + 1 + (DYN ? 3 : 0);  // colours, dL/dgro, Q, opacity, time dL/dgro
    constexpr int kChunks = (K + 15) / 16;
    // Totals kept until the batch's end: all, or (colours read from HBM) those after the colours', whose
    // totals are added at once
    constexpr int KO = CL > 0 ? 0 : CDIM, KT = K - KO;
    constexpr int G0 = CDIM - KO;  // the first total after the colours'
    constexpr int NWB = NT / 64, NSB = NWB * PX;
    // Gaussians per batch: one per thread, or 64 where a slot holds many channels and larger batches' LDS would
    // leave a SIMD one wavefront (32 channels, two wavefronts per tile: 31 KB instead of 54; 16 channels, four: 84)
    constexpr int NB = CL > 16 || (CL == 16 && NT > 128) ? 64 : NT;
    constexpr int NBW = NB / 64;
    // A Gaussian's slot: its staged values (rows and colours), then, once the workgroup's one wavefront has
    // composited it, its K totals
    constexpr int kRec4 = 3 + C4;
    constexpr int kSlot4 = NWB > 1 || kRec4 > (KT + 3) / 4 ? kRec4 : (KT + 3) / 4;
    __shared__ float4 s_slot[NB * kSlot4];
    __shared__ float s_tot[NWB > 1 ? NB * KT : 1];  // the totals when several wavefronts read the slots
    __shared__ uint64_t s_did[NWB][NBW];           // [wavefront][staging wavefront]: Gaussians with totals
    __shared__ int32_t s_id[NB];
    __shared__ float s_op[NB];                        // any origins: the opacity
    __shared__ float4 s_vel[DYN ? NB : 1], s_mv[DYN ? NB : 1];  // and vel, M vel
    __shared__ float4 s_box[NSB];
    __shared__ int s_vote[NWB];
    __shared__ TileFrame s_frame;
    __shared__ float s_slack[2][NWB];
    __shared__ int s_max[NWB];
    __shared__ int32_t s_sbf[NSB];              // largest last id of each strip's pixels
    __shared__ uint64_t s_mask[NSB][NBW];       // [strip][staging wavefront]: Gaussians it evaluates
    __shared__ uint64_t s_high[NBW];
    // where the totals go: the k-th one's array (in bytes from v_means) and its bytes per Gaussian. Looked up, the
    // five arrays' addresses do not sit in scalar registers across the pair loops.
    __shared__ int64_t s_dst[KT];
    __shared__ uint32_t s_step[KT];
    __shared__ __align__(16) float s_red[NWB][(K < 16 ? K : 16) * kRedRow];  // per wavefront: the gradient reduction

    const TileGrid& g = p.g;
    const int n_tiles = g.n_tiles_w * g.n_tiles_h;
    const int nblocks = n_tiles * g.n_cams;
    const int order = xcd_tile((int)blockIdx.x, nblocks);
    const int logical = p.tile_order ? p.tile_order[order] : order;
    const int cam = logical / n_tiles, tile = logical - cam * n_tiles;
    const int bs = g.tile_w * g.tile_h;
    const int tr = threadIdx.x;
    const int wave = tr >> 6, lane = tr & 63;
    const int nwb = (int)(blockDim.x >> 6);
    const int nb = min(NB, (int)blockDim.x), nbw = nb >> 6;  // Gaussians per batch, wavefronts that stage them
    const int trow = tile / g.n_tiles_w, tcol = tile - trow * g.n_tiles_w;
    const int32_t range_start = p.offsets[logical];  // utils.h:48-58
    const int32_t range_end = (logical == nblocks - 1) ? (int32_t)g.n_isects : p.offsets[logical + 1];
    const int64_t hw = (int64_t)g.width * g.height;
    if (past_image(g, trow, tcol)) return;

    // strip h's pixel of this lane: its index in the [cams, H, W] images (utils.h:32-44), -1 outside;
    // recomputed where needed rather than kept in registers (opaque: or the compiler keeps it)
    auto pixel_at = [&](int q) -> int64_t {
        const int ty = q / g.tile_w, tx = q - ty * g.tile_w;
        const int i = trow * g.tile_h + ty, j = tcol * g.tile_w + tx;
        return q < bs && i < g.height && j < g.width ? (int64_t)cam * hw + (int64_t)i * g.width + j : -1;
    };
    auto pixel_of = [&](int h) { return pixel_at((wave * PX + h) * 64 + opaque(lane)); };
    for (int k = tr; k < KT; k += (int)blockDim.x) {
        const int kk = KO + k;
        const float* dst;
        int step = 3;
        if (kk < CDIM) {  // colour gradients of camera cam start at cam * (n * CDIM - col_shift)
            dst = p.v_colors + (int64_t)cam * (g.n * CDIM - p.col_shift) + kk;
            step = CDIM;
        } else if (kk < CDIM + 3) {
            dst = p.v_means + (kk - CDIM);
        } else if (kk < CDIM + 9) {
            dst = p.v_mt + (kk - CDIM - 3);
            step = 6;
        } else if (kk == CDIM + 9) {
            dst = p.v_opac;
            step = 1;
        } else {
            dst = p.v_velocity + (kk - CDIM - 10);
        }
        s_dst[k] = reinterpret_cast<const char*>(dst) - reinterpret_cast<const char*>(p.v_means);
        s_step[k] = 4 * step;
    }
    // The left end of the tile's middle row, and that row's middle pixel (which stands in for those outside)
    const int64_t ps = (int64_t)cam * hw + (int64_t)min(trow * g.tile_h + g.tile_h / 2, g.height - 1) * g.width + tcol * g.tile_w;
    const int64_t pm = ps + min(g.tile_w / 2, g.width - 1 - tcol * g.tile_w);
    // The pixels' state and rays, loaded before the basis pixel's is looked at (their latencies overlap)
    BwdPixel<CS> px[PX];
    f3 ray_o[PX], ray_d[PX];
    float ray_t[PX];
    bool inside[PX];
#pragma unroll
    for (int h = 0; h < PX; ++h) {
        BwdPixel<CS>& q = px[h];
        const int64_t pix = pixel_of(h);
        inside[h] = pix >= 0;
        const int64_t at = inside[h] ? pix : pm;
        ray_o[h] = ld3(p.ray_o + 3 * at);
        ray_d[h] = ld3(p.ray_d + 3 * at);
        ray_t[h] = 0.f;
        if constexpr (DYN) ray_t[h] = p.rtd[at];
        const float T_final = 1.0f - p.render_alpha[at];
        q.T = T_final;
#pragma unroll
        for (int k = 0; k < CS; ++k) q.v_c[k] = 0.f;
#pragma unroll
        for (int k = 0; k < CDIM; ++k) q.v_c[k] = inside[h] ? p.v_rgb[at * CDIM + k] : 0.0f;
        q.v_d = inside[h] ? p.v_depth[at] : 0.0f;
        q.buf = inside[h] ? -T_final * p.v_alpha[at] : 0.0f;
        q.bin_final = inside[h] ? p.last_ids[at] : -1;
        q.v_ro = mk3(0.f, 0.f, 0.f);
        q.v_rd = mk3(0.f, 0.f, 0.f);
    }
    // the forward's tile set-up: basis, boxes, whether the rays share one origin
    const f3 side = ld3(p.ray_d + 3 * ps);
    const BasisPixel mid = basis_pixel<DYN>(p.ray_o, p.ray_d, p.rtd, pm, bs, pixel_at);
    const f3 o0 = mid.o;
    const float rt0 = mid.t;
    const TileBasis basis = uniform_basis(tile_basis(mid.d, side));
    if (tr == 0) put_basis(s_frame, basis);
    bool same = true, some = false;
    int bare = 0;  // strips
    float far2 = 0.f, late = 0.f;
    int32_t wave_bin_final = -1;
#pragma unroll
    for (int h = 0; h < PX; ++h) {
        BwdPixel<CS>& q = px[h];
        const f3 away = ray_o[h] - o0;
        const float rt = ray_t[h] - rt0;
        float ik;
        const bool ray = ray_xy(basis, ray_d[h], q.x, q.y, ik) && finite3(away) && isfinite(rt) && inside[h];
        const float4 box = strip_box(ray, q.x, q.y);
        same = same && (!ray || (__float_as_uint(ray_o[h].x) == __float_as_uint(o0.x) &&
                                 __float_as_uint(ray_o[h].y) == __float_as_uint(o0.y) &&
                                 __float_as_uint(ray_o[h].z) == __float_as_uint(o0.z)));
        some = some || ray;
        far2 = ray ? fmaxf(far2, dot(away, away)) : far2;
        late = ray ? fmaxf(late, fabsf(rt)) : late;
        q.x = ray ? q.x : 0.f;
        q.y = ray ? q.y : 0.f;
        q.v_t = ray ? ik : 0.f;  // until the mode is known
        if (__ballot(inside[h] && !ray) != 0) bare |= 1 << (wave * PX + h);
        const int m = wave_max(q.bin_final);
        if (lane == 0) {
            s_box[wave * PX + h] = box;
            s_sbf[wave * PX + h] = m;
        }
        wave_bin_final = max(wave_bin_final, m);
    }
    {
        const int v = tile_vote(__ballot(!same) == 0, __ballot(some) != 0, bare);
        const float f = wave_max_f(far2), l = DYN ? wave_max_f(late) : 0.f;
        if (lane == 0) {
            s_vote[wave] = v;
            s_slack[0][wave] = f;
            s_slack[1][wave] = l;
            s_max[wave] = wave_bin_final;
        }
    }
    __syncthreads();
    int vote = -1, tile_max = -1;
    for (int k = 0; k < nwb; ++k) {
        vote &= s_vote[k];
        tile_max = max(tile_max, s_max[k]);
    }
    if (tr == 0) tile_bounds(s_frame, s_box, nwb * PX, s_slack[0], s_slack[1], nwb);
    __syncthreads();
    vote = __builtin_amdgcn_readfirstlane(vote);
    const bool fixed = !DYN && (vote & (kVoteOneOrigin | kVoteNoRay)) == kVoteOneOrigin;
    bare = bare_strips(vote);

    uint64_t n_eval = 0, n_contrib = 0;  // evaluated / composited pixel-pairs of the wave, when counting
    int32_t eff_end;
    int num_batches;
    auto list_up_to = [&](int32_t last) {  // the tile's list up to its pixels' largest last id
        eff_end = min(range_end - 1, __builtin_amdgcn_readfirstlane(last));
        const int32_t n_eff = eff_end - range_start + 1;
        num_batches = n_eff > 0 ? (n_eff + nb - 1) / nb : 0;
    };
    list_up_to(tile_max);

    // the whole sweep is instantiated for both origin modes, so that neither carries the other's registers
    auto sweep = [&](auto fixed_c) {
        constexpr bool FIXED = decltype(fixed_c)::value;
#pragma unroll
        for (int h = 0; h < PX; ++h) {
            if constexpr (FIXED) {
                px[h].v_d = -px[h].v_d * px[h].v_t;
                px[h].bin_final = px[h].v_t != 0.f ? px[h].bin_final : -1;
            }
            px[h].v_t = 0.f;
        }
        f3 px_rd[FIXED ? 1 : PX], px_ro[FIXED ? 1 : PX];  // the pixels' rays and times
        float px_rt[FIXED ? 1 : PX];
        if constexpr (!FIXED) {
#pragma unroll
            for (int h = 0; h < PX; ++h) {
                const int64_t pix = pixel_of(h);
                px_rd[h] = pix >= 0 ? ld3(p.ray_d + 3 * pix) : mk3(0.f, 0.f, 0.f);
                px_ro[h] = pix >= 0 ? ld3(p.ray_o + 3 * pix) : mk3(0.f, 0.f, 0.f);
                px_rt[h] = 0.f;
                if constexpr (DYN) px_rt[h] = pix >= 0 ? p.rtd[pix] : 0.f;
            }
        }
        // the flatten id a thread stages in the next batch, loaded one batch ahead (its latency then
        // overlaps the pair loop instead of preceding the Gaussian's own loads)
        int32_t fid_next = 0;
        if (num_batches > 0 && tr < nb && eff_end - tr >= range_start) fid_next = p.flatten[eff_end - tr];
        for (int b = 0; b < num_batches; ++b) {
            const int32_t batch_end = eff_end - nb * b;
            const int32_t idx = batch_end - tr;
            const bool staged = tr < nb && idx >= range_start;
            StripCull cg;
            bool high = false;
            const int32_t fid = fid_next;
            if (tr < nb && idx - nb >= range_start) fid_next = p.flatten[idx - nb];
            float4* slot = s_slot + (tr < NB ? tr : 0) * kSlot4;
            if (staged) {
                const int64_t gid = fid - (int64_t)cam * g.n;
                s_id[tr] = fid;
                const f3 mu = ld3(p.means + 3 * gid);
                const float4 q = p.quats[gid];
                const f3 sc = ld3(p.scales + 3 * gid);
                const float op = p.opac[gid];
                const CullInput in = cull_input(mu, sc, q, op);
                f3 r0, r1, r2;
                iscl_rot_rows(q, sc, r0, r1, r2);
                f3 vel = mk3(0.f, 0.f, 0.f), at = mu;  // at: where the Gaussian is at the basis pixel's time
                if constexpr (DYN) {
                    vel = ld3(p.velocity + 3 * gid);
                    at = mu + rt0 * vel;
                }
                if constexpr (FIXED) {
                    const RayFrame f = ray_frame(r0, r1, r2, at, o0, get_basis(s_frame));
                    slot[0] = make_float4(f.a1.x, f.a1.y, f.a1.z, f.D * f.D * -0.72134752f);
                    slot[1] = make_float4(f.a2.x, f.a2.y, f.a2.z, f.D);
                    slot[2] = make_float4(f.au.x, f.au.y, f.au.z, op);
                    cg = strip_cull(f, in, s_frame.hx, s_frame.hy);
                } else {
                    slot[0] = make_float4(r0.x, r0.y, r0.z, mu.x);
                    slot[1] = make_float4(r1.x, r1.y, r1.z, mu.y);
                    slot[2] = make_float4(r2.x, r2.y, r2.z, mu.z);
                    s_op[tr] = op;
                    if constexpr (DYN) {
                        const f3 mv = rows_mul(r0, r1, r2, vel);
                        s_vel[tr] = make_float4(vel.x, vel.y, vel.z, 0.f);
                        s_mv[tr] = make_float4(mv.x, mv.y, mv.z, 0.f);
                    }
                    cg = strip_cull_moving(r0, r1, r2, at, sc, in, o0,
                                           s_frame.slack_o + s_frame.slack_t * __builtin_amdgcn_sqrtf(dot(vel, vel)), s_frame);
                }
                // alphas may reach the clamp, or be no number
                high = !(op <= kMaxAlpha) || cg.keep_all || (!FIXED && bare != 0);
                if constexpr (CL > 0) {
                    const float* cp = p.colors + ((int64_t)fid * CDIM - (int64_t)cam * p.col_shift);
#pragma unroll
                    for (int k4 = 0; k4 < C4; ++k4) {
                        float v[4];
#pragma unroll
                        for (int j = 0; j < 4; ++j) v[j] = (4 * k4 + j < CL) ? cp[4 * k4 + j] : 0.f;
                        slot[3 + k4] = make_float4(v[0], v[1], v[2], v[3]);
                    }
                }
            }
            // which strips evaluate this Gaussian: those with a pixel at or past it (last ids) that the
            // Gaussian can reach; one ballot per strip
            for (int k = 0; k < nwb * PX; ++k) {
                const bool keep = staged && idx <= s_sbf[k] &&
                                  ((!FIXED && ((bare >> k) & 1) != 0) || ((FIXED || !fixed) && strip_keep(s_box[k], cg)));
                const uint64_t m = __ballot(keep);
                if (lane == 0 && wave < nbw) s_mask[k][wave] = m;
            }
            {
                const uint64_t m = __ballot(high);
                if (lane == 0 && wave < nbw) s_high[wave] = m;
            }
            if constexpr (NWB > 1)
                for (int k = tr; k < nb * KT; k += (int)blockDim.x) s_tot[k] = 0.f;
            __syncthreads();
            uint64_t did = 0;
            for (int w2 = 0; w2 < nbw; ++w2) {
                uint64_t sm[PX], any = 0;
                did = 0;
#pragma unroll
                for (int h = 0; h < PX; ++h) {
                    sm[h] = uniform_u64(s_mask[wave * PX + h][w2]);
                    any |= sm[h];
                }
                const uint64_t high_m = uniform_u64(s_high[w2]);
                for (uint64_t m = any; m != 0; m &= m - 1) {
                    const int bit = (int)__builtin_ctzll(m), t = (w2 << 6) + bit;
                    const uint64_t bit_m = 1ull << bit;
                    const float4* rec = s_slot + t * kSlot4;
                    BwdGauss gs;
                    gs.a = rec[0]; gs.b = rec[1]; gs.c = rec[2];
                    if constexpr (FIXED) {
                        gs.op = gs.c.w;
                    } else {
                        gs.op = s_op[t];
                        if constexpr (DYN) {
                            gs.vel = mk3(s_vel[t].x, s_vel[t].y, s_vel[t].z);
                            gs.mv = mk3(s_mv[t].x, s_mv[t].y, s_mv[t].z);
                        }
                    }
                    const int32_t gidx = batch_end - t;
                    float rgb[CS];
#pragma unroll
                    for (int k = 0; k < CS; ++k) rgb[k] = 0.f;
                    if constexpr (CL > 0) {
#pragma unroll
                        for (int k4 = 0; k4 < C4; ++k4) {
                            const float4 v = rec[3 + k4];
                            if (4 * k4 + 0 < CDIM) rgb[4 * k4 + 0 < CS ? 4 * k4 + 0 : 0] = v.x;
                            if (4 * k4 + 1 < CDIM) rgb[4 * k4 + 1 < CS ? 4 * k4 + 1 : 0] = v.y;
                            if (4 * k4 + 2 < CDIM) rgb[4 * k4 + 2 < CS ? 4 * k4 + 2 : 0] = v.z;
                            if (4 * k4 + 3 < CDIM) rgb[4 * k4 + 3 < CS ? 4 * k4 + 3 : 0] = v.w;
                        }
                    } else if constexpr (CDIM > 0) {
                        const float* cp = p.colors + ((int64_t)s_id[t] * CDIM - (int64_t)cam * p.col_shift);
#pragma unroll
                        for (int k = 0; k < CDIM; ++k) rgb[k] = cp[k];
                    }
                    auto eval = [&](auto high_c, int h, float& rt) {
                        constexpr bool HIGH = decltype(high_c)::value;
                        BwdEval e;
                        if constexpr (FIXED) {
                            const RayEval v = ray_eval(gs.a, gs.b, gs.c, px[h].x, px[h].y);
                            e.vis = v.e;
                            e.grd = mk3(v.x, v.y, v.u);
                            e.inv_dd = v.inv_dd;
                            const float di = gs.b.w * v.inv_dd;
                            e.hit = di * v.u;
                            e.p = mk3(-e.hit * v.x, -e.hit * v.y, di * v.tt);
                        } else {
                            const f3 r0 = mk3(gs.a.x, gs.a.y, gs.a.z), r1 = mk3(gs.b.x, gs.b.y, gs.b.z),
                                     r2 = mk3(gs.c.x, gs.c.y, gs.c.z);
                            rt = px_rt[h];
                            f3 mu = mk3(gs.a.w, gs.b.w, gs.c.w);
                            if constexpr (DYN) mu = mu + rt * gs.vel;
                            e.gro = rows_mul(r0, r1, r2, px_ro[h] - mu);
                            e.grd = rows_mul(r0, r1, r2, px_rd[h]);
                            e.inv_dd = fminf(__builtin_amdgcn_rcpf(dot(e.grd, e.grd)), 3.40282347e38f);
                            const f3 c = cross(e.grd, e.gro);
                            e.vis = __builtin_amdgcn_exp2f(dot(c, c) * (e.inv_dd * -0.72134752f));
                            e.hit = -dot(e.gro, e.grd) * e.inv_dd;
                            // p = gro + hit_t grd in exact arithmetic; from the cross product its float32
                            // error is smaller (the direct sum moved per-pixel ray gradients beyond tolerance)
                            e.p = cross(c, e.grd) * e.inv_dd;
                        }
                        const float araw = gs.op * e.vis;
                        // (an alpha that is no number is kMaxAlpha, as the reference's min gives)
                        const bool reach = (HIGH ? fminf(kMaxAlpha, araw) : araw) >= 1.f / 255.f;
                        e.valid = gidx <= px[h].bin_final && reach;
                        e.araw = e.valid ? araw : 0.0f;
                        if constexpr (COUNT) {  // wave totals, scalar
                            n_eval += (uint64_t)__popcll(__builtin_amdgcn_ballot_w64(gidx <= px[h].bin_final));
                            n_contrib += (uint64_t)__popcll(__builtin_amdgcn_ballot_w64(e.valid));
                        }
                        return e;
                    };
                    // each strip evaluated, then composited, in turn (one evaluation live at a time), if a
                    // pixel of it takes the pair (eval3d_bwd.cu:209-212 skips pairs below the alpha
                    // threshold; an invalid pair adds exact zeros, so skipping whole strips changes nothing)
                    float acc[K];
#pragma unroll
                    for (int k = 0; k < K; ++k) acc[k] = 0.f;
                    bool some = false;
                    auto strips = [&](auto high_c) {
#pragma unroll
                        for (int h = 0; h < PX; ++h) {
                            if ((sm[h] & bit_m) == 0) continue;
                            float rt = 0.f;
                            const BwdEval e = eval(high_c, h, rt);
                            if (__builtin_amdgcn_ballot_w64(e.valid) == 0) continue;
                            some = true;
                            bwd_pair<CDIM, CS, K, DYN, RG, FIXED, decltype(high_c)::value>(px[h], rt, gs, e, rgb, acc);
                        }
                    };
                    // (two copies of the loop body where it is small; elsewhere the code costs more than the
                    // few instructions of the clamp)
                    if (!kBwdSplit<CDIM, DYN, RG, PX> || (high_m & bit_m) != 0) strips(std::true_type{});
                    else strips(std::false_type{});
                    if (!some) continue;  // nothing to reduce (wave-uniform)
                    did |= bit_m;
                    // wave totals by reduce-scatter: lane l ends with component 16 * chunk + (l >> 2)
                    float* out = reinterpret_cast<float*>(s_slot + t * kSlot4);
#pragma unroll
                    for (int ch = 0; ch < kChunks; ++ch) {
                        float chunk[16];
#pragma unroll
                        for (int k = 0; k < 16; ++k) chunk[k] = (16 * ch + k < K) ? acc[16 * ch + k] : 0.f;
                        const float tot = wave_reduce_scatter16_lds(chunk, min(16, K - 16 * ch), s_red[wave]);
                        const int kk = 16 * ch + (lane >> 2);
                        if ((lane & 3) == 0 && kk < K) {
                            if (kk < KO)
                                unsafeAtomicAdd(p.v_colors + ((int64_t)s_id[t] * CDIM - (int64_t)cam * p.col_shift) + kk, tot);
                            else if constexpr (NWB > 1) atomicAdd(&s_tot[t * KT + kk - KO], tot);
                            else out[kk - KO] = tot;
                        }
                    }
                }
                if constexpr (NWB > 1)
                    if (lane == 0) s_did[wave][w2] = did;
            }
            // The totals of wavefront w2's staged Gaussians, finished by one wavefront: its own (the only one)
            int w2 = 0;
            if constexpr (NWB > 1) {
                __syncthreads();
                w2 = wave;
                did = 0;
                if (wave < nbw)
                    for (int k = 0; k < nwb; ++k) did |= uniform_u64(s_did[k][w2]);
            } else {
                wave_lds_order();
            }
            if (did != 0) {
                // one lane per Gaussian: the totals in the original frame and world space
                const int t = (w2 << 6) + lane;
                float* tot = NWB > 1 ? s_tot + t * KT : reinterpret_cast<float*>(s_slot + t * kSlot4);
                if ((did >> lane) & 1) {
                    const int64_t gid = s_id[t] - (int64_t)cam * g.n;
                    const float4 q = p.quats[gid];
                    const f3 sc = ld3(p.scales + 3 * gid);
                    f3 r0, r1, r2;
                    iscl_rot_rows(q, sc, r0, r1, r2);
                    f3 vg = mk3(tot[G0], tot[G0 + 1], tot[G0 + 2]);
                    float Q[6];
#pragma unroll
                    for (int k = 0; k < 6; ++k) Q[k] = tot[G0 + 3 + k];
                    if constexpr (FIXED) {
                        turn_back(r0, r1, r2, ld3(p.means + 3 * gid), o0, vg, Q);
#pragma unroll
                        for (int k = 0; k < 6; ++k) tot[G0 + 3 + k] = Q[k];
                    }
                    f3 vm = rows_tmul(r0, r1, r2, vg);
                    tot[G0] = -vm.x; tot[G0 + 1] = -vm.y; tot[G0 + 2] = -vm.z;
                    tot[G0 + 9] = tot[G0 + 9] != 0.f ? tot[G0 + 9] / p.opac[gid] : 0.f;
                    if constexpr (DYN) {
                        vm = rows_tmul(r0, r1, r2, mk3(tot[G0 + 10], tot[G0 + 11], tot[G0 + 12]));
                        tot[G0 + 10] = -vm.x; tot[G0 + 11] = -vm.y; tot[G0 + 12] = -vm.z;
                    }
                }
                wave_lds_order();
                // 16 lanes per Gaussian: one atomic instruction per chunk of 16 components of four Gaussians
                const int kk0 = lane & 15;
#pragma unroll 1
                for (int s4 = 0; s4 < 64; s4 += 4) {
                    if (((did >> s4) & 15) == 0) continue;
                    const int bit = s4 + (lane >> 4);
                    const int tt = (w2 << 6) + bit;
                    const bool on = ((did >> bit) & 1) != 0;
                    const float* src = NWB > 1 ? s_tot + tt * KT : reinterpret_cast<const float*>(s_slot + tt * kSlot4);
                    const int32_t fid2 = s_id[tt];
                    const uint32_t gid = (uint32_t)(fid2 - (int64_t)cam * g.n);
#pragma unroll
                    for (int ch = 0; ch < (KT + 15) / 16; ++ch) {
                        const int k = 16 * ch + kk0;
                        if (!on || k >= KT) continue;
                        char* dst = reinterpret_cast<char*>(p.v_means) + s_dst[k] + (uint64_t)gid * s_step[k];
                        unsafeAtomicAdd(reinterpret_cast<float*>(dst), src[k]);
                    }
                }
            }
            __syncthreads();  // the slots are free for the next batch
        }
    };
    if constexpr (!DYN) {
        if (fixed) {
            sweep(std::true_type{});
            if constexpr (RG) {  // in the tile's basis, and dL/dgrd times k
                const TileBasis basis = get_basis(s_frame);
                const f3 ba = to32(basis.a), bx = to32(basis.x), by = to32(basis.y);
#pragma unroll
                for (int h = 0; h < PX; ++h) {
                    const int64_t pix = pixel_of(h);
                    if (pix < 0) continue;
                    float x, y, ik;
                    ray_xy(basis, ld3(p.ray_d + 3 * pix), x, y, ik);
                    f3 v = px[h].v_ro;
                    px[h].v_ro = v.x * ba + v.y * bx + v.z * by;
                    v = px[h].v_rd;
                    px[h].v_rd = (px[h].bin_final >= 0 ? ik : 0.f) * (v.x * ba + v.y * bx + v.z * by);
                }
            }
            if (bare != 0) {  // the pixels without a ray, left out above (last id -1), with their own last ids
#pragma unroll
                for (int h = 0; h < PX; ++h) {
                    const int64_t pix = pixel_of(h);
                    const bool in = pix >= 0 && px[h].bin_final < 0;
                    px[h].bin_final = in ? p.last_ids[pix] : -1;
                    px[h].v_d = in ? p.v_depth[pix] : 0.f;
                    const int m = wave_max(px[h].bin_final);
                    if (lane == 0) s_sbf[wave * PX + h] = m;
                }
                __syncthreads();
                int32_t last = -1;
                for (int k = 0; k < nwb * PX; ++k) last = max(last, s_sbf[k]);
                list_up_to(last);
            }
        }
    }
    if (DYN || !fixed || bare != 0) sweep(std::false_type{});
    if (COUNT && lane == 0) {  // one atomic per wave and counter
        atomicAdd(p.pair_counts, (unsigned long long)n_eval);
        atomicAdd(p.pair_counts + 1, (unsigned long long)n_contrib);
    }
    if constexpr (RG || DYN) {
#pragma unroll
        for (int h = 0; h < PX; ++h) {
            const int64_t pix = pixel_of(h);
            if (pix >= 0) {
                if constexpr (RG) {
                    st3(p.v_ray_o + 3 * pix, px[h].v_ro);
                    st3(p.v_ray_d + 3 * pix, px[h].v_rd);
                }
                if constexpr (DYN) p.v_time[pix] = px[h].v_t;
            }
        }
    }
}

// Variants without per-pixel ray gradients exist for CDIM <= kBwdNoRayCdim; larger CDIMs always compute
// them, two pixels per thread (the C-ABI then needs the ray-gradient buffers). Tiles of more than 256 pixels
// (up to kMaxTilePixels) take four pixels per thread in workgroups of up to 256 threads, with and without
// ray gradients. A tile of at most 128 pixels is one wavefront: its workgroup's LDS is sized for that (8 KB instead
// of 23 at three channels, where 23 leave a SIMD two wavefronts) and needs no totals shared between wavefronts
// (1280x800, 16x8 tiles: 424 -> 277 us). Channels read from HBM share few totals and keep the one variant.
constexpr int64_t kBwdFullGridWaves = 3 * 1024;

// one launch, with or without the pair counters
template <int CDIM, bool DYN, bool RG, int PX, int NT>
void launch_bwd(int n_blocks, int threads, const Eval3dParams& p, hipStream_t s) {
    if (p.pair_counts) eval3d_bwd_kernel<CDIM, DYN, RG, PX, NT, true><<<n_blocks, threads, 0, s>>>(p);
    else eval3d_bwd_kernel<CDIM, DYN, RG, PX, NT, false><<<n_blocks, threads, 0, s>>>(p);
}

}  // namespace

template <int CDIM>
int eval3d_bwd_cdim(bool dyn, bool ray_grads, const Eval3dParams& p, hipStream_t s) {
    const int n_blocks = p.g.n_tiles_w * p.g.n_tiles_h * p.g.n_cams;
    const int tile_px = p.g.tile_w * p.g.tile_h;
    // whole wavefronts (the reduction uses every lane)
    const int strips = (tile_px + 63) / 64;
    const int bs2 = (strips + 1) / 2 * 64;
    const int bs4 = (strips + 3) / 4 * 64;
    constexpr int T = kTileThreads;
    constexpr bool wide = CDIM > kBwdNoRayCdim;
    if (tile_px > T) {
        if (ray_grads || wide) {
            if (!p.v_ray_o || !p.v_ray_d)
                return xsg_fail(XSG_ERR_INVALID, "ray gradient buffers are required for cdim %d", CDIM);
            if (dyn) launch_bwd<CDIM, true, true, 4, T>(n_blocks, bs4, p, s);
            else launch_bwd<CDIM, false, true, 4, T>(n_blocks, bs4, p, s);
        } else if constexpr (!wide) {
            if (dyn) launch_bwd<CDIM, true, false, 4, T>(n_blocks, bs4, p, s);
            else launch_bwd<CDIM, false, false, 4, T>(n_blocks, bs4, p, s);
        }
        return XSG_OK;
    }
    if constexpr (!wide) {
        if (!ray_grads) {
            // four pixels per lane when the grid gives each of the 1024 SIMDs three waves of them (three
            // channels, 100 k Gaussians: 3432 tiles 181 us against 231, 8160 tiles 329 against 411); a small
            // grid (a 2048x128 lidar's 1024 tiles) runs two per lane on twice the waves (1000 tiles 132
            // against 155). From 1900 tiles four are ahead by 3 to 8 % there, but with motion or more channels
            // that was not measured. The caller may fix either
            const bool px4 = p.px_hint == 4 ||
                             (p.px_hint == 0 && (int64_t)n_blocks * (bs4 / 64) >= kBwdFullGridWaves);
            if (tile_px > 128 && px4) {
                if (dyn) launch_bwd<CDIM, true, false, 4, T / 4>(n_blocks, bs4, p, s);
                else launch_bwd<CDIM, false, false, 4, T / 4>(n_blocks, bs4, p, s);
            } else if (bs2 == 64) {
                if (dyn) launch_bwd<CDIM, true, false, 2, T / 4>(n_blocks, bs2, p, s);
                else launch_bwd<CDIM, false, false, 2, T / 4>(n_blocks, bs2, p, s);
            } else {
                if (dyn) launch_bwd<CDIM, true, false, 2, T / 2>(n_blocks, bs2, p, s);
                else launch_bwd<CDIM, false, false, 2, T / 2>(n_blocks, bs2, p, s);
            }
            return XSG_OK;
        }
    }
    if (!p.v_ray_o || !p.v_ray_d) return xsg_fail(XSG_ERR_INVALID, "ray gradient buffers are required for cdim %d", CDIM);
    if constexpr (CDIM <= kBwdColorLdsMax) {
        if (bs2 == 64) {
            if (dyn) launch_bwd<CDIM, true, true, 2, T / 4>(n_blocks, bs2, p, s);
            else launch_bwd<CDIM, false, true, 2, T / 4>(n_blocks, bs2, p, s);
            return XSG_OK;
        }
    }
    if (dyn) launch_bwd<CDIM, true, true, 2, T / 2>(n_blocks, bs2, p, s);
    else launch_bwd<CDIM, false, true, 2, T / 2>(n_blocks, bs2, p, s);
    return XSG_OK;
}

}  // namespace xsg
