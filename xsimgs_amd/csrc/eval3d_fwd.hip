// Forward eval3d compositing: rasterize_eval3d_[dynamic_]fwd_kernel (eval3d_fwd.cu:34-166,
// eval3d_dynamic_fwd.cu:37-173).
//
// Bound: VALU issue. On gfx950 a wave64 FP32 multiply, add or FMA on vector registers issues every two
// cycles, a compare, select, min or any instruction with a scalar-register operand every four, an exp2 or
// reciprocal every eight; a broadcast 16-byte LDS read holds the compute unit's LDS for about four. The
// kernel is laid out for those rates:
//  * a wavefront owns PX strips of 64 consecutive pixels of the tile, one pixel of each per lane, so that
//    the LDS reads and the loop's scalar work of a Gaussian serve PX pixels;
//  * a batch's Gaussians that some pixel of the wavefront can take are listed (their LDS byte offsets)
//    while they are staged, and the pair loop walks the list U at a time: no bit scans, and PX * U
//    independent evaluations in flight;
//  * a pair that is not taken has its alpha cleared by integer arithmetic on the sign of 1/255 - alpha,
//    after which it changes nothing, so nothing else is selected; a pixel whose transmittance has run out
//    is a pixel that no alpha reaches (its threshold becomes infinite). Running out is tested once for the
//    U Gaussians and resolved apart, which each pixel does at most once.
// The whole op against one pixel per lane, a bit scan per Gaussian and every tile evaluated as M (ro - mu), M rd:
// 1920x1080, 1 M Gaussians 240 -> 188-197 us; six cameras of 1600x900 886 -> 655-716; 1237x701 115 -> 85; 2048x128
// lidar 72 -> 49-54; 256x256 63 -> 25; 32 channels at 640x480 170 -> 88; moving origins, which keep that form, 154 -> 154.
#include <type_traits>

#include "xsg_eval3d.h"

namespace xsg {
namespace {

// Channels staged in LDS: up to 33 (wider colours are read from HBM, as scalars, at half the FMA rate), up
// to 8 in the workgroups of large tiles, whose batches are larger.
constexpr int kFwdColorLdsMax = 33;
template <int NT>
constexpr int kFwdLdsColors = NT > kTileThreads ? 8 : kFwdColorLdsMax;

// Pixels per lane (PX) and Gaussians per step (U). Two pixels per lane halve the LDS reads and the loop's
// scalar work of a pair, but a tile is then half as many wavefronts, each twice as long, and its strips share
// one list: worth it once the grid has many rounds of wavefronts (16 k of two pixels at 1920x1080: 190 us
// against 194; 68 k for six 1600x900 cameras: 667 against 700; but 6.9 k at 1237x701: 99 against 92), and only
// where the tile's strips pair up. Where the grid leaves at most four wavefronts per SIMD, the length of a
// wavefront's chain counts, and U = 4 keeps four evaluations of it in flight (256x256: 24 us against 29).
constexpr int64_t kFwdTwoPixelWaves = 8 * 1024;
constexpr int64_t kFwdDeepWaves = 4 * 1024;

// Wavefronts per SIMD the compiler is asked to fit: five (96 registers; a few set-up values spill) for up to
// four channels, four with U = 4, whose grids bring no more; wider colours take what registers they need.
template <int CDIM, int U, int NT>
constexpr int kFwdWaves = CDIM > 4 || NT > kTileThreads ? 1 : U > 1 ? 4 : 5;

template <int CDIM, bool DYN, int PX, int U, int NT, bool COUNT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(kFwdWaves<CDIM, U, NT>))) void eval3d_fwd_kernel(
    Eval3dParams p) {
    constexpr int CL = (CDIM > 0 && CDIM <= kFwdLdsColors<NT>) ? CDIM : 0;  // channels staged in LDS
    constexpr int C4 = (CL + 3) / 4;                                       // float4 slots of them
    constexpr int CS = CDIM > 0 ? CDIM : 1;
    constexpr int NW = NT / 64;
    constexpr int NS = NW * PX;  // strips
    // The opacity rides in the last colour float4's first free component when there is one
    constexpr bool OP_IN_COL = CL > 0 && (CL & 3) != 0;
    // Every per-Gaussian slot is an array indexed by the batch position, so that one address register (16
    // times the position) serves all reads of a Gaussian; position NT holds a Gaussian no pixel takes,
    // which fills the lists up to whole steps. One origin: the affine rows with -log2(e) / 2 D^2, D and the
    // opacity in the fourth components; else the rows of M with the mean there.
    __shared__ float4 s_m0[NT + 1], s_m1[NT + 1], s_m2[NT + 1];
    __shared__ float4 s_op[OP_IN_COL ? 1 : NT + 1];  // opacity, when no colour slot has room
    __shared__ float4 s_vel[DYN ? NT + 1 : 1];
    __shared__ float4 s_col[C4 > 0 ? C4 : 1][NT + 1];
    __shared__ int32_t s_id[CL > 0 || CDIM == 0 ? 1 : NT];
    static_assert(U == 1 || CL > 0 || CDIM == 0, "the lists' filling has no colours in HBM");
    __shared__ float4 s_box[NS];                        // the strips' boxes of (x, y)
    __shared__ float s_ik[DYN ? 1 : PX][DYN ? 1 : NT];  // each pixel's 1 / k, 0 without a ray
    __shared__ TileFrame s_frame;
    __shared__ float s_slack[2][NW];  // largest distance from the basis pixel's origin, and time from its own
    // [wavefront][staging wavefront]: the Gaussians it evaluates, and their number
    __shared__ uint16_t s_list[NW][NW][64 + 2 * U];
    __shared__ int s_cnt[NW][NW];
    __shared__ int s_vote[NW];

    const TileGrid& g = p.g;
    const int n_tiles = g.n_tiles_w * g.n_tiles_h;
    const int nblocks = n_tiles * g.n_cams;
    const int logical = xcd_tile((int)blockIdx.x, nblocks);
    const int cam = logical / n_tiles, tile = logical - cam * n_tiles;
    const int tr = threadIdx.x;
    const int bs = g.tile_w * g.tile_h;
    const int nw = (int)(blockDim.x >> 6);  // whole wavefronts; strips past the tile's pixels hold none
    const int wave = tr >> 6, lane = tr & 63;
    const int trow = tile / g.n_tiles_w, tcol = tile - trow * g.n_tiles_w;
    const int32_t range_start = p.offsets[logical];  // utils.h:48-58
    const int32_t range_end = (logical == nblocks - 1) ? (int32_t)g.n_isects : p.offsets[logical + 1];
    const int64_t hw = (int64_t)g.width * g.height;
    if (past_image(g, trow, tcol)) {
        if (p.tile_work && tr == 0) p.tile_work[logical] = 0;
        return;
    }

    // strip h's pixel of this lane: its index in the [cams, H, W] images (utils.h:32-44), -1 outside;
    // recomputed where needed rather than kept in registers (opaque: or the compiler keeps it)
    auto pixel_at = [&](int q) -> int64_t {
        const int ty = q / g.tile_w, tx = q - ty * g.tile_w;
        const int i = trow * g.tile_h + ty, j = tcol * g.tile_w + tx;
        return q < bs && i < g.height && j < g.width ? (int64_t)cam * hw + (int64_t)i * g.width + j : -1;
    };
    auto pixel_of = [&](int h) { return pixel_at((wave * PX + h) * 64 + opaque(lane)); };
    // the conjunction of the wavefronts' votes, written to s_vote before the last barrier
    auto votes = [&]() {
        int v = -1;
        for (int k = 0; k < nw; ++k) v &= s_vote[k];
        return __builtin_amdgcn_readfirstlane(v);
    };
    const int32_t n_range = range_end - range_start;
    const int nthr = (int)blockDim.x;  // Gaussians per batch
    const int num_batches = n_range > 0 ? (n_range + nthr - 1) / nthr : 0;
    auto staged_at = [&](int b) { return (uint32_t)range_start + (uint32_t)(nthr * b + tr) < (uint32_t)range_end; };
    // The flatten id a thread stages in the next batch is loaded one batch ahead, and the first batch's
    // Gaussian before the tile's set-up: their latencies then overlap the pair loop and the set-up.
    struct Raw {
        f3 mu, sc, vel;
        float4 q;
        float op;
    };
    int32_t fid_next = 0;
    auto load_raw = [&](bool some) {
        Raw r = {mk3(0.f, 0.f, 0.f), mk3(1.f, 1.f, 1.f), mk3(0.f, 0.f, 0.f), make_float4(1.f, 0.f, 0.f, 0.f), 0.f};
        if (some) {
            const int64_t gid = fid_next - (int64_t)cam * g.n;
            r.mu = ld3(p.means + 3 * gid);
            r.op = p.opac[gid];
            r.q = p.quats[gid];
            r.sc = ld3(p.scales + 3 * gid);
            if constexpr (DYN) {
                if (p.velocity) r.vel = ld3(p.velocity + 3 * gid);
            }
        }
        return r;
    };
    if (num_batches > 0 && staged_at(0)) fid_next = p.flatten[(uint32_t)range_start + (uint32_t)tr];
    Raw raw = load_raw(num_batches > 0 && staged_at(0));
    bool inside[PX];
    float px[PX], py[PX];  // the pixels' (x, y)
    if (tr == 0) {
        s_m0[NT] = s_m1[NT] = s_m2[NT] = make_float4(0.f, 0.f, 0.f, 0.f);
        if constexpr (!OP_IN_COL) s_op[NT] = make_float4(0.f, 0.f, 0.f, 0.f);
        if constexpr (DYN) s_vel[NT] = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int k4 = 0; k4 < C4; ++k4) s_col[k4][NT] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    // The pixels' rays and times, loaded before the basis pixel's is looked at (their latencies overlap)
    f3 ray_o[PX], ray_d[PX];
    float ray_t[PX];
#pragma unroll
    for (int h = 0; h < PX; ++h) {
        const int64_t pix = pixel_of(h);
        inside[h] = pix >= 0;
        ray_o[h] = inside[h] ? ld3(p.ray_o + 3 * pix) : mk3(0.f, 0.f, 0.f);
        ray_d[h] = inside[h] ? ld3(p.ray_d + 3 * pix) : mk3(0.f, 0.f, 0.f);
        ray_t[h] = 0.f;
        if constexpr (DYN) ray_t[h] = inside[h] && p.rtd ? p.rtd[pix] : 0.f;
    }
    // the left end of the tile's middle row, and the pixel its basis is built on
    const int64_t ps = (int64_t)cam * hw + (int64_t)min(trow * g.tile_h + g.tile_h / 2, g.height - 1) * g.width + tcol * g.tile_w;
    const f3 side = ld3(p.ray_d + 3 * ps);
    const BasisPixel mid = basis_pixel<DYN>(p.ray_o, p.ray_d, p.rtd, ps + min(g.tile_w / 2, g.width - 1 - tcol * g.tile_w), bs, pixel_at);
    const f3 o0 = mid.o;
    const float rt0 = mid.t;
    const TileBasis basis = uniform_basis(tile_basis(mid.d, side));
    if (tr == 0) put_basis(s_frame, basis);
    bool same = true, some = false, ray[PX];
    int bare = 0;  // strips
    float far2 = 0.f, late = 0.f;
#pragma unroll
    for (int h = 0; h < PX; ++h) {
        const f3 away = ray_o[h] - o0;
        const float rt = ray_t[h] - rt0;
        float ik;
        ray[h] = ray_xy(basis, ray_d[h], px[h], py[h], ik) && finite3(away) && isfinite(rt) && inside[h];
        const float4 box = strip_box(ray[h], px[h], py[h]);
        same = same && (!ray[h] || (__float_as_uint(ray_o[h].x) == __float_as_uint(o0.x) &&
                                    __float_as_uint(ray_o[h].y) == __float_as_uint(o0.y) &&
                                    __float_as_uint(ray_o[h].z) == __float_as_uint(o0.z)));
        some = some || ray[h];
        far2 = ray[h] ? fmaxf(far2, dot(away, away)) : far2;
        late = ray[h] ? fmaxf(late, fabsf(rt)) : late;
        px[h] = ray[h] ? px[h] : 0.f;
        py[h] = ray[h] ? py[h] : 0.f;
        if (__ballot(inside[h] && !ray[h]) != 0) bare |= 1 << (wave * PX + h);
        if (lane == 0) s_box[wave * PX + h] = box;
        if constexpr (!DYN) s_ik[h][tr] = ray[h] ? ik : 0.f;
    }
    {
        const int v = tile_vote(__ballot(!same) == 0, __ballot(some) != 0, bare);
        if (lane == 0) s_vote[wave] = v;
        const float f = wave_max_f(far2), l = DYN ? wave_max_f(late) : 0.f;
        if (lane == 0) { s_slack[0][wave] = f; s_slack[1][wave] = l; }
    }
    __syncthreads();
    const int vote = votes();
    // one origin (as float32 values): the pairs in the turned frame's affine form
    const bool fixed = !DYN && (vote & (kVoteOneOrigin | kVoteNoRay)) == kVoteOneOrigin;
    bare = bare_strips(vote);
    if (tr == 0) tile_bounds(s_frame, s_box, nw * PX, s_slack[0], s_slack[1], nw);
    __syncthreads();

    // A pixel takes a pair when alpha > thr: the largest float below 1/255 while the pixel is open, then
    // infinity (also outside the image, and in the other form's sweep).
    constexpr float kOpen = 0.00392156839370728f;  // 1.f / 255.f less one ulp
    float T[PX], depth[PX], thr[PX], acc[PX][CS];
    uint64_t open[PX];  // the wavefront's open pixels
    int32_t cur_idx[PX];
    uint64_t n_eval = 0, n_contrib = 0;  // wave totals (uniform) when counting
#pragma unroll
    for (int h = 0; h < PX; ++h) {
        T[h] = 1.f; depth[h] = 0.f; cur_idx[h] = 0;
        const bool in = fixed ? ray[h] : inside[h];
        thr[h] = in ? kOpen : __builtin_inff();
        open[h] = __ballot(in);
#pragma unroll
        for (int k = 0; k < CS; ++k) acc[h][k] = 0.f;
    }
    auto any_open = [&]() {
        uint64_t m = open[0];
#pragma unroll
        for (int h = 1; h < PX; ++h) m |= open[h];
        return m != 0;
    };

    // the whole sweep is instantiated for both origin modes, so that neither carries the other's registers
    auto sweep = [&](auto fixed_c) {
        constexpr bool FIXED = decltype(fixed_c)::value;
        for (int b = 0; b < num_batches;) {
            const uint32_t batch_start = (uint32_t)range_start + (uint32_t)(nthr * b);
            const bool staged = staged_at(b);
            const int32_t fid = fid_next;
            if (staged_at(b + 1)) fid_next = p.flatten[batch_start + (uint32_t)(nthr + tr)];
            StripCull cg;
            if (staged) {
                const f3 mu = raw.mu, sc = raw.sc;
                const float4 q = raw.q;
                const float op = raw.op;
                const CullInput in = cull_input(mu, sc, q, op);
                f3 r0, r1, r2;
                iscl_rot_rows(q, sc, r0, r1, r2);
                f3 vel = mk3(0.f, 0.f, 0.f);
                if constexpr (DYN) {
                    vel = raw.vel;
                    s_vel[tr] = make_float4(vel.x, vel.y, vel.z, 0.f);
                }
                f3 at = mu;  // where the Gaussian is at the basis pixel's time
                if constexpr (DYN) at = mu + rt0 * vel;
                if constexpr (FIXED) {
                    const RayFrame f = ray_frame(r0, r1, r2, at, o0, get_basis(s_frame));
                    s_m0[tr] = make_float4(f.a1.x, f.a1.y, f.a1.z, f.D * f.D * -0.72134752f);
                    s_m1[tr] = make_float4(f.a2.x, f.a2.y, f.a2.z, f.D);
                    s_m2[tr] = make_float4(f.au.x, f.au.y, f.au.z, op);
                    cg = strip_cull(f, in, s_frame.hx, s_frame.hy);
                } else {
                    s_m0[tr] = make_float4(r0.x, r0.y, r0.z, mu.x);
                    s_m1[tr] = make_float4(r1.x, r1.y, r1.z, mu.y);
                    s_m2[tr] = make_float4(r2.x, r2.y, r2.z, mu.z);
                    if constexpr (!OP_IN_COL) s_op[tr].x = op;
                    cg = strip_cull_moving(r0, r1, r2, at, sc, in, o0,
                                           s_frame.slack_o + s_frame.slack_t * __builtin_amdgcn_sqrtf(dot(vel, vel)), s_frame);
                }
                if constexpr (CL > 0) {
                    const float* cp = p.colors + ((int64_t)fid * CDIM - (int64_t)cam * p.col_shift);
#pragma unroll
                    for (int k4 = 0; k4 < C4; ++k4) {
                        float v[4];
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            v[j] = (4 * k4 + j < CL) ? cp[4 * k4 + j] : (OP_IN_COL && 4 * k4 + j == CL) ? op : 0.f;
                        s_col[k4][tr] = make_float4(v[0], v[1], v[2], v[3]);
                    }
                } else if constexpr (CDIM > 0) {
                    s_id[tr] = fid;
                }
            }
            // the lists of the Gaussians each wavefront evaluates, in order, filled up to whole steps
            for (int k = 0; k < nw; ++k) {
                bool keep = false;
                if (staged) {
#pragma unroll 1
                    for (int h = 0; h < PX; ++h)
                        keep = keep || (!FIXED && ((bare >> (k * PX + h)) & 1) != 0) ||
                               ((FIXED || !fixed) && strip_keep(s_box[k * PX + h], cg));
                }
                const uint64_t m = __ballot(keep);
                const int cnt = (int)__popcll(m);
                uint16_t* list = s_list[k][wave];
                if (keep) list[(int)__popcll(m & ((1ull << lane) - 1))] = (uint16_t)(16 * tr);
                if (lane < U) list[cnt + lane] = (uint16_t)(16 * NT);
                if (lane == 0) s_cnt[k][wave] = cnt;
            }
            __syncthreads();

            int32_t cur[PX];  // byte offset of the last pair taken in this batch
#pragma unroll
            for (int h = 0; h < PX; ++h) cur[h] = -1;
            // the lists' pairs for the strips [H0, H0 + NH)
            auto pairs = [&](auto h0_c, auto nh_c) {
            constexpr int H0 = decltype(h0_c)::value, H1 = H0 + decltype(nh_c)::value;
            auto some_open = [&]() {
                uint64_t m = open[H0];
#pragma unroll
                for (int h = H0 + 1; h < H1; ++h) m |= open[h];
                return m != 0;
            };
            f3 rd[FIXED ? 1 : PX], ro[FIXED ? 1 : PX];
            float rt[FIXED ? 1 : PX];
            if constexpr (!FIXED) {
#pragma unroll
                for (int h = H0; h < H1; ++h) {
                    const int64_t pix = pixel_of(h);
                    rd[h] = pix >= 0 ? ld3(p.ray_d + 3 * pix) : mk3(0.f, 0.f, 0.f);
                    ro[h] = pix >= 0 ? ld3(p.ray_o + 3 * pix) : mk3(0.f, 0.f, 0.f);
                    rt[h] = 0.f;
                    if constexpr (DYN) rt[h] = (pix >= 0 && p.rtd) ? p.rtd[pix] : 0.0f;
                }
            }
            for (int w2 = 0; w2 < nw; ++w2) {
                int cnt = __builtin_amdgcn_readfirstlane(s_cnt[wave][w2]);
                const uint16_t* list = s_list[wave][w2];
                uint32_t off[U];
#pragma unroll
                for (int u = 0; u < U; ++u) off[u] = list[u];
                for (int i = 0; i < cnt; i += U) {
                    const int n_step = min(U, cnt - i);  // without the filling
                    float alpha[U][PX], hit[U][PX];
                    int32_t took[U][PX];  // all ones where the pair is taken
                    float4 cl[U][C4 > 0 ? C4 : 1];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        auto at = [&](const float4* base) {
                            return *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(base) + off[u]);
                        };
                        const float4 a = at(s_m0), bq = at(s_m1), cq = at(s_m2);
                        const f3 r0 = mk3(a.x, a.y, a.z), r1 = mk3(bq.x, bq.y, bq.z), r2 = mk3(cq.x, cq.y, cq.z);
#pragma unroll
                        for (int k4 = 0; k4 < C4; ++k4) cl[u][k4] = at(s_col[k4]);
                        float op;
                        if constexpr (FIXED) {
                            op = cq.w;
                        } else if constexpr (OP_IN_COL) {
                            const float4 last = cl[u][C4 - 1];
                            op = (CL & 3) == 1 ? last.y : (CL & 3) == 2 ? last.z : last.w;
                        } else {
                            op = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(s_op) + off[u]);
                        }
                        f3 vel = mk3(0.f, 0.f, 0.f);
                        if constexpr (DYN) {
                            const float4 v = at(s_vel);
                            vel = mk3(v.x, v.y, v.z);
                        }
#pragma unroll
                        for (int h = H0; h < H1; ++h) {
                            float e;
                            if constexpr (FIXED) {
                                const RayEval v = ray_eval(a, bq, cq, px[h], py[h]);
                                e = v.e;
                                hit[u][h] = bq.w * (v.u * v.inv_dd);  // -k hit_t
                            } else {
                                f3 mu = mk3(a.w, bq.w, cq.w);
                                if constexpr (DYN) mu = mu + rt[h] * vel;
                                const f3 gro = rows_mul(r0, r1, r2, ro[h] - mu);
                                const f3 grd = rows_mul(r0, r1, r2, rd[h]);
                                // 1/|grd|^2, capped so that grd = 0 gives power 0 as safe_normalize does
                                const float inv_dd = fminf(__builtin_amdgcn_rcpf(dot(grd, grd)), 3.40282347e38f);
                                // |n x gro|^2 = |grd x gro|^2 / |grd|^2; exp(-x/2) = exp2(x * -log2(e)/2)
                                const f3 cr = cross(grd, gro);
                                e = __builtin_amdgcn_exp2f(dot(cr, cr) * (inv_dd * -0.72134752f));
                                hit[u][h] = -dot(gro, grd) * inv_dd;
                            }
                            const float al = fminf(0.999f, op * e);
                            took[u][h] = opaque(__float_as_int(thr[h] - al) >> 31);
                            alpha[u][h] = __int_as_float(__float_as_int(al) & took[u][h]);
                        }
                    }
                    uint32_t off_now[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        off_now[u] = off[u];
                        off[u] = list[i + U + u];  // past the list's end at most once, and then unused
                    }
                    if constexpr (COUNT) {
#pragma unroll
                        for (int h = H0; h < H1; ++h)
                            n_eval += (uint64_t)__popcll(open[h]) * (uint64_t)n_step;
                    }
#pragma unroll
                    for (int h = H0; h < H1; ++h) {
                        // termination is exclusive (eval3d_fwd.cu:135-139): the pair that would bring the
                        // transmittance to 1e-4 closes the pixel and is not taken
                        float t = T[h];
#pragma unroll
                        for (int u = 0; u < U; ++u) t = fmaf(-alpha[u][h], t, t);
                        if (__ballot(t <= 1e-4f) != 0) {
                            float tc = T[h];
#pragma unroll
                            for (int u = 0; u < U; ++u) {
                                const float next = fmaf(-alpha[u][h], tc, tc);
                                const bool ends = next <= 1e-4f;
                                if constexpr (COUNT)  // the pairs after a pixel's last are not evaluated
                                    n_eval -= (uint64_t)__popcll(__ballot(ends)) * (uint64_t)max(0, n_step - u - 1);
                                thr[h] = ends ? __builtin_inff() : thr[h];
#pragma unroll
                                for (int v = u; v < U; ++v) {
                                    alpha[v][h] = ends ? 0.f : alpha[v][h];
                                    took[v][h] = ends ? 0 : took[v][h];
                                }
                                tc = ends ? tc : next;
                            }
                            open[h] = __ballot(thr[h] == kOpen);
                            if (!some_open()) cnt = 0;  // the last step of this wavefront
                        }
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        float wide[CL == 0 && CDIM > 0 ? CDIM : 1];
                        if constexpr (CL == 0 && CDIM > 0) {
                            const int32_t id = *reinterpret_cast<const int32_t*>(reinterpret_cast<const char*>(s_id) + off_now[u] / 4);
                            const float* cp = p.colors + ((int64_t)id * CDIM - (int64_t)cam * p.col_shift);
#pragma unroll
                            for (int k = 0; k < CDIM; ++k) wide[k] = cp[k];
                        }
#pragma unroll
                        for (int h = H0; h < H1; ++h) {
                            const float vis = alpha[u][h] * T[h];
                            T[h] = fmaf(-alpha[u][h], T[h], T[h]);
                            depth[h] = fmaf(vis, hit[u][h], depth[h]);
#pragma unroll
                            for (int k = 0; k < CDIM; ++k) {
                                float c;
                                if constexpr (CL > 0) {
                                    const float4 cv = cl[u][k / 4];
                                    c = (k & 3) == 0 ? cv.x : (k & 3) == 1 ? cv.y : (k & 3) == 2 ? cv.z : cv.w;
                                } else {
                                    c = wide[k];
                                }
                                acc[h][k] = fmaf(c, vis, acc[h][k]);
                            }
                            cur[h] = (took[u][h] & (int32_t)off_now[u]) | (~took[u][h] & cur[h]);
                            if constexpr (COUNT) n_contrib += (uint64_t)__popcll(__ballot(took[u][h] != 0));
                        }
                    }
                }
                if (!some_open()) break;
            }
            };
            if constexpr (FIXED || PX == 1) {
                if (any_open()) pairs(std::integral_constant<int, 0>{}, std::integral_constant<int, PX>{});
            } else {  // a strip at a time: the pixels' origins and times would take too many registers
                if (open[0]) pairs(std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{});
                if (open[1]) pairs(std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{});
            }
#pragma unroll
            for (int h = 0; h < PX; ++h) cur_idx[h] = cur[h] >= 0 ? (int32_t)batch_start + (cur[h] >> 4) : cur_idx[h];
            if (++b == num_batches) break;
            if (lane == 0) s_vote[wave] = any_open() ? 0 : 1;
            __syncthreads();  // also ends the reads of this batch
            if (votes() != 0) break;
            raw = load_raw(staged_at(b));
        }
    };
    if constexpr (!DYN) {
        if (fixed) {
            sweep(std::true_type{});
#pragma unroll
            for (int h = 0; h < PX; ++h) depth[h] = -depth[h] * s_ik[h][tr];
            if (bare != 0) {  // the pixels without a ray, which took nothing yet
                __syncthreads();
#pragma unroll
                for (int h = 0; h < PX; ++h) {
                    const bool in = pixel_of(h) >= 0 && s_ik[h][tr] == 0.f;
                    thr[h] = in ? kOpen : __builtin_inff();
                    open[h] = __ballot(in);
                }
                if (num_batches > 0 && staged_at(0)) fid_next = p.flatten[(uint32_t)range_start + (uint32_t)tr];
                raw = load_raw(num_batches > 0 && staged_at(0));
            }
        }
    }
    if (DYN || !fixed || bare != 0) sweep(std::false_type{});
    if (COUNT && lane == 0) {  // one atomic per wave and counter
        atomicAdd(p.pair_counts, (unsigned long long)n_eval);
        atomicAdd(p.pair_counts + 1, (unsigned long long)n_contrib);
    }
#pragma unroll
    for (int h = 0; h < PX; ++h) {
        const int64_t pix = pixel_of(h);
        if (pix >= 0) {
            p.out_alpha[pix] = 1.0f - T[h];
            p.out_depth[pix] = depth[h];
#pragma unroll
            for (int k = 0; k < CDIM; ++k) p.out_rgb[pix * CDIM + k] = acc[h][k];
            p.out_last[pix] = cur_idx[h];
        }
    }
    if (p.tile_work) {  // the tile's backward work: its intersections up to the largest last id
        __shared__ int s_last[NW];
        int m = -1;
#pragma unroll
        for (int h = 0; h < PX; ++h) m = pixel_of(h) >= 0 ? max(m, cur_idx[h]) : m;
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) m = max(m, __shfl_xor(m, off, 64));
        if (lane == 0) s_last[wave] = m;
        __syncthreads();
        if (tr == 0) {
            for (int k = 1; k < nw; ++k) m = max(m, s_last[k]);
            p.tile_work[logical] = max(0, min(range_end - 1, m) - range_start + 1);
        }
    }
}

template <int CDIM>
int launch_cdim(bool dyn, const Eval3dParams& p, hipStream_t s) {
    const int n_blocks = p.g.n_tiles_w * p.g.n_tiles_h * p.g.n_cams;
    const int tile_px = p.g.tile_w * p.g.tile_h;
    const int strips = (tile_px + 63) / 64;
    const int nt1 = 64 * strips, nt2 = 64 * ((strips + 1) / 2);  // threads with one / two pixels per lane
    constexpr int T = kTileThreads;
    auto go = [&](auto count_c, auto dyn_c) {
        constexpr bool C = decltype(count_c)::value, D = decltype(dyn_c)::value;
        constexpr bool two = CDIM <= kFwdColorLdsMax;  // wider colours' sums fill the registers of one pixel
        // large tiles: the general form takes its strips one at a time, which reads colours from HBM twice
        // (32x32 tiles with motion: 16 channels 416 us against 333; but 9 channels 259 against 305)
        constexpr int big = two && !(D && CDIM >= 16) ? 2 : 1;
        constexpr int U4 = CDIM <= 4 ? 4 : 1;
        // With more than 16 channels in LDS a workgroup of one or two wavefronts takes arrays of its own size:
        // those of four leave a compute unit four workgroups (17 channels, 37 KB; 1280x800 in 8x8 tiles: 370 us
        // against 146)
        constexpr bool sized = CDIM > 16 && CDIM <= kFwdColorLdsMax;
        if (tile_px > T)  // up to the reference's 1024 pixels (eval3d_fwd.cu:204-221)
            eval3d_fwd_kernel<CDIM, D, big, 1, kMaxTilePixels / big, C><<<n_blocks, big == 2 ? nt2 : nt1, 0, s>>>(p);
        else if (two && !D && strips % 2 == 0 && (int64_t)n_blocks * (nt2 / 64) >= kFwdTwoPixelWaves)
            eval3d_fwd_kernel<CDIM, false, two ? 2 : 1, 1, T / (two ? 2 : 1), C>
                <<<n_blocks, two ? nt2 : nt1, 0, s>>>(p);
        else if (sized && strips == 1)
            eval3d_fwd_kernel<CDIM, D, 1, 1, sized ? T / 4 : T, C><<<n_blocks, nt1, 0, s>>>(p);
        else if (sized && strips == 2)
            eval3d_fwd_kernel<CDIM, D, 1, 1, sized ? T / 2 : T, C><<<n_blocks, nt1, 0, s>>>(p);
        else if ((int64_t)n_blocks * strips > kFwdDeepWaves)
            eval3d_fwd_kernel<CDIM, D, 1, 1, T, C><<<n_blocks, nt1, 0, s>>>(p);
        else
            eval3d_fwd_kernel<CDIM, D, 1, U4, T, C><<<n_blocks, nt1, 0, s>>>(p);
    };
    auto with_dyn = [&](auto count_c) {
        if (dyn) go(count_c, std::true_type{});
        else go(count_c, std::false_type{});
    };
    if (p.pair_counts) with_dyn(std::true_type{});
    else with_dyn(std::false_type{});
    return XSG_OK;
}

}  // namespace

int eval3d_fwd_launch(int cdim, bool dyn, const Eval3dParams& p, hipStream_t s) {
    switch (cdim) {
#define XSG_CASE(C) case C: return launch_cdim<C>(dyn, p, s);
        XSG_CDIM_LIST(XSG_CASE)
#undef XSG_CASE
        default: return xsg_fail(XSG_ERR_INVALID, "Unsupported number of channels: %d", cdim);
    }
}

}  // namespace xsg
