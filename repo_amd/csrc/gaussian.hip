// 2D Gaussian splats: the kernels behind GsRenderFunction
// (tilelang_renderer.py:149-490) and the op-level functions of
// ops/forward2d.py, ops/backward2d.py, ops/intersects.py and ops/rasterize.py.
//
//   k_gs_project      forward2d.py:14-164, one thread per Gaussian
//   k_gs_pack         per-Gaussian 48-byte raster records (GsRec)
//   k_gs_raster_fwd   rasterize.py:18-157: one workgroup per tile, one or two
//                     pixels per lane; each wave tests 64 list entries at a
//                     time against its pixels' rectangle, one entry per lane,
//                     visits those whose ellipse meets it with scalar loads
//                     of their records, and leaves the list when all of its
//                     pixels are done
//   k_gs_raster_bwd   rasterize.py:160-529: each wave walks back from the
//                     largest final index of its pixels over the same
//                     entries; per entry the wave sums its pixels' nine terms
//                     with DPP reductions into LDS, and adds them 64 at a
//                     time with float atomics
//   k_gs_project_bwd  backward2d.py:8-151 (with the meta scaling of
//                     tilelang_renderer.py:111-116)
//   k_gs_map_ref      intersects.py:12-226 in the reference's int64 layout
//
// Arithmetic follows the spec shared with oracle/gs_oracle.c (cs_common.h):
// the forward's outputs are bit-identical to it.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/cubicsplat_hip.h"
#include "cs_common.h"

namespace cs {

constexpr int kGsThreads = 256;
constexpr float kGsAlphaCapFwd = (float)0.999;  // rasterize.py:49
constexpr float kGsAlphaCapBwd = (float)0.99;   // rasterize.py:246
constexpr float kGsAlphaMin = (float)(1.0 / 255.0);
constexpr float kGsTStop = (float)1e-4;

static_assert(sizeof(GsRec) == 48, "GsRec is read as 12 dwords");

__global__ __launch_bounds__(kGsThreads) void k_gs_project(
    const float2* __restrict__ means, const float2* __restrict__ scales,
    const float* __restrict__ rot, int n, int img_h, int img_w, int block_x, int block_y,
    int tbx, int tby, float2* __restrict__ xys, float* __restrict__ depths,
    int32_t* __restrict__ radii, float* __restrict__ conics, int32_t* __restrict__ tiles_hit) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float ox = 0.5f * (float)img_w, oy = 0.5f * (float)img_h;
    const float2 m = means[i], s = scales[i];
    const float cx = ox * m.x + ox, cy = oy * m.y + oy;
    float sr, cr;
    spec_sincosf(rot[i], &sr, &cr);
    const float m00 = cr * s.x, m01 = sr * s.y, m10 = -sr * s.x, m11 = cr * s.y;
    const float cxx = m00 * m00 + m01 * m01;
    const float cxy = m00 * m10 + m01 * m11;
    const float cyy = m10 * m10 + m11 * m11;
    const float det = cxx * cyy - cxy * cxy;
    float ox_ = 0.0f, oy_ = 0.0f, q0 = 0.0f, q1 = 0.0f, q2 = 0.0f;
    int32_t rad = 0, area = 0;
    if (det != 0.0f) {
        const float inv_det = 1.0f / det;
        const float qx = cyy * inv_det, qy = -cxy * inv_det, qz = cxx * inv_det;
        const float b = 0.5f * (cxx + cyy);
        const float delta = fmaxf(0.1f, b * b - det);
        const float sd = __builtin_sqrtf(delta);
        const float radius = __builtin_ceilf(3.0f * __builtin_sqrtf(fmaxf(b + sd, b - sd)));
        const int4 r = gs_tile_rect(cx, cy, qx, qy, qz, radius, block_x, block_y, tbx, tby);
        const int32_t a = (r.z - r.x) * (r.w - r.y);
        if (a > 0) {
            ox_ = cx;
            oy_ = cy;
            q0 = qx;
            q1 = qy;
            q2 = qz;
            rad = f2i_sat(radius);
            area = a;
        }
    }
    xys[i] = make_float2(ox_, oy_);
    depths[i] = 0.0f;
    radii[i] = rad;
    conics[3 * i] = q0;
    conics[3 * i + 1] = q1;
    conics[3 * i + 2] = q2;
    tiles_hit[i] = area;
}

__global__ __launch_bounds__(kGsThreads) void k_gs_pack(const float2* __restrict__ xys,
                                                        const float* __restrict__ conics,
                                                        const float* __restrict__ colors,
                                                        const float* __restrict__ opac, int n,
                                                        GsRec* __restrict__ recs) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n) return;
    const float2 p = xys[g];
    const float qa = conics[3 * g], qb = conics[3 * g + 1], qc = conics[3 * g + 2];
    const float o = opac[g];
    float4* dst = reinterpret_cast<float4*>(recs + g);
    dst[0] = make_float4(p.x, p.y, 0.5f * qa, qb);
    dst[1] = make_float4(0.5f * qc, o, gs_alpha_cut(o), colors[3 * g]);
    dst[2] = make_float4(colors[3 * g + 1], colors[3 * g + 2], qa, qc);
}

// A wave's pixels: KP per lane, pixels 64 KP wv .. 64 KP (wv + 1) - 1 of the
// tile's block_x x block_y in row-major order, lane l's p-th at 64 p + l, at
// (px, py) = (j, i) (rasterize.py:84-88).  [x0, x1] x [y0, y1] holds them all
// (those inside the image).
template <int KP>
struct GsPixels {
    int i[KP], j[KP];
    bool inside[KP];
    float px[KP], py[KP];
    float x0, x1, y0, y1;
};

template <int KP>
__device__ __forceinline__ GsPixels<KP> gs_pixels(int tile, int tbx, int bx, int by, int img_h,
                                                  int img_w) {
    GsPixels<KP> P;
    const int ty = tile / tbx, tx = tile - ty * tbx;
    const int lane = threadIdx.x & (kWave - 1);
    const int k0 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * (KP * kWave);
#pragma unroll
    for (int p = 0; p < KP; ++p) {
        const int k = k0 + p * kWave + lane;
        const int ly = k / bx, lx = k - ly * bx;
        P.i[p] = ty * by + ly;
        P.j[p] = tx * bx + lx;
        P.inside[p] = k < bx * by && P.i[p] < img_h && P.j[p] < img_w;
        P.px[p] = (float)P.j[p];
        P.py[p] = (float)P.i[p];
    }
    P.x0 = (float)(tx * bx);
    P.x1 = (float)min(tx * bx + bx - 1, img_w - 1);
    P.y0 = (float)(ty * by + k0 / bx);
    P.y1 = (float)min(ty * by + min(by - 1, (k0 + KP * kWave - 1) / bx), img_h - 1);
    return P;
}

// sigma = dx (a dx + b dy) + c dy^2, the spec form of rasterize.py:111-114.
__device__ __forceinline__ float gs_sigma(const GsRec& R, float px, float py, float& dx,
                                          float& dy) {
    dx = R.x - px;
    dy = R.y - py;
    return __builtin_fmaf(dx, __builtin_fmaf(R.a, dx, R.b * dy), (R.c * dy) * dy);
}

// Whether no pixel of the rectangle can reach alpha 1/255: the least sigma
// over it exceeds the record's cut.  For a positive definite conic with its
// centre outside the rectangle the least value lies on a side that faces the
// centre, where the other coordinate is minimised and clamped.  The margin
// 2^-18 M (M: the largest sum of the form's absolute terms over the
// rectangle) covers the rounding here and in gs_sigma, which is a few 2^-24
// of M; the cut itself lies 1/64 above the threshold.  Kept (false): a centre
// inside, a form that is not clearly definite, and NaN or overflow anywhere
// (every comparison with them fails).
__device__ __forceinline__ bool gs_culled(const float4& r0, const float4& r1, float x0, float x1,
                                          float y0, float y1) {
    const float a = r0.z, b = r0.w, c = r1.x, cut = r1.z;
    const float xl = r0.x - x1, xh = r0.x - x0, yl = r0.y - y1, yh = r0.y - y0;
    const float xn = fminf(fmaxf(0.0f, xl), xh), yn = fminf(fmaxf(0.0f, yl), yh);
    const float yv = fminf(fmaxf(-0.5f * b * xn * __builtin_amdgcn_rcpf(c), yl), yh);
    const float xv = fminf(fmaxf(-0.5f * b * yn * __builtin_amdgcn_rcpf(a), xl), xh);
    const float sv = a * xn * xn + b * xn * yv + c * yv * yv;
    const float sh = a * xv * xv + b * xv * yn + c * yn * yn;
    const float low = xn != 0.0f ? (yn != 0.0f ? fminf(sv, sh) : sv) : sh;
    const float mx = fmaxf(fabsf(xl), fabsf(xh)), my = fmaxf(fabsf(yl), fabsf(yh));
    const float M = a * mx * mx + fabsf(b) * mx * my + c * my * my;
    const float ac4 = 4.0f * a * c;
    return (xn != 0.0f || yn != 0.0f) && a > 0.0f && c > 0.0f && ac4 - b * b > 1e-5f * ac4 &&
           sv - sv == 0.0f && sh - sh == 0.0f && low > cut + M * 0x1p-18f;
}

// exp(-sigma) for sigma <= cut: spec_expf, through spec_expf_mid where that is
// the same (mid: the record's cut, which is wave-uniform, keeps sigma in its
// range).
__device__ __forceinline__ float gs_exp(float sigma, bool mid) {
    return mid ? spec_expf_mid(-sigma) : spec_expf(-sigma);
}

// Forward.  Bound by the vector instructions of the visited entries (about 35
// a pixel) and, with few waves, by the latency of one entry after the other.
// The cull leaves out the entries whose tile rectangle holds the tile but
// whose ellipse misses the wave's pixels.  KP = 2 halves the scalar work and
// the record loads per pixel and is taken when that still fills the chip
// (gs_two_pixels).  100000 Gaussians at 1024 x 1024, 16 x 8 tiles: 171 -> 132
// us, all of it issue time of its vector instructions (VALU busy 99%).
template <int KP>
__global__ __launch_bounds__(1024 / KP) void k_gs_raster_fwd(
    const int32_t* __restrict__ ids, const int32_t* __restrict__ bins_g,
    const GsRec* __restrict__ recs_g, const float* __restrict__ bg, int img_h, int img_w, int bx,
    int by, int tbx, int ntiles, float* __restrict__ out, float* __restrict__ final_T,
    int32_t* __restrict__ final_idx) {
    const int tile = xcd_tile(blockIdx.x, ntiles);
    const GsPixels<KP> P = gs_pixels<KP>(tile, tbx, bx, by, img_h, img_w);
    const cptr<GsRec> recs = as_const(recs_g);
    const cptr<int32_t> bins = as_const(bins_g);
    const int lane = threadIdx.x & (kWave - 1);
    const int g0 = bins[2 * tile], g1 = bins[2 * tile + 1];
    float T[KP], c0[KP], c1[KP], c2[KP];
    int cur[KP];
    bool done[KP];
#pragma unroll
    for (int p = 0; p < KP; ++p) {
        T[p] = 1.0f;
        c0[p] = c1[p] = c2[p] = 0.0f;
        cur[p] = 0;
        done[p] = !P.inside[p];
    }
    bool finished = false;
    for (int ec = g0; ec < g1 && !finished; ec += kWave) {
        const bool in = ec + lane < g1;
        const int id_l = in ? ids[ec + lane] : 0;
        const float4* rl = reinterpret_cast<const float4*>(recs_g + id_l);
        const float4 r0 = rl[0], r1 = rl[1];
        uint64_t todo = __ballot(in && !gs_culled(r0, r1, P.x0, P.x1, P.y0, P.y1));
        while (todo) {
            bool live = false;
#pragma unroll
            for (int p = 0; p < KP; ++p) live |= !done[p];
            if (__ballot(live) == 0) {
                finished = true;
                break;
            }
            const int k = (int)__builtin_ctzll(todo);
            todo &= todo - 1;
            const GsRec R = recs[__builtin_amdgcn_readlane(id_l, k)];
            const bool mid = R.cut <= 80.0f;
            float sigma[KP];
            bool on[KP], any = false;
#pragma unroll
            for (int p = 0; p < KP; ++p) {
                float dx, dy;
                sigma[p] = gs_sigma(R, P.px[p], P.py[p], dx, dy);
                on[p] = !done[p] && !(sigma[p] < 0.0f) && !(sigma[p] > R.cut);
                any |= on[p];
            }
            if (__ballot(any) == 0) continue;
#pragma unroll
            for (int p = 0; p < KP; ++p) {
                const float alpha = fminf(kGsAlphaCapFwd, R.opac * gs_exp(sigma[p], mid));
                const bool take = on[p] && !(alpha < kGsAlphaMin);
                const float vis = alpha * T[p];
                const float nT = T[p] * (1.0f - alpha);
                c0[p] = take ? __builtin_fmaf(R.r, vis, c0[p]) : c0[p];
                c1[p] = take ? __builtin_fmaf(R.g, vis, c1[p]) : c1[p];
                c2[p] = take ? __builtin_fmaf(R.bl, vis, c2[p]) : c2[p];
                T[p] = take ? nT : T[p];
                cur[p] = take ? ec + k : cur[p];
                done[p] = done[p] || (take && nT <= kGsTStop);
            }
        }
    }
#pragma unroll
    for (int p = 0; p < KP; ++p) {
        if (!P.inside[p]) continue;
        const size_t q = (size_t)P.i[p] * img_w + P.j[p];
        final_T[q] = T[p];
        final_idx[q] = cur[p];
        out[3 * q] = __builtin_fmaf(T[p], bg[0], c0[p]);
        out[3 * q + 1] = __builtin_fmaf(T[p], bg[1], c1[p]);
        out[3 * q + 2] = __builtin_fmaf(T[p], bg[2], c2[p]);
    }
}

// A wave's gradient sums waiting in LDS: (destination, value) pairs, added
// with one 64-lane atomic instruction per 64 of them.  (One counter tracks a
// wave's loads and atomics alike: added entry by entry, each entry's atomics
// would stand before the next entry's loads.)
struct GsAdd {
    float* dst;
    float v;
};
constexpr int kGsAdds = 128;   // 2 KiB of LDS per wave

__device__ __forceinline__ void gs_flush(GsAdd* buf, int& n) {
    const int lane = threadIdx.x & (kWave - 1);
    for (int i = lane; i < n; i += kWave) {
        const GsAdd r = buf[i];
        if (r.dst) atomicAdd(r.dst, r.v);
    }
    n = 0;
}

// Pushes v from the lanes with `on` (at most `count`, at their slots 0 .. count
// - 1; a null dst is skipped).
__device__ __forceinline__ void gs_push(GsAdd* buf, int& n, int count, bool on, int slot,
                                        float* dst, float v) {
    if (n + count > kGsAdds) gs_flush(buf, n);
    if (on) buf[n + slot] = GsAdd{dst, v};
    n += count;
}

// Backward: the visited entries of the forward, in reverse.  Bound by vector
// instructions: per entry about 45 a pixel and 60 for the reductions, which
// KP = 2 halves per pixel.  CONTRIB: contribution outputs are asked for.
// Same scene: 493 -> 244 us.
template <int KP, bool CONTRIB>
__global__ __launch_bounds__(1024 / KP) void k_gs_raster_bwd(
    const int32_t* __restrict__ ids, const int32_t* __restrict__ meta_g,
    const int32_t* __restrict__ bins_g, const GsRec* __restrict__ recs_g,
    const float* __restrict__ bg, int img_h, int img_w, int bx, int by, int tbx, int ntiles,
    const float* __restrict__ final_T, const int32_t* __restrict__ final_idx,
    const float* __restrict__ v_out, const float* __restrict__ v_out_alpha,
    float* __restrict__ v_xy, float* __restrict__ v_conic, float* __restrict__ v_rgb,
    float* __restrict__ v_opac, float* __restrict__ contrib_rgb,
    float* __restrict__ isect_contrib) {
    extern __shared__ GsAdd adds_all[];
    const int tile = xcd_tile(blockIdx.x, ntiles);
    const GsPixels<KP> P = gs_pixels<KP>(tile, tbx, bx, by, img_h, img_w);
    const cptr<GsRec> recs = as_const(recs_g);
    const cptr<int32_t> bins = as_const(bins_g);
    const int lane = threadIdx.x & (kWave - 1);
    GsAdd* const adds = adds_all + (threadIdx.x >> 6) * kGsAdds;
    int nadd = 0;
    const int g0 = bins[2 * tile], g1 = bins[2 * tile + 1];
    float T[KP], v0[KP], v1[KP], v2[KP], b0[KP], b1[KP], b2[KP], bgT[KP];
    int fidx[KP], fmax = -1;
#pragma unroll
    for (int p = 0; p < KP; ++p) {
        T[p] = v0[p] = v1[p] = v2[p] = b0[p] = b1[p] = b2[p] = bgT[p] = 0.0f;
        fidx[p] = -1;
        if (P.inside[p]) {
            const size_t q = (size_t)P.i[p] * img_w + P.j[p];
            T[p] = final_T[q];
            fidx[p] = final_idx[q];
            v0[p] = v_out[3 * q];
            v1[p] = v_out[3 * q + 1];
            v2[p] = v_out[3 * q + 2];
            const float va = v_out_alpha ? v_out_alpha[q] : 0.0f;
            // T_final ra (va - bg.v) is the background's share of d alpha.
            bgT[p] = T[p] * (va - (bg[0] * v0[p] + bg[1] * v1[p] + bg[2] * v2[p]));
        }
        fmax = max(fmax, fidx[p]);
    }
    // The value this lane adds per entry: lanes 8..15 one of wave_reduce8's
    // totals, lane 63 the ninth; the address of Gaussian g's is base + stride g.
    const bool adder = (lane & ~7) == 8, ninth = lane == kWave - 1;
    const int slot = ninth ? 8 : reduce8_slot(lane & 7);
    const int stride = slot < 3 ? 3 : slot == 3 ? 1 : slot < 7 ? 3 : 2;
    float* const base = slot < 3 ? v_rgb + slot
                      : slot == 3 ? v_opac
                      : slot < 7 ? v_conic + (slot - 4)
                                 : v_xy + (slot - 7);
    const float scale = slot >= 4 && slot < 7 ? 0.5f : 1.0f;   // v_conic: half the moments
    const int gstart = min(g1 - 1, __builtin_amdgcn_readfirstlane(wave_max_i(fmax)));
    for (int ec = gstart; ec >= g0; ec -= kWave) {
        const bool in = ec - lane >= g0;
        const int id_l = in ? ids[ec - lane] : 0;
        const int geom_l = in && meta_g ? meta_g[ec - lane] : 1;
        const float4* rl = reinterpret_cast<const float4*>(recs_g + id_l);
        const float4 r0 = rl[0], r1 = rl[1];
        uint64_t todo = __ballot(in && !gs_culled(r0, r1, P.x0, P.x1, P.y0, P.y1));
        for (; todo; todo &= todo - 1) {
            const int k = (int)__builtin_ctzll(todo);
            const int e = ec - k;
            const int g = __builtin_amdgcn_readlane(id_l, k);
            const GsRec R = recs[g];
            const bool mid = R.cut <= 80.0f;
            float sigma[KP], dx[KP], dy[KP];
            bool valid[KP], any = false;
#pragma unroll
            for (int p = 0; p < KP; ++p) {
                sigma[p] = gs_sigma(R, P.px[p], P.py[p], dx[p], dy[p]);
                valid[p] = e <= fidx[p] && !(sigma[p] < 0.0f) && !(sigma[p] > R.cut);
                any |= valid[p];
            }
            if (__ballot(any) == 0) continue;
            float vis[KP], alpha[KP];
            any = false;
#pragma unroll
            for (int p = 0; p < KP; ++p) {
                vis[p] = gs_exp(sigma[p], mid);
                alpha[p] = fminf(kGsAlphaCapBwd, R.opac * vis[p]);
                valid[p] = valid[p] && alpha[p] >= kGsAlphaMin;
                any |= valid[p];
            }
            if (__ballot(any) == 0) continue;
            const bool geom = __builtin_amdgcn_readlane(geom_l, k) != 0;
            float pv[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
            float py9 = 0.0f, cv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int p = 0; p < KP; ++p) {
                if (!valid[p]) continue;
                const float ra = __builtin_amdgcn_rcpf(1.0f - alpha[p]);
                T[p] = T[p] * ra;
                const float fac = alpha[p] * T[p];
                pv[0] = __builtin_fmaf(fac, v0[p], pv[0]);
                pv[1] = __builtin_fmaf(fac, v1[p], pv[1]);
                pv[2] = __builtin_fmaf(fac, v2[p], pv[2]);
                if constexpr (CONTRIB) {
                    const float cr = fac * R.r, cg = fac * R.g, cb = fac * R.bl;
                    cv[0] += cr;
                    cv[1] += cg;
                    cv[2] += cb;
                    cv[3] += cr + cg + cb;
                }
                float va = __builtin_fmaf(R.r, T[p], -(b0[p] * ra)) * v0[p];
                va = __builtin_fmaf(__builtin_fmaf(R.g, T[p], -(b1[p] * ra)), v1[p], va);
                va = __builtin_fmaf(__builtin_fmaf(R.bl, T[p], -(b2[p] * ra)), v2[p], va);
                va = __builtin_fmaf(bgT[p], ra, va);
                b0[p] = __builtin_fmaf(R.r, fac, b0[p]);
                b1[p] = __builtin_fmaf(R.g, fac, b1[p]);
                b2[p] = __builtin_fmaf(R.bl, fac, b2[p]);
                pv[3] = __builtin_fmaf(vis[p], va, pv[3]);
                const float v_sigma = -R.opac * vis[p] * va;
                const float sx = v_sigma * dx[p], sy = v_sigma * dy[p];
                pv[4] = __builtin_fmaf(sx, dx[p], pv[4]);
                pv[5] = __builtin_fmaf(sx, dy[p], pv[5]);
                pv[6] = __builtin_fmaf(sy, dy[p], pv[6]);
                pv[7] = __builtin_fmaf(v_sigma, __builtin_fmaf(R.pad0, dx[p], R.b * dy[p]),
                                       pv[7]);
                py9 = __builtin_fmaf(v_sigma, __builtin_fmaf(R.b, dx[p], R.pad1 * dy[p]), py9);
            }
            const float t = wave_reduce8(pv);
            const float t9 = wave_sum_lane63(py9);
            gs_push(adds, nadd, 9, adder || ninth, slot,
                    geom || slot < 4 ? base + (int64_t)stride * g : nullptr,
                    scale * (ninth ? t9 : t));
            if constexpr (CONTRIB) {
                const float cw[8] = {cv[0], cv[1], cv[2], cv[3], 0.0f, 0.0f, 0.0f, 0.0f};
                const float ct = wave_reduce8(cw);
                gs_push(adds, nadd, 4, adder && slot < 4, slot,
                        slot < 3 ? (contrib_rgb ? contrib_rgb + 3 * (size_t)g + slot : nullptr)
                                 : (isect_contrib ? isect_contrib + e : nullptr),
                        ct);
            }
        }
    }
    gs_flush(adds, nadd);
}

__global__ __launch_bounds__(kGsThreads) void k_gs_project_bwd(
    const float2* __restrict__ scales, const float* __restrict__ rot,
    const int32_t* __restrict__ radii, const float* __restrict__ conics,
    const float2* __restrict__ v_xy, const float* __restrict__ v_conic,
    const int32_t* __restrict__ meta, int n, int img_h, int img_w, float* __restrict__ v_cov2d,
    float2* __restrict__ v_mean, float2* __restrict__ v_scale, float* __restrict__ v_rot) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float g11 = 0.0f, g12 = 0.0f, g22 = 0.0f, vs0 = 0.0f, vs1 = 0.0f, vr = 0.0f;
    float vm0 = 0.0f, vm1 = 0.0f;
    if (radii[i] > 0) {
        // tilelang_renderer.py:111-116: v_xy and v_conic times the meta flag.
        const float keep = meta ? (float)meta[i] : 1.0f;
        const float c0 = conics[3 * i], c1 = conics[3 * i + 1], c2 = conics[3 * i + 2];
        const float q0 = v_conic[3 * i] * keep, q1 = v_conic[3 * i + 1] * keep,
                    q2 = v_conic[3 * i + 2] * keep;
        const float h00 = c0 * q0 + c1 * q1, h01 = c0 * q1 + c1 * q2;
        const float h10 = c1 * q0 + c2 * q1, h11 = c1 * q1 + c2 * q2;
        g11 = -(h00 * c0 + h01 * c1);
        g12 = -(h10 * c0 + h11 * c1) - (h00 * c1 + h01 * c2);
        g22 = -(h10 * c1 + h11 * c2);
        const float2 s = scales[i];
        float sn, cs_;
        spec_sincosf(rot[i], &sn, &cs_);
        vs0 = g11 * (2.0f * s.x * cs_ * cs_) + 2.0f * g12 * (-2.0f * s.x * sn * cs_) +
              g22 * (2.0f * s.x * sn * sn);
        vs1 = g11 * (2.0f * s.y * sn * sn) + 2.0f * g12 * (2.0f * s.y * cs_ * sn) +
              g22 * (2.0f * s.y * cs_ * cs_);
        const float m00 = cs_ * s.x, m01 = sn * s.y, m10 = -sn * s.x, m11 = cs_ * s.y;
        const float a00 = -sn * s.x, a01 = cs_ * s.y, a10 = -cs_ * s.x, a11 = -sn * s.y;
        const float t1_00 = a00 * m00 + a01 * m01, t1_10 = a10 * m00 + a11 * m01,
                    t1_11 = a10 * m10 + a11 * m11;
        const float b00 = m00 * s.x, b01 = m01 * s.y, b10 = m10 * s.x, b11 = m11 * s.y;
        const float t2_00 = b00 * -sn + b01 * cs_, t2_10 = b10 * -sn + b11 * cs_,
                    t2_11 = b10 * -cs_ + b11 * -sn;
        vr = g11 * (t1_00 + t2_00) + 2.0f * g12 * (t1_10 + t2_10) + g22 * (t1_11 + t2_11);
        const float2 vx = v_xy[i];
        vm0 = vx.x * keep * (0.5f * (float)img_w);
        vm1 = vx.y * keep * (0.5f * (float)img_h);
    }
    if (v_cov2d) {
        v_cov2d[3 * i] = g11;
        v_cov2d[3 * i + 1] = g12;
        v_cov2d[3 * i + 2] = g22;
    }
    v_mean[i] = make_float2(vm0, vm1);
    v_scale[i] = make_float2(vs0, vs1);
    v_rot[i] = vr;
}

// intersects.py:12-226: Gaussian g writes its rectangle's tiles row-major at
// [cum[g-1], cum[g-1] + area), key (tile << 32) | depth bits.  Writes outside
// [0, num_intersects) are dropped (the reference assumes they cannot occur).
__global__ __launch_bounds__(kGsThreads) void k_gs_map_ref(
    const float* __restrict__ xys, const float* __restrict__ conics,
    const float* __restrict__ depths, const int32_t* __restrict__ radii,
    const int32_t* __restrict__ cum, int n, int64_t num_isects, int bx, int by, int tbx,
    int tby, int64_t* __restrict__ isect_ids, int32_t* __restrict__ gauss_ids) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n || radii[g] <= 0) return;
    const float rf = (float)radii[g];
    const int4 r = conics ? gs_tile_rect(xys[2 * g], xys[2 * g + 1], conics[3 * g],
                                         conics[3 * g + 1], conics[3 * g + 2], rf, bx, by, tbx,
                                         tby)
                          : gs_tile_rect(xys[2 * g], xys[2 * g + 1], 0.0f, 0.0f, 0.0f, rf, bx,
                                         by, tbx, tby);
    const int w = r.z - r.x, h = r.w - r.y;
    if (w * h <= 0) return;
    const int64_t base = g == 0 ? 0 : (int64_t)cum[g - 1];
    const int64_t key_lo = (int64_t)__builtin_bit_cast(uint32_t, depths[g]);
    for (int row = 0; row < h; ++row) {
        for (int col = 0; col < w; ++col) {
            const int64_t o = base + (int64_t)row * w + col;
            if (o < 0 || o >= num_isects) continue;
            const int64_t t = (int64_t)(r.y + row) * tbx + r.x + col;
            isect_ids[o] = (t << 32) | key_lo;
            gauss_ids[o] = g;
        }
    }
}

}  // namespace cs

using namespace cs;

static inline int gs_blocks(int64_t n) { return (int)((n + kGsThreads - 1) / kGsThreads); }

static int gs_status() { return hipGetLastError() == hipSuccess ? CS_OK : CS_ERR_HIP; }

static bool gs_dims_ok(int32_t img_h, int32_t img_w, int32_t block_x, int32_t block_y) {
    return img_h > 0 && img_w > 0 && block_x > 0 && block_y > 0 && block_x * block_y <= 1024;
}

static bool al(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

extern "C" int cs_gs_project_forward(const float* means2d, const float* scales2d,
                                     const float* rotation, int32_t n, int32_t img_h,
                                     int32_t img_w, int32_t block_x, int32_t block_y, float* xys,
                                     float* depths, int32_t* radii, float* conics,
                                     int32_t* num_tiles_hit, hipStream_t stream) {
    if (n < 0 || !gs_dims_ok(img_h, img_w, block_x, block_y) || !al(means2d, 8) ||
        !al(scales2d, 8) || !al(xys, 8))
        return CS_ERR_ARGS;
    if (n == 0) return CS_OK;
    const int tbx = (img_w + block_x - 1) / block_x, tby = (img_h + block_y - 1) / block_y;
    hipLaunchKernelGGL(k_gs_project, dim3(gs_blocks(n)), dim3(kGsThreads), 0, stream,
                       reinterpret_cast<const float2*>(means2d),
                       reinterpret_cast<const float2*>(scales2d), rotation, n, img_h, img_w,
                       block_x, block_y, tbx, tby, reinterpret_cast<float2*>(xys), depths, radii,
                       conics, num_tiles_hit);
    return gs_status();
}

extern "C" int cs_gs_pack_records(const float* xys, const float* conics, const float* colors,
                                  const float* opacities, int32_t n, void* records,
                                  hipStream_t stream) {
    if (n < 0 || !al(xys, 8) || !al(records, 16)) return CS_ERR_ARGS;
    if (n == 0) return CS_OK;
    hipLaunchKernelGGL(k_gs_pack, dim3(gs_blocks(n)), dim3(kGsThreads), 0, stream,
                       reinterpret_cast<const float2*>(xys), conics, colors, opacities, n,
                       reinterpret_cast<GsRec*>(records));
    return gs_status();
}

// Threads of a tile's workgroup at kp pixels per lane.
static inline int gs_wg(int32_t block_x, int32_t block_y, int kp) {
    const int per_wave = kWave * kp;
    return (block_x * block_y + per_wave - 1) / per_wave * kWave;
}

// Two pixels per lane where that halves the waves and leaves at least
// `min_waves`; with fewer, a launch lasts as long as its longest list, and one
// pixel per lane shortens each entry.  The forward needs six waves for each of
// the chip's 1024 SIMDs, the backward, which has more to share between two
// pixels, two.  Measured, one against two (us; 16 x 8 tiles, a Gaussian of up to
// 8 pixels per 10 pixels | of up to 20 per 100):
//   waves of two     forward                    backward
//       1536     54 /  68 | 30 / 34         114 / 113 |  84 /  70
//       2048     60 /  71 | 30 / 33         129 / 118 |  83 /  67
//       4096     83 /  97 | 44 / 43         227 / 156 | 132 /  90
//       5120    102 / 107 | 48 / 49         292 / 174 | 147 / 103
//       6144    116 / 120 | 54 / 54         339 / 211 | 171 / 116
//       8192    147 / 145 | 64 / 64         402 / 260 | 185 / 124
// (16 x 16 tiles: the forward 101 / 111 at 5120 and 116 / 114 at 6144, the
// backward 105 / 116 at 1536 and 127 / 121 at 2048.)
constexpr int kGsTwoForward = 6144, kGsTwoBackward = 2048;

static inline bool gs_two_pixels(int32_t block_x, int32_t block_y, int ntiles, int min_waves) {
    const int two = gs_wg(block_x, block_y, 2);
    return gs_wg(block_x, block_y, 1) == 2 * two && (int64_t)ntiles * (two / kWave) >= min_waves;
}

extern "C" int cs_gs_rasterize_forward(const int32_t* gaussian_ids_sorted,
                                       const int32_t* tile_bins, const void* records,
                                       const float* background, int32_t img_h, int32_t img_w,
                                       int32_t block_x, int32_t block_y, float* out_img,
                                       float* final_Ts, int32_t* final_idx,
                                       hipStream_t stream) {
    if (!gs_dims_ok(img_h, img_w, block_x, block_y) || !al(records, 16)) return CS_ERR_ARGS;
    const int tbx = (img_w + block_x - 1) / block_x, tby = (img_h + block_y - 1) / block_y;
    const int ntiles = tbx * tby;
    const bool two = gs_two_pixels(block_x, block_y, ntiles, kGsTwoForward);
    hipLaunchKernelGGL(two ? k_gs_raster_fwd<2> : k_gs_raster_fwd<1>, dim3(ntiles),
                       dim3(gs_wg(block_x, block_y, two ? 2 : 1)), 0, stream,
                       gaussian_ids_sorted, tile_bins, reinterpret_cast<const GsRec*>(records),
                       background, img_h, img_w, block_x, block_y, tbx, ntiles, out_img,
                       final_Ts, final_idx);
    return gs_status();
}

extern "C" int cs_gs_rasterize_backward(
    const int32_t* gaussian_ids_sorted, const int32_t* intersect_meta_sorted,
    const int32_t* tile_bins, const void* records, const float* background, int32_t img_h,
    int32_t img_w, int32_t block_x, int32_t block_y, const float* final_Ts,
    const int32_t* final_idx, const float* v_output, const float* v_output_alpha, float* v_xy,
    float* v_conic, float* v_rgb, float* v_opacity, float* contrib_rgb, float* isect_contrib,
    hipStream_t stream) {
    if (!gs_dims_ok(img_h, img_w, block_x, block_y) || !al(records, 16)) return CS_ERR_ARGS;
    const int tbx = (img_w + block_x - 1) / block_x, tby = (img_h + block_y - 1) / block_y;
    const int ntiles = tbx * tby;
    const bool two = gs_two_pixels(block_x, block_y, ntiles, kGsTwoBackward);
    const int threads = gs_wg(block_x, block_y, two ? 2 : 1);
    auto kern = contrib_rgb || isect_contrib
                    ? (two ? k_gs_raster_bwd<2, true> : k_gs_raster_bwd<1, true>)
                    : (two ? k_gs_raster_bwd<2, false> : k_gs_raster_bwd<1, false>);
    hipLaunchKernelGGL(kern, dim3(ntiles), dim3(threads),
                       threads / kWave * kGsAdds * sizeof(GsAdd), stream,
                       gaussian_ids_sorted, intersect_meta_sorted, tile_bins,
                       reinterpret_cast<const GsRec*>(records), background, img_h, img_w,
                       block_x, block_y, tbx, ntiles, final_Ts, final_idx, v_output,
                       v_output_alpha, v_xy, v_conic, v_rgb, v_opacity, contrib_rgb,
                       isect_contrib);
    return gs_status();
}

extern "C" int cs_gs_project_backward(const float* scales2d, const float* rotation,
                                      const int32_t* radii, const float* conics,
                                      const float* v_xy, const float* v_conic,
                                      const int32_t* gaussian_meta, int32_t n, int32_t img_h,
                                      int32_t img_w, float* v_cov2d, float* v_mean2d,
                                      float* v_scale, float* v_rot, hipStream_t stream) {
    if (n < 0 || img_h <= 0 || img_w <= 0 || !al(scales2d, 8) || !al(v_xy, 8) ||
        !al(v_mean2d, 8) || !al(v_scale, 8))
        return CS_ERR_ARGS;
    if (n == 0) return CS_OK;
    hipLaunchKernelGGL(k_gs_project_bwd, dim3(gs_blocks(n)), dim3(kGsThreads), 0, stream,
                       reinterpret_cast<const float2*>(scales2d), rotation, radii, conics,
                       reinterpret_cast<const float2*>(v_xy), v_conic, gaussian_meta, n, img_h,
                       img_w, v_cov2d, reinterpret_cast<float2*>(v_mean2d),
                       reinterpret_cast<float2*>(v_scale), v_rot);
    return gs_status();
}

extern "C" int cs_gs_map_to_intersects(const float* xys, const float* conics,
                                       const float* depths, const int32_t* radii,
                                       const int32_t* cum_tiles_hit, int32_t n,
                                       int64_t num_intersects, int32_t tile_bound_x,
                                       int32_t tile_bound_y, int32_t block_x, int32_t block_y,
                                       int64_t* isect_ids, int32_t* gaussian_ids,
                                       hipStream_t stream) {
    if (n < 0 || num_intersects < 0 || tile_bound_x <= 0 || tile_bound_y <= 0 || block_x <= 0 ||
        block_y <= 0)
        return CS_ERR_ARGS;
    if (n == 0 || num_intersects == 0) return CS_OK;
    hipLaunchKernelGGL(k_gs_map_ref, dim3(gs_blocks(n)), dim3(kGsThreads), 0, stream, xys, conics,
                       depths, radii, cum_tiles_hit, n, num_intersects, block_x, block_y,
                       tile_bound_x, tile_bound_y, isect_ids, gaussian_ids);
    return gs_status();
}
