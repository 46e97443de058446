// Texture edit (texture_edit.cu:11-227 semantics): splat a per-pixel edit
// canvas back onto the Gaussians' texel charts.
//
// For every pair the forward would composite (same alpha, skip and stop
// rules; blur from settings bit 0 as in the reference edit kernel) whose view
// depth lies in the pixel's [depth_lower, depth_upper], the bilinear weights
// of the pair's texel quad (always bilinear, replicate padding) times
// (r*a, g*a, b*a, a, 1) are added to channels 0..4 of the output, a being the
// pixel's edit alpha.  The walk is the forward's: quadrant waves, 64-entry
// windows with screen-box culling, SMEM records.  The values reach the output
// through matrix instructions for a shared texel quad or a window of up to 3x3
// texels, else by DPP-merged lanes into an LDS accumulator or direct float
// atomics.
//
// Bound by VALU issue (0.8 of the issue slots).  500k Gaussians on a 1080p
// canvas: 897 us with wave reductions of all taps x 5 values in a branch of the
// live lanes, 711 with wave masks in the branch's place and 2x3 and 3x2
// windows, 609 with the matrix instructions (280 of it the walk).  The plain
// kernels are held to 96 VGPRs, five waves per SIMD (four: 748 against 711).
#include <type_traits>

#include "raster_common.hpp"

namespace gstex {

struct EditIn {
    const float* upd_img;      // (H, W, 3)
    const float* upd_alpha;    // (H, W)
    const float* depth_lower;  // (H, W)
    const float* depth_upper;  // (H, W)
    float* out;                // (X, C), C >= 5
};

// Adds to the texels of one window the sums over the wave's pixels of weight x
// (4 channels, 1): rows[r] holds the weights of window row r's texels (of all
// four texels of a quad, R = 1, Q = 4), value the channels of the pixel quad.
// at(r, q): the texel's first value.  Channel 4: lane i of a pixel quad sums
// texel i's weights over the quad.  A zero sum is not added; window rows and
// columns past the chart carry no weight.
template <int R, int Q, typename At>
__device__ __forceinline__ void window_add(const float (&rows)[R][4], const float (&value)[4],
                                           int lane, float* chart, At at) {
    constexpr int N = R * Q;
    float v[N + R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        quad_sums<Q>(rows[r], value, v + Q * r);
        v[N + r] = (rows[r][0] + rows[r][1]) + (rows[r][2] + rows[r][3]);
    }
    const float tot = quad_reduce_scatter(v, lane);
    const int code = quad_slot<N + R>(lane), j = lane & 3;
    const bool one = code >= N;  // bit 6 (a copy) makes it larger still
    const int r = one ? code - N : code / Q, q = one ? j : code - Q * (code / Q);
    if (code < 64 && q < Q && tot != 0.f) unsafeAtomicAdd(chart + at(r, q) + (one ? 4 : j), tot);
}

// Chart::ok of chart_of (float values).
__device__ __forceinline__ bool chart_inside(const Splat& s, int C, int num_texels) {
    const uint32_t h = (uint32_t)s.h, w = (uint32_t)s.w, n = h * w, X = (uint32_t)num_texels;
    const uint32_t over = __umulhi(h, w) | __umulhi(n, 4u * C) | ((n * 4u * C) >> 31);
    return (over == 0) & (max(h - 1u, w - 1u) < 0xffffffu) & (n <= X) & ((uint32_t)s.start <= X - n);
}

template <bool BLUR, bool PRECISE>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(PRECISE ? 1 : 5))) void k_texture_edit(RasterArgs a, EditIn ed) {
    const int tile = blockIdx.x;
    const int ty = tile / a.tiles_x, tx = tile - ty * a.tiles_x;
    const int lane = threadIdx.x & (kWave - 1);
    int lx, ly;
    bool in_tile;
    lane_pixel(a.bw, threadIdx.x, lx, ly, in_tile);
    const int j = tx * a.bw + lx, i = ty * a.bw + ly;
    const bool inside = in_tile && i < a.img_h && j < a.img_w;
    const PixelRay pr = pixel_ray(a.c2w, a.viewmat, a.fx, a.fy, a.cx, a.cy, j, i);
    const int C = a.channels;
    float val[5] = {0.f, 0.f, 0.f, 0.f, 1.f};
    float lo = 0.f, hi = -1.f;
    if (inside) {
        const int pid = i * a.img_w + j;
        const float al = ed.upd_alpha[pid];
        val[0] = ed.upd_img[3 * pid] * al;
        val[1] = ed.upd_img[3 * pid + 1] * al;
        val[2] = ed.upd_img[3 * pid + 2] * al;
        val[3] = al;
        lo = ed.depth_lower[pid];
        hi = ed.depth_upper[pid];
    }
    int r0, r1;
    tile_range(a, tile, r0, r1);
    float T = 1.f;
    // culling rectangle of the live pixels (shrinks as pixels finish, as in
    // k_raster_forward)
    WaveRect rect = wave_rect(inside, j, i);
    uint64_t live = lanes_where(inside);  // pixels still compositing
    int live_n = __popcll(live);
    // wave-private texel accumulator, kept zero between Gaussians by the flush
    __shared__ float tex_acc[256 / kWave][kTexAccFloats];
    float* acc = tex_acc[wave_index()];
    for (int k = lane; k < kTexAccFloats; k += kWave) acc[k] = 0.f;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    // a pixel with T (1 - 1/255) <= 1e-4 can take no further entry (each one
    // with alpha >= 1/255 ends it), so it stops at once and culled entries
    // never matter (as in k_raster_forward)
    constexpr float kKeep = 1.f - 1.f / 255.f;
    const bool cull = a.boxes != nullptr;

    // products with the zero weights of other pixels' texels need finite values
    const bool finite = lanes_where(!(fabsf(val[0]) < INFINITY && fabsf(val[1]) < INFINITY &&
                                      fabsf(val[2]) < INFINITY && fabsf(val[3]) < INFINITY)) == 0;
    // channels 0..3 of the pixels of this lane's quad, channel lane & 3
    float quad_val[4];
    {
        const float rgba[4] = {val[0], val[1], val[2], val[3]};
        quad_transpose(rgba, lane, quad_val);
    }

    // One list entry: Gaussian g with record s.  The pair math runs for every
    // lane (finite for any pixel ray); the live, composited and hitting pixels
    // are wave masks.
    auto entry = [&](const Splat& s) {
        const Pair p = pair_eval(s, pr, BLUR, PRECISE);
        const float next_T = T * (1.f - p.alpha);
        live &= ~lanes_where(next_T <= 1e-4f);
        const uint64_t comp = live & ~skip_lanes(p);
        if (comp == 0) return;
        const float t_view = p.t * pr.view_depth;
        const uint64_t hm = comp & lanes_where(t_view >= lo) & lanes_where(t_view <= hi);
        const bool composited = __builtin_amdgcn_inverse_ballot_w64(comp);
        T = composited ? next_T : T;
        live &= ~(comp & lanes_where(next_T * kKeep <= 1e-4f));
        // out has the texture's (X, C) float layout; charts outside it get nothing
        if (hm == 0 || !chart_inside(s, C, a.num_texels)) return;
        const bool hit = __builtin_amdgcn_inverse_ballot_w64(hm);
        float* const out_chart = ed.out + (size_t)s.start * C;
        const int first = __ffsll((unsigned long long)hm) - 1;
        // How the (taps x 5) values reach the output (wave-uniform choice):
        //   quad    every hitting lane samples one texel quad (a 1x1 chart too),
        //   window  or its taps lie inside one 2x3, 3x2 or 3x3 texel window:
        //           matrix instructions (window_add), one atomic per texel
        //           and value
        //   lds     charts of up to kTexAccFloats / 5 texels: merged lanes
        //           add into the wave's LDS accumulator, then flush
        //   direct  one atomic per tap and value (all entries of a wave with
        //           a value that is not finite: only its own texels take it)
        auto quad = [&](float y, float x, int ou, int ov) {
            QuadWeights qw;
            qw.set(y, x, hit ? 1.f : 0.f, lane);
            const float rows[1][4] = {{qw.w[0], qw.w[1], qw.w[2], qw.w[3]}};
            const int o = ou * s.w + ov;
            window_add<1, 4>(rows, quad_val, lane, out_chart,
                             [&](int, int q) { return (o + (q & 1) + (q >> 1) * s.w) * C; });
        };
        if (s.h * s.w == 1 && finite) {
            quad(0.f, 0.f, 0, 0);
            return;
        }
        // position in texels, with replicate padding: past the last texel's
        // centre both taps are that texel, as at its centre
        float u, v;
        splat_uv(s, p.delta, u, v);
        const float tu = fminf((float)s.h * u, (float)(s.h - 1));
        const float tv = fminf((float)s.w * v, (float)(s.w - 1));
        const float flu = floorf(tu), flv = floorf(tv);
        // position relative to the first hitting lane's taps
        const float au = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(flu), first));
        const float av = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(flv), first));
        const float y0 = tu - au, x0 = tv - av;
        const int iu0 = (int)au, iv0 = (int)av;
        auto outside = [&](float t, float top) {
            return lanes_where(fminf(fmaxf(t, 0.f), top) != t) & hm;
        };
        const bool ou1 = outside(y0, 1.f) != 0, ov1 = outside(x0, 1.f) != 0;
        if (finite && !ou1 && !ov1) {
            quad(y0, x0, iu0, iv0);
            return;
        }
        // window origin: one texel lower where some hitting lane lies below
        const bool lu = (lanes_where(y0 < 0.f) & hm) != 0, lv = (lanes_where(x0 < 0.f) & hm) != 0;
        const float y = y0 + (lu ? 1.f : 0.f), x = x0 + (lv ? 1.f : 0.f);
        if (finite && !(outside(y, 2.f) | outside(x, 2.f))) {
            const int o = (iu0 - (lu ? 1 : 0)) * s.w + iv0 - (lv ? 1 : 0);
            auto at = [&](int r, int q) { return (o + r * s.w + q) * C; };
            // a pixel that does not hit has no column weights
            const float xh = hit ? x : 8.f;
            auto window = [&](auto R, auto Q) {
                float a[R.value];
                row_weights(y, a);
                WindowWeights<R.value> ww;
                ww.set(a, xh, lane);
                window_add<R.value, Q.value>(ww.w, quad_val, lane, out_chart, at);
            };
            using two = std::integral_constant<int, 2>;
            using three = std::integral_constant<int, 3>;
            if (!outside(y, 1.f)) window(two{}, three{});
            else if (!outside(x, 1.f)) window(three{}, two{});
            else window(three{}, three{});
            return;
        }
        const int iu = (int)flu, iv = (int)flv;  // tap rows and columns
        const int ju = min(iu + 1, s.h - 1), jv = min(iv + 1, s.w - 1);
        const float fu = tu - flu, fv = tv - flv;
        const float a0 = hit ? 1.f - fu : 0.f, a1 = hit ? fu : 0.f;
        const float wt[4] = {a0 * (1.f - fv), a0 * fv, a1 * (1.f - fv), a1 * fv};
        const int tix[4] = {iu * s.w + iv, iu * s.w + jv, ju * s.w + iv, ju * s.w + jv};
        if (!finite) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int k = 0; k < 5; ++k)
                    if (wt[t] != 0.f)
                        unsafeAtomicAdd(out_chart + (size_t)tix[t] * C + k, wt[t] * val[k]);
            return;
        }
        const QuadMerge qm = quad_merge_setup(hit ? tix[0] : -1, lane);
        if (s.h * s.w * 5 <= kTexAccFloats) {
            // charts of up to kTexAccFloats / 5 texels: merged lanes add into
            // the wave's LDS accumulator (5 values per texel), then the texels
            // some lane touched go out with one atomic each
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                float q[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) q[t] = quad_merge(wt[t] * val[k], qm);
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    if (q[t] != 0.f) atomicAdd(acc + tix[t] * 5 + k, q[t]);
            }
            // tap 0 is the lowest texel of a lane's quad, tap 3 the highest
            const int tlo = wave_min(hit ? tix[0] : 0x7fffffff);
            const int thi = wave_max(hit ? tix[3] : -1);
            // every lane's LDS adds precede these reads in the wave's LDS queue
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            const int nv = (thi - tlo + 1) * 5;
            for (int idx = lane; idx < nv; idx += kWave) {
                const int tx = tlo + idx / 5, k = idx - (idx / 5) * 5;
                const float v = acc[tx * 5 + k];
                if (v != 0.f) {
                    unsafeAtomicAdd(out_chart + (size_t)tx * C + k, v);
                    acc[tx * 5 + k] = 0.f;
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            return;
        }
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            float q[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) q[t] = quad_merge(wt[t] * val[k], qm);
#pragma unroll
            for (int t = 0; t < 4; ++t)
                if (q[t] != 0.f) unsafeAtomicAdd(out_chart + (size_t)tix[t] * C + k, q[t]);
        }
    };

    for (int base = r0 & ~63; base < r1 && live != 0; base += 64) {
        const int now = __popcll(live);
        if (now < live_n) {
            live_n = now;
            rect = wave_rect(__builtin_amdgcn_inverse_ballot_w64(live), j, i);
        }
        const Window w = window_candidates<BLUR>(a, base, r0, r1 - 1, rect, lane, cull);
        uint64_t cand = w.cand;
        while (cand != 0 && live != 0) {
            const int bit = __ffsll((unsigned long long)cand) - 1;
            cand &= cand - 1;
            entry(splat_record(a, __builtin_amdgcn_readlane(w.gid, bit)));
        }
    }
}

size_t texture_edit_workspace_bytes(int n) { return splat_records_bytes(n) + 256; }

hipError_t texture_edit(const RasterCall& c, const float* upd_img, const float* upd_alpha,
                        const float* depth_lower, const float* depth_upper, float* out,
                        void* ws, size_t ws_bytes, hipStream_t s) {
    if (ws_bytes < texture_edit_workspace_bytes(c.num_points)) return hipErrorInvalidValue;
    hipError_t e = fill_f32(out, (size_t)c.num_texels * (size_t)c.channels, 0.f, s);
    if (e != hipSuccess) return e;
    float* records = (float*)ws;
    if ((e = build_raster_records(c, records, s)) != hipSuccess) return e;
    const RasterArgs a = make_raster_args(c, records);
    const int tiles = a.tiles_x * a.tiles_y;
    if (tiles <= 0) return hipSuccess;
    const EditIn ed{upd_img, upd_alpha, depth_lower, depth_upper, out};
    const dim3 block(raster_block_threads(a.bw));
    auto* const kernel = c.settings & 1 ? (a.precise_edge ? k_texture_edit<true, true>
                                                          : k_texture_edit<true, false>)
                                        : (a.precise_edge ? k_texture_edit<false, true>
                                                          : k_texture_edit<false, false>);
    kernel<<<tiles, block, 0, s>>>(a, ed);
    return hipGetLastError();
}

}  // namespace gstex
