// Raster kernels for small tile grids: one wave per 4x4 pixels, four list
// entries at a time.
//
// The kernels of raster.hip and raster_bwd.hip give a wave 8x8 pixels and walk
// its list one entry at a time.  On a grid of few tiles that leaves most of
// the chip idle and the time is the longest wave's walk: one entry after the
// other, each a chain of a record read, the pair math, texel reads and (in the
// backward) two reductions, with few other waves on the SIMD to fill its
// waits.  Here the 64 lanes of a wave are four slots of 16 pixels.  Slot s
// (lanes 16 s .. 16 s + 15, a DPP row) evaluates the s-th of four consecutive
// entries, so the pair math, the texel reads, the gradient seeds and the
// reductions serve four entries per instruction; only the transmittance
// recursion runs through the four entries in order, on every lane, from values
// exchanged between the rows by permlane swaps.  A tile has 16 such waves instead of four, and a
// wave meets only the entries of its own 4x4 pixels.
//
// The forward runs the same float32 operations in the same order as the 8x8
// kernels, so its outputs are theirs bit for bit: row r of a pixel holds a
// part of its sums (colour, normal, texture), and the slots' values are
// transposed across the rows and added in list order.
//
// A block is one 8x8 quadrant: its four waves scan the list together, 256
// entries a step, and keep the entries that meet the quadrant in LDS with
// their culling data; batches of up to 64 of them have their records staged in
// LDS, and each wave takes those that meet its own pixels, four at a time.  So
// the walk itself waits for no list or record read, and the backward's
// per-Gaussian sums of the four waves meet in LDS and go out once a batch.
#include "raster_common.hpp"

namespace gstex {

constexpr int kSlots = 4;

// The values of the four rows (slots) of x at this lane's position in the row,
// on every lane.
__device__ __forceinline__ void rows4(float x, float (&r)[kSlots]) {
    const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                    false);
    const auto lo = __builtin_amdgcn_permlane16_swap(h[0], h[0], false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(h[1], h[1], false, false);
    r[0] = __uint_as_float(lo[0]);
    r[1] = __uint_as_float(lo[1]);
    r[2] = __uint_as_float(hi[0]);
    r[3] = __uint_as_float(hi[1]);
}

// Lane mask of slot s's lanes, and the 16 bits of slot s of a lane mask
// repeated in every row.
__device__ __forceinline__ constexpr uint64_t row_lanes(int s) { return 0xffffull << (16 * s); }
__device__ __forceinline__ uint64_t row_bits(uint64_t m, int s) {
    const uint32_t x = (uint32_t)(m >> (16 * s)) & 0xffffu;
    const uint32_t y = x | (x << 16);
    return ((uint64_t)y << 32) | y;
}
__device__ __forceinline__ bool lane_of(uint64_t m) {
    return __builtin_amdgcn_inverse_ballot_w64(m);
}

// The lanes of every row that holds a set bit of m.
__device__ __forceinline__ uint64_t rows_with(uint64_t m) {
    uint64_t r = 0;
#pragma unroll
    for (int s = 0; s < kSlots; ++s)
        if (m & row_lanes(s)) r |= row_lanes(s);
    return r;
}

__device__ __forceinline__ int row_min(int v) {
    v = min(v, dpp_i<kDppRowMirror>(v));
    v = min(v, dpp_i<kDppRowHalfMirror>(v));
    v = min(v, dpp_i<kDppQuadXor2>(v));
    return min(v, dpp_i<kDppQuadXor1>(v));
}

// Transpose across the rows: on return row r holds, in v[q], what row q held in
// v[r].
__device__ __forceinline__ void rows_transpose(float (&v)[kSlots]) {
    auto swap32 = [](float& a, float& b) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b),
                                                        false, false);
        a = __uint_as_float(r[0]);
        b = __uint_as_float(r[1]);
    };
    auto swap16 = [](float& a, float& b) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b),
                                                        false, false);
        a = __uint_as_float(r[0]);
        b = __uint_as_float(r[1]);
    };
    swap32(v[0], v[2]);
    swap32(v[1], v[3]);
    swap16(v[0], v[1]);
    swap16(v[2], v[3]);
}

// Reduce-scatter of N <= 16 values over each row of 16 lanes (the DPP rounds
// of ReduceScatter), and the value a lane ends with (bit 6 set when a lower
// lane of its row holds the same).
template <int N>
__device__ __forceinline__ float row_reduce_scatter(const float (&v)[N], int lane) {
    static_assert(N <= 16, "one value per lane of a row");
    return ReduceScatter<N, 2>::run(v, lane);
}
template <int N>
__device__ __forceinline__ int row_slot(int lane) {
    int ns[6];
    ns[2] = N;
#pragma unroll
    for (int r = 3; r < 6; ++r) ns[r] = ns[r - 1] - ns[r - 1] / 2;
    int pos = 0, dup = 0;
#pragma unroll
    for (int r = 5; r >= 2; --r) {
        const int h = ns[r] / 2, np = ns[r] - h;
        const int bit = (lane >> (5 - r)) & 1;
        if (pos < h) pos += bit ? np : 0;
        else dup |= bit;
    }
    return pos | (dup << 6);
}

// Tile, 8x8 quadrant and pixel of this lane.  Blocks go to the eight XCDs in
// turn, so the quadrants of one tile are eight blocks apart: they share one L2.
struct NarrowPixel {
    int tile, quad, j, i, sub;
    bool inside;
};

inline int narrow_grid(int tiles) { return ((tiles + 7) / 8) * 32; }

__device__ __forceinline__ NarrowPixel narrow_pixel(const RasterArgs& a, int wave, int lane) {
    NarrowPixel p;
    const int b = blockIdx.x, k = b >> 3;
    p.tile = (k >> 2) * 8 + (b & 7);
    p.quad = k & 3;
    const int ty = p.tile / a.tiles_x, tx = p.tile - ty * a.tiles_x;
    p.j = tx * 16 + (p.quad & 1) * 8 + (wave & 1) * 4 + (lane & 3);
    p.i = ty * 16 + (p.quad >> 1) * 8 + (wave >> 1) * 4 + ((lane >> 2) & 3);
    p.sub = lane >> 4;
    p.inside = p.i < a.img_h && p.j < a.img_w;
    return p;
}

// A lane's chart: byte offset of its first texel in the texture, ok false for
// a chart that does not lie inside the texture (see chart_of; the launch
// requires the texture's size in bytes to be below 2^31).
template <bool TB>
__device__ __forceinline__ int chart_offset(const Splat& s, int C, int num_texels, bool& ok) {
    constexpr int E = TB ? 2 : 4;
    const uint32_t h = (uint32_t)s.h, w = (uint32_t)s.w, n = h * w;
    ok = s.start >= 0 && s.h > 0 && s.w > 0 && h < (1u << 24) && w < (1u << 24) &&
         __umulhi(h, w) == 0 && n <= (uint32_t)num_texels &&
         (uint32_t)s.start <= (uint32_t)num_texels - n;
    return ok ? s.start * (C * E) : 0;
}

// Bilinear taps of a lane's chart: as chart_taps_ij (weights, fractions, tap
// rows and columns), with texel indices inside the chart.
__device__ __forceinline__ void narrow_taps(const Splat& s, float u, float v, float& fu, float& fv,
                                            int& iu, int& iv, int& ju, int& jv, float (&wt)[4],
                                            int (&at)[4]) {
    const float tu = (float)s.h * u, tv = (float)s.w * v;
    const int iu0 = f2i_trunc(tu), iv0 = f2i_trunc(tv);
    fu = __builtin_amdgcn_fractf(tu);
    fv = __builtin_amdgcn_fractf(tv);
    iu = min(iu0, s.h - 1);
    iv = min(iv0, s.w - 1);
    ju = min(iu0 + 1, s.h - 1);
    jv = min(iv0 + 1, s.w - 1);
    wt[0] = (1.f - fu) * (1.f - fv);
    wt[1] = (1.f - fu) * fv;
    wt[2] = fu * (1.f - fv);
    wt[3] = fu * fv;
    at[0] = iu * s.w + iv;
    at[1] = iu * s.w + jv;
    at[2] = ju * s.w + iv;
    at[3] = ju * s.w + jv;
}

template <int CM, bool TB>
__device__ __forceinline__ void narrow_texels(__amdgpu_buffer_rsrc_t rsrc, int base, bool ok,
                                              const int (&at)[4], float (&tv)[4][CM]) {
    constexpr int E = TB ? 2 : 4;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        // 2^31 is past the resource, which reads as 0 (the hardware range check)
        const int off = ok ? base + at[k] * (CM * E) : (int)0x80000000;
#pragma unroll
        for (int c = 0; c < CM; ++c) {
            if constexpr (TB)
                tv[k][c] = __uint_as_float(
                    (unsigned)(unsigned short)__builtin_amdgcn_raw_buffer_load_b16(
                        rsrc, off + c * E, 0, 0)
                    << 16);
            else
                tv[k][c] = __uint_as_float(
                    __builtin_amdgcn_raw_buffer_load_b32(rsrc, off + c * E, 0, 0));
        }
    }
}

template <int CM, bool TB>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t texture_rsrc(const RasterArgs& a) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.texture), (short)0,
                                             a.num_texels * (CM * (TB ? 2 : 4)), kBufferWord3);
}

// The entries of one step that meet the quadrant, in walking order, with the
// culling data the waves test against their own pixels; and the records of a
// batch of them (rows padded to 36 floats: the four rows of a wave read
// different banks).
constexpr int kStep = 256, kBatch = 64, kRecStride = 36, kScan = 64;
struct NarrowList {
    float4 el[kStep];
    uint2 box[kStep];
    float ec[kStep];
    int g[kStep], e[kStep];
    float rec[kBatch * kRecStride];
    int cnt[4];
};

// Appends this thread's entry (cand) to the list, in the order of waves and,
// in a wave, of lanes (descending with BACK); returns the list's length.  Two
// barriers; the list is complete after the second.
template <bool BACK>
__device__ __forceinline__ int list_append(NarrowList& L, bool cand, int g, int e, uint2 box,
                                           float4 el, float ec, int wave, int lane) {
    const uint64_t m = lanes_where(cand);
    if (lane == 0) L.cnt[wave] = __popcll(m);
    __syncthreads();
    int off = 0, n = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const int c = L.cnt[w];
        if (w < wave) off += c;
        n += c;
    }
    if (cand) {
        const uint64_t before = BACK ? (lane == 63 ? 0ull : m >> (lane + 1))
                                     : m & ((1ull << lane) - 1ull);
        const int at = off + __popcll(before);
        L.g[at] = g;
        L.e[at] = e;
        L.box[at] = box;
        L.el[at] = el;
        L.ec[at] = ec;
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(n);
}

// Copies the records of list entries [b0, b0 + nb) into LDS (no barrier).
__device__ __forceinline__ void stage_batch(NarrowList& L, const float* records, int b0, int nb) {
    const float4* src = reinterpret_cast<const float4*>(records);
    for (int k = threadIdx.x; k < nb * (kRecordFloats / 4); k += 256) {
        const int i = k / (kRecordFloats / 4), c = k % (kRecordFloats / 4);
        *reinterpret_cast<float4*>(&L.rec[i * kRecStride + 4 * c]) =
            src[(size_t)L.g[b0 + i] * (kRecordFloats / 4) + c];
    }
}

// The batch entries (bit i: entry b0 + i) that can meet the wave's rectangle.
template <bool BLUR>
__device__ __forceinline__ uint64_t batch_meets(const NarrowList& L, int b0, int nb, bool cull,
                                                const WaveRect& rect, int lane) {
    bool meets = lane < nb;
    if (cull && meets) {
        const int i = b0 + lane;
        meets = box_meets(L.box[i], rect);
        if (meets && !ellipse_meets(L.el[i], L.ec[i], rect))
            meets = BLUR && blur_disc_meets(&L.rec[lane * kRecStride], rect);
    }
    return lanes_where(meets);
}

// A list entry's culling test against a rectangle, and its data.
template <bool BLUR>
__device__ __forceinline__ bool entry_meets(const RasterArgs& a, bool cull, int gid,
                                            const WaveRect& rect, uint2& box, float4& el,
                                            float& ec) {
    box = make_uint2(0u, 0u);
    el = make_float4(0.f, 0.f, -1.f, 0.f);
    ec = 0.f;
    if (!cull) return true;
    box = a.boxes[gid];
    el = a.ellipses[gid];
    ec = a.ellipse_c[gid];
    if (!box_meets(box, rect)) return false;
    if (ellipse_meets(el, ec, rect)) return true;
    if constexpr (BLUR) return blur_disc_meets(a.records + (size_t)gid * kRecordFloats, rect);
    return false;
}

__device__ __forceinline__ int list_id(const RasterArgs& a, int e) {
    return min(max(a.ids_sorted[e], 0), a.num_points - 1);
}

// Up to four batch entries for the four slots: takes them off `cand` (lowest
// bits first); returns the bit of this lane's slot (slot 0's for a slot
// without an entry) and the number taken.
__device__ __forceinline__ int take_four(uint64_t& cand, int (&bit)[kSlots], int& n, int sub) {
    n = 0;
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
        if (cand != 0) {
            bit[s] = __ffsll((unsigned long long)cand) - 1;
            cand &= cand - 1;
            n = s + 1;
        } else {
            bit[s] = bit[0];
        }
    }
    int b = bit[0];
#pragma unroll
    for (int s = 1; s < kSlots; ++s) b = sub == s ? bit[s] : b;
    return b;
}

// ------------------------------------------------------------------ forward
template <int CM, bool BLUR, bool TB>
__global__ __launch_bounds__(256) void k_raster_forward_narrow(RasterArgs a, FwdOut o) {
    __shared__ NarrowList L;
    __shared__ int s_rect[4][4];
    __shared__ uint32_t s_mask[kStep / 32];
    __shared__ int s_last[2];
    const int lane = threadIdx.x & (kWave - 1), wave = wave_index();
    const NarrowPixel px = narrow_pixel(a, wave, lane);
    const int tile = px.tile, sub = px.sub;
    if (tile >= a.tiles_x * a.tiles_y) return;
    const bool inside = px.inside;
    const PixelRay pr = pixel_ray(a.c2w, a.viewmat, a.fx, a.fy, a.cx, a.cy, px.j, px.i);
    const bool flip = a.settings & kSetNormalFlip;
    int r0, r1;
    tile_range(a, tile, r0, r1);
    const int mword0 = (r0 >> 6) + tile, mentry0 = r0 & ~63;
    uint64_t* const mplane =
        a.wave_masks ? a.wave_masks + (size_t)px.quad * a.mask_plane + mword0 : nullptr;
    const __amdgpu_buffer_rsrc_t rsrc = texture_rsrc<CM, TB>(a);

    // pixel state, the same on the four lanes of a pixel
    bool done = !inside;
    float T = 1.f, pdepth = 0.f, preg = 0.f, s0 = 0.f, s1 = 0.f, s2 = 0.f;
    int cur_idx = 0, pdi = -1;
    // this row's part of the pixel's sums: colour (row 0), normal (row 1), the
    // first three texture channels (row 2), the fourth in acc[0] of row 3
    float acc[3] = {0.f, 0.f, 0.f};

    // culling rectangle of the wave's live pixels (shrinks as pixels finish,
    // as in k_raster_forward); the scan uses the union over the waves
    WaveRect rect = wave_rect(inside, px.j, px.i);
    int live = __popcll(lanes_where(inside));
    constexpr float kKeep = 1.f - 1.f / 255.f;
    const bool cull = a.boxes != nullptr;
    int sb = mentry0;
    int gid_next = 0;
    {
        const int e = sb + (int)threadIdx.x;
        if (e >= r0 && e < r1) gid_next = list_id(a, e);
    }
    while (sb < r1) {
        if (lane == 0) {
            s_rect[wave][0] = rect.x0;
            s_rect[wave][1] = rect.x1;
            s_rect[wave][2] = rect.y0;
            s_rect[wave][3] = rect.y1;
        }
        __syncthreads();
        // (after the barrier: every thread has read the last step's words)
        if (threadIdx.x < kStep / 32) s_mask[threadIdx.x] = 0u;
        WaveRect all = {0x7fffffff, -0x7fffffff, 0x7fffffff, -0x7fffffff};
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            all.x0 = min(all.x0, s_rect[w][0]);
            all.x1 = max(all.x1, s_rect[w][1]);
            all.y0 = min(all.y0, s_rect[w][2]);
            all.y1 = max(all.y1, s_rect[w][3]);
        }
        if (all.x1 < all.x0) break;  // every pixel of the block is done
        const int e = sb + (int)threadIdx.x;
        const int gid = gid_next;
        const bool in_range = e >= r0 && e < r1;
        uint2 box;
        float4 el;
        float ec;
        bool cand = entry_meets<BLUR>(a, cull, gid, all, box, el, ec);
        cand = cand && in_range;
        const int e_last = min(sb + kStep, r1) - 1;
        if (e >= e_last - 1 && e <= e_last) s_last[e_last - e] = e >= r0 ? gid : -1;
        {
            const int en = e + kStep;  // the next step's ids, read ahead
            gid_next = en >= r0 && en < r1 ? list_id(a, en) : 0;
        }
        const int n = list_append<false>(L, cand, gid, e, box, el, ec, wave, lane);
        for (int b0 = 0; b0 < n; b0 += kBatch) {
            const int nb = min(kBatch, n - b0);
            if (b0) __syncthreads();
            stage_batch(L, a.records, b0, nb);
            __syncthreads();
            uint64_t cand_m = batch_meets<BLUR>(L, b0, nb, cull, rect, lane);
            const int e_lane = L.e[b0 + min(lane, nb - 1)];
            uint64_t comp_all = 0;
            while (cand_m != 0) {
                if (!any_lane(!done)) break;
                int bit[kSlots], ns;
                const int mybit = take_four(cand_m, bit, ns, sub);
                const Splat s = load_splat(&L.rec[mybit * kRecStride]);
                const Pair p = pair_eval(s, pr, BLUR);
                const uint64_t skip_m = skip_lanes(p);
                float A[kSlots], D[kSlots];
                rows4(p.alpha, A);
                rows4(p.t, D);
                float vis[kSlots];
                uint64_t comp_m[kSlots];
#pragma unroll
                for (int q = 0; q < kSlots; ++q) {
                    comp_m[q] = 0;
                    vis[q] = 0.f;
                    if (q >= ns) continue;
                    // the 8x8 kernel's step for entry q: its operations and
                    // their contraction (a product that feeds one sum is
                    // fused there)
                    const float next_T = T * (1.f - A[q]);
                    done = done || next_T <= 1e-4f;
                    const bool comp = !done && !lane_of(row_bits(skip_m, q));
                    comp_m[q] = lanes_where(comp);
                    if (comp_m[q] == 0) continue;
                    const int eq = __builtin_amdgcn_readlane(e_lane, bit[q]);
                    comp_all |= 1ull << bit[q];
                    if (comp) {
                        const float d = D[q];
                        vis[q] = A[q] * T;
                        preg = fmaf(fmaf(-s1, d + d, fmaf(s0, d * d, s2)), vis[q], preg);
                        if constexpr (BLUR) {
#pragma clang fp contract(off)
                            s0 = s0 + vis[q];
                        } else {
                            s0 = fmaf(A[q], T, s0);
                        }
                        s1 = fmaf(d, vis[q], s1);
                        s2 = fmaf(d, d * vis[q], s2);
                        if (T > 0.5f) {
                            pdepth = d * pr.view_depth;
                            pdi = eq;
                        }
                        T = next_T;
                        cur_idx = eq;
                        if (T * kKeep <= 1e-4f) done = true;
                    }
                }
                uint64_t my_comp = 0;
#pragma unroll
                for (int q = 0; q < kSlots; ++q) my_comp |= comp_m[q] & row_lanes(q);
                if (my_comp == 0) continue;
                float val[4] = {0.f, 0.f, 0.f, 0.f};
                if (lane_of(my_comp)) {
                    float u, v, fu, fv, wt[4], tv[4][CM];
                    int iu, iv, ju, jv, at[4];
                    bool ok;
                    splat_uv(s, p.delta, u, v);
                    const int base_off = chart_offset<TB>(s, CM, a.num_texels, ok);
                    narrow_taps(s, u, v, fu, fv, iu, iv, ju, jv, wt, at);
                    narrow_texels<CM, TB>(rsrc, base_off, ok, at, tv);
#pragma unroll
                    for (int c = 0; c < CM; ++c)
                        val[c] = fmaf(wt[3], tv[3][c],
                                      fmaf(wt[2], tv[2][c],
                                           fmaf(wt[0], tv[0][c], wt[1] * tv[1][c])));
                }
                // the facing normal: the flip's sign is exact
                const float sg = (flip && dot3(pr.r, s.a3) > 0.f) ? -1.f : 1.f;
                float x[3][kSlots] = {{s.rgb.x, sg * s.a3.x, val[0], val[3]},
                                      {s.rgb.y, sg * s.a3.y, val[1], 0.f},
                                      {s.rgb.z, sg * s.a3.z, val[2], 0.f}};
#pragma unroll
                for (int k = 0; k < 3; ++k) rows_transpose(x[k]);
#pragma unroll
                for (int q = 0; q < kSlots; ++q)
                    if (lane_of(comp_m[q])) {
#pragma unroll
                        for (int k = 0; k < 3; ++k) acc[k] = fmaf(x[k][q], vis[q], acc[k]);
                    }
            }
            if (lane_of(comp_all))
                atomicOr(&s_mask[(e_lane - sb) >> 5], 1u << (e_lane & 31));
        }
        {
            const int now = __popcll(lanes_where(!done));
            if (now < live) {
                live = now;
                rect = wave_rect(!done, px.j, px.i);
            }
        }
        __syncthreads();  // the step's mask words are complete, its lists consumed
        if (mplane && threadIdx.x < kStep / 64 && sb + 64 * (int)threadIdx.x < r1)
            mplane[((sb - mentry0) >> 6) + threadIdx.x] =
                ((uint64_t)s_mask[2 * threadIdx.x + 1] << 32) | s_mask[2 * threadIdx.x];
        // Copies of the step's last entry in a row (see k_raster_forward): if
        // it changed no pixel (evaluated or culled), neither do its copies, so
        // stretches of 8 steps that hold nothing else are passed over.
        const int dup_g = s_last[0];
        const bool copies = s_last[1] == dup_g && e_last > r0 &&
                            !((s_mask[(e_last - sb) >> 5] >> (e_last & 31)) & 1u);
        sb += kStep;
        if (copies) {
            bool moved = false;
            while (sb < r1) {
                bool same = true;
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const int ek = sb + kStep * k + (int)threadIdx.x;
                    same = same && (ek >= r1 || a.ids_sorted[ek] == dup_g);
                }
                if (!__syncthreads_and(same)) break;
                if (mplane && threadIdx.x < 8 * kStep / 64 && sb + 64 * (int)threadIdx.x < r1)
                    mplane[((sb - mentry0) >> 6) + threadIdx.x] = 0ull;
                sb += 8 * kStep;
                moved = true;
            }
            if (moved) {
                const int en = sb + (int)threadIdx.x;
                gid_next = en >= r0 && en < r1 ? list_id(a, en) : 0;
            }
        }
    }
    if (!inside) return;
    // each row writes its part of the pixel's outputs
    const int pid = px.i * a.img_w + px.j;
    if (sub == 0) {
#pragma unroll
        for (int k = 0; k < 3; ++k)
            o.out_img[3 * pid + k] = fmaf(T, a.background[k], acc[k]);
        o.out_depth[pid] = pdepth;
    } else if (sub == 1) {
#pragma unroll
        for (int k = 0; k < 3; ++k) o.out_normal[3 * pid + k] = acc[k];
        o.out_reg[pid] = preg;
    } else if (sub == 2) {
#pragma unroll
        for (int c = 0; c < (CM < 3 ? CM : 3); ++c) o.out_texture[(size_t)pid * CM + c] = acc[c];
        o.final_Ts[pid] = T;
        o.final_idx[pid] = cur_idx;
        o.depth_idx[pid] = pdi;
    } else {
        if constexpr (CM == 4) o.out_texture[(size_t)pid * CM + 3] = acc[0];
        o.out_reg_s[3 * pid + 0] = s0;
        o.out_reg_s[3 * pid + 1] = s1;
        o.out_reg_s[3 * pid + 2] = s2;
    }
}

// ------------------------------------------------------------------ backward
// A batch entry's texel gradients meet in LDS too: a window of 4x4 texels of
// its chart, whose corner the first row to reach the entry sets (kNoAnchor:
// not yet set), one texel before that row's own taps.  An entry with a row
// whose taps do not fit (a splat seen edge-on runs over many texels in a few
// pixels) takes a copy of its whole chart from a pool; with the pool used up
// the taps go to memory directly.  Waves must not wait for memory here: loads
// and atomics of a wave complete in order, so the next group's texel reads
// would wait for these atomics' round trip.
constexpr int kTexWin = 4, kTexPool = 3072;
constexpr unsigned long long kNoAnchor = ~0ull;
constexpr int kPoolUnset = -1, kPoolNone = -2;  // not asked for yet; being taken, or none left
constexpr int kGradSums = G_EXTRA + 2;          // per-Gaussian sums and the two blur values

template <int CM, bool BLUR, bool TB>
__global__ __launch_bounds__(256) void k_raster_backward_narrow(RasterArgs a, BwdIn b) {
    __shared__ NarrowList L;
    __shared__ float s_grad[kBatch * kGradSums];  // the batch's per-Gaussian sums
    __shared__ float s_tex[kBatch * kTexWin * kTexWin * CM];  // and its texel windows
    __shared__ unsigned long long s_anchor[kBatch];
    __shared__ float s_pool[kTexPool];  // zero between batches
    __shared__ int s_pool_at[kBatch], s_pool_list[kBatch], s_pool_used, s_pool_count;
    __shared__ uint64_t s_word[kScan];
    __shared__ int s_win[kScan];
    __shared__ int s_wave[4][5];
    const int lane = threadIdx.x & (kWave - 1), wave = wave_index();
    const NarrowPixel px = narrow_pixel(a, wave, lane);
    const int tile = px.tile, sub = px.sub;
    if (tile >= a.tiles_x * a.tiles_y) return;
    const bool inside = px.inside;
    const PixelRay pr = pixel_ray(a.c2w, a.viewmat, a.fx, a.fy, a.cx, a.cy, px.j, px.i);
    const bool prop_uv = a.settings & kSetUvGrad;
    const int pid = inside ? px.i * a.img_w + px.j : 0;
    const __amdgpu_buffer_rsrc_t rsrc = texture_rsrc<CM, TB>(a);

    float T = 1.f, S0 = 0.f, S1 = 0.f, S2 = 0.f, vdep = 0.f, vreg = 0.f, vT = 0.f;
    V3 vo = v3(0.f, 0.f, 0.f), vn = v3(0.f, 0.f, 0.f);
    int dfin = -1, bfin = -1;
    float vtex[CM];
#pragma unroll
    for (int c = 0; c < CM; ++c) vtex[c] = 0.f;
    if (inside) {
        T = b.final_Ts[pid];
        S0 = b.final_s[3 * pid];
        S1 = b.final_s[3 * pid + 1];
        S2 = b.final_s[3 * pid + 2];
        dfin = b.depth_idx[pid];
        bfin = b.final_idx[pid];
        vo = v3(b.v_img[3 * pid], b.v_img[3 * pid + 1], b.v_img[3 * pid + 2]);
        vn = v3(b.v_normal[3 * pid], b.v_normal[3 * pid + 1], b.v_normal[3 * pid + 2]);
        vdep = b.v_depth[pid];
        vreg = b.v_reg[pid];
#pragma unroll
        for (int c = 0; c < CM; ++c) vtex[c] = b.v_texture_out[(size_t)pid * CM + c];
        if constexpr (CM == 3) {
            if (b.loss_target) {  // vo, vtex hold out_img, out_texture
                const float* tg = b.loss_target + 3 * pid;
                const float g0 = l2_cotangent(vo.x, vtex[0], tg[0], b.loss_scale);
                const float g1 = l2_cotangent(vo.y, vtex[1], tg[1], b.loss_scale);
                const float g2 = l2_cotangent(vo.z, vtex[2], tg[2], b.loss_scale);
                vo = v3(g0, g1, g2);
                vtex[0] = g0;
                vtex[1] = g1;
                vtex[2] = g2;
            }
        }
        vT = a.background[0] * vo.x + a.background[1] * vo.y + a.background[2] * vo.z -
             b.v_alpha[pid];
    }
    // pixels with a texture cotangent that is not finite: a window's sums weigh
    // texels which they do not sample by zero
    bool finite = true;
#pragma unroll
    for (int c = 0; c < CM; ++c) finite = finite && fabsf(vtex[c]) < INFINITY;
    const uint64_t bad = lanes_where(!finite);
    for (int k = threadIdx.x; k < kTexPool; k += 256) s_pool[k] = 0.f;
    int r0, r1;
    tile_range(a, tile, r0, r1);
    const int wave_last = wave_max(bfin);
    const int last_e = inside ? bfin : -1;
    const bool cull = a.boxes != nullptr;
    const WaveRect rect = wave_rect(inside, px.j, px.i);
    if (lane == 0) {
        s_wave[wave][0] = rect.x0;
        s_wave[wave][1] = rect.x1;
        s_wave[wave][2] = rect.y0;
        s_wave[wave][3] = rect.y1;
        s_wave[wave][4] = wave_last;
    }
    __syncthreads();
    WaveRect all = {0x7fffffff, -0x7fffffff, 0x7fffffff, -0x7fffffff};
    int block_last = -1;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        all.x0 = min(all.x0, s_wave[w][0]);
        all.x1 = max(all.x1, s_wave[w][1]);
        all.y0 = min(all.y0, s_wave[w][2]);
        all.y1 = max(all.y1, s_wave[w][3]);
        block_last = max(block_last, s_wave[w][4]);
    }
    const int e_hi = __builtin_amdgcn_readfirstlane(min(r1 - 1, block_last));
    // Four entries of a batch: this lane's is batch entry mybit, list entry e.
    auto four = [&](const int ns, const int mybit, const int e) {
        const Splat s = load_splat(&L.rec[mybit * kRecStride]);
        const Pair p = pair_eval(s, pr, BLUR);
        const uint64_t has = ns == kSlots ? ~0ull : (1ull << (16 * ns)) - 1ull;
        const uint64_t vmask = lanes_where(e <= last_e) & ~skip_lanes(p) & has;
        if (vmask == 0) return;
        const bool valid = lane_of(vmask);

        bool ok;
        float u, v, fu, fv, wt[4], tv[4][CM];
        int iu, iv, ju, jv, at[4];
        splat_uv(s, p.delta, u, v);
        const int base_off = chart_offset<TB>(s, CM, a.num_texels, ok);
        narrow_taps(s, u, v, fu, fv, iu, iv, ju, jv, wt, at);
        narrow_texels<CM, TB>(rsrc, base_off, ok, at, tv);
        float D[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < CM; ++c)
#pragma unroll
            for (int k = 0; k < 4; ++k) D[k] = fmaf(tv[k][c], vtex[c], D[k]);
        float vvis = dot3(s.rgb, vo) + dot3(s.a3, vn);
        // (every fused product below is the one the 8x8 kernel forms: several of
        // these terms cancel, and optimisers divide by a gradient's size)
        vvis += fmaf(wt[1], D[1], wt[0] * D[0]) + fmaf(wt[3], D[3], wt[2] * D[2]);
        const float dval = p.t;
        const float vw = (fmaf(S0, dval * dval, -(2.f * dval * S1)) + S2) * vreg;

        // the transmittance and its cotangent through the four entries
        float A[kSlots], V[kSlots], W[kSlots];
        rows4(p.alpha, A);
        rows4(vvis, V);
        rows4(vw, W);
        float my_T = 0.f, my_vT = 0.f;
#pragma unroll
        for (int q = 0; q < kSlots; ++q) {
            if (q >= ns) break;
            const bool val_q = lane_of(row_bits(vmask, q));
            if (val_q) T = T * __builtin_amdgcn_rcpf(1.f - A[q]);
            if (lane_of(row_lanes(q))) {
                my_T = T;
                my_vT = vT;
            }
            const float vTn = fmaf(W[q], A[q], fmaf(A[q], V[q] - vT, vT));
            if (val_q) vT = vTn;
        }

        const float vis = valid ? p.alpha * my_T : 0.f;
        float vu = 0.f, vv = 0.f;
        if (prop_uv) {
            vu = vis * (float)s.h * fmaf(1.f - fv, D[2] - D[0], fv * (D[3] - D[1]));
            vv = vis * (float)s.w * fmaf(1.f - fu, D[1] - D[0], fu * (D[3] - D[2]));
        }
        if (!valid) vu = vv = 0.f;  // NaN-safe zero seeds
        const float vd_val = 2.f * fmaf(S0, vis * dval, -(vis * S1)) * vreg;
        float valpha = fmaf(vw, my_T, my_T * (vvis - my_vT));
        valpha = valid ? valpha : 0.f;
        const float vtview = (e == dfin && dfin != -1) ? vdep : 0.f;
        float vt = fmaf(pr.view_depth, vtview, vd_val);
        vt = valid ? vt : 0.f;

        float gr[16], ge[BLUR ? 6 : 4];
        gr[G_RGB + 0] = vis * vo.x;
        gr[G_RGB + 1] = vis * vo.y;
        gr[G_RGB + 2] = vis * vo.z;
        gr[G_OPAC] = (p.blur_sel ? p.Gb : p.G) * valpha;
        const float vsigma = p.blur_sel ? 0.f : -s.opac * p.G * valpha;
        const float vl1 = vsigma * s.iq1 * p.l1;
        const float vl2 = vsigma * s.iq2 * p.l2;
        auto vd = [&](float a1, float a2, float um, float vm) {
            return fmaf(vm, vv, fmaf(um, vu, fmaf(vl1, a1, vl2 * a2)));
        };
        const V3 vdelta = v3(vd(s.a1.x, s.a2.x, s.umap.x, s.vmap.x),
                             vd(s.a1.y, s.a2.y, s.umap.y, s.vmap.y),
                             vd(s.a1.z, s.a2.z, s.umap.z, s.vmap.z));
        vt += dot3(vdelta, pr.r);
        const float vnum = vt * __builtin_amdgcn_rcpf(p.den);
        const float vden = -vnum * p.t;
        gr[G_P11] = vl1 * p.l1;
        gr[G_P12] = vl1 * p.l2;
        gr[G_P21] = vl2 * p.l1;
        gr[G_P22] = vl2 * p.l2;
        gr[G_U1] = vu * p.l1;
        gr[G_U2] = vu * p.l2;
        ge[G_V1 - 16] = vv * p.l1;
        ge[G_V2 - 16] = vv * p.l2;
        gr[G_VL1] = vl1;
        gr[G_VL2] = vl2;
        ge[G_VU - 16] = vu;
        ge[G_VV - 16] = vv;
        gr[G_VNUM] = vnum;
        gr[G_AX3X + 0] = fmaf(vis, vn.x, vden * pr.r.x);
        gr[G_AX3X + 1] = fmaf(vis, vn.y, vden * pr.r.y);
        gr[G_AX3X + 2] = fmaf(vis, vn.z, vden * pr.r.z);
        if constexpr (BLUR) {
            const float vsb = p.blur_sel ? -s.opac * p.Gb * valpha : 0.f;
            ge[4] = 2.0f * vsb * (s.pix_x - pr.px);
            ge[5] = 2.0f * vsb * (s.pix_y - pr.py);
        }
        {
            // rows without a valid lane add nothing
            const bool add = lane_of(rows_with(vmask));
            float* const grec = s_grad + mybit * kGradSums;
            const float t0 = row_reduce_scatter<16>(gr, lane);
            const int c0 = row_slot<16>(lane);
            if (add && t0 != 0.f) unsafeAtomicAdd(grec + c0, t0);
            constexpr int NE = BLUR ? 6 : 4;
            const float t1 = row_reduce_scatter<NE>(ge, lane);
            const int c1 = row_slot<NE>(lane);
            if (add && c1 < 64 && t1 != 0.f)
                unsafeAtomicAdd(grec + 16 + c1, t1);
        }

        // Texel gradients.  A row whose valid lanes' taps lie in one 3x3
        // texel window (2x2 where that holds for every such row) inside its
        // entry's 4x4 window reduces the values of its texels and adds them
        // there; the lanes of other rows, and of rows with a pixel of `bad`, add
        // their own taps.
        const uint64_t okmask = vmask & lanes_where(ok);
        if (okmask == 0) return;
        const bool part = lane_of(okmask);
        const int ou = row_min(part ? iu : 0x3fffffff), ov = row_min(part ? iv : 0x3fffffff);
        unsigned long long anchor = 0;
        if ((lane & 15) == 0 && lane_of(rows_with(okmask))) {
            const int wu = min(max(ou - 1, 0), max(s.h - kTexWin, 0));
            const int wv = min(max(ov - 1, 0), max(s.w - kTexWin, 0));
            const unsigned long long want = ((unsigned long long)(unsigned)wu << 32) | (unsigned)wv;
            anchor = atomicCAS(&s_anchor[mybit], kNoAnchor, want);
            if (anchor == kNoAnchor) anchor = want;
        }
        const int au = __shfl((int)(anchor >> 32), lane & 48), av = __shfl((int)anchor, lane & 48);
        const int ri = iu - ou, rj = ju - ou, ci = iv - ov, cj = jv - ov;
        const uint64_t far =
            okmask & (bad | lanes_where(((uint32_t)ri | (uint32_t)ci) > 1u) |
                      lanes_where((uint32_t)(iu - au) >= (uint32_t)kTexWin) |
                      lanes_where((uint32_t)(ju - au) >= (uint32_t)kTexWin) |
                      lanes_where((uint32_t)(iv - av) >= (uint32_t)kTexWin) |
                      lanes_where((uint32_t)(jv - av) >= (uint32_t)kTexWin));
        uint64_t direct = 0;
        if (far != 0) direct = rows_with(far);
        const uint64_t win = okmask & ~direct;
        float vval[CM];
#pragma unroll
        for (int c = 0; c < CM; ++c) vval[c] = vis * vtex[c];
        if (win != 0) {
            const bool at0 = ri == 0, bt0 = ci == 0, samea = rj == ri, sameb = cj == ci;
            const float a1 = samea ? 1.f : 1.f - fu, a2 = samea ? 0.f : fu;
            const float b1 = sameb ? 1.f : 1.f - fv, b2 = sameb ? 0.f : fv;
            const float Wa[3] = {at0 ? a1 : 0.f, at0 ? a2 : a1, at0 ? 0.f : a2};
            const float Wb[3] = {bt0 ? b1 : 0.f, bt0 ? b2 : b1, bt0 ? 0.f : b2};
            float vk[CM];
#pragma unroll
            for (int c = 0; c < CM; ++c) vk[c] = lane_of(win) ? vval[c] : 0.f;
            const bool row_ok = lane_of(rows_with(win));
            float* const tex = s_tex + mybit * (kTexWin * kTexWin * CM);
            // window texel (r, q), channel c; one past the 4x4 window carries
            // no weight
            auto add = [&](int code, int r, int q, int c, float tot) {
                const int wr = ou + r - au, wq = ov + q - av;
                if (code < 64 && tot != 0.f && row_ok && wr < kTexWin && wq < kTexWin)
                    unsafeAtomicAdd(tex + (wr * kTexWin + wq) * CM + c, tot);
            };
            if (!((lanes_where(rj == 2) | lanes_where(cj == 2)) & win)) {
                float vals[4 * CM];
#pragma unroll
                for (int r = 0; r < 2; ++r)
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const float ab = Wa[r] * Wb[q];
#pragma unroll
                        for (int c = 0; c < CM; ++c) vals[(2 * r + q) * CM + c] = ab * vk[c];
                    }
                const float tot = row_reduce_scatter<4 * CM>(vals, lane);
                const int code = row_slot<4 * CM>(lane), rq = (code & 63) / CM;
                add(code, rq >> 1, rq & 1, (code & 63) - CM * rq, tot);
            } else {
#pragma unroll
                for (int r = 0; r < 3; ++r) {
                    float vals[3 * CM];
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        const float ab = Wa[r] * Wb[q];
#pragma unroll
                        for (int c = 0; c < CM; ++c) vals[q * CM + c] = ab * vk[c];
                    }
                    const float tot = row_reduce_scatter<3 * CM>(vals, lane);
                    const int code = row_slot<3 * CM>(lane), q = (code & 63) / CM;
                    add(code, r, q, (code & 63) - CM * q, tot);
                }
            }
        }
        if (direct == 0) return;
        // the row's pool space, taken by the first row that needs it
        int pool = kPoolNone;
        if ((lane & 15) == 0 && lane_of(direct)) {
            pool = atomicCAS(&s_pool_at[mybit], kPoolUnset, kPoolNone);
            if (pool == kPoolUnset) {
                const int size = s.h * s.w <= kTexPool / CM ? s.h * s.w * CM : kTexPool + 1;
                const int at0 = atomicAdd(&s_pool_used, min(size, kTexPool + 1));
                pool = at0 + size <= kTexPool ? at0 : kPoolNone;
                if (pool >= 0) {
                    s_pool_at[mybit] = pool;
                    s_pool_list[atomicAdd(&s_pool_count, 1)] = mybit;
                }
            }
        }
        pool = __shfl(pool, lane & 48);
        if (lane_of(okmask & direct)) {
            float* const chart = b.v_texture + (size_t)s.start * CM;
            if (pool >= 0) {
#pragma unroll
                for (int k = 0; k < 4; ++k)
#pragma unroll
                    for (int c = 0; c < CM; ++c) {
                        const float add = wt[k] * vval[c];
                        if (add != 0.f) unsafeAtomicAdd(s_pool + pool + at[k] * CM + c, add);
                    }
                return;
            }
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int c = 0; c < CM; ++c) {
                    const float add = wt[k] * vval[c];
                    if (add != 0.f) unsafeAtomicAdd(chart + at[k] * CM + c, add);
                }
        }
    };

    // Back to front over [r0, e_hi]: the entries the forward composited in this
    // quadrant (all of them without masks) whose screen bounds meet it.  Mask
    // words are read 64 windows at a time and the windows with entries kept in
    // s_win, so empty windows cost no read of their ids.
    const int mword0 = (r0 >> 6) + tile, mentry0 = r0 & ~63;
    const uint64_t* const mplane =
        a.wave_masks ? a.wave_masks + (size_t)px.quad * a.mask_plane + mword0 : nullptr;
    const int top = e_hi >= r0 ? ((e_hi & ~63) - mentry0) >> 6 : -1;
    for (int wt = top; wt >= 0; wt -= kScan) {
        // every wave reads the same words; the first keeps them
        const int wi = wt - lane;
        const uint64_t word = wi < 0 ? 0ull : mplane ? mplane[wi] : ~0ull;
        const uint64_t nz = lanes_where(word != 0);
        const int nw = __popcll(nz);
        __syncthreads();  // the previous windows are consumed
        if (wave == 0 && word != 0) {
            const int at = __popcll(nz & ((1ull << lane) - 1ull));
            s_win[at] = wi;
            s_word[at] = word;
        }
        __syncthreads();
        for (int w0 = 0; w0 < nw; w0 += 4) {
            // one window a wave
            bool cand = false;
            int e = 0, gid = 0;
            uint2 box = make_uint2(0u, 0u);
            float4 el = make_float4(0.f, 0.f, -1.f, 0.f);
            float ec = 0.f;
            if (w0 + wave < nw) {
                e = mentry0 + (s_win[w0 + wave] << 6) + lane;
                cand = ((s_word[w0 + wave] >> lane) & 1ull) && e >= r0 && e <= e_hi;
                if (cand) {
                    gid = list_id(a, e);
                    cand = entry_meets<BLUR>(a, cull, gid, all, box, el, ec);
                }
            }
            const int n = list_append<true>(L, cand, gid, e, box, el, ec, wave, lane);
            for (int b0 = 0; b0 < n; b0 += kBatch) {
                const int nb = min(kBatch, n - b0);
                if (b0) __syncthreads();
                stage_batch(L, a.records, b0, nb);
                for (int k = threadIdx.x; k < nb * kGradSums; k += 256) s_grad[k] = 0.f;
                for (int k = threadIdx.x; k < nb * kTexWin * kTexWin * CM; k += 256) s_tex[k] = 0.f;
                if (threadIdx.x < kBatch) {
                    s_anchor[threadIdx.x] = kNoAnchor;
                    s_pool_at[threadIdx.x] = kPoolUnset;
                }
                if (threadIdx.x == 0) s_pool_used = s_pool_count = 0;
                __syncthreads();
                uint64_t m = batch_meets<BLUR>(L, b0, nb, cull, rect, lane);
                const int e_lane = L.e[b0 + min(lane, nb - 1)];
                while (m != 0) {
                    int bit[kSlots], ns;
                    const int mybit = take_four(m, bit, ns, sub);
                    four(ns, mybit, __shfl(e_lane, mybit));
                }
                __syncthreads();
                for (int k = threadIdx.x; k < nb * kGradSums; k += 256) {
                    const float v = s_grad[k];
                    if (v == 0.f) continue;
                    const int i = k / kGradSums, slot = k - i * kGradSums;
                    unsafeAtomicAdd(b.grad_rec + (size_t)L.g[b0 + i] * kGradFloats +
                                        (slot < G_EXTRA ? slot : G_PIX + (slot - G_EXTRA)),
                                    v);
                }
                for (int k = threadIdx.x; k < nb * kTexWin * kTexWin * CM; k += 256) {
                    const float v = s_tex[k];
                    if (v == 0.f) continue;
                    const int i = k / (kTexWin * kTexWin * CM), t = k - i * (kTexWin * kTexWin * CM);
                    const int wr = t / (kTexWin * CM), wq = (t / CM) % kTexWin, c = t % CM;
                    const float* rec = &L.rec[i * kRecStride];
                    const int h = __float_as_int(rec[R_TEX_H]), w = __float_as_int(rec[R_TEX_W]);
                    const unsigned long long anchor = s_anchor[i];
                    const int r = (int)(anchor >> 32) + wr, q = (int)anchor + wq;
                    if (r < h && q < w)  // (always, where weight was added)
                        unsafeAtomicAdd(b.v_texture +
                                            ((size_t)__float_as_int(rec[R_TEX_START]) +
                                             (size_t)r * w + q) * CM + c,
                                        v);
                }
                for (int j = 0; j < s_pool_count; ++j) {
                    const int i = s_pool_list[j];
                    const float* rec = &L.rec[i * kRecStride];
                    const int size = __float_as_int(rec[R_TEX_H]) * __float_as_int(rec[R_TEX_W]) * CM;
                    float* const chart =
                        b.v_texture + (size_t)__float_as_int(rec[R_TEX_START]) * CM;
                    float* const from = s_pool + s_pool_at[i];
                    for (int k = threadIdx.x; k < size; k += 256) {
                        const float v = from[k];
                        if (v == 0.f) continue;
                        unsafeAtomicAdd(chart + k, v);
                        from[k] = 0.f;
                    }
                }
            }
            __syncthreads();  // the lists are consumed
        }
    }
}

// ------------------------------------------------------------------ launchers
// The narrow kernels take 16-pixel tiles, up to four channels, bilinear taps
// and the plain or the blur alpha, on textures whose float32 gradient is below
// 2^31 bytes (one buffer resource); the sizes they are used for are beside
// kNarrowTiles.
static bool narrow_supported(const RasterArgs& a) {
    const long long bytes = (long long)a.num_texels * a.channels * 4;  // also of v_texture
    return a.bw == 16 && a.tiles_x * a.tiles_y <= kNarrowTiles && a.channels >= 1 && a.channels <= 4 && a.num_points > 0 &&
           !(a.settings & (kSetNearest | kSetNdc | kSetAlphaViz)) && !a.precise_edge &&
           bytes < 0x7fffffffll;
}

bool raster_forward_is_narrow(const RasterArgs& a) {
    return narrow_supported(a) && a.num_ids <= kNarrowForwardIds;
}
bool raster_backward_is_narrow(const RasterArgs& a) {
    if (!narrow_supported(a)) return false;
    const int tiles = a.tiles_x * a.tiles_y;
    const bool many = tiles > kNarrowManyTiles;
    if (a.num_ids > (many ? kNarrowManyTilesIds : kNarrowBackwardIds)) return false;
    const double chart = (double)a.channels * a.num_texels / a.num_points;  // mean values
    const bool one_size = a.num_texels % a.num_points == 0 && chart <= kNarrowChartOneSize;
    if (many && a.num_ids < (one_size || tiles <= kNarrowSparseTiles ? 6 : 12) * tiles)
        return false;
    if (one_size) return true;
    if (!many && chart <= kNarrowChartMean) return true;
    return a.num_ids * chart <= kNarrowBackwardValues;
}

template <int CM>
static hipError_t launch_fwd(const RasterArgs& a, const FwdOut& o, hipStream_t s) {
    const int grid = narrow_grid(a.tiles_x * a.tiles_y);
    const bool blur = a.settings & kSetBlur;
    if (a.texture_bf16) {
        if (blur) k_raster_forward_narrow<CM, true, true><<<grid, 256, 0, s>>>(a, o);
        else k_raster_forward_narrow<CM, false, true><<<grid, 256, 0, s>>>(a, o);
    } else {
        if (blur) k_raster_forward_narrow<CM, true, false><<<grid, 256, 0, s>>>(a, o);
        else k_raster_forward_narrow<CM, false, false><<<grid, 256, 0, s>>>(a, o);
    }
    return hipGetLastError();
}

template <int CM>
static hipError_t launch_bwd(const RasterArgs& a, const BwdIn& b, hipStream_t s) {
    const int grid = narrow_grid(a.tiles_x * a.tiles_y);
    const bool blur = a.settings & kSetBlur;
    if (a.texture_bf16) {
        if (blur) k_raster_backward_narrow<CM, true, true><<<grid, 256, 0, s>>>(a, b);
        else k_raster_backward_narrow<CM, false, true><<<grid, 256, 0, s>>>(a, b);
    } else {
        if (blur) k_raster_backward_narrow<CM, true, false><<<grid, 256, 0, s>>>(a, b);
        else k_raster_backward_narrow<CM, false, false><<<grid, 256, 0, s>>>(a, b);
    }
    return hipGetLastError();
}

hipError_t raster_forward_narrow(const RasterArgs& a, const FwdOut& o, hipStream_t s) {
    switch (a.channels) {
        case 1: return launch_fwd<1>(a, o, s);
        case 2: return launch_fwd<2>(a, o, s);
        case 3: return launch_fwd<3>(a, o, s);
        case 4: return launch_fwd<4>(a, o, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t raster_backward_narrow(const RasterArgs& a, const BwdIn& b, hipStream_t s) {
    switch (a.channels) {
        case 1: return launch_bwd<1>(a, b, s);
        case 2: return launch_bwd<2>(a, b, s);
        case 3: return launch_bwd<3>(a, b, s);
        case 4: return launch_bwd<4>(a, b, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace gstex
