// ff_tiles.hip -- several iterations of one stage in a launch (gfx950): upwind
// propagation, box smoothing and Lax-Wendroff propagation on tiles held in
// registers (ff_tile.hpp), for the stage classes and the differentiable form.
//
// One launch per X or Y pass reads and writes every field once per pass, 2 n
// times for n iterations, with a launch's latency each. Here a workgroup loads
// a buffer of 64 columns by waves * 4 rows once, runs the
// iterations in registers, and writes the tile inside it that neighbouring
// pixels beyond the buffer cannot have reached. The iterations cost VALU
// instructions and a barrier each (plus those of the halo), so a launch is
// bound by HBM up to about four propagation iterations and by the VALU beyond.
// Results are those of the single passes bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "ff_device.hpp"
#include "ff_kernels.hpp"
#include "ff_per_device.hpp"
#include "ff_runtime.hpp"
#include "ff_tile.hpp"

namespace ffamd {

namespace {

using namespace tile;

// Rows per thread; 16 waves of 4 rows need 64 VGPRs for the five fields of a
// propagation with payloads, so two workgroups (all 32 wave slots) share a CU.
constexpr int kTileRows = 4;

// Tiles of an image: buffer of 64 x rows with a halo on every side; an image
// no wider (taller) than the buffer is one tile across (down).
struct Tiling {
    int W, H, TW, TH, tiles_x, tiles_y, halo;
};
Tiling tiling(int H, int W, int halo, int rows) {
    Tiling t;
    t.W = W;
    t.H = H;
    t.halo = halo;
    t.TW = W <= LANES ? W : LANES - 2 * halo;
    t.TH = H <= rows ? H : rows - 2 * halo;
    t.tiles_x = (W + t.TW - 1) / t.TW;
    t.tiles_y = (H + t.TH - 1) / t.TH;
    return t;
}
// Waves per workgroup: 16, or 8 (a buffer of half the height, more of it
// halo) where the taller tiles would leave CUs without a workgroup.
int waves_for(int B, int H, int W, int halo) {
    const Tiling t = tiling(H, W, halo, 16 * kTileRows);
    return (long long)B * t.tiles_x * t.tiles_y < 256 ? 8 : 16;
}

// A workgroup's tile: its buffer's place, clamped into the image, and the
// output range. Blocks of one XCD (dealt round-robin) form bands of the image.
struct TilePos {
    Geo g;
    int x0, y0, ox0, ox1, oy0, oy1;
    bool xedge, xinside, yinside;
    int rlast;
    __device__ __forceinline__ bool out_row(int r) const { return g.yw + r >= oy0 && g.yw + r < oy1; }
};
__device__ __forceinline__ TilePos tile_pos(const Tiling& t, int nw, int border) {
    constexpr int R = kTileRows;
    TilePos p;
    const int i = xcd_tile((int)blockIdx.x, t.tiles_x * t.tiles_y);
    const int ty = i / t.tiles_x, tx = i - ty * t.tiles_x;
    p.ox0 = tx * t.TW;
    p.ox1 = min(p.ox0 + t.TW, t.W);
    p.oy0 = ty * t.TH;
    p.oy1 = min(p.oy0 + t.TH, t.H);
    p.x0 = clampi(p.ox0 - t.halo, 0, t.W - LANES);
    p.y0 = clampi(p.oy0 - t.halo, 0, t.H - nw * R);
    Geo& g = p.g;
    g.lane = lane_id();
    g.wave = wave_id();
    g.x = p.x0 + g.lane;
    g.xl = min(g.x, t.W - 1);
    g.xlast = t.W - 1 - p.x0;
    g.yw = p.y0 + g.wave * R;
    g.xin = g.x >= border && g.x < t.W - border;
    p.xedge = p.x0 == 0 || p.x0 + LANES >= t.W;
    p.xinside = g.xlast < LANES - 1;
    p.yinside = p.y0 + nw * R > t.H;
    p.rlast = t.H - 1 - g.yw;
    return p;
}

// Image b of a batch of B images one after the other.
template <class T>
__device__ __forceinline__ Rsrc image_rsrc(T* p, int pitch, int H, int b) {
    return rsrc((const char*)p + (size_t)b * pitch * H, pitch * H);
}

// ------------------------------------------------------------ propagation

struct PassParams {
    float dt;
    int border, H;
};

// n upwind iterations of the flow and, with PAY, a scalar and a vector
// payload; with a middle output, the fields after `mid` iterations are written
// too. Needs border >= 1: the pixels next to an image edge then keep their
// values, so the lanes and rows beyond the image are never read by others.
// Four iterations with payloads at 3840x2160: 116 us for 332 MB (66 us at a
// copy's rate; the rest is VALU), 138 us with the middle output's 166 MB.
template <bool PAY>
__global__ void __launch_bounds__(1024, 8) k_propagate_tile(PropFields in, PropFields mid, PropFields out, Tiling tl,
                                                            int n, int after, float dt, int border) {
    constexpr int R = kTileRows;
    extern __shared__ float xch[];
    const int nw = (int)blockDim.x / LANES, b = (int)blockIdx.y;
    const TilePos p = tile_pos(tl, nw, border);
    const Geo& g = p.g;
    const PassParams pp{dt, border, tl.H};
    State<PAY, R> s;
    {
        const Rsrc rf = image_rsrc(in.f, in.fp, tl.H, b), rs = image_rsrc(in.s, in.sp, tl.H, b),
                   rv = image_rsrc(in.v, in.vp, tl.H, b);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int y = min(g.yw + r, tl.H - 1);
            const float2 f = ld2(rf, y * in.fp + g.xl * 8);
            s.fu[r] = f.x;
            s.fv[r] = f.y;
            if constexpr (PAY) {
                s.sa[r] = ld1(rs, y * in.sp + g.xl * 4);
                const float2 v = ld2(rv, y * in.vp + g.xl * 8);
                s.du[r] = v.x;
                s.dv[r] = v.y;
            }
        }
    }
    auto store = [&](const PropFields& o) {
        // the column from the lane's number anew, so that nothing of the
        // addresses is held through the iterations
        int x;
        asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(x));
        x += p.x0;
        const bool ox = x >= p.ox0 && x < p.ox1;
        const Rsrc rf = image_rsrc(o.f, o.fp, tl.H, b), rs = image_rsrc(o.s, o.sp, tl.H, b),
                   rv = image_rsrc(o.v, o.vp, tl.H, b);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int y = g.yw + r;
            const bool ok = ox && p.out_row(r);
            st2(rf, ok ? y * o.fp + x * 8 : OOB, s.fu[r], s.fv[r]);
            if constexpr (PAY) {
                st1(rs, ok ? y * o.sp + x * 4 : OOB, s.sa[r]);
                st2(rv, ok ? y * o.vp + x * 8 : OOB, s.du[r], s.dv[r]);
            }
        }
    };
    const bool inner = p.x0 >= border && p.x0 + LANES - 1 < tl.W - border && p.y0 >= border &&
                       p.y0 + nw * R - 1 < tl.H - border;
    int slot = 0, todo = n;
    // (a loop of its own for each form of the passes: where two forms join,
    // the compiler hoists what they share, and spilled 40 registers)
    auto iterate = [&](auto interior, int count) {
        constexpr bool INNER = decltype(interior)::value;
        for (int it = 0; it < count; ++it) {
            prop_x<PAY, !INNER, R>(s, g, pp);
            put_rows<PAY, R>(s, xch, nw, slot, g.wave, g.lane);
            __syncthreads();
            Edge5 ea = own_row<PAY, R>(s, 0), eb = own_row<PAY, R>(s, R - 1);
            if (g.wave > 0) get_row<PAY>(ea, xrow(xch, nw, slot, g.wave - 1) + 5 * LANES, g.lane);
            if (g.wave < nw - 1) get_row<PAY>(eb, xrow(xch, nw, slot, g.wave + 1), g.lane);
            slot ^= 1;
            prop_y<PAY, !INNER, R>(s, g, pp, ea, eb);
        }
    };
    // the iterations up to the middle output, if there is one, then the rest
    for (bool middle = mid.f != nullptr;; middle = false) {
        const int count = middle ? after : todo;
        todo -= count;
        if (inner) iterate(std::true_type{}, count);
        else iterate(std::false_type{}, count);
        store(middle ? mid : out);
        if (!middle) break;
    }
}

// --------------------------------------------------------- a whole level

// What the passes, the update and the outputs of a level read (as the fused
// frame kernel's job).
struct LevelParams {
    float dt;
    int border, H;
    float gamma, maxflow;
    float2* flow_upd;
};

// One level of one frame of the differentiable form, images of a batch: n
// propagation iterations of the old flow (on a delta level with the old
// brightness and delta flow as payloads; without PROP none, what is read being
// propagated already), the image model, the update and K smoothing iterations,
// as the fused frame kernel's tiles. SAVE: what the adjoints read is written as
// well: the fields after every two iterations but the last (f.mid_*, images of a
// batch one after the other, then the next two iterations'), the propagated
// fields and the image gradient. Halo: max(n, 2) + 2 K, an error's way in from
// the buffer's edge.
//
// What bounds it: without PROP, HBM and the latency of its four phases (3840x2160
// delta level, K = 2: 95 us for 316 MB, with the gradient 117 us for 382 MB; the
// launches it replaces, image model, update and smoothing, took 149 us). With
// PROP, the VALU: n = 4 193 us, n = 8 338 us, the halo being 8 and 12 of 64
// columns. 16 x 512x512, n = 4: 101 us (161 in four launches).
template <bool DELTA, bool SAVE, bool PROP>
__global__ void __launch_bounds__(1024, 8) k_level_tile(LevelFields f, Tiling tl, int Hu, int Wu, int n, int K,
                                                        LevelParams lp) {
    constexpr int R = kTileRows;
    extern __shared__ float xch[];
    const int nw = (int)blockDim.x / LANES, b = (int)blockIdx.y, B = (int)gridDim.y;
    const TilePos p = tile_pos(tl, nw, lp.border);
    const Geo& g = p.g;
    const int pa = tl.W * 4, pf = tl.W * 8;  // row pitches in bytes
    State<DELTA, R> s;
    {
        const Rsrc rf = image_rsrc(f.flow, pf, tl.H, b), rs = image_rsrc(f.bright, pa, tl.H, b),
                   rv = image_rsrc(f.dflow, pf, tl.H, b);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int y = min(g.yw + r, tl.H - 1);
            if constexpr (PROP || !DELTA) {
                const float2 v = ld2(rf, y * pf + g.xl * 8);
                s.fu[r] = v.x;
                s.fv[r] = v.y;
            }
            if constexpr (DELTA) {
                s.sa[r] = ld1(rs, y * pa + g.xl * 4);
                const float2 d = ld2(rv, y * pf + g.xl * 8);
                s.du[r] = d.x;
                s.dv[r] = d.y;
            }
        }
    }
    // this lane's column, from the lane's number anew, so that nothing of the
    // addresses is held through the iterations
    auto column = [&] {
        int x;
        asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(x));
        return x + p.x0;
    };
    // (null pointers are skipped)
    auto store = [&](float* of, float* os, float* ov, int image) {
        const int x = column();
        const bool ox = x >= p.ox0 && x < p.ox1;
        const Rsrc rf = image_rsrc(of, pf, tl.H, image), rs = image_rsrc(os, pa, tl.H, image),
                   rv = image_rsrc(ov, pf, tl.H, image);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int y = g.yw + r;
            const bool ok = ox && p.out_row(r);
            if (of) st2(rf, ok ? y * pf + x * 8 : OOB, s.fu[r], s.fv[r]);
            if constexpr (DELTA) {
                st1(rs, ok ? y * pa + x * 4 : OOB, s.sa[r]);
                st2(rv, ok ? y * pf + x * 8 : OOB, s.du[r], s.dv[r]);
            }
        }
    };
    const bool inner = p.x0 >= lp.border && p.x0 + LANES - 1 < tl.W - lp.border && p.y0 >= lp.border &&
                       p.y0 + nw * R - 1 < tl.H - lp.border;
    int slot = 0;
    // (a loop of its own for each form of the passes, as in k_propagate_tile)
    auto iterate = [&](auto interior, int count) {
        constexpr bool INNER = decltype(interior)::value;
        for (int it = 0; it < count; ++it) {
            prop_x<DELTA, !INNER, R>(s, g, lp);
            put_rows<DELTA, R>(s, xch, nw, slot, g.wave, g.lane);
            __syncthreads();
            Edge5 ea = own_row<DELTA, R>(s, 0), eb = own_row<DELTA, R>(s, R - 1);
            if (g.wave > 0) get_row<DELTA>(ea, xrow(xch, nw, slot, g.wave - 1) + 5 * LANES, g.lane);
            if (g.wave < nw - 1) get_row<DELTA>(eb, xrow(xch, nw, slot, g.wave + 1), g.lane);
            slot ^= 1;
            prop_y<DELTA, !INNER, R>(s, g, lp, ea, eb);
        }
    };
    for (int done = 0; PROP && done < n;) {
        const int count = SAVE ? min(2, n - done) : n;
        if (inner) iterate(std::true_type{}, count);
        else iterate(std::false_type{}, count);
        done += count;
        if constexpr (SAVE) {
            if (done < n) store(f.mid_flow, f.mid_scalar, f.mid_vector, (done / 2 - 1) * B + b);
            else store(DELTA ? nullptr : f.prop_flow, f.prop_scalar, f.prop_vector, b);
        }
    }
    // image model and update
    {
        const int x = column(), xl = min(x, tl.W - 1);
        const bool ox = x >= p.ox0 && x < p.ox1;
        float im[R + 4];
        const Rsrc ri = image_rsrc(f.image, pa, tl.H, b);
#pragma unroll
        for (int j = 0; j < R + 4; ++j) im[j] = ld1(ri, clampi(g.yw - 2 + j, 0, tl.H - 1) * pa + xl * 4);
        float aold[R];
        float2 up[R];
        int offa[R], offf[R];
        const Rsrc ra = image_rsrc(f.bright, pa, tl.H, b), ru = image_rsrc(f.upper, Wu * 8, Hu, b);
        const int xm = DELTA ? f.xmap[xl] * 8 : 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int y = g.yw + r, yl = min(y, tl.H - 1);
            const bool out = ox && p.out_row(r);
            offa[r] = out ? y * pa + x * 4 : OOB;
            offf[r] = out ? y * pf + x * 8 : OOB;
            aold[r] = DELTA ? 0.f : ld1(ra, yl * pa + xl * 4);
            up[r] = DELTA ? ld2(ru, f.ymap[yl] * Wu * 8 + xm) : make_float2(0.f, 0.f);
        }
        const Rsrc rao = image_rsrc(f.bright_out, pa, tl.H, b), rdf = image_rsrc(f.dflow_out, pf, tl.H, b),
                   rfu = image_rsrc(f.flow_upd, pf, tl.H, b), rg = image_rsrc(f.grad, pf, tl.H, b);
        auto gradient = [&](int r, float gx, float gy) {
            if constexpr (SAVE) st2(rg, offf[r], gx, gy);
        };
        if (p.xedge) model_update<DELTA, true, R>(s, im, aold, up, lp, rao, rdf, rfu, offa, offf, gradient);
        else model_update<DELTA, false, R>(s, im, aold, up, lp, rao, rdf, rfu, offa, offf, gradient);
    }
    for (int it = 0; it < K; ++it) {
        if (p.xinside) copy_last_column<R>(s.fu, s.fv, g.lane, g.xlast);
        if (p.xedge) smooth_x<true, R>(s.fu, s.fv);
        else smooth_x<false, R>(s.fu, s.fv);
        const Edge2 e = exchange_smooth_rows<R>(s.fu, s.fv, xch, nw, slot, g.wave, g.lane);
        slot ^= 1;
        if (p.yinside) smooth_y<true, R>(s.fu, s.fv, e, p.rlast);
        else smooth_y<false, R>(s.fu, s.fv, e, p.rlast);
    }
    const int x = column();
    const bool ox = x >= p.ox0 && x < p.ox1;
    const Rsrc ro = image_rsrc(f.flow_out, pf, tl.H, b);
#pragma unroll
    for (int r = 0; r < R; ++r)
        st2(ro, ox && p.out_row(r) ? (g.yw + r) * pf + x * 8 : OOB, s.fu[r], s.fv[r]);
}

// -------------------------------------------------------------- smoothing

// n iterations of the box smoother (an X and a Y pass each), halo 2 n.
__global__ void __launch_bounds__(1024, 8) k_smooth_tile(const float2* in, int ip, float2* out, int op, Tiling tl,
                                                         int n) {
    constexpr int R = kTileRows;
    extern __shared__ float xch[];
    const int nw = (int)blockDim.x / LANES, b = (int)blockIdx.y;
    const TilePos p = tile_pos(tl, nw, 0);
    const Geo& g = p.g;
    float fu[R], fv[R];
    const Rsrc ri = image_rsrc(in, ip, tl.H, b);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float2 f = ld2(ri, min(g.yw + r, tl.H - 1) * ip + g.xl * 8);
        fu[r] = f.x;
        fv[r] = f.y;
    }
    for (int it = 0; it < n; ++it) {
        if (p.xinside) copy_last_column<R>(fu, fv, g.lane, g.xlast);
        if (p.xedge) smooth_x<true, R>(fu, fv);
        else smooth_x<false, R>(fu, fv);
        const Edge2 e = exchange_smooth_rows<R>(fu, fv, xch, nw, it & 1, g.wave, g.lane);
        if (p.yinside) smooth_y<true, R>(fu, fv, e, p.rlast);
        else smooth_y<false, R>(fu, fv, e, p.rlast);
    }
    const Rsrc ro = image_rsrc(out, op, tl.H, b);
    const bool ox = g.x >= p.ox0 && g.x < p.ox1;
#pragma unroll
    for (int r = 0; r < R; ++r)
        st2(ro, ox && p.out_row(r) ? (g.yw + r) * op + g.x * 8 : OOB, fu[r], fv[r]);
}

// ------------------------------------------------- adjoints of 5-tap passes

// Adjoint of a 5-tap correlation with clamped reads at one position of a
// line, from the output gradients at the five positions around it (0 outside
// the line): output i's tap c reads position clamp(i + c), so the first
// (last) position also receives the taps of the outputs near it that the
// clamp sends there. Outputs in ascending order, each one's taps in
// ascending order, as a sum over all outputs and taps would take them.
template <bool EDGE, class Wf>
__device__ __forceinline__ float adjoint5(float m2, float m1, float z, float p1, float p2, bool first, bool last,
                                          Wf w) {
    float a = fmaf(w(4), m2, 0.0f);
    a = fmaf(w(3), m1, a);
    if constexpr (EDGE) {
        a = fmaf(w(4), last ? m1 : 0.0f, a);
        a = fmaf(w(0), first ? z : 0.0f, a);
        a = fmaf(w(1), first ? z : 0.0f, a);
    }
    a = fmaf(w(2), z, a);
    if constexpr (EDGE) {
        a = fmaf(w(3), last ? z : 0.0f, a);
        a = fmaf(w(4), last ? z : 0.0f, a);
        a = fmaf(w(0), first ? p1 : 0.0f, a);
    }
    a = fmaf(w(1), p1, a);
    a = fmaf(w(0), p2, a);
    return a;
}
template <bool EDGE, class Wf>
__device__ __forceinline__ float adjoint5_x(float v, const TilePos& p, int W, Wf w) {
    const float m = zshr(v), q = zshl(v);
    return adjoint5<EDGE>(zshr(m), m, v, q, zshl(q), p.g.x == 0, p.g.x == W - 1, w);
}
// Row r's adjoint along y: v the strip's rows, e0, e1 the two rows above it and
// e2, e3 below.
template <bool EDGE, int R, class Wf>
__device__ __forceinline__ float adjoint5_y(const float (&v)[R], const float (&e)[4], int r, int y, int H, Wf w) {
    const float m2 = r >= 2 ? v[r >= 2 ? r - 2 : 0] : e[r], m1 = r >= 1 ? v[r >= 1 ? r - 1 : 0] : e[1];
    const float p1 = r + 1 < R ? v[r + 1 < R ? r + 1 : 0] : e[2], p2 = r + 2 < R ? v[r + 2 < R ? r + 2 : 0] : e[r + 4 - R];
    return adjoint5<EDGE>(m2, m1, v[r], p1, p2, y == 0, y == H - 1, w);
}
// The two rows above and below each strip, of field k of K in `rows` (LDS, 4 K
// rows a wave): 0 beyond the first and last strip, where the buffer ends at
// the image's edge (elsewhere that is halo).
template <int K, int R>
__device__ __forceinline__ void put_edges(const float (&v)[R], float* rows, int k, const Geo& g) {
    float* my = rows + (g.wave * 4 * K + 4 * k) * LANES + g.lane;
    my[0] = v[0];
    my[LANES] = v[1];
    my[2 * LANES] = v[R - 2];
    my[3 * LANES] = v[R - 1];
}
template <int K>
__device__ __forceinline__ void get_edges(float (&e)[4], const float* rows, int k, int nw, const Geo& g) {
    e[0] = e[1] = e[2] = e[3] = 0.0f;
    if (g.wave > 0) {
        const float* o = rows + ((g.wave - 1) * 4 * K + 4 * k) * LANES + g.lane;
        e[0] = o[2 * LANES];
        e[1] = o[3 * LANES];
    }
    if (g.wave < nw - 1) {
        const float* o = rows + ((g.wave + 1) * 4 * K + 4 * k) * LANES + g.lane;
        e[2] = o[0];
        e[3] = o[LANES];
    }
}

// Adjoint of the image model on B float images (a0 = Sx(sy), gx = Dx(sy), gy =
// Dy(sx) with sy = Sy(I), sx = Sx(I)):
//   g_I = Sy^T g_sy + Sx^T g_sx,  g_sy = Sx^T g_a0 + Dx^T g_gx,  g_sx = Dy^T g_gy.
// One pass over memory (12 bytes in, 4 out per pixel); as two kernels with
// g_sy and g_sx in between and a gather that tests every tap's clamp, a
// 3840x2160 image took 204 us.
template <bool EDGE>
__device__ __forceinline__ void image_model_adjoint(const float* ga0, const float2* gg, float* gI, const Tiling& tl,
                                                    int acc, const TilePos& p, int nw, float* xch) {
    constexpr int R = kTileRows;
    const Geo& g = p.g;
    float sy[R], gy[R];
    const size_t image = (size_t)blockIdx.y * tl.H;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const size_t row = (image + min(g.yw + r, tl.H - 1)) * tl.W;
        float a = ga0[row + g.xl];
        float2 d = gg[row + g.xl];
        if (EDGE && (g.x >= tl.W || g.yw + r >= tl.H)) a = d.x = d.y = 0.0f;
        const float s = adjoint5_x<EDGE>(a, p, tl.W, WSmooth{});
        sy[r] = s + adjoint5_x<EDGE>(d.x, p, tl.W, WDiff{});
        gy[r] = d.y;
    }
    put_edges<2, R>(sy, xch, 0, g);
    put_edges<2, R>(gy, xch, 1, g);
    __syncthreads();
    float es[4], eg[4];
    get_edges<2>(es, xch, 0, nw, g);
    get_edges<2>(eg, xch, 1, nw, g);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int y = g.yw + r;
        const float sx = adjoint5_y<EDGE, R>(gy, eg, r, y, tl.H, WDiff{});
        const float v = adjoint5_y<EDGE, R>(sy, es, r, y, tl.H, WSmooth{}) + adjoint5_x<EDGE>(sx, p, tl.W, WSmooth{});
        if (g.x >= p.ox0 && g.x < p.ox1 && p.out_row(r)) {
            float* o = gI + (image + y) * tl.W + g.x;
            *o = acc ? *o + v : v;
        }
    }
}
__global__ void __launch_bounds__(1024, 8) k_image_model_adjoint(const float* ga0, const float2* gg, float* gI,
                                                                 Tiling tl, int acc) {
    extern __shared__ float xch[];
    const int nw = (int)blockDim.x / LANES;
    const TilePos p = tile_pos(tl, nw, 0);
    if (p.xedge || p.y0 == 0 || p.y0 + nw * kTileRows >= tl.H) image_model_adjoint<true>(ga0, gg, gI, tl, acc, p, nw, xch);
    else image_model_adjoint<false>(ga0, gg, gI, tl, acc, p, nw, xch);
}

// Adjoint of n smoothing iterations for the output gradient gout + gout2
// (gout2 may be null): of each the Y pass's adjoint, then the X pass's.
template <bool EDGE>
__device__ __forceinline__ void smooth_adjoint(const float2* gout, const float2* gout2, float2* gin, const Tiling& tl,
                                               int n, int acc, const TilePos& p, int nw, float* xch) {
    constexpr int R = kTileRows;
    const Geo& g = p.g;
    float u[R], v[R];
    const size_t image = (size_t)blockIdx.y * tl.H;
    // what lies outside the image contributes nothing
    auto clear = [&](int r) {
        if (EDGE && (g.x >= tl.W || g.yw + r >= tl.H)) u[r] = v[r] = 0.0f;
    };
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const size_t i = (image + min(g.yw + r, tl.H - 1)) * tl.W + g.xl;
        float2 f = gout[i];
        if (gout2) {
            const float2 h = gout2[i];
            f.x += h.x;
            f.y += h.y;
        }
        u[r] = f.x;
        v[r] = f.y;
        clear(r);
    }
    for (int it = 0; it < n; ++it) {
        float* rows = xch + (it & 1) * nw * 8 * LANES;
        put_edges<2, R>(u, rows, 0, g);
        put_edges<2, R>(v, rows, 1, g);
        __syncthreads();
        float eu[4], ev[4], a[R], b[R];
        get_edges<2>(eu, rows, 0, nw, g);
        get_edges<2>(ev, rows, 1, nw, g);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            a[r] = adjoint5_y<EDGE, R>(u, eu, r, g.yw + r, tl.H, WBox{});
            b[r] = adjoint5_y<EDGE, R>(v, ev, r, g.yw + r, tl.H, WBox{});
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            u[r] = adjoint5_x<EDGE>(a[r], p, tl.W, WBox{});
            v[r] = adjoint5_x<EDGE>(b[r], p, tl.W, WBox{});
            clear(r);
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
        if (g.x >= p.ox0 && g.x < p.ox1 && p.out_row(r)) {
            float2* o = gin + (image + g.yw + r) * tl.W + g.x;
            const float2 old = acc ? *o : make_float2(0.f, 0.f);
            *o = acc ? make_float2(old.x + u[r], old.y + v[r]) : make_float2(u[r], v[r]);
        }
}
__global__ void __launch_bounds__(1024, 8) k_smooth_adjoint(const float2* gout, const float2* gout2, float2* gin,
                                                            Tiling tl, int n, int acc) {
    extern __shared__ float xch[];
    const int nw = (int)blockDim.x / LANES;
    const TilePos p = tile_pos(tl, nw, 0);
    if (p.xedge || p.y0 == 0 || p.y0 + nw * kTileRows >= tl.H) smooth_adjoint<true>(gout, gout2, gin, tl, n, acc, p, nw, xch);
    else smooth_adjoint<false>(gout, gout2, gin, tl, n, acc, p, nw, xch);
}

// ------------------------------------------------------------ Lax-Wendroff

// n iterations (a Y and an X pass each, as in LaxWendroffPropagator) of a
// scalar image along a flow, halo n.
__global__ void __launch_bounds__(1024, 8) k_lax_wendroff_tile(DevImg flow, DevImg in, DevImg out, Tiling tl, int n,
                                                               float dt) {
    constexpr int R = kTileRows;
    extern __shared__ float xch[];
    const int nw = (int)blockDim.x / LANES;
    const TilePos p = tile_pos(tl, nw, 0);
    const Geo& g = p.g;
    float cx[R], cy[R], a[R];  // Courant numbers, image
    const Rsrc rf = rsrc(flow.data, (int)flow.pitch * tl.H), ri = rsrc(in.data, (int)in.pitch * tl.H);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int y = min(g.yw + r, tl.H - 1);
        const float2 f = ld2(rf, y * (int)flow.pitch + g.xl * 8);
        cx[r] = dt * f.x;
        cy[r] = dt * f.y;
        a[r] = ld1(ri, y * (int)in.pitch + g.xl * 4);
    }
    for (int it = 0; it < n; ++it) {
        // rows next to the strip
        float* my = xch + ((it & 1) * nw + g.wave) * 2 * LANES + g.lane;
        my[0] = a[0];
        my[LANES] = a[R - 1];
        __syncthreads();
        float above = a[0], below = a[R - 1];
        if (g.wave > 0) above = my[-2 * LANES + LANES];
        if (g.wave < nw - 1) below = my[2 * LANES];
        float m = above;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float z = a[r];
            float q = r + 1 < R ? a[r + 1] : below;
            if (p.yinside) q = r + 1 <= p.rlast ? q : z;  // clamped at the last row
            a[r] = lw_scalar<1>(m, z, q, cy[r]);
            m = z;
        }
        if (p.xinside) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const float e = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(a[r]), g.xlast));
                a[r] = g.lane > g.xlast ? e : a[r];
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) a[r] = lw_scalar<0>(cshr(a[r]), a[r], cshl(a[r]), cx[r]);
    }
    const Rsrc ro = rsrc(out.data, (int)out.pitch * tl.H);
    const bool ox = g.x >= p.ox0 && g.x < p.ox1;
#pragma unroll
    for (int r = 0; r < R; ++r)
        st1(ro, ox && p.out_row(r) ? (g.yw + r) * (int)out.pitch + g.x * 4 : OOB, a[r]);
}

size_t exchange_bytes(int nw) { return (size_t)2 * nw * 10 * LANES * sizeof(float); }

// The dynamic LDS of a launch is above the default limit, which is lifted for
// each kernel on each device.
template <class... K>
void allow_lds(OncePerDevice& once, K... kernels) {
    int dev = 0;
    FF_HIP(hipGetDevice(&dev));
    once.run(dev, [&] {
        for (const void* k : {(const void*)kernels...})
            FF_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)exchange_bytes(16)));
    });
}

bool fits(long long pitch, int H) { return pitch * H < 0x7fffffffLL; }

}  // namespace

bool propagate_tile_supported(const PropFields& in, const PropFields& out, int H, int W, int border) {
    return border >= 1 && H > 0 && W > 0 && fits(in.fp, H) && fits(in.sp, H) && fits(in.vp, H) && fits(out.fp, H) &&
           fits(out.sp, H) && fits(out.vp, H);
}

void launch_propagate_tile(const PropFields& in, const PropFields& mid, int after, const PropFields& out, int n, int B,
                           int H, int W, float dt, int border, hipStream_t s) {
    if (n < 1 || n > kMaxPropIters) throw logic_error("propagation: iterations of one launch out of range");
    static OncePerDevice once;
    allow_lds(once, k_propagate_tile<true>, k_propagate_tile<false>);
    const int nw = waves_for(B, H, W, n);
    const Tiling tl = tiling(H, W, n, nw * kTileRows);
    const dim3 grid(tl.tiles_x * tl.tiles_y, B), blk(nw * LANES);
    if (in.s)
        hipLaunchKernelGGL(k_propagate_tile<true>, grid, blk, exchange_bytes(nw), s, in, mid, out, tl, n, after, dt,
                           border);
    else
        hipLaunchKernelGGL(k_propagate_tile<false>, grid, blk, exchange_bytes(nw), s, in, mid, out, tl, n, after, dt,
                           border);
}

// A level's halo, and waves per workgroup: 16, or 8 where the taller tiles
// would leave CUs without one and the halo is at most half of the shorter
// buffer.
namespace {
int level_halo(int n, int K) { return std::max(n, 2) + 2 * K; }
int level_waves(int B, int H, int W, int halo) {
    return 4 * halo <= 8 * kTileRows ? waves_for(B, H, W, halo) : 16;
}
}  // namespace

bool level_tile_supported(int H, int W, int n, int K) {
    return H > 0 && W > 0 && n >= 0 && K >= 0 && fits((long long)W * 8, H) && n < LANES && K < LANES &&
           2 * level_halo(n, K) < 16 * kTileRows;
}

void launch_level_tile(const LevelFields& f, int B, int H, int W, int Hu, int Wu, int n, int K, int border, float dt,
                       float gamma, float maxflow, hipStream_t s) {
    if (!level_tile_supported(H, W, n, K)) throw logic_error("level: iterations or size of one launch out of range");
    static OncePerDevice once;
    allow_lds(once, k_level_tile<true, true, true>, k_level_tile<true, false, true>, k_level_tile<false, true, true>,
              k_level_tile<false, false, true>, k_level_tile<true, true, false>, k_level_tile<true, false, false>,
              k_level_tile<false, true, false>, k_level_tile<false, false, false>);
    const int halo = level_halo(n, K), nw = level_waves(B, H, W, halo);
    const Tiling tl = tiling(H, W, halo, nw * kTileRows);
    const dim3 grid(tl.tiles_x * tl.tiles_y, B), blk(nw * LANES);
    const LevelParams lp{dt, border, H, gamma, maxflow, (float2*)f.flow_upd};
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, blk, exchange_bytes(nw), s, f, tl, Hu, Wu, n, K, lp);
    };
    auto form = [&](auto delta, auto save) {
        if (n) launch(k_level_tile<decltype(delta)::value, decltype(save)::value, true>);
        else launch(k_level_tile<decltype(delta)::value, decltype(save)::value, false>);
    };
    const std::true_type yes;
    const std::false_type no;
    if (f.dflow) f.grad ? form(yes, yes) : form(yes, no);
    else f.grad ? form(no, yes) : form(no, no);
}

void launch_smooth_tile(const void* in, int in_pitch, void* out, int out_pitch, int n, int B, int H, int W,
                        hipStream_t s) {
    if (n < 1 || n > kMaxSmoothIters) throw logic_error("smoothing: iterations of one launch out of range");
    static OncePerDevice once;
    allow_lds(once, k_smooth_tile);
    const int nw = waves_for(B, H, W, 2 * n);
    const Tiling tl = tiling(H, W, 2 * n, nw * kTileRows);
    hipLaunchKernelGGL(k_smooth_tile, dim3(tl.tiles_x * tl.tiles_y, B), dim3(nw * LANES), exchange_bytes(nw), s,
                       (const float2*)in, in_pitch, (float2*)out, out_pitch, tl, n);
}

void launch_image_model_adjoint(const float* ga0, const float* gg, float* gI, int B, int H, int W, int acc,
                                hipStream_t s) {
    const int nw = waves_for(B, H, W, 2);
    const Tiling tl = tiling(H, W, 2, nw * kTileRows);
    hipLaunchKernelGGL(k_image_model_adjoint, dim3(tl.tiles_x * tl.tiles_y, B), dim3(nw * LANES),
                       (size_t)nw * 8 * LANES * sizeof(float), s, ga0, (const float2*)gg, gI, tl, acc);
}

void launch_smooth_adjoint(const float* gout, const float* gout2, float* gin, int n, int B, int H, int W, int acc,
                           hipStream_t s) {
    if (n < 1 || n > kMaxSmoothIters) throw logic_error("smoothing adjoint: iterations of one launch out of range");
    static OncePerDevice once;
    allow_lds(once, k_smooth_adjoint);
    const int nw = waves_for(B, H, W, 2 * n);
    const Tiling tl = tiling(H, W, 2 * n, nw * kTileRows);
    hipLaunchKernelGGL(k_smooth_adjoint, dim3(tl.tiles_x * tl.tiles_y, B), dim3(nw * LANES),
                       (size_t)2 * nw * 8 * LANES * sizeof(float), s, (const float2*)gout, (const float2*)gout2,
                       (float2*)gin, tl, n, acc);
}

// The launches of n iterations, at most `most` each, as evenly as they go:
// run(first, count, last). The results of the last go to `y`, those of the
// one before to `x`, and so on, so that no launch writes what it reads.
namespace {
template <class F>
void in_chunks(int n, int most, F run) {
    const int chunks = (n + most - 1) / most;
    for (int c = 0, done = 0; c < chunks; ++c) {
        const int k = (n - done + chunks - c - 1) / (chunks - c);
        run(c == 0, k, (chunks - 1 - c) % 2 == 0);
        done += k;
    }
}
}  // namespace

bool launch_propagate(const PropFields& in, const PropFields& x, const PropFields& y, int n, int H, int W, float dt,
                      int border, hipStream_t s) {
    if (!propagate_tile_supported(in, y, H, W, border) || !propagate_tile_supported(x, y, H, W, border)) return false;
    // an input that is one of the buffers is read and written pass by pass
    for (const PropFields* o : {&x, &y})
        if (in.f == o->f || (in.s && (in.s == o->s || in.v == o->v))) return false;
    PropFields from = in;
    in_chunks(n, kMaxPropIters, [&](bool, int k, bool to_y) {
        const PropFields& to = to_y ? y : x;
        ProfileScope ps(in.s ? "propagate_payload_tile" : "propagate_tile", s);
        launch_propagate_tile(from, PropFields{}, 0, to, k, 1, H, W, dt, border, s);
        from = to;
    });
    return true;
}

bool launch_smooth(const DevImg& in, const DevImg& x, const DevImg& y, int n, hipStream_t s) {
    const int H = in.h, W = in.w;
    // (FlowSmoother's buffers are new with every input, so none is its input)
    if (H <= 0 || W <= 0 || in.data == x.data || in.data == y.data) return false;
    for (const DevImg* d : {&in, &x, &y})
        if (!fits((long long)d->pitch, H)) return false;
    DevImg from = in;
    in_chunks(n, kMaxSmoothIters, [&](bool, int k, bool to_y) {
        const DevImg& to = to_y ? y : x;
        ProfileScope ps("smooth_tile", s);
        launch_smooth_tile(from.data, (int)from.pitch, to.data, (int)to.pitch, k, 1, H, W, s);
        from = to;
    });
    return true;
}

bool launch_lax_wendroff(const DevImg& flow, const DevImg& in, const DevImg& x, const DevImg& y, int n, float dt,
                         hipStream_t s) {
    const int H = in.h, W = in.w;
    if (H <= 0 || W <= 0) return true;
    for (const DevImg* d : {&flow, &in, &x, &y})
        if (!fits((long long)d->pitch, H)) return false;
    for (const DevImg* d : {&x, &y})
        if (in.data == d->data || flow.data == d->data) return false;
    constexpr int kMost = 8;  // 48 of the buffer's 64 columns are output
    DevImg from = in;
    in_chunks(n, kMost, [&](bool, int k, bool last) {
        const DevImg& to = last ? x : y;  // the propagated image is the X pass's buffer
        const int nw = waves_for(1, H, W, k);
        const Tiling tl = tiling(H, W, k, nw * kTileRows);
        ProfileScope ps("lax_wendroff_tile", s);
        hipLaunchKernelGGL(k_lax_wendroff_tile, dim3(tl.tiles_x * tl.tiles_y), dim3(nw * LANES),
                           (size_t)2 * nw * 2 * LANES * sizeof(float), s, flow, from, to, tl, k, dt);
        from = to;
    });
    return true;
}

}  // namespace ffamd
