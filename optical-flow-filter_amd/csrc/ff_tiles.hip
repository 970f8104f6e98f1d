// ff_tiles.hip -- several iterations of one stage in a launch (gfx950): upwind
// propagation, box smoothing and Lax-Wendroff propagation on tiles held in
// registers (ff_tile.hpp), for the stage classes and the differentiable form.
//
// One launch per X or Y pass reads and writes every field once per pass, 2 n
// times for n iterations, with a launch's latency each. Here a workgroup loads
// a buffer of 64 columns by waves * 4 rows once, runs up to kMaxIters
// iterations in registers, and writes the tile inside it that neighbouring
// pixels beyond the buffer cannot have reached. The iterations cost VALU
// instructions and a barrier each (plus those of the halo), so a launch is
// bound by HBM up to about four propagation iterations and by the VALU beyond.
// Results are those of the single passes bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "ff_device.hpp"
#include "ff_kernels.hpp"
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
    g.wave_in = p.x0 >= border && p.x0 + LANES - 1 < t.W - border && g.yw >= border && g.yw + R - 1 < t.H - border;
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
// Four iterations with payloads at 3840x2160: see kMaxPropIters.
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

// The dynamic LDS of a launch is above the default limit.
template <class K>
void allow_lds(K kernel) {
    const hipError_t e =
        hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)exchange_bytes(16));
    if (e != hipSuccess) throw_hip(e, "hipFuncSetAttribute", __FILE__, __LINE__);
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
    static const bool once = [] {
        allow_lds(k_propagate_tile<true>);
        allow_lds(k_propagate_tile<false>);
        return true;
    }();
    (void)once;
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

bool smooth_tile_supported(int in_pitch, int out_pitch, int H, int W) {
    return H > 0 && W > 0 && fits(in_pitch, H) && fits(out_pitch, H);
}

void launch_smooth_tile(const void* in, int in_pitch, void* out, int out_pitch, int n, int B, int H, int W,
                        hipStream_t s) {
    if (n < 1 || n > kMaxSmoothIters) throw logic_error("smoothing: iterations of one launch out of range");
    static const bool once = [] {
        allow_lds(k_smooth_tile);
        return true;
    }();
    (void)once;
    const int nw = waves_for(B, H, W, 2 * n);
    const Tiling tl = tiling(H, W, 2 * n, nw * kTileRows);
    hipLaunchKernelGGL(k_smooth_tile, dim3(tl.tiles_x * tl.tiles_y, B), dim3(nw * LANES), exchange_bytes(nw), s,
                       (const float2*)in, in_pitch, (float2*)out, out_pitch, tl, n);
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
        launch_propagate_tile(from, PropFields{}, 0, to, k, 1, H, W, dt, border, s);
        from = to;
    });
    return true;
}

bool launch_smooth(const DevImg& in, const DevImg& x, const DevImg& y, int n, hipStream_t s) {
    const int H = in.h, W = in.w;
    if (!smooth_tile_supported((int)in.pitch, (int)y.pitch, H, W) || !smooth_tile_supported((int)x.pitch, (int)y.pitch, H, W) ||
        in.data == x.data || in.data == y.data)
        return false;
    ProfileScope ps("smooth_tile", s);
    DevImg from = in;
    in_chunks(n, kMaxSmoothIters, [&](bool, int k, bool to_y) {
        const DevImg& to = to_y ? y : x;
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
    ProfileScope ps("lax_wendroff_tile", s);
    constexpr int kMost = 8;  // 48 of the buffer's 64 columns are output
    DevImg from = in;
    in_chunks(n, kMost, [&](bool, int k, bool last) {
        const DevImg& to = last ? x : y;  // the propagated image is the X pass's buffer
        const int nw = waves_for(1, H, W, k);
        const Tiling tl = tiling(H, W, k, nw * kTileRows);
        hipLaunchKernelGGL(k_lax_wendroff_tile, dim3(tl.tiles_x * tl.tiles_y), dim3(nw * LANES),
                           (size_t)2 * nw * 2 * LANES * sizeof(float), s, flow, from, to, tl, k, dt);
        from = to;
    });
    return true;
}

}  // namespace ffamd
