// ff_tile.hpp -- device code of the kernels that run several stencil passes
// on a tile held in registers (gfx950).
//
// A workgroup is nw waves stacked vertically; lane l of every wave owns column
// l of a 64-column buffer and R consecutive rows of its wave's strip. X
// neighbours come from lane shifts, Y neighbours from the thread's own
// registers, and the rows above and below a strip are exchanged through LDS
// once per Y pass. The arithmetic per pixel is the reference's, operation by
// operation.
#pragma once

#include <hip/hip_runtime.h>

#include "ff_device.hpp"
#include "ff_kernels.hpp"

namespace ffamd {
namespace tile {

constexpr int LANES = 64;
constexpr int OOB = (int)0x80000000;  // buffer offset beyond any image: access dropped

__device__ __forceinline__ int lane_id() { return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); }

// ------------------------------------------------------------ buffer access

typedef __amdgpu_buffer_rsrc_t Rsrc;
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ Rsrc rsrc(const void* p, int bytes) {
    // word 3 of the buffer descriptor for gfx9-family raw (untyped) buffers
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}
__device__ __forceinline__ float ld1(Rsrc r, int off) {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
__device__ __forceinline__ float2 ld2(Rsrc r, int off) {
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
    return make_float2(__uint_as_float(v.x), __uint_as_float(v.y));
}
__device__ __forceinline__ unsigned ldb(Rsrc r, int off) { return __builtin_amdgcn_raw_buffer_load_b8(r, off, 0, 0); }
__device__ __forceinline__ unsigned ldh(Rsrc r, int off) { return __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0); }
// Cache policy sc1: stores write through this XCD's L2 and such loads do
// not hit a stale line in its caches (device-coherent, as for agent-scope
// atomics).
constexpr int kCoherent = 16;
// Every store writes through. A frame's state is written once and read by
// the next launch only, so dirty lines kept in L2 save nothing, and they
// cost time: 55.8 us per 2048x1088 two-level frame with write-back stores,
// 52.8 us with write-through ones (streaming stores and loads, policy nt,
// were slower than either). The write-through also publishes the top
// level's unsmoothed flow to the tiles of the level below, which read it
// within the same launch with ld2_coherent.
__device__ __forceinline__ void st1(Rsrc r, int off, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, off, 0, kCoherent);
}
__device__ __forceinline__ void st2(Rsrc r, int off, float a, float b) {
    const u32x2 v = {__float_as_uint(a), __float_as_uint(b)};
    __builtin_amdgcn_raw_buffer_store_b64(v, r, off, 0, kCoherent);
}
__device__ __forceinline__ float2 ld2_coherent(Rsrc r, int off) {
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, kCoherent);
    return make_float2(__uint_as_float(v.x), __uint_as_float(v.y));
}

// ---------------------------------------------------------- lane shifts
// Lane i receives lane i-1 (shr) or lane i+1 (shl). The zero-filling forms
// give 0 to the lane without a source; the clamping forms let it keep its
// own value (the clamp-to-edge read at an image edge).
__device__ __forceinline__ float zshr(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float zshl(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));
}
__device__ __forceinline__ float cshr(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), 0x138, 0xf, 0xf, false));
}
__device__ __forceinline__ float cshl(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), 0x130, 0xf, 0xf, false));
}
// Lane i receives lane i-1's v; lane 0 receives `own`. (A select between a
// shifted value and a lane's own value must not be written as a condition:
// the compiler may then run the shift with some lanes disabled, and a lane
// reading a disabled lane receives 0.)
__device__ __forceinline__ unsigned shr_or(unsigned v, unsigned own) {
    return (unsigned)__builtin_amdgcn_update_dpp((int)own, (int)v, 0x138, 0xf, 0xf, false);
}
template <bool CLAMP>
__device__ __forceinline__ float shr(float v) {
    if constexpr (CLAMP) return cshr(v);
    else return zshr(v);
}
template <bool CLAMP>
__device__ __forceinline__ float shl(float v) {
    if constexpr (CLAMP) return cshl(v);
    else return zshl(v);
}

// Lane shifts folded into the instruction that uses the shifted value, where
// the compiler does not fold them (a lane shift into a select; a lane shift
// into a product with a constant). Every lane must be active. An instruction
// that reads a register of other lanes must come two instructions after the
// one that wrote it: the leading s_nop covers the writer before the block,
// the order inside each block its own. (Both forms took the 2048x1088
// two-level launch from 52.2 to 49.0 us and a 64-stream batch from 975 to
// 930; the image model's x taps written so too gained nothing and spilled.)

#define FF_PICK(k) "v_cndmask_b32_dpp %" #k ", %" #k ", %" #k ", vcc wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
#define FF_PICK_HEAD(k) "v_cmp_le_f32 vcc, 0, %" #k "\n\ts_nop 1\n\t"
// Where the speed is not >= 0 (negative or NaN), each value becomes that of
// lane i + 1 (0 without such a lane). With the backward differences z[i] -
// z[i-1] of an upwind pass this selects between them and the forward
// differences.
__device__ __forceinline__ void pick(float speed, float& a, float& b) {
    asm(FF_PICK_HEAD(2) FF_PICK(0) FF_PICK(1) : "+v"(a), "+v"(b) : "v"(speed) : "vcc");
}
__device__ __forceinline__ void pick(float speed, float& a, float& b, float& c, float& d) {
    asm(FF_PICK_HEAD(4) FF_PICK(0) FF_PICK(1) FF_PICK(2) FF_PICK(3)
        : "+v"(a), "+v"(b), "+v"(c), "+v"(d)
        : "v"(speed)
        : "vcc");
}
__device__ __forceinline__ void pick(float speed, float& a, float& b, float& c, float& d, float& e) {
    asm(FF_PICK_HEAD(5) FF_PICK(0) FF_PICK(1) FF_PICK(2) FF_PICK(3) FF_PICK(4)
        : "+v"(a), "+v"(b), "+v"(c), "+v"(d), "+v"(e)
        : "v"(speed)
        : "vcc");
}
#undef FF_PICK
#undef FF_PICK_HEAD

#define FF_DPP_SHR " wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
#define FF_DPP_SHL " wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
// Two 5-tap sums along x, of u and of v, with weights wo, wi, wc, wi, wo:
// taps_x<false>'s products and order, with the outer neighbours shifted
// inside their multiply-adds (7 instructions instead of 9).
__device__ __forceinline__ void taps_x2(float& u, float& v, float wo, float wi, float wc) {
    float mu, pu, mv, pv, a, b;
    asm("s_nop 1\n\t"
        "v_mov_b32_dpp %2, %0" FF_DPP_SHR "v_mov_b32_dpp %4, %1" FF_DPP_SHR
        "v_mov_b32_dpp %3, %0" FF_DPP_SHL "v_mov_b32_dpp %5, %1" FF_DPP_SHL
        "v_mul_f32_dpp %6, %2, %8" FF_DPP_SHR "v_mul_f32_dpp %7, %4, %8" FF_DPP_SHR
        "v_fmac_f32 %6, %9, %2\n\t"
        "v_fmac_f32 %7, %9, %4\n\t"
        "v_fmac_f32 %6, %10, %0\n\t"
        "v_fmac_f32 %7, %10, %1\n\t"
        "v_fmac_f32 %6, %9, %3\n\t"
        "v_fmac_f32 %7, %9, %5\n\t"
        "v_fmac_f32_dpp %6, %3, %8" FF_DPP_SHL "v_fmac_f32_dpp %7, %5, %8" FF_DPP_SHL
        : "+v"(u), "+v"(v), "=&v"(mu), "=&v"(pu), "=&v"(mv), "=&v"(pv), "=&v"(a), "=&v"(b)
        : "v"(wo), "s"(wi), "s"(wc));
    u = a;
    v = b;
}
#undef FF_DPP_SHR
#undef FF_DPP_SHL

// 5-tap correlation along x in the order of the reference loops (c = -2..2):
// acc = 0; acc = fma(w[c], v(x+c), acc).
template <bool CLAMP, class Wf>
__device__ __forceinline__ float taps_x(float v, Wf w) {
    const float m1 = shr<CLAMP>(v), p1 = shl<CLAMP>(v);
    float a = 0.0f;
    a = fmaf(w(0), shr<CLAMP>(m1), a);
    a = fmaf(w(1), m1, a);
    a = fmaf(w(2), v, a);
    a = fmaf(w(3), p1, a);
    a = fmaf(w(4), shl<CLAMP>(p1), a);
    return a;
}

struct WSmooth {
    __device__ __forceinline__ float operator()(int i) const { return smooth_w(i); }
};
struct WDiff {
    __device__ __forceinline__ float operator()(int i) const { return diff_w(i); }
};
struct WBox {
    __device__ __forceinline__ float operator()(int) const { return kBox; }
};

// Map a job's tile index so that the tiles of one XCD (blocks are dealt
// round-robin over the 8 XCDs) form a contiguous band of the image.
__device__ __forceinline__ int xcd_tile(int b, int nt) {
    const int q = nt / 8;
    if (b >= 8 * q) return b;
    return (b % 8) * q + b / 8;
}

// Per-thread view of the tile.
struct Geo {
    int lane, wave, x, yw;
    int xl;        // column read: x, or the last column for x beyond the image
    int xlast;     // lane of the image's last column (>= LANES - 1: not in the buffer)
    bool xin;      // column strictly inside the propagation border
    bool wave_in;  // every pixel of the wave strictly inside the border
};

// Registers of the level state: flow (fu, fv) and, on delta levels, the
// scalar (old brightness) and vector (delta flow) payloads.
template <bool DELTA, int R>
struct State {
    float fu[R], fv[R];
    float sa[DELTA ? R : 1], du[DELTA ? R : 1], dv[DELTA ? R : 1];
};

// One upwind X pass (flowPropagateX_k / flowPropagatePayloadX_k,
// propagation_k.cu:16-72, 134-232). p: dt, border and H. LAST: the final iteration of a delta
// level, whose propagated flow is read only as the Y pass's speed (the
// delta update consumes the payloads): the u component is not advanced.
template <bool DELTA, bool BORDER, int R, bool LAST = false, class P>
__device__ __forceinline__ void prop_x(State<DELTA, R>& s, const Geo& g, const P& p) {
    constexpr bool kSkipU = DELTA && LAST;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float zu = s.fu[r], zv = s.fv[r];
        const float mu = zshr(zu), pu = zshl(zu);
        const float Ud = (fabsf(pu) - fabsf(mu)) > 0.0f ? pu : mu;
        const float nd = -(p.dt * Ud);
        // the upwind difference of each field: its backward difference here,
        // or, where the flow comes from the right, the one of the next lane
        // (26 instructions per pixel with both differences and a select, 21
        // so)
        float ou = zu, ov = zv, os = 0.f, odu = 0.f, odv = 0.f;
        float bu = zu - mu, bv = zv - zshr(zv);
        if constexpr (DELTA) {
            float bs = s.sa[r] - zshr(s.sa[r]), bdu = s.du[r] - zshr(s.du[r]), bdv = s.dv[r] - zshr(s.dv[r]);
            if constexpr (kSkipU) pick(Ud, bv, bs, bdu, bdv);
            else pick(Ud, bu, bv, bs, bdu, bdv);
            os = fmaf(nd, bs, s.sa[r]);
            odu = fmaf(nd, bdu, s.du[r]);
            odv = fmaf(nd, bdv, s.dv[r]);
        } else {
            pick(Ud, bu, bv);
        }
        if constexpr (!kSkipU) ou = fmaf(nd, bu, zu);
        ov = fmaf(nd, bv, zv);
        if constexpr (BORDER) {
            const int y = g.yw + r;
            const bool in = g.xin && y >= p.border && y < p.H - p.border;
            if constexpr (!kSkipU) ou = in ? ou : zu;
            ov = in ? ov : zv;
            if constexpr (DELTA) {
                os = in ? os : s.sa[r];
                odu = in ? odu : s.du[r];
                odv = in ? odv : s.dv[r];
            }
        }
        s.fu[r] = ou;
        s.fv[r] = ov;
        if constexpr (DELTA) {
            s.sa[r] = os;
            s.du[r] = odu;
            s.dv[r] = odv;
        }
    }
}

// Rows above (a) and below (b) a wave's strip for one Y pass.
struct Edge5 {
    float u, v, s, du, dv;
};

// One upwind Y pass (flowPropagateY_k / flowPropagatePayloadY_k,
// propagation_k.cu:75-131, 235-334); rows top-down, m* keep the old values
// of row r-1. LAST: the final pass of a delta level, whose propagated flow
// is dead (only the payloads feed the delta update): the flow is not
// advanced, only read for the speed Vd.
template <bool DELTA, bool BORDER, int R, bool LAST = false, class P>
__device__ __forceinline__ void prop_y(State<DELTA, R>& s, const Geo& g, const P& p, const Edge5& a, const Edge5& b) {
    constexpr bool kSkipF = DELTA && LAST;
    float mu = a.u, mv = a.v, ms = a.s, mdu = a.du, mdv = a.dv;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float zu = s.fu[r], zv = s.fv[r];
        const float pu = r + 1 < R ? s.fu[r + 1] : b.u;
        const float pv = r + 1 < R ? s.fv[r + 1] : b.v;
        const float Vd = (fabsf(pv) - fabsf(mv)) > 0.0f ? pv : mv;
        const float nd = -(p.dt * Vd);
        const bool back = Vd >= 0.0f;
        float ou = kSkipF ? zu : upwind(mu, zu, pu, back, nd);
        float ov = kSkipF ? zv : upwind(mv, zv, pv, back, nd);
        mu = zu;
        mv = zv;
        bool in = true;
        if constexpr (BORDER) {
            const int y = g.yw + r;
            in = g.xin && y >= p.border && y < p.H - p.border;
            if constexpr (!kSkipF) {
                ou = in ? ou : zu;
                ov = in ? ov : zv;
            }
        }
        s.fu[r] = ou;
        s.fv[r] = ov;
        if constexpr (DELTA) {
            const float zs = s.sa[r], zdu = s.du[r], zdv = s.dv[r];
            const float ps = r + 1 < R ? s.sa[r + 1] : b.s;
            const float pdu = r + 1 < R ? s.du[r + 1] : b.du;
            const float pdv = r + 1 < R ? s.dv[r + 1] : b.dv;
            float os = upwind(ms, zs, ps, back, nd);
            float odu = upwind(mdu, zdu, pdu, back, nd);
            float odv = upwind(mdv, zdv, pdv, back, nd);
            ms = zs;
            mdu = zdu;
            mdv = zdv;
            if constexpr (BORDER) {
                os = in ? os : zs;
                odu = in ? odu : zdu;
                odv = in ? odv : zdv;
            }
            s.sa[r] = os;
            s.du[r] = odu;
            s.dv[r] = odv;
        }
    }
}

// Image model (imagePrefilter_k / imageModel_k, imagemodel_k.cu:31-133) and
// update (flowUpdate_k, update_k.cu:15-79, or deltaFlowUpdate_k, :82-173)
// of every row of the thread. im[j] is image row yw-2+j (clamped reads),
// aold[r] the old brightness (top level) and up[r] the upper-level flow
// (delta level) of row r. Writes the new brightness (and delta flow) of the
// tile's output pixels; leaves the updated flow in s.fu/s.fv. p: gamma, maxflow
// and flow_upd. gradient(r, gx, gy) is called for each row.
template <bool DELTA, bool CLAMP, int R, class P, class G>
__device__ __forceinline__ void model_update(State<DELTA, R>& s, const float (&im)[R + 4], const float (&aold)[R],
                                             const float2 (&up)[R], const P& p, const Rsrc& ra0,
                                             const Rsrc& rdf, const Rsrc& rfu, const int (&offa)[R],
                                             const int (&offf)[R], G&& gradient) {
    float sx[R + 4];
#pragma unroll
    for (int j = 0; j < R + 4; ++j) sx[j] = taps_x<CLAMP>(im[j], WSmooth{});
#pragma unroll
    for (int r = 0; r < R; ++r) {
        float sy = 0.0f;
#pragma unroll
        for (int k = 0; k < 5; ++k) sy = fmaf(smooth_w(k), im[r + k], sy);
        const float a0 = taps_x<CLAMP>(sy, WSmooth{});
        const float gx = taps_x<CLAMP>(sy, WDiff{});
        float gy = 0.0f;
#pragma unroll
        for (int k = 0; k < 5; ++k) gy = fmaf(diff_w(k), sx[r + k], gy);
        gradient(r, gx, gy);
        float ox, oy;
        if constexpr (DELTA) {
            const float Yt = s.sa[r] - a0;
            solve2x2(gx, gy, Yt, s.du[r], s.dv[r], p.gamma, ox, oy);
            ox = not_finite(ox) ? 0.0f : ox;
            oy = not_finite(oy) ? 0.0f : oy;
            const float half = 0.5f * p.maxflow;
            ox = fmaxf(-half, fminf(ox, half));
            oy = fmaxf(-half, fminf(oy, half));
            float fx = ox + 2.0f * up[r].x, fy = oy + 2.0f * up[r].y;
            fx = fmaxf(-p.maxflow, fminf(fx, p.maxflow));
            fy = fmaxf(-p.maxflow, fminf(fy, p.maxflow));
            st1(ra0, offa[r], a0);
            st2(rdf, offf[r], ox, oy);
            ox = fx;
            oy = fy;
        } else {
            const float Yt = aold[r] - a0;
            solve2x2(gx, gy, Yt, s.fu[r], s.fv[r], p.gamma, ox, oy);
            ox = fmaxf(-p.maxflow, fminf(ox, p.maxflow));
            oy = fmaxf(-p.maxflow, fminf(oy, p.maxflow));
            ox = not_finite(ox) ? 0.0f : ox;
            oy = not_finite(oy) ? 0.0f : oy;
            st1(ra0, offa[r], a0);
            if (p.flow_upd) st2(rfu, offf[r], ox, oy);
        }
        s.fu[r] = ox;
        s.fv[r] = oy;
    }
}

// Lanes beyond the image's last column (lane xlast) take its values.
template <int R>
__device__ __forceinline__ void copy_last_column(float (&fu)[R], float (&fv)[R], int lane, int xlast) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float eu = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fu[r]), xlast));
        const float ev = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fv[r]), xlast));
        fu[r] = lane > xlast ? eu : fu[r];
        fv[r] = lane > xlast ? ev : fv[r];
    }
}

// X pass of the box smoother (flowSmoothX_k, flowsmoothing_k.cu:21-53).
template <bool CLAMP, int R>
__device__ __forceinline__ void smooth_x(float (&fu)[R], float (&fv)[R]) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if constexpr (CLAMP) {
            fu[r] = taps_x<CLAMP>(fu[r], WBox{});
            fv[r] = taps_x<CLAMP>(fv[r], WBox{});
        } else {
            taps_x2(fu[r], fv[r], kBox, kBox, kBox);
        }
    }
}

// Two rows above (a2, a1) and below (b1, b2) a strip of a vector field.
struct Edge2 {
    float a2u, a2v, a1u, a1v, b1u, b1v, b2u, b2v;
};

// Y pass of the box smoother (flowSmoothY_k, flowsmoothing_k.cu:55-87) over
// the thread's rows; e: the rows above and below. With
// YCLAMP, rows after rlast (outside the image) are replaced by row rlast, the
// clamped read; rows after rlast themselves are not needed.
template <bool YCLAMP, int R>
__device__ __forceinline__ void smooth_y(float (&fu)[R], float (&fv)[R], const Edge2& e, int rlast) {
    float m2u = e.a2u, m2v = e.a2v, m1u = e.a1u, m1v = e.a1v;  // old rows r-2, r-1
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float zu = fu[r], zv = fv[r];
        float p1u = r + 1 < R ? fu[r + 1] : e.b1u, p1v = r + 1 < R ? fv[r + 1] : e.b1v;
        float p2u = r + 2 < R ? fu[r + 2] : (r + 2 == R ? e.b1u : e.b2u);
        float p2v = r + 2 < R ? fv[r + 2] : (r + 2 == R ? e.b1v : e.b2v);
        if constexpr (YCLAMP) {
            p2u = r + 2 <= rlast ? p2u : (r + 1 <= rlast ? p1u : zu);
            p2v = r + 2 <= rlast ? p2v : (r + 1 <= rlast ? p1v : zv);
            p1u = r + 1 <= rlast ? p1u : zu;
            p1v = r + 1 <= rlast ? p1v : zv;
        }
        float su = 0.0f, sv = 0.0f;
        su = fmaf(kBox, m2u, su);
        sv = fmaf(kBox, m2v, sv);
        su = fmaf(kBox, m1u, su);
        sv = fmaf(kBox, m1v, sv);
        su = fmaf(kBox, zu, su);
        sv = fmaf(kBox, zv, sv);
        su = fmaf(kBox, p1u, su);
        sv = fmaf(kBox, p1v, sv);
        su = fmaf(kBox, p2u, su);
        sv = fmaf(kBox, p2v, sv);
        m2u = m1u;
        m2v = m1v;
        m1u = zu;
        m1v = zv;
        fu[r] = su;
        fv[r] = sv;
    }
}

// Row exchange buffer of the workgroup: [2][nw][10][LANES] floats (double
// buffered; 10 rows of each wave: its first and last rows of up to five
// fields).
__device__ __forceinline__ float* xrow(float* xch, int nw, int slot, int wave) {
    return xch + ((slot * nw + wave) * 10) * LANES;
}

// The rows next to each strip, for a Y pass: every wave leaves its first and
// last rows in LDS (put_rows, the half `slot` of the exchange buffer), and
// after a barrier takes the last row of the wave above (row_above) and the
// first of the wave below (row_below). The first (last) wave gets its own
// first (last) row: the clamp-to-edge read at an image edge.
template <bool DELTA, int R>
__device__ __forceinline__ void put_rows(const State<DELTA, R>& s, float* xch, int nw, int slot, int wave, int lane) {
    float* my = xrow(xch, nw, slot, wave);
    my[0 * LANES + lane] = s.fu[0];
    my[1 * LANES + lane] = s.fv[0];
    my[5 * LANES + lane] = s.fu[R - 1];
    my[6 * LANES + lane] = s.fv[R - 1];
    if constexpr (DELTA) {
        my[2 * LANES + lane] = s.sa[0];
        my[3 * LANES + lane] = s.du[0];
        my[4 * LANES + lane] = s.dv[0];
        my[7 * LANES + lane] = s.sa[R - 1];
        my[8 * LANES + lane] = s.du[R - 1];
        my[9 * LANES + lane] = s.dv[R - 1];
    }
}
template <bool DELTA, int R>
__device__ __forceinline__ Edge5 own_row(const State<DELTA, R>& s, int r) {
    Edge5 e{s.fu[r], s.fv[r], 0.f, 0.f, 0.f};
    if constexpr (DELTA) {
        e.s = s.sa[r];
        e.du = s.du[r];
        e.dv = s.dv[r];
    }
    return e;
}
template <bool DELTA>
__device__ __forceinline__ void get_row(Edge5& e, const float* o, int lane) {
    e.u = o[0 * LANES + lane];
    e.v = o[1 * LANES + lane];
    if constexpr (DELTA) {
        e.s = o[2 * LANES + lane];
        e.du = o[3 * LANES + lane];
        e.dv = o[4 * LANES + lane];
    }
}

// Those rows of each strip, for a Y pass of the smoother, as above.
template <int R>
__device__ __forceinline__ Edge2 exchange_smooth_rows(const float (&fu)[R], const float (&fv)[R], float* xch, int nw,
                                                      int slot, int wave, int lane) {
    {
        float* my = xrow(xch, nw, slot, wave);
        my[0 * LANES + lane] = fu[0];
        my[1 * LANES + lane] = fv[0];
        my[2 * LANES + lane] = fu[1];
        my[3 * LANES + lane] = fv[1];
        my[4 * LANES + lane] = fu[R - 2];
        my[5 * LANES + lane] = fv[R - 2];
        my[6 * LANES + lane] = fu[R - 1];
        my[7 * LANES + lane] = fv[R - 1];
    }
    __syncthreads();
    Edge2 e{fu[0], fv[0], fu[0], fv[0], fu[R - 1], fv[R - 1], fu[R - 1], fv[R - 1]};
    if (wave > 0) {
        const float* o = xrow(xch, nw, slot, wave - 1);
        e.a2u = o[4 * LANES + lane];
        e.a2v = o[5 * LANES + lane];
        e.a1u = o[6 * LANES + lane];
        e.a1v = o[7 * LANES + lane];
    }
    if (wave < nw - 1) {
        const float* o = xrow(xch, nw, slot, wave + 1);
        e.b1u = o[0 * LANES + lane];
        e.b1v = o[1 * LANES + lane];
        e.b2u = o[2 * LANES + lane];
        e.b2v = o[3 * LANES + lane];
    }
    return e;
}

}  // namespace tile
}  // namespace ffamd
