// ff_fused.hip -- the fused frame kernel for gfx950.
//
// One launch advances every level of a frame. Each level is a job; its
// output tiles are workgroups of the launch. A tile runs the whole per-level
// recurrence of the reference (FlowFilter::compute, src/gpu/flowfilter.cu:
// 125-153, and the DeltaFlowFilter update path, :429-503): N upwind
// propagation iterations of the previous smoothed flow (with the old
// brightness and delta flow as payloads on delta levels), the image model,
// the 2x2 update and K box smoothing iterations. State is read once and
// written once per frame; everything in between stays in registers.
//
// Jobs and their order. The top level of a pyramid comes first; the level
// below it reads the top level's unsmoothed flow of the same frame
// (flowfilter.cu:663-672), so its tiles wait, after their propagation
// phase and before the update, until the few top-level tiles that cover
// them have signalled completion (flags in device memory, wait_upper). Blocks
// are dispatched in order on each XCD and producers never wait, so every
// producer a consumer waits for is running or finished; the wait is also
// bounded by a spin limit. Lower levels read the previous frame's flow of the level above (the
// reference's ascending update order) and do not wait.
//
// Tile geometry: a workgroup is nw waves stacked vertically (nw is a launch
// parameter, picked by timing the candidates); lane l of every wave owns
// buffer column l (64 columns), and each thread owns R consecutive rows of
// its wave's strip (R = 8, or 4 on a top level that the level below waits
// for), so the buffer is 64 x (nw*R) pixels. The output
// tile is the buffer minus a halo h0 = max(N, 2 + e) + 2K on every side (the
// distance an error at the buffer edge travels inward: one pixel per
// propagation pass, two per smoothing pass, two for the image model's x
// taps, plus e = 1 when the image is reduced while loading, because then
// the buffer's first column also lacks its left source pixel).
//  - X neighbours come from DPP wave shifts; Y neighbours are registers of
//    the same thread, and the rows above and below a wave's strip are
//    exchanged through LDS once per Y pass.
//  - On levels at least as large as the buffer every buffer lies inside the
//    image: buffers at the image edges are clamped against the edge and
//    their output range extends to it. At an
//    image edge the missing neighbour must be the clamp-to-edge read of the
//    reference: the first/last wave use their own first/last row, and the
//    x taps of the image model and smoothing use DPP shifts in which the
//    edge lane keeps its own value. The propagation passes use zero-filling
//    shifts (a single instruction the compiler folds into the arithmetic):
//    with border >= 1 the pixels next to an image edge keep their value, so
//    the filled lane only affects pixels inside the halo.
//  - All global accesses are buffer instructions with 32-bit offsets; stores
//    of pixels outside the tile's output range use an offset beyond the
//    buffer's size, which the hardware discards (no branches).
//  - Image rows, the upper-level flow and the old brightness are loaded
//    before they are needed so their latency overlaps computation.
//  - A level narrower or shorter than the buffer is a single tile across or
//    down; the buffer then extends past the image's last column or row,
//    whose values the loads replicate (see level_tile).
//  The fused path needs border >= 1.
//
// Arithmetic per pixel is the reference's (same operations, order and
// rounding points as the stage kernels and the CPU oracle); results are
// bitwise identical to the stage-by-stage path.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <stdexcept>
#include <string>
#include <type_traits>

#include "ff_device.hpp"
#include "ff_kernels.hpp"
#include "ff_per_device.hpp"
#include "ff_runtime.hpp"
#include "ff_tile.hpp"

namespace ffamd {

namespace {

using namespace tile;

constexpr int kSpinLimit = 1 << 23;   // polls before a wait gives up: about 2 s at s_sleep 8

// One level of one frame, as the kernel reads it. Blocks first_block ..
// first_block + tiles_x * tiles_y - 1 of the launch are its tiles.
struct LevelJob {
    const void* img;
    const float2* flow_in;
    const float* a0_in;
    const float2* dflow_in;
    float2* flow_out;
    float* a0_out;
    float2* dflow_out;
    float2* flow_upd;  // may be null on a top level
    const float2* upper;
    const int* xmap;
    const int* ymap;
    // row pitches in bytes
    int img_pitch, flow_in_pitch, a0_in_pitch, dflow_in_pitch, flow_out_pitch, a0_out_pitch, dflow_out_pitch,
        flow_upd_pitch, upper_pitch;
    int W, H, Hu, Hsrc;  // level size, upper level height, image height
    int N, K, border, h0, TW, TH, tiles_x, tiles_y;
    int delta, img_mode, first_block;
    // wait_job >= 0: wait for tiles of that job of the table, which has
    // wait_tx tiles across and its first tile's flags at wait_flags. Which
    // of them: the first and last row (words wait_rows + 2 r and + 2 r + 1 of
    // the block map) for this job's tile row r, and the first and last column
    // (from word wait_rows + 2 (tiles_y + c)) for its tile column c. flags
    // >= 0: the job's tiles are waited for; tile t's flags are at flags + t.
    // frame_slot >= 0: the level's image is a filter's input frame, which a
    // launch may pass in place as its frame frame_slot (read where the
    // caller keeps it).
    int wait_job, wait_tx, wait_flags, wait_rows, flags, frame_slot;
    float dt, gamma, maxflow;
};


// A job in the constant address space: its fields are read with scalar loads
// wherever they are used.
#define FF_CONSTANT __attribute__((address_space(4)))

// --------------------------------------------------- tiles waited for

// Flags of the top-level tiles that a launch's other tiles wait for: a word
// each, which the launch sets to its sequence number `epoch` (1, 2, ... since
// the host last cleared the flags) when the tile is done, so that nothing is
// reset in the kernel. `started` (may be null) counts all such tiles of all
// launches on the device as they start (WaitingLaunch).
struct TileFlags {
    unsigned* done;
    unsigned* timeouts;  // count of the waits that gave up
    unsigned* started;
    unsigned epoch;
};

// Blocks are grouped by tile body: top levels with float, u8, reduced u8
// and twice-reduced u8 images, then delta levels with float, u8 and reduced
// u8 images; ends[i] is the first block after group i. (Selecting the body
// from the block index rather than from a job field also keeps the
// compiler's register allocation of each body as tight as in a kernel of
// its own.)
struct GroupEnds {
    int e[6];
};

// Arguments of the frame kernel, in one struct that any place reads from the
// kernel's argument segment (launch_args).
struct WaitArgs {
    int spin_limit;
    unsigned bias;
};
struct FrameArgs {
    const unsigned char* ptr[kMaxLaunchFrames];
    int pitch[kMaxLaunchFrames];
};
struct LaunchArgs {
    const LevelJob* jobs;
    const int* block_job;
    TileFlags fl;
    GroupEnds ends;
    int nw;
    WaitArgs wa;
    FrameArgs frames;
};
__device__ __forceinline__ const LaunchArgs& launch_args() {
    auto* q = (const FF_CONSTANT LaunchArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    return *(const LaunchArgs*)q;
}

__device__ __forceinline__ unsigned flag_load(const unsigned* f) {
    return __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void flag_store(unsigned* f, unsigned v) {
    __hip_atomic_store(f, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void flag_add(unsigned* f) {
    __hip_atomic_fetch_add(f, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The tiles of the upper level that tile t waits for: first, first + 1, ..,
// nx of them across, n in all.
struct UpperTiles {
    int first, nx, n;
    // the i-th of them
    __device__ __forceinline__ int tile(int i, const LevelJob& p) const { return first + i / nx * p.wait_tx + i % nx; }
};
__device__ __forceinline__ UpperTiles upper_tiles(const LevelJob& p, int t) {
    const int ty = t / p.tiles_x, tx = t - ty * p.tiles_x;
    const auto* w = (const FF_CONSTANT int*)launch_args().block_job + p.wait_rows;
    const auto *rows = w + 2 * ty, *cols = w + 2 * (p.tiles_y + tx);
    const int ty0 = rows[0], ty1 = rows[1], tx0 = cols[0], tx1 = cols[1];
    const int nx = tx1 - tx0 + 1;
    return UpperTiles{ty0 * p.wait_tx + tx0, nx, (ty1 - ty0 + 1) * nx};
}

// Wait for the tiles u of the upper level. Waiting for these few alone lets a
// tile go on as soon as they are there, whatever the rest of the level does
// (a 2048x1088 two-level launch took 54.6 us when every tile waited for the
// whole level, 52.2 us so). The first wave polls, a lane per tile, with
// relaxed loads (the flow the producers published is read with
// device-coherent loads after the wait, so no cache needs invalidating), and
// the barrier holds the others. The wait gives up after `spin_limit` polls
// and counts a timeout (the host reports it as an error). `bias` is added to
// the number waited for (0, or what no launch writes, which a test uses to
// make the wait give up).
__device__ __forceinline__ void wait_upper(const LevelJob& p, const UpperTiles& u, const Geo& g) {
    if (g.wave == 0) {
        const TileFlags& fl = launch_args().fl;
        const int spin_limit = launch_args().wa.spin_limit;
        const unsigned bias = launch_args().wa.bias;
        int spins = 0;
        for (int first = 0; first < u.n; first += LANES) {
            const unsigned* done = fl.done + p.wait_flags + u.tile(min(first + g.lane, u.n - 1), p);
            while (__ballot(flag_load(done) != fl.epoch + bias)) {
                __builtin_amdgcn_s_sleep(8);
                if (++spins > spin_limit) {
                    if (g.lane == 0) flag_add(fl.timeouts);
                    first = u.n;
                    break;
                }
            }
        }
    }
    __syncthreads();
}

// Count an awaited tile as started.
__device__ __forceinline__ void signal_started(const Geo& g) {
    unsigned* started = launch_args().fl.started;
    if (started && g.wave == 0 && g.lane == 0) flag_add(started);
}

// Mark tile t as done once its device-coherent stores have completed: every
// wave waits for its outstanding stores (vmcnt 0; the immediate leaves the
// other counters unwaited), the barrier joins the waves, and one thread
// writes the flag.
__device__ __forceinline__ void signal_done(const LevelJob& p, int t, const Geo& g) {
    const TileFlags& fl = launch_args().fl;
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    if (g.wave == 0 && g.lane == 0) flag_store(fl.done + p.flags + t, fl.epoch);
}

// ------------------------------------------------------------ tile body

// Image rows yw-2 .. yw+R+1 (clamped to the level) at the thread's column.
// load_image issues the loads; finish_image turns them into normalized
// values once they are needed, so the latency of the F32 and U8 loads
// overlaps the propagation phase.
//  IMG_F32:     the float texel.
//  IMG_U8:      the u8 texel.
//  IMG_U8_DOWN: the texel of the level one pyramid step below (twice the
//               size): imageDownX_uint8_k then imageDownY_uint8_k
//               (pyramid_k.cu:14-78) evaluated for this texel. Row yy needs
//               source rows 2yy-1 (clamped), 2yy, 2yy+1; each of those the
//               source columns 2x-1 (clamped), 2x, 2x+1, read as one 16-bit
//               load of columns 2x, 2x+1 and the high byte of the left
//               lane's load. With W = Wsrc/2 and H = Hsrc/2 (integer
//               halving) the columns 2x+1 and rows 2yy+1 are always inside
//               the source image. The reduction runs right after the loads
//               (three source rows per texel would not fit in registers
//               through the propagation phase).

// One pyramid step along x of a source row: columns 2x-1 (clamped), 2x, 2x+1.
// Column 2x-1 is the high byte of the left lane's pair; lane 0 takes its own
// low byte instead, which is the clamped read when x = 0 (for a buffer that
// does not start at the image edge lane 0 lies in the halo).
__device__ __forceinline__ unsigned down_x(unsigned pair) {
    const unsigned lo = pair & 0xffu, hi = pair >> 8;
    const unsigned left = (shr_or(pair, pair << 8) >> 8) & 0xffu;
    return down_u8(left, lo, hi);
}

// Registers holding the image rows between the loads and their use: the
// float texels, or the u8 texels packed four to a register (the byte
// conversion instructions read them in place).
template <int MODE, int R>
struct ImageRegs {
    static constexpr int kN = MODE == IMG_F32 ? R + 4 : (R + 4 + 3) / 4;
    unsigned v[kN];
};

// The level's source image: the job's, or the frame passed to the launch.
struct ImgSrc {
    const void* data;
    int pitch;
};

template <int MODE, int R>
__device__ __forceinline__ void load_image(ImageRegs<MODE, R>& ir, const LevelJob& p, const Geo& g, ImgSrc src) {
    const Rsrc rimg = rsrc(src.data, src.pitch * p.Hsrc);
    const int ipitch = src.pitch;
    if constexpr (MODE == IMG_F32) {
#pragma unroll
        for (int j = 0; j < R + 4; ++j) {
            const int yc = clampi(g.yw - 2 + j, 0, p.H - 1);
            ir.v[j] = __builtin_amdgcn_raw_buffer_load_b32(rimg, yc * ipitch + g.xl * 4, 0, 0);
        }
        return;
    } else {
        unsigned t[R + 4];
        if constexpr (MODE == IMG_U8_DOWN2) {
            // source rows 4yy-3 .. 4yy+3 (level-1 rows 2yy-1 .. 2yy+1, each
            // from its three source rows), one 32-bit load of columns
            // 4x .. 4x+3 per row
            const int H1 = p.Hsrc / 2;
#pragma unroll
            for (int j = 0; j < R + 4; ++j) {
                const int yy = clampi(g.yw - 2 + j, 0, p.H - 1);
                unsigned l1a[3], l1b[3];  // level-1 texels at columns 2x, 2x+1 of rows 2yy-1+k
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const int r1 = clampi(2 * yy - 1 + k, 0, H1 - 1);
                    unsigned xa[3], xb[3];
#pragma unroll
                    for (int m = 0; m < 3; ++m) {
                        const int r0 = max(2 * r1 - 1 + m, 0);
                        const unsigned wd = __builtin_amdgcn_raw_buffer_load_b32(rimg, r0 * ipitch + 4 * g.xl, 0, 0);
                        const unsigned b0 = wd & 0xffu, b1 = (wd >> 8) & 0xffu, b2 = (wd >> 16) & 0xffu, b3 = wd >> 24;
                        const unsigned left = (shr_or(wd, wd << 24) >> 24) & 0xffu;  // column 4x-1 (clamped)
                        xa[m] = down_u8(left, b0, b1);
                        xb[m] = down_u8(b1, b2, b3);
                    }
                    l1a[k] = down_u8(xa[0], xa[1], xa[2]);
                    l1b[k] = down_u8(xb[0], xb[1], xb[2]);
                }
                unsigned yv[3];
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    // level-1 column 2x-1 is the left lane's 2x+1 (clamped at x = 0)
                    const unsigned lm = shr_or(l1b[k], l1a[k]);
                    yv[k] = down_u8(lm, l1a[k], l1b[k]);
                }
                t[j] = down_u8(yv[0], yv[1], yv[2]);
            }
        } else if constexpr (MODE == IMG_U8_DOWN) {
            unsigned src[R + 4][3];
#pragma unroll
            for (int j = 0; j < R + 4; ++j) {
                const int r1 = 2 * clampi(g.yw - 2 + j, 0, p.H - 1);
                const int r0 = r1 > 0 ? r1 - 1 : 0;
                src[j][0] = ldh(rimg, r0 * ipitch + 2 * g.xl);
                src[j][1] = ldh(rimg, r1 * ipitch + 2 * g.xl);
                src[j][2] = ldh(rimg, (r1 + 1) * ipitch + 2 * g.xl);
            }
#pragma unroll
            for (int j = 0; j < R + 4; ++j) t[j] = down_u8(down_x(src[j][0]), down_x(src[j][1]), down_x(src[j][2]));
        } else {
#pragma unroll
            for (int j = 0; j < R + 4; ++j) {
                const int yc = clampi(g.yw - 2 + j, 0, p.H - 1);
                t[j] = ldb(rimg, yc * ipitch + g.xl);
            }
        }
        if constexpr (MODE == IMG_U8_DOWN || MODE == IMG_U8_DOWN2) {
            // lanes beyond the last column: copies of it (their own reduction
            // would combine a clamped centre with an unclamped left column)
            if (g.xlast < LANES - 1) {
#pragma unroll
                for (int j = 0; j < R + 4; ++j) {
                    const unsigned e = (unsigned)__builtin_amdgcn_readlane((int)t[j], g.xlast);
                    t[j] = g.lane > g.xlast ? e : t[j];
                }
            }
        }
#pragma unroll
        for (int k = 0; k < ImageRegs<MODE, R>::kN; ++k) {
            unsigned w = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (4 * k + i < R + 4) w |= t[4 * k + i] << (8 * i);
            // pack here: left to the compiler, the bytes (or, reduced on
            // load, three source values per row) would stay in separate
            // registers through the propagation phase
            asm volatile("" : "+v"(w));
            ir.v[k] = w;
        }
    }
}

template <int MODE, int R>
__device__ __forceinline__ void finish_image(const ImageRegs<MODE, R>& ir, float (&im)[R + 4]) {
#pragma unroll
    for (int j = 0; j < R + 4; ++j) {
        if constexpr (MODE == IMG_F32) im[j] = __uint_as_float(ir.v[j]);
        else im[j] = unorm8((ir.v[j / 4] >> (8 * (j % 4))) & 0xffu);
    }
}

// INNER: a tile whose every pixel lies inside the border, away from the
// image edges (every wave inside, no edge lanes, no clamped rows, no
// column or row beyond the image): one straight-line body with no per-wave
// choice of pass forms, so no register copies where two forms of a pass
// would join; it computes what the general body computes for such a tile.
// ALLOW_INNER: interior tiles take that body (a kernel instantiation of
// its own, since the second body changes the register allocation of the
// first). Other tiles choose per wave.
// t: the tile, row by row from the top.
template <bool DELTA, int MODE, int R, bool ALLOW_INNER, bool INNER = false>
__device__ __forceinline__ void level_tile(const LevelJob& p, int t, float* xch, int nw, ImgSrc frame) {
    Geo g;
    // the lane from the hardware's count, so that threadIdx.x takes no
    // register beyond the next line
    g.lane = lane_id();
    g.wave = wave_id();
    if constexpr (!DELTA && !INNER)
        if (p.flags >= 0) signal_started(g);
    // output range of the tile and the buffer around it, clamped into the image
    const int tyi = t / p.tiles_x, txi = t - tyi * p.tiles_x;
    const int ox0 = txi * p.TW, ox1 = min(ox0 + p.TW, p.W);
    const int oy0 = tyi * p.TH, oy1 = min(oy0 + p.TH, p.H);
    const int x0 = clampi(ox0 - p.h0, 0, p.W - LANES);
    const int y0 = clampi(oy0 - p.h0, 0, p.H - nw * R);
    if constexpr (ALLOW_INNER && !INNER) {
        // at least one column and row from each image edge, also when the
        // propagation border is 0
        const int bb = max(p.border, 1);
        if (x0 >= bb && x0 + LANES - 1 < p.W - bb && y0 >= bb && y0 + nw * R - 1 < p.H - bb) {
            level_tile<DELTA, MODE, R, true, true>(p, t, xch, nw, frame);
            return;
        }
    }
    g.x = x0 + g.lane;
    g.xl = min(g.x, p.W - 1);
    g.yw = y0 + g.wave * R;  // image row of this thread's first row (wave-uniform)
    const int b = p.border;
    g.xin = g.x >= b && g.x < p.W - b;
    g.wave_in = (x0 >= b) && (x0 + LANES - 1 < p.W - b) && (g.yw >= b) && (g.yw + R - 1 < p.H - b);
    // an image edge at or inside the buffer's left/right edge
    const bool xedge = (x0 == 0) || (x0 + LANES >= p.W);
    // Images narrower than the buffer (a single tile across): the lanes
    // beyond the last column hold copies of it, loaded by clamped reads, so
    // the image model's taps and the propagation (which keeps pixels within
    // the border) see the reference's clamp-to-edge reads; the smoothing
    // passes re-copy the last column before every X pass and clamp their row
    // neighbours at the last row (rlast: the thread's last row inside the
    // image, relative to its first row).
    const int xlast = p.W - 1 - x0;  // lane of the last column
    const bool xinside = xlast < LANES - 1;
    g.xlast = xlast;
    const int rlast = p.H - 1 - g.yw;
    const bool yinside = y0 + nw * R > p.H;
    const int lane = g.lane, wave = g.wave;
    const bool out_x = g.x >= ox0 && g.x < ox1;

    const Rsrc rfi = rsrc(p.flow_in, p.flow_in_pitch * p.H);
    const Rsrc rai = rsrc(p.a0_in, p.a0_in_pitch * p.H);

    // (looked up here, so that the wait is one load from the flags)
    UpperTiles u{0, 1, 0};
    if (DELTA && p.wait_job >= 0) u = upper_tiles(p, t);

    State<DELTA, R> s;

    // ------------------------------------- load the state and the image rows
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int y = min(g.yw + r, p.H - 1);
        const float2 f = ld2(rfi, y * p.flow_in_pitch + g.xl * 8);
        s.fu[r] = f.x;
        s.fv[r] = f.y;
        if constexpr (DELTA) {
            s.sa[r] = ld1(rai, y * p.a0_in_pitch + g.xl * 4);
            const float2 d = ld2(rsrc(p.dflow_in, p.dflow_in_pitch * p.H), y * p.dflow_in_pitch + g.xl * 8);
            s.du[r] = d.x;
            s.dv[r] = d.y;
        }
    }
    ImageRegs<MODE, R> ir;
    load_image<MODE, R>(ir, p, g, frame.data ? frame : ImgSrc{p.img, p.img_pitch});

    int slot = 0;

    // ---------------------------------------------------------- propagation
    // N iterations of an X and a Y pass; the last one separately, since on
    // a delta level part of its flow output is dead
    auto iteration = [&](auto last) {
        constexpr bool LAST = decltype(last)::value;
        if (INNER || g.wave_in) prop_x<DELTA, false, R, LAST>(s, g, p);
        else prop_x<DELTA, true, R, LAST>(s, g, p);
        put_rows<DELTA, R>(s, xch, nw, slot, wave, lane);
        __syncthreads();
        Edge5 ea = own_row<DELTA, R>(s, 0), eb = own_row<DELTA, R>(s, R - 1);
        if (wave > 0) get_row<DELTA>(ea, xrow(xch, nw, slot, wave - 1) + 5 * LANES, lane);
        if (wave < nw - 1) get_row<DELTA>(eb, xrow(xch, nw, slot, wave + 1), lane);
        slot ^= 1;
        if (INNER || g.wave_in) prop_y<DELTA, false, R, LAST>(s, g, p, ea, eb);
        else prop_y<DELTA, true, R, LAST>(s, g, p, ea, eb);
    };
    for (int it = 0; it + 1 < p.N; ++it) iteration(std::false_type{});
    iteration(std::true_type{});

    // ------------------------------------------------ image model + update
    if (DELTA && p.wait_job >= 0) wait_upper(p, u, g);
    float aold[R];  // unused (and removed) on delta levels
    float2 up[R];
    int offa[R], offf[R];
    const Rsrc rao = rsrc(p.a0_out, p.a0_out_pitch * p.H);
    const Rsrc rdf = rsrc(p.dflow_out, p.dflow_out_pitch * p.H);
    const Rsrc rfu = rsrc(p.flow_upd, p.flow_upd_pitch * p.H);
    const int xmx = DELTA ? p.xmap[g.xl] : 0;
    const Rsrc rup = rsrc(p.upper, p.upper_pitch * p.Hu);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int y = g.yw + r;
        const bool out = out_x && y >= oy0 && y < oy1;
        const int yl = min(y, p.H - 1);
        offa[r] = out ? y * p.a0_out_pitch + g.x * 4 : OOB;
        if constexpr (DELTA) {
            offf[r] = out ? y * p.dflow_out_pitch + g.x * 8 : OOB;
            up[r] = ld2_coherent(rup, p.ymap[yl] * p.upper_pitch + xmx * 8);
            aold[r] = 0.f;
        } else {
            offf[r] = out ? y * p.flow_upd_pitch + g.x * 8 : OOB;
            // (looked up anew: held from the start it spills)
            aold[r] = ld1(rsrc(p.a0_in, p.a0_in_pitch * p.H), yl * p.a0_in_pitch + g.xl * 4);
            up[r] = make_float2(0.f, 0.f);
        }
    }
    float im[R + 4];
    finish_image<MODE, R>(ir, im);
    const auto none = [](int, float, float) {};
    if (!INNER && xedge) model_update<DELTA, true, R>(s, im, aold, up, p, rao, rdf, rfu, offa, offf, none);
    else model_update<DELTA, false, R>(s, im, aold, up, p, rao, rdf, rfu, offa, offf, none);

    // ------------------------------------------------------------ smoothing
    // flowSmoothX_k / flowSmoothY_k (flowsmoothing_k.cu:21-87), K times.
    for (int it = 0; it < p.K; ++it) {
        if (!INNER && xinside) copy_last_column<R>(s.fu, s.fv, g.lane, xlast);
        if (!INNER && xedge) smooth_x<true, R>(s.fu, s.fv);
        else smooth_x<false, R>(s.fu, s.fv);
        const Edge2 e = exchange_smooth_rows<R>(s.fu, s.fv, xch, nw, slot, wave, lane);
        slot ^= 1;
        if (!INNER && yinside) smooth_y<true, R>(s.fu, s.fv, e, rlast);
        else smooth_y<false, R>(s.fu, s.fv, e, rlast);
    }

    // ------------------------------------------------- write the new state
    const Rsrc rfo = rsrc(p.flow_out, p.flow_out_pitch * p.H);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int y = g.yw + r;
        const bool out = out_x && y >= oy0 && y < oy1;
        st2(rfo, out ? y * p.flow_out_pitch + g.x * 8 : OOB, s.fu[r], s.fv[r]);
    }
    if (!DELTA && p.flags >= 0) signal_done(p, t, g);
}

// Rows per thread of a tile body: RLOW, except for top levels reduced on
// load (the top level of a pyramid, which the level below waits for), which
// use RTOP; both are parameters of the kernel, chosen per launch by the
// tuner among kShapes. RTOP 4: the top level's tiles are more and shorter
// and finish sooner (a pyramid launched alone is faster); 8: they carry less
// halo (a 64-stream batch is 1.4 % faster). RLOW 4 with 16 waves covers
// the same 64-row tile as RLOW 8 with 8 waves, in half the registers per
// thread: that kernel is held to 64 VGPRs, so two 16-wave workgroups (32
// waves) fit a CU instead of two 8-wave ones, for about 8 % more VALU
// instructions per pixel (each wave exchanges its edge rows for half as
// many rows).
constexpr int kRows = 8;
constexpr int kTopRowChoices[] = {4, 8};
struct TileShape {
    int rtop, rlow;
    bool inner;  // interior tiles in a body of their own (k_fused_frame's INNER)
};
constexpr TileShape kShapes[] = {{4, 8, false}, {8, 8, false}, {4, 4, false}, {4, 4, true}};

// The job of block b, its tile there, and its input frame if the launch passes
// it in place (frame_slot is uniform, so is the selection).
__device__ __forceinline__ const LevelJob& job_of_block(unsigned b) {
    const LaunchArgs& a = launch_args();
    return *(const LevelJob*)((const FF_CONSTANT LevelJob*)a.jobs + ((const FF_CONSTANT int*)a.block_job)[b]);
}
__device__ __forceinline__ int job_tile(const LevelJob& p, unsigned b) {
    return xcd_tile((int)b - p.first_block, p.tiles_x * p.tiles_y);
}
__device__ __forceinline__ ImgSrc frame_of(const LevelJob& p) {
    if (p.frame_slot < 0) return ImgSrc{nullptr, 0};
    const FrameArgs& f = launch_args().frames;
    return ImgSrc{f.ptr[p.frame_slot], f.pitch[p.frame_slot]};
}

template <int RTOP, int RLOW = kRows, bool INNER = false>
__global__ void __launch_bounds__(1024, RLOW == 4 ? 8 : 1) k_fused_frame(LaunchArgs) {
    // row exchange between the waves of the workgroup (2 * nw * 10 * LANES floats)
    extern __shared__ float xch[];
    const unsigned b = blockIdx.x;
    const LevelJob& q = job_of_block(b);
    const int t = job_tile(q, b);
    const ImgSrc fr = frame_of(q);
    const int nw = launch_args().nw;
    const GroupEnds& ends = launch_args().ends;
    if (b < (unsigned)ends.e[0]) level_tile<false, IMG_F32, RLOW, INNER>(q, t, xch, nw, fr);
    else if (b < (unsigned)ends.e[1]) level_tile<false, IMG_U8, RLOW, INNER>(q, t, xch, nw, fr);
    else if (b < (unsigned)ends.e[2]) level_tile<false, IMG_U8_DOWN, RTOP, INNER>(q, t, xch, nw, fr);
    else if (b < (unsigned)ends.e[3]) level_tile<false, IMG_U8_DOWN2, RTOP, INNER>(q, t, xch, nw, fr);
    else if (b < (unsigned)ends.e[4]) level_tile<true, IMG_F32, RLOW, INNER>(q, t, xch, nw, fr);
    else if (b < (unsigned)ends.e[5]) level_tile<true, IMG_U8, RLOW, INNER>(q, t, xch, nw, fr);
    else level_tile<true, IMG_U8_DOWN, RLOW, INNER>(q, t, xch, nw, fr);
}

// (The stream behind it goes on either way, so that its work ends; the count
// makes the filter's next check an error.)
__global__ void __launch_bounds__(LANES) k_wait_started(const unsigned* word, unsigned target, int spin_limit,
                                                        unsigned* timeouts, unsigned* gave_up) {
    int spins = 0;
    while ((int)(flag_load(word) - target) < 0) {
        __builtin_amdgcn_s_sleep(8);
        if (++spins <= spin_limit) continue;
        if (lane_id() == 0) {
            flag_add(timeouts);
            __hip_atomic_store(gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        break;
    }
}

__global__ void k_clear_flags(unsigned* c, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) c[i] = 0u;
}

constexpr int kMaxWaves = 16;  // waves per workgroup, at most
// Waves per workgroup the autotuner tries: 16 and 15 (one workgroup per CU),
// 8 (two), 5 (three) and 4 (four); the register budget allows 16 waves per
// CU.
constexpr int kWaveChoices[] = {16, 15, 8, 5, 4};

// Whether a job runs a top-level body reduced on load (rows per thread
// RTOP).
bool top_rows_body(const LevelArgs& a) { return !a.delta && (a.img_mode == IMG_U8_DOWN || a.img_mode == IMG_U8_DOWN2); }

// Rows per thread of a job's tile body (see k_fused_frame).
int rows_per_thread(const LevelArgs& a, int rtop, int rlow = kRows) { return top_rows_body(a) ? rtop : rlow; }

size_t lds_bytes(int nw) { return (size_t)2 * nw * 10 * LANES * sizeof(float); }

// Level size of a job (the image is larger when reduced on load).
void level_size(const LevelArgs& a, int& H, int& W) {
    H = a.flow_s_in.h;
    W = a.flow_s_in.w;
}

int halo_of(const LevelArgs& a) {
    const int lo = (a.img_mode == IMG_U8_DOWN || a.img_mode == IMG_U8_DOWN2) ? 3 : 2;
    return (a.prop_iters > lo ? a.prop_iters : lo) + 2 * a.smooth_iters;
}

bool fits_i32(const DevImg& d) {
    return (unsigned long long)d.pitch * (unsigned long long)(d.h > 0 ? d.h : 0) < 0x7fffffffULL;
}

// The tiling of a level with buffers of `rows` rows leaves a non-empty
// output tile (or the level fits in one tile).
bool tiles_with(const LevelArgs& a, int rows) {
    int H, W;
    level_size(a, H, W);
    const int h0 = halo_of(a);
    return !((W > LANES && 2 * h0 >= LANES) || (H > rows && 2 * h0 >= rows));
}

}  // namespace

void launch_wait_started(const unsigned* word, unsigned target, int spin_limit, unsigned* timeouts, unsigned* gave_up,
                         hipStream_t s) {
    hipLaunchKernelGGL(k_wait_started, dim3(1), dim3(LANES), 0, s, word, target, spin_limit, timeouts, gave_up);
}

bool fused_level_supported(const LevelArgs& a) {
    if (a.border < 1 || a.prop_iters < 1 || a.smooth_iters < 1) return false;
    int H, W;
    level_size(a, H, W);
    if (H < 1 || W < 1) return false;
    if (!tiles_with(a, kMaxWaves * rows_per_thread(a, kTopRowChoices[0]))) return false;
    if (!a.img.data || !a.flow_s_in.data || !a.a0_in.data || !a.flow_s_out.data || !a.a0_out.data) return false;
    switch (a.img_mode) {
    case IMG_F32:
    case IMG_U8:
        if (a.img.h != H || a.img.w != W) return false;
        break;
    case IMG_U8_DOWN:
        if (a.img.h / 2 != H || a.img.w / 2 != W) return false;
        break;
    case IMG_U8_DOWN2:
        if ((a.img.h / 2) / 2 != H || (a.img.w / 2) / 2 != W || a.delta) return false;
        break;
    default:
        return false;
    }
    if (a.delta && (!a.dflow_in.data || !a.dflow_out.data || !a.upper.data || !a.xmap || !a.ymap ||
                    a.upper.h <= 0 || a.upper.w <= 0))
        return false;
    if (!a.delta && a.wait_on >= 0) return false;
    for (const DevImg* d : {&a.a0_in, &a.flow_s_out, &a.a0_out})
        if (d->h != H || d->w != W) return false;
    if (a.delta)
        for (const DevImg* d : {&a.dflow_in, &a.dflow_out})
            if (d->h != H || d->w != W) return false;
    if (a.flow_upd_out.data && (a.flow_upd_out.h != H || a.flow_upd_out.w != W)) return false;
    // every buffer must be addressable with 32-bit offsets
    for (const DevImg* d : {&a.img, &a.flow_s_in, &a.a0_in, &a.dflow_in, &a.flow_s_out, &a.a0_out, &a.dflow_out,
                            &a.flow_upd_out, &a.upper})
        if (!fits_i32(*d)) return false;
    return true;
}

// ------------------------------------------------------------- FusedFrame

namespace {
constexpr int kGroups = 7;
// Tile body group of a job (the order of the kernel's dispatch).
int body_group(const LevelArgs& a) {
    if (!a.delta) return a.img_mode;  // IMG_F32 .. IMG_U8_DOWN2: groups 0 .. 3
    return 4 + a.img_mode;            // IMG_F32 .. IMG_U8_DOWN: groups 4 .. 6
}

// What the tiling choice depends on: the shape and halo of every level.
std::vector<int> tune_key(const std::vector<LevelArgs>& jobs) {
    std::vector<int> k;
    for (const LevelArgs& a : jobs) {
        int H, W;
        level_size(a, H, W);
        k.insert(k.end(), {H, W, halo_of(a), a.prop_iters, a.smooth_iters, a.delta, a.img_mode, a.wait_on});
    }
    return k;
}
}  // namespace

struct FusedFrame::Impl {
    struct Table {
        std::vector<char> key;  // job records + block map + launch shape, as uploaded
        DeviceArray dev;
        int njobs = 0, blocks = 0, nw = 0;
        GroupEnds ends{};
        int rtop = 0, rlow = kRows;
        bool inner = false;  // launched as k_fused_frame<4, 4, true>
        size_t map_offset = 0;
        unsigned long long token = 0;
        int awaited = 0;  // tiles that others wait for
    };
    Table slot[2];
    int next = 0;
    unsigned long long uploads = 0;
    // Flags of the tiles waited for: per table slot (the two slots alternate
    // when a filter's state buffers ping-pong between frames) nflags words;
    // then the count of the waits that gave up.
    DeviceArray flags;
    int nflags = 0;
    // per slot: launches since its flags were last cleared, and the table
    // they were for (0: clear before the next launch)
    unsigned epoch[2] = {0, 0};
    unsigned long long counted[2] = {0, 0};
    // waves per workgroup, top-level rows per thread, other rows per thread;
    // 0: autotune
    int fixed = 0, fixed_rtop = 0, fixed_rlow = 0;
    int fixed_inner = 0;  // 0: tuned, 1: interior tiles in their own body, 2: not
    std::vector<int> tuned_for;
    int tuned = 0, tuned_rtop = 0, tuned_rlow = kRows;
    bool tuned_inner = false;
    std::shared_ptr<WaitWatch> watch = std::make_shared<WaitWatch>();
    int test_spins = 0;  // > 0: the waits give up after this many polls (test hook)

    int table(const std::vector<LevelArgs>& jobs, int nw, int rtop, int rlow, bool inner, hipStream_t s);
    unsigned* region(int si) const { return (unsigned*)flags.data() + (size_t)si * nflags; }
    unsigned* timeout_word() const { return (unsigned*)flags.data() + (size_t)2 * nflags; }
    // the waits of the test hook wait for what no launch writes
    WaitArgs wait_args() const {
        return test_spins > 0 ? WaitArgs{test_spins, 0x40000000u} : WaitArgs{kSpinLimit, 0u};
    }
    AwaitedTiles awaited(const Table& t) const {
        const WaitArgs wa = wait_args();
        return AwaitedTiles{t.awaited, timeout_word(), wa.spin_limit, wa.bias};
    }
    void clear_flags(int si, hipStream_t s) const;
    void run(int t, hipStream_t s, const FrameRef* frames = nullptr, int nframes = 0);
    void tune(const std::vector<LevelArgs>& jobs, hipStream_t s);
};

FusedFrame::FusedFrame() : impl_(new Impl) {}
FusedFrame::~FusedFrame() { delete impl_; }
FusedFrame::FusedFrame(FusedFrame&& o) noexcept : impl_(o.impl_) { o.impl_ = new Impl; }
FusedFrame& FusedFrame::operator=(FusedFrame&& o) noexcept {
    std::swap(impl_, o.impl_);
    return *this;
}

// Job table of `jobs` tiled with nw waves per workgroup and rtop rows per
// thread on reduced top levels: found among the two resident tables or
// built and uploaded (after waiting for stream s, the stream of every launch
// of this FusedFrame, since the slot it replaces may be in use).
int FusedFrame::Impl::table(const std::vector<LevelArgs>& jobs, int nw, int rtop, int rlow, bool inner,
                            hipStream_t s) {
    // launch order: grouped by tile body, stable within a group; every top
    // level precedes every delta level, so producers precede consumers
    std::vector<int> order(jobs.size()), pos(jobs.size());
    for (size_t i = 0; i < jobs.size(); ++i) order[i] = (int)i;
    std::stable_sort(order.begin(), order.end(),
                     [&](int x, int y) { return body_group(jobs[x]) < body_group(jobs[y]); });
    for (size_t i = 0; i < order.size(); ++i) pos[order[i]] = (int)i;
    std::vector<LevelJob> rec(jobs.size());
    int blocks = 0;
    int ends[kGroups - 1] = {0, 0, 0, 0, 0, 0};
    for (size_t i = 0; i < jobs.size(); ++i) {
        const LevelArgs& a = jobs[order[i]];
        const int rows = nw * rows_per_thread(a, rtop, rlow);
        if (!fused_level_supported(a) || !tiles_with(a, rows))
            throw logic_error("fused frame: unsupported level parameters");
        LevelJob& p = rec[i];
        std::memset(&p, 0, sizeof(p));
        p.img = a.img.data;
        p.img_pitch = (int)a.img.pitch;
        p.flow_in = (const float2*)a.flow_s_in.data;
        p.flow_in_pitch = (int)a.flow_s_in.pitch;
        p.a0_in = (const float*)a.a0_in.data;
        p.a0_in_pitch = (int)a.a0_in.pitch;
        p.dflow_in = (const float2*)a.dflow_in.data;
        p.dflow_in_pitch = (int)a.dflow_in.pitch;
        p.flow_out = (float2*)a.flow_s_out.data;
        p.flow_out_pitch = (int)a.flow_s_out.pitch;
        p.a0_out = (float*)a.a0_out.data;
        p.a0_out_pitch = (int)a.a0_out.pitch;
        p.dflow_out = (float2*)a.dflow_out.data;
        p.dflow_out_pitch = (int)a.dflow_out.pitch;
        p.flow_upd = (float2*)a.flow_upd_out.data;
        p.flow_upd_pitch = (int)a.flow_upd_out.pitch;
        p.upper = (const float2*)a.upper.data;
        p.upper_pitch = (int)a.upper.pitch;
        p.xmap = a.xmap;
        p.ymap = a.ymap;
        level_size(a, p.H, p.W);
        p.Hu = a.upper.h;
        p.Hsrc = a.img.h;
        p.N = a.prop_iters;
        p.K = a.smooth_iters;
        p.border = a.border;
        p.h0 = halo_of(a);
        // a level no wider (taller) than the buffer is one tile across (down)
        p.TW = p.W <= LANES ? p.W : LANES - 2 * p.h0;
        p.TH = p.H <= rows ? p.H : rows - 2 * p.h0;
        p.tiles_x = (p.W + p.TW - 1) / p.TW;
        p.tiles_y = (p.H + p.TH - 1) / p.TH;
        p.delta = a.delta;
        p.img_mode = a.img_mode;
        p.first_block = blocks;
        p.wait_job = -1;
        p.flags = -1;
        p.frame_slot = a.frame_slot < kMaxLaunchFrames ? a.frame_slot : -1;
        p.dt = a.dt;
        p.gamma = a.gamma;
        p.maxflow = a.maxflow;
        blocks += p.tiles_x * p.tiles_y;
        for (int g = body_group(a); g < kGroups - 1; ++g) ends[g] = blocks;
    }
    for (size_t i = 0; i < jobs.size(); ++i) {
        const int k = jobs[i].wait_on;
        if (k < 0) continue;
        if (k >= (int)i) throw logic_error("fused frame: a level waits on a later level");
        if (!jobs[i].delta || jobs[k].delta) throw logic_error("fused frame: only delta levels wait on a top level");
        LevelJob& c = rec[pos[i]];
        LevelJob& q = rec[pos[k]];
        // top levels come first, so their block indices are compact
        q.flags = q.first_block;
        c.wait_job = pos[k];
        c.wait_tx = q.tiles_x;
        c.wait_flags = q.flags;
    }
    std::vector<int> map(blocks);
    for (size_t i = 0; i < rec.size(); ++i)
        for (int b = 0; b < rec[i].tiles_x * rec[i].tiles_y; ++b) map[rec[i].first_block + b] = (int)i;
    // the upper level's tiles that each tile row and column waits for: the
    // results of a tile's update reach 2 K pixels further (the smoothing), and
    // the upper flow read beyond that, finished or not, reaches no output
    for (LevelJob& c : rec) {
        if (c.wait_job < 0) continue;
        const LevelJob& q = rec[c.wait_job];
        c.wait_rows = (int)map.size();
        auto ranges = [&](int tiles, int size, int n, int nu, int upper_size) {
            for (int i = 0; i < tiles; ++i) {
                const int lo = std::max(i * size - 2 * c.K, 0), hi = std::min(std::min(i * size + size, n) - 1 + 2 * c.K, n - 1);
                map.push_back(upper_index(lo, n, nu) / upper_size);
                map.push_back(upper_index(hi, n, nu) / upper_size);
            }
        };
        ranges(c.tiles_y, c.TH, c.H, q.H, q.TH);
        ranges(c.tiles_x, c.TW, c.W, q.W, q.TW);
    }

    const size_t jobs_bytes = rec.size() * sizeof(LevelJob);
    const size_t map_offset = (jobs_bytes + 255) & ~size_t(255);
    std::vector<char> key(map_offset + map.size() * sizeof(int), 0);
    std::memcpy(key.data(), rec.data(), jobs_bytes);
    std::memcpy(key.data() + map_offset, map.data(), map.size() * sizeof(int));
    // launch shape: part of the table's identity
    for (int g = 0; g < kGroups - 1; ++g) {
        const char* e = reinterpret_cast<const char*>(&ends[g]);
        key.insert(key.end(), e, e + sizeof(int));
    }
    key.insert(key.end(), reinterpret_cast<const char*>(&nw), reinterpret_cast<const char*>(&nw) + sizeof(int));
    key.insert(key.end(), reinterpret_cast<const char*>(&rtop), reinterpret_cast<const char*>(&rtop) + sizeof(int));
    key.insert(key.end(), reinterpret_cast<const char*>(&rlow), reinterpret_cast<const char*>(&rlow) + sizeof(int));
    key.push_back(inner ? 1 : 0);

    for (int i = 0; i < 2; ++i)
        if (slot[i].key == key) {
            next = i ^ 1;  // the one used less recently is replaced
            return i;
        }

    // a table (or the flags) may be in use by launches still in flight on
    // the stream
    FF_HIP(hipStreamSynchronize(s));
    const int need = ends[3];  // tiles of top levels
    if (nflags < need || !flags.data()) {
        const int n = std::max(need, 256);
        // the timed-out waits counted so far are kept
        watch->stream = s;
        watch->read();
        std::vector<unsigned> zero(2 * (size_t)n + 1, 0u);
        flags.assign(zero.data(), zero.size() * sizeof(unsigned));
        nflags = n;
        watch->retire(timeout_word());
        // launches recorded with the old flags must not be replayed, and the
        // new ones count from the start
        for (Table& o : slot) o.token = ++uploads;
    }
    const int si = next;
    Table& t = slot[si];
    t.dev.assign(key.data(), key.size());
    t.key = std::move(key);
    t.njobs = (int)rec.size();
    t.blocks = blocks;
    t.nw = nw;
    t.rtop = rtop;
    t.rlow = rlow;
    t.inner = inner;
    t.map_offset = map_offset;
    t.awaited = 0;
    for (const LevelJob& r : rec)
        if (r.flags >= 0) t.awaited += r.tiles_x * r.tiles_y;
    for (int g = 0; g < kGroups - 1; ++g) t.ends.e[g] = ends[g];
    t.token = ++uploads;
    next ^= 1;
    return si;
}

void FusedFrame::Impl::clear_flags(int si, hipStream_t s) const {
    const int n = nflags;
    hipLaunchKernelGGL(k_clear_flags, dim3((n + 255) / 256), dim3(256), 0, s, region(si), n);
}

void FusedFrame::Impl::run(int ti, hipStream_t s, const FrameRef* frames, int nframes) {
    const int si = ti & 1;
    const Table& t = slot[si];
    if (!t.blocks) throw logic_error("fused frame: launch of an unprepared table");
    // (the limit of the dynamic LDS is a device's)
    int dev = 0;
    FF_HIP(hipGetDevice(&dev));
    static OncePerDevice once;
    once.run(dev, [] {
        for (const void* k : {(const void*)k_fused_frame<4>, (const void*)k_fused_frame<8>,
                              (const void*)k_fused_frame<4, 4>, (const void*)k_fused_frame<4, 4, true>})
            FF_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes(kMaxWaves)));
    });
    // Sequence number of this launch for its slot's flags. A launch recorded
    // into a graph clears them itself and counts as the first, so every
    // replay is self-contained; direct launches count up from the last
    // clear, which happens whenever the region served another table or a
    // replay (replayed()) in between.
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    FF_HIP(hipStreamIsCapturing(s, &cs));
    unsigned e;
    if (cs != hipStreamCaptureStatusNone) {
        if (t.awaited) clear_flags(si, s);
        e = 1;
        counted[si] = 0;
    } else {
        if (counted[si] != t.token || epoch[si] == 0x3fffffffu) {
            if (t.awaited) clear_flags(si, s);
            epoch[si] = 0;
            counted[si] = t.token;
        }
        e = ++epoch[si];
    }
    const WaitArgs wa = wait_args();
    FrameArgs fa;
    std::memset(&fa, 0, sizeof(fa));
    for (int k = 0; k < nframes; ++k) {
        fa.ptr[k] = (const unsigned char*)frames[k].ptr;
        fa.pitch[k] = (int)frames[k].pitch;
    }
    watch->stream = s;
    if (t.awaited) watch->pending = true;
    const WaitingLaunch order(s, awaited(t));
    ProfileScope ps("fused_frame", s);
    const char* base = (const char*)t.dev.data();
    const TileFlags fl{region(si), timeout_word(), order.started(), e};
    const LaunchArgs args{(const LevelJob*)base, (const int*)(base + t.map_offset), fl, t.ends, t.nw, wa, fa};
    const void* kernel = t.rlow == 4 ? (t.inner ? (const void*)k_fused_frame<4, 4, true> : (const void*)k_fused_frame<4, 4>)
                                     : (t.rtop == 8 ? (const void*)k_fused_frame<8> : (const void*)k_fused_frame<4>);
    void* argv[] = {(void*)&args};
    const hipError_t err = hipLaunchKernel(kernel, dim3(t.blocks), dim3(t.nw * LANES), argv, lds_bytes(t.nw), s);
    if (err != hipSuccess) {
        (void)hipGetLastError();  // reported here
        throw_hip(err, "the fused frame's launch", __FILE__, __LINE__);
    }
    if (cs == hipStreamCaptureStatusNone) order.launched();
}

// Time the launches of every candidate tiling (waves per workgroup and, when
// a job runs a reduced top-level body, its rows per thread) on the actual
// job table and keep the fastest; a fixed choice is not varied. A launch
// reads the current state and writes the next one without committing it, so
// repeated launches recompute the same output; every tiling gives bitwise
// the same results.
void FusedFrame::Impl::tune(const std::vector<LevelArgs>& jobs, hipStream_t s) {
    bool reduced_top = false;
    for (const LevelArgs& a : jobs) reduced_top = reduced_top || top_rows_body(a);
    int best_nw = 0, best_rtop = 0, best_rlow = kRows;
    bool best_inner = false;
    float best_ms = 0.0f;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    FF_HIP(hipEventCreate(&e0));
    FF_HIP(hipEventCreate(&e1));
    try {
        for (const TileShape& sh : kShapes) {
            const int rtop = sh.rtop, rlow = sh.rlow;
            if (fixed_rtop ? rtop != fixed_rtop : (!reduced_top && rtop != kTopRowChoices[0])) continue;
            if (fixed_rlow && rlow != fixed_rlow) continue;
            if (fixed_inner && sh.inner != (fixed_inner == 1)) continue;
            for (int nw : kWaveChoices) {
                if (fixed && nw != fixed) continue;
                // four rows per thread only in the tallest workgroups (the
                // 64-row tiles of eight waves of eight rows)
                if (rlow == 4 && nw < 15) continue;
                bool ok = true;
                for (const LevelArgs& a : jobs) ok = ok && tiles_with(a, nw * rows_per_thread(a, rtop, rlow));
                if (!ok) continue;
                const int t = table(jobs, nw, rtop, rlow, sh.inner, s);
                run(t, s);  // warm-up
                constexpr int kReps = 3;
                FF_HIP(hipEventRecord(e0, s));
                for (int r = 0; r < kReps; ++r) run(t, s);
                FF_HIP(hipEventRecord(e1, s));
                FF_HIP(hipEventSynchronize(e1));
                float ms = 0.0f;
                FF_HIP(hipEventElapsedTime(&ms, e0, e1));
                if (!best_nw || ms < best_ms) {
                    best_nw = nw;
                    best_rtop = rtop;
                    best_rlow = rlow;
                    best_inner = sh.inner;
                    best_ms = ms;
                }
            }
        }
    } catch (...) {
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        throw;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (!best_nw && fixed_inner == 1)
        throw invalid_argument("fused frame: the interior tile body needs four rows per thread and 16 or 15 waves per "
                               "workgroup, which the fixed part of the tiling excludes");
    if (!best_nw) throw logic_error("fused frame: no tiling fits the levels");
    tuned = best_nw;
    tuned_rtop = best_rtop;
    tuned_rlow = best_rlow;
    tuned_inner = best_inner;
}

int FusedFrame::prepare(const std::vector<LevelArgs>& jobs, hipStream_t s) {
    if (jobs.empty()) throw invalid_argument("fused frame: no levels");
    // the rows below the top level default to eight when the tile height
    // and the top rows are both fixed; otherwise the tuner picks them too
    int nw = impl_->fixed, rtop = impl_->fixed_rtop, rlow = impl_->fixed_rlow ? impl_->fixed_rlow : kRows;
    bool inner = impl_->fixed_inner == 1;
    if (rlow == 4 && nw && nw < 15)
        throw invalid_argument("fused frame: four rows per thread need 16 or 15 waves per workgroup, got " +
                               std::to_string(nw));
    if (inner && nw && rtop && rlow != 4)
        throw invalid_argument("fused frame: the interior tile body needs four rows per thread below the top level");
    if (!nw || !rtop) {
        // tuned per set of level shapes and per fixed part of the choice
        std::vector<int> k = tune_key(jobs);
        k.push_back(impl_->fixed);
        k.push_back(impl_->fixed_rtop);
        k.push_back(impl_->fixed_rlow);
        k.push_back(impl_->fixed_inner);
        if (k != impl_->tuned_for || !impl_->tuned) {
            impl_->tune(jobs, s);
            impl_->tuned_for = std::move(k);
        }
        nw = impl_->tuned;
        rtop = impl_->tuned_rtop;
        rlow = impl_->tuned_rlow;
        inner = impl_->tuned_inner;
    }
    return impl_->table(jobs, nw, rtop, rlow, inner, s);
}

void FusedFrame::launch(int table, hipStream_t s, const FrameRef* frames, int nframes) {
    if (nframes < 0 || nframes > kMaxLaunchFrames) throw invalid_argument("fused frame: too many frames in place");
    for (int k = 0; k < nframes; ++k)
        if (frames[k].ptr && (frames[k].pitch > 0x7fffffffu || frames[k].pitch % 4 || (uintptr_t)frames[k].ptr % 4))
            throw invalid_argument("fused frame: a frame in place needs a pitch and address that are multiples of 4 "
                                   "and a pitch below 2^31");
    impl_->run(table, s, frames, nframes);
}

void FusedFrame::replayed(int table, hipStream_t s) {
    impl_->counted[0] = impl_->counted[1] = 0;
    if (!impl_->slot[table & 1].awaited) return;
    impl_->watch->stream = s;
    impl_->watch->pending = true;
}

int FusedFrame::blocks(int table) const { return impl_->slot[table & 1].blocks; }
unsigned long long FusedFrame::token(int table) const { return impl_->slot[table & 1].token; }
AwaitedTiles FusedFrame::awaited(int table) const { return impl_->awaited(impl_->slot[table & 1]); }

void FusedFrame::setWaves(int nw) {
    bool ok = nw == 0;
    for (int c : kWaveChoices) ok = ok || c == nw;
    if (!ok)
        throw invalid_argument("fused frame: waves per workgroup must be 0 (autotune), 16, 15, 8, 5 or 4, got " +
                               std::to_string(nw));
    impl_->fixed = nw;
}

int FusedFrame::waves() const { return impl_->fixed ? impl_->fixed : impl_->tuned; }

void FusedFrame::setTopRows(int rows) {
    bool ok = rows == 0;
    for (int c : kTopRowChoices) ok = ok || c == rows;
    if (!ok)
        throw invalid_argument("fused frame: top-level rows per thread must be 0 (autotune), 4 or 8, got " +
                               std::to_string(rows));
    impl_->fixed_rtop = rows;
}

int FusedFrame::topRows() const { return impl_->fixed_rtop ? impl_->fixed_rtop : impl_->tuned_rtop; }
int FusedFrame::rows() const {
    if (impl_->fixed_rlow) return impl_->fixed_rlow;
    return impl_->fixed && impl_->fixed_rtop ? kRows : impl_->tuned_rlow;
}

void FusedFrame::setInterior(int mode) {
    if (mode < 0 || mode > 2)
        throw invalid_argument("fused frame: interior tile body must be 0 (autotune), 1 (on) or 2 (off), got " +
                               std::to_string(mode));
    impl_->fixed_inner = mode;
}

int FusedFrame::interior() const {
    if (impl_->fixed_inner) return impl_->fixed_inner;
    return impl_->tuned ? (impl_->tuned_inner ? 1 : 2) : 0;
}

void FusedFrame::setRows(int rows) {
    if (rows != 0 && rows != 4 && rows != 8)
        throw invalid_argument("fused frame: rows per thread must be 0 (autotune), 4 or 8, got " +
                               std::to_string(rows));
    impl_->fixed_rlow = rows;
}

unsigned long long FusedFrame::timeouts() const { return impl_->watch->read(); }

const std::shared_ptr<WaitWatch>& FusedFrame::watch() const { return impl_->watch; }

void FusedFrame::setWaitTest(int spins) {
    if (spins < 0) throw invalid_argument("fused frame: wait test spins must be >= 0");
    impl_->test_spins = spins;
}

int FusedFrame::waitTest() const { return impl_->test_spins; }

// ------------------------------------------------------------- WaitWatch

WaitWatch::~WaitWatch() {
    if (host) (void)hipHostFree(host);
}

unsigned long long WaitWatch::read() {
    if (!pending || !word) return total;
    if (!host) FF_HIP(hipHostMalloc((void**)&host, sizeof(unsigned), hipHostMallocDefault));
    FF_HIP(hipMemcpyAsync(host, word, sizeof(unsigned), hipMemcpyDeviceToHost, stream));
    FF_HIP(hipStreamSynchronize(stream));
    total = base + *host;
    pending = false;
    return total;
}

void WaitWatch::retire(const unsigned* next) {
    base = total;
    word = next;
}

void WaitCheck::follow(const std::shared_ptr<WaitWatch>& w) {
    if (watch == w) return;
    watch = w;
    seen = w ? w->total : 0;
}

void WaitCheck::check(const char* who) {
    if (!watch) return;
    const unsigned long long n = watch->read();
    if (n > seen) {
        const unsigned long long d = n - seen;
        seen = n;
        throw runtime_error(std::string(who) + ": " + std::to_string(d) +
                            " wait(s) of the fused frame kernel (for the level above, or for a launch on another "
                            "stream) gave up after the spin limit since the last check; the flow of those frames is "
                            "not valid");
    }
}

}  // namespace ffamd
