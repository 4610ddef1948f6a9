// Observation pre-/post-processing either side of the forward pass, on the device:
// /root/reference/test.py:88-201 (`_resize_with_pad`, `_normalize_image`, `_normalize_state`, `_digitize_state`,
// `_unnormalize_actions`, and the delta-to-absolute step of `infer`), which the reference runs in numpy / Pillow on
// the host per observation.
//
// The resize reproduces Pillow's `Image.resize(..., BILINEAR)` bit for bit: triangle filter with the support stretched
// by the shrink factor, double-precision weights normalised per output pixel, 22-bit fixed point, a horizontal pass to
// an 8-bit intermediate and a vertical pass, each rounded to nearest and clipped.  The weights are derived in the kernel
// (a dozen double operations per tap), so there are no coefficient tables to upload and the kernels can be captured in a
// graph.  This file is compiled with floating-point contraction off: a fused
// multiply-add would round the weights differently from the C code being matched.
#include "../../include/rtvla.h"
#include "kernels.h"
#include <atomic>
#include <math.h>

namespace {

constexpr int PRECISION_BITS = 32 - 8 - 2;
constexpr int MAX_TAPS = 64;            // ceil(scale) * 2 + 1 taps: shrink factors up to 31

struct Window { int first, count; double center, ss, ww; };

// one direction of a resize (Resample.c: precompute_coeffs): source pixels per output pixel, reach of the filter and its reciprocal
struct Axis { double scale, support, ss; int in; };

RTVLA_DEVICE void window_bounds(const Axis& d, int xx, int* first, int* end) {
    const double center = 0.0 + (xx + 0.5) * d.scale;
    const int xmin = (int)(center - d.support + 0.5), xmax = (int)(center + d.support + 0.5);
    *first = xmin < 0 ? 0 : xmin; *end = xmax > d.in ? d.in : xmax;
}
// the source window and weight sum of output index xx
RTVLA_DEVICE Window window_of(const Axis& d, int xx) {
    Window w;
    int end;
    window_bounds(d, xx, &w.first, &end);
    w.center = 0.0 + (xx + 0.5) * d.scale;
    w.ss = d.ss;
    w.count = end - w.first;
    double ww = 0.0;
    for (int x = 0; x < w.count; ++x) {
        double a = (x + w.first - w.center + 0.5) * w.ss;
        if (a < 0.0) a = -a;
        ww += a < 1.0 ? 1.0 - a : 0.0;
    }
    w.ww = ww;
    return w;
}

RTVLA_DEVICE int tap_weight(const Window& w, int x) {
    double a = (x + w.first - w.center + 0.5) * w.ss;
    if (a < 0.0) a = -a;
    double k = a < 1.0 ? 1.0 - a : 0.0;
    if (w.ww != 0.0) k /= w.ww;
    return k < 0 ? (int)(-0.5 + k * (double)(1 << PRECISION_BITS)) : (int)(0.5 + k * (double)(1 << PRECISION_BITS));
}

RTVLA_DEVICE int clip8(int v) { v >>= PRECISION_BITS; return v < 0 ? 0 : (v > 255 ? 255 : v); }

// One launch per frame: resize, pad, x / 255 * 2 - 1 -> bf16 NHWC.  A workgroup owns 32 x TH pixels of the 224 x 224 canvas.  It derives
// the weights of its 32 columns and TH rows once (one thread per tap, into LDS), resamples the source rows its output rows need
// across into an 8-bit LDS tile, and that tile down into the output.  Neighbouring row blocks resample the rows they share twice
// ((TH + 2) / TH of the work for TH output rows); in exchange nothing but the frame is read and nothing but the result written, and the
// second launch with its round trip through memory is gone.  Measured (480 x 640 uint8, one frame): two launches, each thread deriving the
// weights of its own pixel, 11.7 us; this one 4.4 us.  TH = 4 gives large frames (many taps per pixel) twice the workgroups.
enum FrameFormat { FRAME_U8_HWC = 0, FRAME_F32_HWC, FRAME_F32_CHW, FRAME_U8_CHW };
constexpr int TW = 32;                      // columns of a workgroup
// Threads: a thread takes a column of every (threads / TW)-th source row, and all wait for the loads of one row before those of their next.  With 1 024 instead of 512 a frame of bytes
// of 300 x 400, 480 x 640, 719 x 1 279, 1 080 x 1 920 takes 3.99, 4.38, 5.45, 7.4 instead of 3.90, 4.56, 5.63, 8.6 us: from 24 source rows a block on (the first has 22, the second 30).
// Not so where the blocks that hold a part of the picture are more than the CUs and have many rows: 1 920 x 1 920 (47 rows) 9.1 / 9.9, 2 448 x 2 448 (58) 11.9 / 12.0, 2 160 x 2 880 (68) 15.6 / 14.4,
// 3 000 x 4 000 (95) 27.3 / 24.6, channels first 42.8 / 38.5; 2 250 x 4 000 (95 as well, 224 blocks) 17.0 / 20.3.  Nor for float frames that are not staged: 1 440 x 2 560 37.4 / 33.9, 2 160 x 3 840
// 105 / 92, channels first 68 / 63.
// Staged float frames, whose loads are all on the way at once and whose bytes it converts: 4.43, 4.91, 7.24, 10.8 instead of 4.58, 5.60, 8.30, 12.8 (1 200 x 1 600 13.4 instead of 13.2).
// (All figures of this file: launches in a graph, four frames in turn.)
constexpr int NT_MANY_ROWS = 24, NT_TOO_MANY_ROWS = 60, CUS = 256, STAGED_NT = 1024;
struct FrameP { const uint8_t* src; int h, w, rw, rh, pad_top, pad_left, taps_x, taps_y, max_rows, pitch; bf16_t* dst; Axis x, y; };      // taps: rounded up to 4

// numpy's / torch's float -> uint8: truncation to an integer, low byte
RTVLA_DEVICE int to_u8(float x) {
    const float v = 255.0f * x;
    int i = (int)v;
    if (__builtin_expect(!(fabsf(v) < 2147483648.0f), 0)) i = (int)(long long)v;
    return i & 255;
}
// four consecutive values, any alignment of 4 bytes; one load unless it would reach past `end`
RTVLA_DEVICE f32x4 load_f4(const float* q, const float* end) {
    f32x4 v;
    if (q + 4 <= end) __builtin_memcpy(&v, q, 16);
    else for (int i = 0; i < 4; ++i) v[i] = q + i < end ? q[i] : 0.f;
    return v;
}

// the second pass, of the 8-bit tile down into the output
template <int TH>
RTVLA_DEVICE void resize_down(const FrameP& p, const Window* win, const bf16_t* value, const int* wy, const unsigned* inter, int lo, int count, int tid, int x0, int y0) {
    const int c = tid & (TW - 1);
    const int rr = tid / TW;
    if (rr >= TH) return;
    int v0 = 0, v1 = 0, v2 = 0;
    const int vfirst = win[TW + rr].first - lo, vcount = win[TW + rr].count;
    if (count > 0 && vcount > 0) {
        int a0 = 1 << (PRECISION_BITS - 1), a1 = a0, a2 = a0;
        for (int t = 0; t < vcount; t += 4)                                    // (past the window: zero weights, and rows that `inter` has room for)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const unsigned e = inter[(vfirst + t + i) * TW + c];
                const int k = wy[(t + i) * TH + rr];
                a0 += __mul24(e & 255, k); a1 += __mul24((e >> 8) & 255, k); a2 += __mul24((e >> 16) & 255, k);
            }
        v0 = clip8(a0); v1 = clip8(a1); v2 = clip8(a2);
    }
    bf16_t* o = p.dst + ((size_t)(y0 + rr) * 224 + x0 + c) * 3;
    o[0] = value[v0]; o[1] = value[v1]; o[2] = value[v2];
}

// Float frames, whose values cost six instructions each to become bytes: the source rectangle of the block is loaded in whole lines, converted once and
// staged in LDS as dwords R G B - (windows overlap by half, and four-tap groups round them up, so resize_kernel loads and converts each value 2.8 times);
// the first loads are on the way while the weights are derived.  us per frame of 300 x 400, 480 x 640, 719 x 1 279, 1 080 x 1 920: 4.8, 6.3, 10.9, 18.3
// without and 4.4, 4.9, 7.25, 10.8 with (1.6 of it the launch).  Frames that are not reduced (4 taps) are as fast or faster without (224 x 224
// 3.8 / 4.0 when this was introduced), as are bytes (480 x 640 4.3 / 4.65), and rectangles of more than half a CU's LDS stay with resize_kernel.
struct Raw4 { f32x4 v[3]; };
template <int FMT>
RTVLA_DEVICE Raw4 load_px4(const FrameP& p, size_t at) {                       // four consecutive pixels; zero past the frame
    Raw4 r;
    const size_t plane = (size_t)p.h * p.w;
    const float* const f = (const float*)p.src;
#pragma unroll
    for (int i = 0; i < 3; ++i) r.v[i] = load_f4(FMT == FRAME_F32_CHW ? f + i * plane + at : f + at * 3 + 4 * i, f + 3 * plane);
    return r;
}
template <int FMT>
RTVLA_DEVICE uint4 px4(const Raw4& r) {
    unsigned o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        unsigned c[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) c[j] = FMT == FRAME_F32_CHW ? to_u8(r.v[j][i]) : to_u8(r.v[(3 * i + j) >> 2][(3 * i + j) & 3]);
        o[i] = c[0] | c[1] << 8 | c[2] << 16;
    }
    return uint4{o[0], o[1], o[2], o[3]};
}

template <int FMT, int TH>
__global__ __launch_bounds__(STAGED_NT) void resize_staged_kernel(FrameP p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    int4* const wx = (int4*)smem;                                              // [taps_x / 4][TW]
    unsigned* const stage = (unsigned*)(wx + (p.taps_x >> 2) * TW);            // [row][pitch] pixels as dwords
    int* const wy = (int*)(stage + p.max_rows * p.pitch);                      // [taps_y][TH]
    unsigned* const inter = (unsigned*)(wy + p.taps_y * TH);                   // [row][TW], three bytes each
    __shared__ Window win[TW + TH];
    __shared__ bf16_t value[256];
    constexpr int NT = STAGED_NT;
    const int tid = threadIdx.x, x0 = blockIdx.x * TW, y0 = blockIdx.y * TH;
    // the source rectangle of this block
    const int rx0 = max(x0 - p.pad_left, 0), rx1 = min(x0 + TW - p.pad_left, p.rw) - 1, ry0 = max(y0 - p.pad_top, 0), ry1 = min(y0 + TH - p.pad_top, p.rh) - 1;
    int lo_x = 0, hi_x = 0, lo = 0, hi = 0, skip;
    if (rx0 <= rx1 && ry0 <= ry1) {
        window_bounds(p.x, rx0, &lo_x, &skip); window_bounds(p.x, rx1, &skip, &hi_x);
        window_bounds(p.y, ry0, &lo, &skip); window_bounds(p.y, ry1, &skip, &hi);
    }
    const int groups = (hi_x - lo_x + 3) >> 2, items = (hi - lo) * groups;
    constexpr int UN = 2;
    Raw4 raw[UN];
    auto pixel = [&](int i) { return (size_t)(lo + i / groups) * p.w + lo_x + 4 * (i % groups); };
#pragma unroll
    for (int j = 0; j < UN; ++j) if (tid + j * NT < items) raw[j] = load_px4<FMT>(p, pixel(tid + j * NT));
    if (tid < 256) value[tid] = f2bf((float)tid / 255.0f * 2.0f - 1.0f);
    if (tid < TW) {
        const int rx = x0 + tid - p.pad_left;
        if (rx >= 0 && rx < p.rw) win[tid] = window_of(p.x, rx); else { win[tid] = Window{}; win[tid].count = 0; }
    } else if (tid >= 64 && tid < 64 + TH) {
        const int ry = y0 + tid - 64 - p.pad_top;
        if (ry >= 0 && ry < p.rh) win[TW + tid - 64] = window_of(p.y, ry); else { win[TW + tid - 64] = Window{}; win[TW + tid - 64].count = 0; }
    }
    __syncthreads();
    for (int i = tid; i < p.taps_x * TW; i += NT) {
        const int c = i % TW, t = i / TW;
        ((int*)wx)[((t >> 2) * TW + c) * 4 + (t & 3)] = t < win[c].count ? tap_weight(win[c], t) : 0;
    }
    for (int i = tid; i < p.taps_y * TH; i += NT) {
        const int rr = i % TH, t = i / TH;
        wy[i] = t < win[TW + rr].count ? tap_weight(win[TW + rr], t) : 0;
    }
    for (int i0 = 0; i0 < items; i0 += UN * NT) {
        if (i0)
#pragma unroll
            for (int j = 0; j < UN; ++j) if (tid + j * NT + i0 < items) raw[j] = load_px4<FMT>(p, pixel(tid + j * NT + i0));
#pragma unroll
        for (int j = 0; j < UN; ++j) {
            const int i = tid + j * NT + i0;
            if (i < items) *(uint4*)(stage + (i / groups) * p.pitch + 4 * (i % groups)) = px4<FMT>(raw[j]);
        }
    }
    __syncthreads();
    const int c = tid & (TW - 1), first = win[c].first - lo_x, count = win[c].count;
    if (count > 0)
        for (int row = tid >> 5; row < hi - lo; row += NT / TW) {
            int a0 = 1 << (PRECISION_BITS - 1), a1 = a0, a2 = a0;
            const unsigned* const e = stage + row * p.pitch + first;
            for (int t = 0; t < count; t += 4) {                               // (past the window: zero weights, pixels of the slack behind the row at most)
                const int4 k4 = wx[(t >> 2) * TW + c];
                const int k[4] = {k4.x, k4.y, k4.z, k4.w};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const unsigned u = e[t + i];
                    a0 += __mul24(u & 255, k[i]); a1 += __mul24((u >> 8) & 255, k[i]); a2 += __mul24((u >> 16) & 255, k[i]);
                }
            }
            inter[row * TW + c] = (unsigned)clip8(a0) | (unsigned)clip8(a1) << 8 | (unsigned)clip8(a2) << 16;
        }
    __syncthreads();
    resize_down<TH>(p, win, value, wy, inter, lo, count, tid, x0, y0);
}

template <int FMT, int TH, int NT>
__global__ __launch_bounds__(NT) void resize_kernel(FrameP p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    int4* const wx = (int4*)smem;                                              // [taps_x / 4][TW]
    int* const wy = (int*)(wx + (p.taps_x >> 2) * TW);                         // [taps_y][TH]
    unsigned* const inter = (unsigned*)(wy + p.taps_y * TH);                   // [row][TW], three bytes each
    __shared__ Window win[TW + TH];
    __shared__ bf16_t value[256];
    const int tid = threadIdx.x, x0 = blockIdx.x * TW, y0 = blockIdx.y * TH;
    if (tid < 256) value[tid] = f2bf((float)tid / 255.0f * 2.0f - 1.0f);
    if (tid < TW) {
        const int rx = x0 + tid - p.pad_left;
        if (rx >= 0 && rx < p.rw) win[tid] = window_of(p.x, rx); else { win[tid] = Window{}; win[tid].count = 0; }
    } else if (tid >= 64 && tid < 64 + TH) {
        const int ry = y0 + tid - 64 - p.pad_top;
        if (ry >= 0 && ry < p.rh) win[TW + tid - 64] = window_of(p.y, ry); else { win[TW + tid - 64] = Window{}; win[TW + tid - 64].count = 0; }
    }
    __syncthreads();
    for (int i = tid; i < p.taps_x * TW; i += NT) {
        const int c = i % TW, t = i / TW;
        ((int*)wx)[((t >> 2) * TW + c) * 4 + (t & 3)] = t < win[c].count ? tap_weight(win[c], t) : 0;
    }
    for (int i = tid; i < p.taps_y * TH; i += NT) {
        const int rr = i % TH, t = i / TH;
        wy[i] = t < win[TW + rr].count ? tap_weight(win[TW + rr], t) : 0;
    }
    // source rows of this block: the windows move down with the output row
    int lo = 1 << 30, hi = 0;
#pragma unroll
    for (int i = 0; i < TH; ++i)
        if (win[TW + i].count > 0) { lo = min(lo, win[TW + i].first); hi = max(hi, win[TW + i].first + win[TW + i].count); }
    __syncthreads();
    const int c = tid & (TW - 1), first = win[c].first, count = win[c].count;
    const uintptr_t last = ((uintptr_t)p.src + (size_t)p.h * p.w * 3 - 1) & ~(uintptr_t)3;      // uint8: the dword that holds the last byte
    if (count > 0)
        for (int row = tid >> 5; row < hi - lo; row += NT / TW) {
            int a0 = 1 << (PRECISION_BITS - 1), a1 = a0, a2 = a0;
            const size_t at = (size_t)(lo + row) * p.w + first;
            if constexpr (FMT == FRAME_U8_CHW) {
                const size_t plane = (size_t)p.h * p.w;
                for (int t = 0; t < count; ++t) {
                    const int k = ((const int*)wx)[((t >> 2) * TW + c) * 4 + (t & 3)];
                    a0 += __mul24((int)p.src[at + t], k); a1 += __mul24((int)p.src[plane + at + t], k); a2 += __mul24((int)p.src[2 * plane + at + t], k);
                }
            } else {
                // Four taps at a time, and the loads of UN such groups before the first is used: with 1 - 2 workgroups per CU the pass is bound
                // by the latency of its loads.  What lies past the window has zero weight.
                constexpr int UN = 4;
                for (int t0 = 0; t0 < p.taps_x; t0 += 4 * UN) {
                    f32x4 v[UN][3];
#pragma unroll
                    for (int j = 0; j < UN; ++j) {
                        const int t = t0 + 4 * j;
                        if (t >= p.taps_x) break;
                        if constexpr (FMT == FRAME_U8_HWC) {                   // 12 bytes, as the dwords they lie in
                            const uintptr_t q = ((uintptr_t)p.src + at * 3 & ~(uintptr_t)3) + t * 3;
                            if (q + 12 <= last) __builtin_memcpy(&v[j][0], (const void*)q, 16);
                            else
#pragma unroll
                                for (int i = 0; i < 4; ++i) v[j][0][i] = *(const float*)min(q + 4 * i, last);
                        } else {
                            const float* const f = (const float*)p.src;
                            const size_t plane = (size_t)p.h * p.w;
#pragma unroll
                            for (int i = 0; i < 3; ++i) v[j][i] = load_f4(FMT == FRAME_F32_CHW ? f + i * plane + at + t : f + (at + t) * 3 + 4 * i, f + 3 * plane);
                        }
                    }
#pragma unroll
                    for (int j = 0; j < UN; ++j) {
                        const int t = t0 + 4 * j;
                        if (t >= p.taps_x) break;
                        const int4 k = wx[(t >> 2) * TW + c];
                        int u[3][4];
                        if constexpr (FMT == FRAME_U8_HWC) {
                            const unsigned sh = (unsigned)(((uintptr_t)p.src + at * 3) & 3);
                            unsigned e[3];
#pragma unroll
                            for (int i = 0; i < 3; ++i) e[i] = __builtin_amdgcn_alignbyte(__float_as_uint(v[j][0][i + 1]), __float_as_uint(v[j][0][i]), sh);
#pragma unroll
                            for (int i = 0; i < 12; ++i) u[i % 3][i / 3] = (e[i >> 2] >> 8 * (i & 3)) & 255;
                        } else {
#pragma unroll
                            for (int i = 0; i < 12; ++i) {
                                if constexpr (FMT == FRAME_F32_CHW) u[i >> 2][i & 3] = to_u8(v[j][i >> 2][i & 3]);
                                else u[i % 3][i / 3] = to_u8(v[j][i >> 2][i & 3]);
                            }
                        }
                        a0 += __mul24(u[0][0], k.x) + __mul24(u[0][1], k.y) + __mul24(u[0][2], k.z) + __mul24(u[0][3], k.w);
                        a1 += __mul24(u[1][0], k.x) + __mul24(u[1][1], k.y) + __mul24(u[1][2], k.z) + __mul24(u[1][3], k.w);
                        a2 += __mul24(u[2][0], k.x) + __mul24(u[2][1], k.y) + __mul24(u[2][2], k.z) + __mul24(u[2][3], k.w);
                    }
                }
            }
            inter[row * TW + c] = (unsigned)clip8(a0) | (unsigned)clip8(a1) << 8 | (unsigned)clip8(a2) << 16;
        }
    __syncthreads();
    resize_down<TH>(p, win, value, wy, inter, lo, count, tid, x0, y0);
}

// state: mode 0 (Pi0) (x - a) / (b + 1e-6), a = mean, b = std; mode 1 (Pi05) (x - a) / (b - a + 1e-6) * 2 - 1, a = q01, b = q99
// (statistics and state zero-padded to 32 like _pad_to_dim); then float32 -> bf16 for the model and the 256-bin index
// This launch and the next are bound by the host: one structure instead of ten arguments takes 0.15 - 0.9 us off a call (3.2 - 4.2 us, by the CPU's clock).
struct State32 { double v[32]; };      // a state handed over by value: no copy to the device, no synchronisation
struct StateP { const double *state, *a, *b; bf16_t* out_bf16; double* out_f64; int32_t* bins; int n, n_stats, mode; State32 by_value; };
__global__ void state_kernel(StateP p) {
    const int i = threadIdx.x;
    if (i >= 32) return;
    const double x = i < p.n ? (p.state ? p.state[i] : p.by_value.v[i]) : 0.0, av = i < p.n_stats ? p.a[i] : 0.0, bv = i < p.n_stats ? p.b[i] : 0.0;
    const double z = p.mode == 0 ? (x - av) / (bv + 1e-6) : (x - av) / (bv - av + 1e-6) * 2.0 - 1.0;
    if (p.out_f64) p.out_f64[i] = z;
    if (p.out_bf16) p.out_bf16[i] = f2bf((float)z);
    if (p.bins) {
        // np.digitize(z, linspace(-1, 1, 257)[:-1]) - 1: number of edges <= z, minus one; edge j is what
        // numpy's linspace yields: -1 + j * (2 / 256) (the step is exact in binary)
        // (by bisection: 256 comparisons one after another were 3.8 of the launch's 5.4 us)
        auto below = [&](int j) { return (-1.0 + j * (2.0 / 256.0)) <= z; };
        int cnt = 0;
#pragma unroll
        for (int s = 128; s; s >>= 1) cnt += below(cnt + s - 1) ? s : 0;
        cnt += cnt == 255 && below(255);
        p.bins[i] = cnt - 1;
    }
}

// actions: bf16 [chunk][32] -> float32 -> un-normalise in double -> first action_dim columns + state, gripper columns
// (every 7th) get the state taken off again, exactly in the reference's order of operations
struct ActionsP { const bf16_t* actions; const double *a, *b, *state; double* out; int chunk, n_stats, mode, action_dim; State32 by_value; };
__global__ void actions_kernel(ActionsP p) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= p.chunk * p.action_dim) return;
    const int r = idx / p.action_dim, d = idx - r * p.action_dim;
    const float x = bf2f(p.actions[r * 32 + d]);
    const double av = d < p.n_stats ? p.a[d] : 0.0, bv = d < p.n_stats ? p.b[d] : 0.0;
    double v;
    if (p.mode == 0) v = (double)x * (bv + 1e-6) + av;                               // a = mean, b = std
    else v = (double)((x + 1.0f) / 2.0f) * (bv - av + 1e-6) + av;                  // a = q01, b = q99; (x + 1) / 2 stays float32
    const double ori = p.state ? p.state[d] : p.by_value.v[d];
    v = v + ori;
    if (d % 7 == 6 && d < (p.action_dim / 7) * 7) v = v - ori;
    p.out[idx] = v;
}

// geometry of test.py:105-116 (Python float arithmetic = C double arithmetic) and limits
int frame_plan(int height, int width, FrameP* p) {
    if (height <= 0 || width <= 0) return RTVLA_ERR_ARG;
    p->h = height; p->w = width; p->rh = p->rw = 224; p->pad_top = p->pad_left = 0;
    if (!(width == 224 && height == 224)) {
        const double rwf = (double)width / 224, rhf = (double)height / 224;
        const double ratio = rwf > rhf ? rwf : rhf;
        p->rh = (int)((double)height / ratio); p->rw = (int)((double)width / ratio);
        p->pad_top = (int)((double)(224 - p->rh) / 2); if (p->pad_top < 0) p->pad_top = 0;
        p->pad_left = (int)((double)(224 - p->rw) / 2); if (p->pad_left < 0) p->pad_left = 0;
    }
    if (p->rh < 1 || p->rw < 1 || p->rh > 224 || p->rw > 224) return RTVLA_ERR_ARG;
    const double sx = (double)width / p->rw, sy = (double)height / p->rh;
    const int tx = (int)ceil(sx > 1.0 ? sx : 1.0) * 2 + 1, ty = (int)ceil(sy > 1.0 ? sy : 1.0) * 2 + 1;
    if (tx > MAX_TAPS || ty > MAX_TAPS) return RTVLA_ERR_LIMIT;
    p->taps_x = (tx + 3) & ~3; p->taps_y = (ty + 3) & ~3;
    p->x = Axis{sx, sx < 1.0 ? 1.0 : sx, 1.0 / (sx < 1.0 ? 1.0 : sx), width};
    p->y = Axis{sy, sy < 1.0 ? 1.0 : sy, 1.0 / (sy < 1.0 ? 1.0 : sy), height};
    return RTVLA_OK;
}

constexpr size_t STAGED_LDS = 76 * 1024;     // two workgroups to a CU
template <int FMT, int TH>
void launch_resize(FrameP p, hipStream_t s) {
    const double sy = (double)p.h / p.rh;
    p.max_rows = (int)((TH - 1) * sy) + p.taps_y + 2;                          // first row of the first window to the last row of the last
    const size_t smem = (size_t)p.taps_x * TW * 4 + (size_t)p.taps_y * TH * 4 + (size_t)p.max_rows * TW * 4;
    // first pixel of the first window to the last of the last, whole groups of four, and the groups that a last window's taps are read in
    p.pitch = ((int)((TW - 1) * ((double)p.w / p.rw)) + p.taps_x + 2 + 3) / 4 * 4 + 4;
    const size_t staged = smem + (size_t)p.max_rows * p.pitch * 4;
    if constexpr (FMT == FRAME_F32_HWC || FMT == FRAME_F32_CHW)
        if (p.taps_x > 4 && staged <= STAGED_LDS) {
            auto kern = resize_staged_kernel<FMT, TH>;
            static std::atomic<uint64_t> done{0};
            if (ensure_dynamic_lds((const void*)kern, STAGED_LDS, done) == 0) { hipLaunchKernelGGL(kern, dim3(224 / TW, 224 / TH), dim3(STAGED_NT), staged, s, p); return; }
            (void)hipGetLastError();                                           // (the refusal is not an error of the launch below, which needs no more than the default)
        }
    if constexpr (FMT == FRAME_U8_HWC || FMT == FRAME_U8_CHW) {
        auto blocks = [](int pad, int n, int per) { return (pad + n - 1) / per - pad / per + 1; };
        if (p.max_rows > NT_MANY_ROWS && (p.max_rows <= NT_TOO_MANY_ROWS || blocks(p.pad_left, p.rw, TW) * blocks(p.pad_top, p.rh, TH) <= CUS)) {
            hipLaunchKernelGGL((resize_kernel<FMT, TH, 1024>), dim3(224 / TW, 224 / TH), dim3(1024), smem, s, p);
            return;
        }
    }
    hipLaunchKernelGGL((resize_kernel<FMT, TH, 512>), dim3(224 / TW, 224 / TH), dim3(512), smem, s, p);
}
template <int FMT>
int launch_frame(const FrameP& p, hipStream_t s) {
    // more than 8 rows of source per output row or column: the across pass dominates, twice the workgroups share it (and LDS stays below 64 KB)
    if (p.taps_x > 12 || p.taps_y > 12) launch_resize<FMT, 4>(p, s); else launch_resize<FMT, 8>(p, s);
    return hipGetLastError() == hipSuccess ? RTVLA_OK : RTVLA_ERR_DEVICE;
}
int preprocess_frame_impl(const void* src, int format, int height, int width, void* dst_bf16, void* stream) {
    if (!src || !dst_bf16) return RTVLA_ERR_ARG;
    FrameP p{};
    if (int rc = frame_plan(height, width, &p)) return rc;
    p.src = (const uint8_t*)src; p.dst = (bf16_t*)dst_bf16;
    switch (format) {
        case FRAME_U8_HWC: return launch_frame<FRAME_U8_HWC>(p, (hipStream_t)stream);
        case FRAME_F32_HWC: return launch_frame<FRAME_F32_HWC>(p, (hipStream_t)stream);
        case FRAME_F32_CHW: return launch_frame<FRAME_F32_CHW>(p, (hipStream_t)stream);
        case FRAME_U8_CHW: return launch_frame<FRAME_U8_CHW>(p, (hipStream_t)stream);
    }
    return RTVLA_ERR_ARG;
}

int launch_state(const double* dev, const double* host, int n, const double* stat_a, const double* stat_b, int n_stats, int mode, void* out_bf16, double* out_f64,
                 int32_t* out_bins, void* stream) {
    if ((!dev && !host) || !stat_a || !stat_b || n < 0 || n > 32 || n_stats < 0 || n_stats > 32 || (mode != 0 && mode != 1)) return RTVLA_ERR_ARG;
    StateP p{dev, stat_a, stat_b, (bf16_t*)out_bf16, out_f64, out_bins, n, n_stats, mode, {}};
    if (!dev) for (int i = 0; i < n; ++i) p.by_value.v[i] = host[i];
    hipLaunchKernelGGL(state_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, p);
    return hipGetLastError() == hipSuccess ? RTVLA_OK : RTVLA_ERR_DEVICE;
}

int launch_actions(const void* actions_bf16, int chunk, const double* stat_a, const double* stat_b, int n_stats, int mode, const double* dev, const double* host, int n_state,
                   int action_dim, double* out, void* stream) {
    if (!actions_bf16 || !stat_a || !stat_b || (!dev && !host) || !out || chunk <= 0 || action_dim <= 0 || action_dim > 32 || n_stats < 0 || n_stats > 32 ||
        n_state < 0 || n_state > 32 || (mode != 0 && mode != 1)) return RTVLA_ERR_ARG;
    ActionsP p{(const bf16_t*)actions_bf16, stat_a, stat_b, dev, out, chunk, n_stats, mode, action_dim, {}};
    if (!dev) for (int i = 0; i < n_state; ++i) p.by_value.v[i] = host[i];
    const int n = chunk * action_dim;
    hipLaunchKernelGGL(actions_kernel, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, p);
    return hipGetLastError() == hipSuccess ? RTVLA_OK : RTVLA_ERR_DEVICE;
}

}  // namespace

extern "C" {

size_t rtvla_preprocess_image_scratch(int height, int width) {
    if (height <= 0 || width <= 0) return 0;
    return ((size_t)height * 224 * 3 + 255) & ~(size_t)255;       // (kept for callers of the ABI: the kernel has no intermediate in memory any more)
}

int rtvla_preprocess_frame(const void* src, int format, int height, int width, void* dst_bf16, void* stream) {
    return preprocess_frame_impl(src, format, height, width, dst_bf16, stream);
}

int rtvla_preprocess_image(const void* src_u8, int height, int width, void* dst_bf16, void* scratch_arg, size_t scratch_bytes, void* stream) {
    if (!scratch_arg || !src_u8 || !dst_bf16) return RTVLA_ERR_ARG;
    FrameP p{};
    if (int rc = frame_plan(height, width, &p)) return rc;
    if (scratch_bytes < (size_t)height * p.rw * 3) return RTVLA_ERR_SIZE;
    return preprocess_frame_impl(src_u8, FRAME_U8_HWC, height, width, dst_bf16, stream);
}

int rtvla_preprocess_image_static(const void* src_u8, int height, int width, void* dst_bf16, void* stream) {
    if (!src_u8 || !dst_bf16) return RTVLA_ERR_ARG;
    FrameP p{};
    if (int rc = frame_plan(height, width, &p)) return rc;
    if ((size_t)height * p.rw * 3 > (size_t)RTVLA_STATIC_SCRATCH_BYTES) return RTVLA_ERR_LIMIT;
    return preprocess_frame_impl(src_u8, FRAME_U8_HWC, height, width, dst_bf16, stream);
}

int rtvla_preprocess_state(const double* state, int n, const double* stat_a, const double* stat_b, int n_stats, int mode,
                           void* out_bf16, double* out_f64, int32_t* out_bins, void* stream) {
    return launch_state(state, nullptr, n, stat_a, stat_b, n_stats, mode, out_bf16, out_f64, out_bins, stream);
}

int rtvla_preprocess_state_host(const double* state_host, int n, const double* stat_a, const double* stat_b, int n_stats, int mode,
                                void* out_bf16, double* out_f64, int32_t* out_bins, void* stream) {
    return launch_state(nullptr, state_host, n, stat_a, stat_b, n_stats, mode, out_bf16, out_f64, out_bins, stream);
}

int rtvla_postprocess_actions(const void* actions_bf16, int chunk, const double* stat_a, const double* stat_b, int n_stats, int mode,
                              const double* ori_state, int action_dim, double* out, void* stream) {
    return launch_actions(actions_bf16, chunk, stat_a, stat_b, n_stats, mode, ori_state, nullptr, 0, action_dim, out, stream);
}

int rtvla_postprocess_actions_host(const void* actions_bf16, int chunk, const double* stat_a, const double* stat_b, int n_stats, int mode,
                                   const double* state_host, int n_state, int action_dim, double* out, void* stream) {
    return launch_actions(actions_bf16, chunk, stat_a, stat_b, n_stats, mode, nullptr, state_host, n_state, action_dim, out, stream);
}

}  // extern "C"
