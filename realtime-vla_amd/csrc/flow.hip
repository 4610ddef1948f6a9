// The action expert's flow-matching loop as ONE resident kernel (replaces the decoder-side launches of
// /root/reference/pi0_infer.py:886-1230, pi05_infer.py:22-523 and dm0_infer.py:763-872).
//
// With at most 128 rows every GEMM of the loop is a few microseconds of latency: as launches, a layer is six dependent ones that
// cost 2.3 us each before they do anything, and every one of them starts with cold L2s, because an XCD's L2 does not carry lines
// across a launch boundary.  Here 256 workgroups, one per CU, stay resident for the whole loop and meet at barriers instead.
//
// Split of the work: the 8 XCDs are the ranks of a tensor-parallel group.  XCD x owns query head x (Pi0 / Pi05: 8 heads, one K/V head
// whose new rows every XCD computes for itself; DM0: K/V head x with its two query heads) and one eighth of the MLP's hidden columns.
// Everything an XCD produces for itself (q, k, v, probabilities, attention output, hidden, the residual stream) stays in memory that
// only this XCD touches and is exchanged through its L2: plain stores, loads that pass the L1 (sc1), a barrier of 32 flags.  Only the
// output and down projections produce sums over XCDs: each XCD writes its fp32 partial through to memory and CU r of every XCD waits
// for the CUs r of the other seven (8 flags), then sums the tiles those eight produced in a fixed order.  A layer is
//   qkv | logits + exp | P V : O partial || sum + residual | gate, up : down partial || sum + residual |      (| XCD barrier, : values that are
// their own flags, || exchange between the 8 CUs of one number)
// Measured on MI355X: XCD barrier 0.35 us (1.02 us with 1 KB stored per workgroup before it and 32 KB read after it, 1.43 us with
// 64 KB), a barrier over all CUs 1.6 us, a dependent launch 2.3 us empty and 4.4-5.0 us as part of a layer.  Of a layer's 21 us
// (Pi0, one view, chunk 50) 6.4 are waits for flags and 5.0 the two exchanges.
//
// A CU holds RH of the 2 RH row tiles (CU parity) and the columns of one of 16 groups, so the activations of a phase are read once
// into half the CUs each and the weights twice per XCD (once from memory).  The eight compute waves split K and reduce through LDS; a
// ninth wave does the waiting, so that the compute waves can have the next phase's weights on the way while it polls.
//
// When the weights are asked for decides a layer's time more than anything else: a CU has one path to its vector cache, and what is in
// it goes before the flags, activations and partial sums asked for later.  Loads of whole lines hardly show (a hot line that takes 0.10 us
// takes 0.15 us beside a wave that streams from HBM), but touching one word of 64 lines holds the path up for all 8 KB of them (0.38 us).
// A tenth wave that touched all weights of the coming phases, spread over the phases, made a layer 2.2 us slower than none at all (Pi0, 1
// view, chunk 50: forward with one vision layer 6 735 us with it, 6 340 us without); so did weights requested ahead of an exchange (+0.7 us
// for the up tiles, +0.6 us for qkv), or K / V^T behind the qkv products (+0.1 us).  What pays: the weights of a phase behind the flag of the
// one before, while the others are waited for; those of the output projection already behind the P V products (-0.3 us); and touches
// by the waiting wave, 8 - 32 KB a phase, where nobody waits for the CU's loads: once the phase's operands have arrived and the products run
// (Cfg::NAP).  Those are a half of the gate tiles in the qkv phase (DM0: all), the other half in P V (DM0: the up tiles), the down projection's
// lines during the output projection, and the next layer's query columns during the down projection: 6 340 -> 6 127 us together.  Twice as much in a
// phase, or the K / V columns too, is slower again.
//
// All workgroups have to be resident at once.  A process keeps one flow kernel per device in flight (rtvla.hip), but another process's
// may be placed on half of the CUs at the same moment.  So no workgroup starts before all 256 have reported: the last one opens the
// gate, and one that has waited too long closes it, after which all of them leave and the CUs are free.  The kernel is therefore
// launched twice; the second launch ends at once if the first one ran, and the limits differ from process to process and from loop to
// loop.  Past the gate every wait still ends after wait_ticks: the wave notes it in `abort` and the kernel runs to its end without
// waiting, so the grid always drains.  Nothing makes the two launches succeed: kernels of others may hold the CUs for as long as they like.  The last launch
// (flow_kernel<.., ALONE>) therefore runs the same program in ONE workgroup, which waits for nobody, if neither finished: the phases one
// after another for the 256 (XCD, number) pairs, with the same sums in the same order, hence the same bits.  That takes 0.7 - 1.0 s
// instead of 4 - 6 ms; otherwise it ends at once (a forward of 8.33, 10.72 or 13.43 ms takes the same with and without it).  The input noise and
// the stream a program starts from are copies that flow_init_kernel made, so that an unfinished launch cannot spoil them.
#include "kernels.h"
#include <algorithm>
#include <atomic>

namespace {

constexpr int FW = 8;                                    // compute waves
constexpr int FLOW_THREADS = (FW + 1) * 64;              // + the wave that polls flags
constexpr float NEG_BIG = -1.0e30f;
constexpr int SQ_BYTES = FW * 4 * 64;
constexpr int ROPE_PITCH = 272;                                       // 256 bytes of a row, and 16 that move the next one to other banks

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef __amdgpu_buffer_rsrc_t rsrc_t;
typedef const __attribute__((address_space(4))) FlowP cFlowP;
constexpr int SC1 = 16, SYS = 17;                        // cache policy of the buffer instructions: past the L1 / through to memory

RTVLA_DEVICE rsrc_t make_rsrc(const void* base, unsigned bytes) { return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)bytes, 0x00027000); }
RTVLA_DEVICE bf16x8 ld16(rsrc_t r, int off) { return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, SC1)); }
RTVLA_DEVICE bf16x4 ld8(rsrc_t r, int off) { return __builtin_bit_cast(bf16x4, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, SC1)); }
RTVLA_DEVICE float ld4(rsrc_t r, int off) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, SC1)); }
RTVLA_DEVICE void st8(rsrc_t r, int off, bf16x4 v) { __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, off, 0, 0); }
RTVLA_DEVICE void st16(rsrc_t r, int off, bf16x8 v) { __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, off, 0, 0); }
// A value that is its own flag: a word of ones means "not there yet", so a pair of NaNs with this pattern loses a bit of its payload.
RTVLA_DEVICE void st8_flag(rsrc_t r, int off, bf16x4 v) {
    u32x2 b = __builtin_bit_cast(u32x2, v);
    b[0] = min(b[0], ~1u); b[1] = min(b[1], ~1u);
    __builtin_amdgcn_raw_buffer_store_b64(b, r, off, 0, 0);
}
RTVLA_DEVICE int ft_off(int row, int col, int cols32) { return (((row >> 4) * cols32 + (col >> 5)) * 64 + (row & 15) + 16 * ((col & 31) >> 3)) * 16 + (col & 7) * 2; }
RTVLA_DEVICE int frag_off(int rt, int kb, int cols32, int lane) { return ((rt * cols32 + kb) * 64 + lane) * 16; }
RTVLA_DEVICE bf16x8 ldw(const bf16_t* tiles, int nb, int kb, int K32p, int lane) { return *(const bf16x8*)(tiles + ((size_t)nb * K32p + kb) * 512 + lane * 8); }
RTVLA_DEVICE bf16x8 cat44(bf16x4 lo, bf16x4 hi) {
    bf16x8 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) { v[j] = lo[j]; v[4 + j] = hi[j]; }
    return v;
}

// The ids a phase starts from, hidden from the optimiser: every address in a phase follows from them, and all of those are loop
// invariants that would be hoisted out of the layer loop into far more registers than there are.
#define FLOW_IDS                                                                                     \
    int lane = lane_, w = w_, x = x_, r = r_;                                                        \
    asm volatile("" : "+v"(lane), "+s"(w), "+s"(x), "+s"(r));                                        \
    [[maybe_unused]] const int g = lane >> 4, lr = lane & 15, half = r & 1, grp = r >> 1

// A wait with an end: after `ticks` (of the 100 MHz counter) the wave notes it in `abort`, stops waiting and runs to the end of the program.
struct Patience {
    unsigned long long t0 = 0;
    int n = 0;
    bool lost = false;
    RTVLA_DEVICE void spin(FlowSync* sync, unsigned ticks, int lane) {
        if ((++n & 255) != 0) return;
        const unsigned long long now = __builtin_amdgcn_s_memrealtime();
        if (n == 256) t0 = now;
        else if (now - t0 > ticks) {
            lost = true;
            if (lane == 0) atomicOr_system(&sync->abort, 1u);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
    }
};

// The gate of one launch (thread 0 of each workgroup): `rank` gets the workgroup's number on its XCD, `gate` what was decided.
enum { GATE_UNDECIDED = 0, GATE_OPEN = 1, GATE_CLOSED = 2, GATE_DONE = 3 };
RTVLA_DEVICE void flow_gate(FlowSync* sync, int attempt, int xcc, unsigned ticks, int* rank, int* gate) {
    auto word = [](unsigned* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    auto decide = [](unsigned* p, unsigned to) {
        unsigned none = GATE_UNDECIDED;
        __hip_atomic_compare_exchange_strong(p, &none, to, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    *rank = 0;
    for (int k = 0; k < attempt; ++k)                                          // (that launch has ended)
        if (word(&sync->gate[k]) == GATE_OPEN) { *gate = GATE_DONE; return; }
    unsigned* const g = &sync->gate[attempt];
    if (ticks == 0) decide(g, GATE_CLOSED);                                    // (before anybody has reported: no patience, no launch)
    *rank = (int)atomicAdd(&sync->rank[attempt][xcc * 32], 1u);
    if (*rank >= 32) decide(g, GATE_CLOSED);                                   // not 32 workgroups per XCD
    else if (atomicAdd(&sync->arrived[attempt], 1u) == 255u) decide(g, GATE_OPEN);
    const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
    unsigned v;
    while ((v = word(g)) == GATE_UNDECIDED) {
        if (__builtin_amdgcn_s_memrealtime() - t0 > ticks) decide(g, GATE_CLOSED);
        __builtin_amdgcn_s_sleep(1);
    }
    *gate = v == GATE_OPEN && *rank >= 32 ? GATE_DONE : (int)v;                // (a launch without its flow_init_kernel finds the gate as the last one left it)
}

// Whether a launch before this one has run the program to its end.
RTVLA_DEVICE bool flow_ran(FlowSync* sync) {
    auto word = [](unsigned* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    bool open = false;
    for (int k = 0; k < FLOW_ATTEMPTS; ++k) open |= word(&sync->gate[k]) == GATE_OPEN;
    return open && word(&sync->abort) == 0;
}

// D[16 x 16] = A[16 x 16] B[16 x 16] of one half (4 elements per lane) of two 16 x 32 fragments
RTVLA_DEVICE f32x4 mfma16k16(bf16x8 a, bf16x8 b, int hi) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    const bf16x4 a4 = {a[4 * hi], a[4 * hi + 1], a[4 * hi + 2], a[4 * hi + 3]}, b4 = {b[4 * hi], b[4 * hi + 1], b[4 * hi + 2], b[4 * hi + 3]};
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a4), __builtin_bit_cast(s16x4, b4), f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
}

// What differs between the models' action experts.  NAP: naps of 64 cycles before the touches of a phase, whatever the number of rows.  Forward
// with one vision layer, us, without naps / a half / as they are / twice as many: Pi0, 1 view, chunk 20 5 549 / 5 477 / 5 431 / 5 644, chunk 50 6 181 /
// 6 154 / 6 028 / 6 193, Pi05, 2 views, chunk 25 6 659 / 6 592 / 6 534 / 6 757, DM0, 1 image 8 308 / 8 292 / 8 100 / 8 343; with three and
// four row tiles per CU they make next to no difference (Pi0, 1 view, chunk 80 7 348 / 7 347 / 7 366 / 7 272, chunk 120 8 290 / 8 305 / 8 299 / 8 284).
template <int MODEL> struct Cfg;
template <> struct Cfg<FLOW_PI0> {
    static constexpr int HD = 256, HEADS = 1, AT = 3, ET = 2, EGRP = 16, FK = 2, FWAVES = 8, HID = 512, WD_K32 = 128, NAP_QKV = 26, NAP = 20;
};
template <> struct Cfg<FLOW_PI05> : Cfg<FLOW_PI0> {};
template <> struct Cfg<FLOW_DM0> {
    static constexpr int HD = 128, HEADS = 2, AT = 2, ET = 1, EGRP = 12, FK = 1, FWAVES = 6, HID = 192, WD_K32 = 64, NAP_QKV = 14, NAP = 14;
};

// ALONE: the last launch, of compute waves only: if the program has not run, one workgroup runs it; then the activations of the last layer
// and step, which a user's program may look at, go from the XCDs' memory to where the loop as launches leaves them.
template <int MODEL, int RH, bool ALONE>
__global__ __launch_bounds__(ALONE ? FW * 64 : FLOW_THREADS)
void flow_kernel(FlowP kernel_args) {
    using C = Cfg<MODEL>;
    constexpr bool PI05 = MODEL == FLOW_PI05, DM0 = MODEL == FLOW_DM0;
    constexpr int RTP = 2 * RH;                          // row tiles of the suffix
    constexpr int QRT = RTP * C::HEADS;                  // row tiles of the queries of one XCD
    constexpr int QRTP = QRT <= 2 ? 2 : QRT <= 4 ? 4 : 8;
    constexpr int KD = C::HD / 32, DT = C::HD / 16, NDT = DT * QRTP / 32;      // d tiles per CU of the P V phase
    // row tiles per pass of a GEMM phase: both of two; of three or four one at a time, which leaves the registers for the pass's loads to be
    // in flight together (layer of 1 view, chunk 80: 31.6 -> 28.5 us, Pi05 32.0 -> 28.2; chunk 120: 33.8 -> 33.3).  Vector registers spilled
    // with two / one at a time: Pi0 with three row tiles 48 / 26, with four 18 / 0, Pi05 12 / 0 and 0 / 0; all other instances none.
    constexpr int MC = RH == 2 ? 2 : 1;
    constexpr int HID32 = C::HID / 32;
    constexpr int AK = (C::AT * RH + 7) / 8, SK = (4 * RH + 7) / 8;            // finished tiles per wave of the qkv and of the 4-column-tile phases
    static_assert(QRT <= 8 && NDT >= 1, "row tiles of one XCD");

    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    f32x4* const red = (f32x4*)smem;                                           // [wave][tile][64]
    float* const sq = (float*)(smem + FW * 4 * RH * 1024);                     // [wave][RH * 16] row sums of squares; [2][wave][16] maxima and sums of P V
    int* const sh = (int*)(smem + FW * 4 * RH * 1024 + SQ_BYTES);
    unsigned char* const rope_lds = smem + FW * 4 * RH * 1024 + SQ_BYTES + 320;       // DM0: the rotary table of the suffix rows, [row][ROPE_PITCH]

    // The parameters are read from the kernel-argument segment where they are used: hoisted out of the loops they would not fit the
    // scalar registers.  prm() hides the pointer from the optimiser so that each phase loads its own.
    auto prm = []() __attribute__((always_inline)) -> cFlowP& {
        auto q = (const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(q));
        return *(cFlowP*)q;
    };

    const int tid = threadIdx.x, lane_ = tid & 63;
    const int w_ = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the XCD this workgroup runs on and its number among the XCD's workgroups (ALONE: both are walked through below)
    if constexpr (ALONE) {
        if (tid == 0) sh[2] = flow_ran(kernel_args.sync) ? GATE_DONE : blockIdx.x == 0 ? GATE_OPEN : GATE_CLOSED;
    } else if (tid == 0) {
        const int xcc = __builtin_amdgcn_s_getreg(20 | (3 << 11)) & 7;         // HW_REG_XCC_ID
        sh[0] = xcc;
        flow_gate(kernel_args.sync, kernel_args.attempt, xcc, kernel_args.gate_ticks, &sh[1], &sh[2]);
    }
    auto load_rope = [&]() __attribute__((always_inline)) {
        if constexpr (DM0)
            for (int i = tid; i < RTP * 16 * 16; i += ALONE ? FW * 64 : FLOW_THREADS)
                *(uint4*)(rope_lds + (i >> 4) * ROPE_PITCH + (i & 15) * 16) = *(const uint4*)(kernel_args.rope + (size_t)min(i >> 4, kernel_args.rows - 1) * 128 + (i & 15) * 8);
    };
    if constexpr (!ALONE) load_rope();                                         // (while others arrive)
    __syncthreads();
    const int gate = __builtin_amdgcn_readfirstlane(sh[2]);
    if (gate != GATE_OPEN && !(ALONE && gate == GATE_DONE)) return;
    int x_ = ALONE ? 0 : __builtin_amdgcn_readfirstlane(sh[0]), r_ = ALONE ? 0 : __builtin_amdgcn_readfirstlane(sh[1]);
    const int step0 = kernel_args.step0, step1 = kernel_args.step1, layer0 = kernel_args.layer0, layer1 = kernel_args.layer1;
    const bool begin = kernel_args.begin != 0, end = kernel_args.end != 0;
    const bool keep_in = layer0 == layer1;                                     // (a single stage: the new stream goes back to the caller's buffer)
    auto bar = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    // ============ the waiting wave polls the flags and meets the compute waves at every barrier
    [[maybe_unused]] auto walk = [&](auto&& local, auto&& ahead) __attribute__((always_inline)) {
        if (!begin) local();
        for (int t = step0; t < step1; ++t) {
            if (begin) {
                local();
                if (!PI05) { bar(); if (!keep_in) local(); }
            }
            for (int l = layer0; l < layer1; ++l) {
                ahead(0, t, l); bar(); local();                                // qkv
                local();                                                       // logits
                ahead(1, t, l); bar(); bar();                                  // P V
                ahead(2, t, l); bar(); local();                                // output projection, exchange, sum
                bar(); bar();                                                  // gate, up
                ahead(3, t, l); bar(); local();                                // down projection, exchange, sum
            }
            if (end) {
                bar(); bar();
                if (t + 1 < step1) local();
            }
        }
    };
    if constexpr (!ALONE) if (w_ == FW) {
        const int lane = lane_, x = x_;
        const unsigned* const flags = kernel_args.sync->lflag + x * 256 + lane * 4;      // 32 workgroups x 8 compute waves, 4 flags per lane
        // One word of every 128-byte line is loaded into a scrap of LDS: the line is then in this XCD's L2 when the compute waves ask for it.
        const unsigned scrap = (unsigned)(FW * 4 * RH * 1024 + SQ_BYTES + 64);
        typedef const __attribute__((address_space(1))) void* gptr_t;
        typedef __attribute__((address_space(3))) void* lptr_t;
        unsigned ep = 0;
        Patience patience;
        if (kernel_args.wait_ticks == 0) {
            patience.lost = true;
            if (lane == 0) atomicOr_system(&kernel_args.sync->abort, 1u);
        }
        walk([&]() __attribute__((always_inline)) {
                 ++ep;
                 while (!patience.lost) {
                     u32x4 v;
                     asm volatile("global_load_dwordx4 %0, %1, off sc1\n\ts_waitcnt vmcnt(0)" : "=v"(v) : "v"(flags) : "memory");
                     if (__all((int)(v[0] - ep) >= 0 && (int)(v[1] - ep) >= 0 && (int)(v[2] - ep) >= 0 && (int)(v[3] - ep) >= 0)) break;
                     patience.spin(kernel_args.sync, kernel_args.wait_ticks, lane);
                 }
                 patience.n = 0;
                 bar();
             },
             [&](int k, int t, int l) __attribute__((always_inline)) {
                 cFlowP& p = prm();
                 auto touch = [&](const bf16_t* base, int kb) __attribute__((always_inline)) {     // kb KB from base
                     for (int i = 0; i < (kb + 7) / 8; ++i)
                         __builtin_amdgcn_global_load_lds((gptr_t)((const char*)base + min((i * 64 + lane) * 128, kb * 1024 - 128)), (lptr_t)(smem + scrap), 4, 0, 0);
                 };
                 if (k == 2) {                                                 // down projection of this layer: this XCD's K slice of two column tiles
#pragma unroll
                     for (int j = 0; j < 2; ++j) touch(p.wd + (size_t)l * p.wd_stride + ((size_t)(2 * r_ + j) * C::WD_K32 + x * HID32) * 512, HID32);
                 } else {                                                      // behind the phase's operands
                     for (int i = 0; i < (k == 0 ? C::NAP_QKV : C::NAP); ++i) __builtin_amdgcn_s_sleep(1);
                     if (k == 3) {                                             // the next layer's query columns: half a tile of every workgroup
                         const int ln = l + 1 < layer1 ? l + 1 : layer0, tn = l + 1 < layer1 || t + 1 == step1 ? t : t + 1;
                         touch(p.wqkv + (size_t)(PI05 ? tn * p.layers + ln : ln) * p.wqkv_stride + (size_t)(x * 32 + r_) * 16 * 512, 16);
                     } else if (r_ < C::HID / 16) {                            // qkv: the gate tiles or their first halves, P V: the others or the up tiles
                         const size_t o = (size_t)(PI05 ? t * p.layers + l : l) * p.wg_stride + (size_t)(x * (C::HID / 16) + r_) * 32 * 512;
                         touch((DM0 && k == 1 ? p.wu : p.wg) + o + (DM0 || k == 0 ? 0 : 16 * 512), DM0 ? 32 : 16);
                     }
                 }
             });
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                       // nothing may land in LDS after the workgroup has ended
        return;
    }
    // ================================================= the compute waves =================================================
    rsrc_t priv = make_rsrc(kernel_args.priv + (size_t)x_ * kernel_args.priv_stride, (unsigned)kernel_args.priv_stride);
    const rsrc_t part = make_rsrc(kernel_args.part, kernel_args.part_bytes);
    const int rows = kernel_args.rows;
    const int KBp = (kernel_args.prefix + 31) >> 5, KB = KBp + ((rows + 31) >> 5);       // 32-key blocks: cached prefix, all
    int vl = kernel_args.prefix;
    if (kernel_args.valid_len) vl = max(0, min(*kernel_args.valid_len, vl));
    const float sc2 = kernel_args.scale * 1.4426950408889634f;
    // this wave's stores are done -> its flag; `pre` runs while the waiting wave polls the flags of the XCD's 256 compute waves
    unsigned ep = 0;
    const unsigned* const my_flag = kernel_args.sync->lflag + x_ * 256 + r_ * FW + w_;
    auto sync = [&](auto&& pre) __attribute__((always_inline)) {
        ++ep;
        asm volatile("s_waitcnt vmcnt(0)\n\tglobal_store_dword %0, %1, off" ::"v"(my_flag), "v"(ep) : "memory");      // (every lane stores the same word)
        pre();
        bar();
    };

    Patience patience;
    patience.lost = !ALONE && kernel_args.wait_ticks == 0;

    // ---- one GEMM phase: NT column tiles x RH row tiles, K of this wave = NK blocks; partial sums to LDS ----
    // `swap`: tile index from which on the product is taken as rows x columns instead of columns x rows; `polled`: the values are their own flags
    auto gemm = [&]<int NT, int NK>(const bf16x8 (&wt)[NT][NK], int a_base, int a_cols32, int kb0, bool with_sq, int swap, bool polled) __attribute__((always_inline)) {
        FLOW_IDS;
#pragma unroll
        for (int m0 = 0; m0 < RH; m0 += MC) {
            bf16x8 a[MC][NK];
#pragma unroll
            for (int m = 0; m < MC; ++m)
#pragma unroll
                for (int i = 0; i < NK; ++i)
                    if (m0 + m < RH) a[m][i] = ld16(priv, a_base + frag_off(half * RH + m0 + m, kb0 + i, a_cols32, lane));
            if (polled && !ALONE) {                                            // what had not arrived is asked for again
                for (;;) {
                    bool missing = false;
#pragma unroll
                    for (int m = 0; m < MC; ++m)
#pragma unroll
                        for (int i = 0; i < NK; ++i) {
                            if (m0 + m >= RH) continue;
                            const u32x4 v = __builtin_bit_cast(u32x4, a[m][i]);
                            if (__any(max(max(v[0], v[1]), max(v[2], v[3])) == ~0u)) { a[m][i] = ld16(priv, a_base + frag_off(half * RH + m0 + m, kb0 + i, a_cols32, lane)); missing = true; }
                        }
                    if (!missing || patience.lost) break;
                    patience.spin(kernel_args.sync, kernel_args.wait_ticks, lane);
                }
                patience.n = 0;
            }
            f32x4 acc[MC][NT];
#pragma unroll
            for (int m = 0; m < MC; ++m)
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < NK; ++i)
#pragma unroll
                for (int m = 0; m < MC; ++m)
#pragma unroll
                    for (int t = 0; t < NT; ++t)
                        if (m0 + m < RH) acc[m][t] = t >= swap ? mfma16(a[m][i], wt[t][i], acc[m][t]) : mfma16(wt[t][i], a[m][i], acc[m][t]);
            if (with_sq) {
#pragma unroll
                for (int m = 0; m < MC; ++m) {
                    if (m0 + m >= RH) continue;
                    float s = 0.f, s1 = 0.f;
#pragma unroll
                    for (int i = 0; i < NK; ++i)
#pragma unroll
                        for (int j = 0; j < 8; j += 4) {
                            const bf16x2 v = {a[m][i][j], a[m][i][j + 1]}, v1 = {a[m][i][j + 2], a[m][i][j + 3]};
                            s = __builtin_amdgcn_fdot2_f32_bf16(v, v, s, false);
                            s1 = __builtin_amdgcn_fdot2_f32_bf16(v1, v1, s1, false);
                        }
                    s = rows_sum(s + s1);
                    if (g == 0) sq[w * (RH * 16) + (m0 + m) * 16 + lr] = s;
                }
            }
#pragma unroll
            for (int m = 0; m < MC; ++m)
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    if (m0 + m < RH) red[((size_t)w * (NT * RH) + t * RH + m0 + m) * 64 + lane] = acc[m][t];
        }
    };
    auto tile_sum = [&](int lane, int ntiles, int u, int waves) __attribute__((always_inline)) {
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ww = 0; ww < FW; ++ww) if (ww < waves) v += red[((size_t)ww * ntiles + u) * 64 + lane];
        return v;
    };
    auto row_factor = [&](int row_in_half) __attribute__((always_inline)) {    // RMS factor of one row of this CU's half
        float t = 0.f;
#pragma unroll
        for (int ww = 0; ww < FW; ++ww) t += sq[ww * (RH * 16) + row_in_half];
        const float f = rsqrtf(t * (1.0f / 1024.0f) + 1e-6f);
        return MODEL == FLOW_PI0 ? round_bf16(f) : f;
    };

    // ---- weights of the phases ----
    auto a_tile = [](int x, int grp, int t) __attribute__((always_inline)) {                  // column tile of the QKV matrix
        if constexpr (DM0) return t == 0 ? x * 16 + grp : (grp < 8 ? 128 + x * 8 + grp : 192 + x * 8 + grp - 8);
        else return t == 0 ? x * 16 + grp : t == 1 ? 128 + grp : 144 + grp;
    };
    auto load_a = [&](cFlowP& p, int t, int l, bf16x8 (&wA)[C::AT][4]) __attribute__((always_inline)) {
        FLOW_IDS;
        const bf16_t* base = p.wqkv + (size_t)(PI05 ? t * p.layers + l : l) * p.wqkv_stride;
#pragma unroll
        for (int j = 0; j < C::AT; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) wA[j][i] = ldw(base, a_tile(x, grp, j), w * 4 + i, 32, lane);
    };
    auto load_c = [&](cFlowP& p, int l, bf16x8 (&wC)[4][1]) __attribute__((always_inline)) {
        FLOW_IDS;
        const bf16_t* base = p.wo + (size_t)l * p.wo_stride;
#pragma unroll
        for (int j = 0; j < 4; ++j) wC[j][0] = ldw(base, grp * 4 + j, x * 8 + w, 64, lane);
    };
    auto load_e = [&](cFlowP& p, int t, int l, int part, bf16x8 (&wE)[2 * C::ET][4]) __attribute__((always_inline)) {
        FLOW_IDS;
        const size_t o = (size_t)(PI05 ? t * p.layers + l : l) * p.wg_stride;
        const int hb = x * (C::HID / 16) + min(grp, C::EGRP - 1) * C::ET;       // (loads are not made conditional anywhere: the compiler spills around it)
#pragma unroll
        for (int j = part * C::ET; j < (part + 1) * C::ET; ++j)                // part 0: gate, 1: up
#pragma unroll
            for (int i = 0; i < 4; ++i) wE[j][i] = ldw((j < C::ET ? p.wg : p.wu) + o, hb + j % C::ET, w * 4 + i, 32, lane);
    };
    auto load_f = [&](cFlowP& p, int l, bf16x8 (&wF)[4][C::FK]) __attribute__((always_inline)) {
        FLOW_IDS;
        const bf16_t* base = p.wd + (size_t)l * p.wd_stride;
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < C::FK; ++i) wF[j][i] = ldw(base, grp * 4 + j, x * HID32 + min(w, C::FWAVES - 1) * C::FK + i, C::WD_K32, lane);
    };

    // ---- qkv: RMS factor (Pi0, Pi05), RoPE, new K / V rows ----
    auto pre_qkv = [&](cFlowP& p, int t, int l, bf16x8 (&wA)[C::AT][4], bf16x4 (&pre_cs)[AK]) __attribute__((always_inline)) {
        FLOW_IDS;
        load_a(p, t, l, wA);
        if constexpr (DM0) {                                                   // norm weights instead (the rotary table is in LDS)
#pragma unroll
            for (int k = 0; k < AK; ++k) pre_cs[k] = load4(((w + 8 * k) / RH == 0 ? p.qnorm : p.knorm) + (size_t)l * 128 + (grp & 7) * 16 + 4 * g);
        } else {
#pragma unroll
            for (int k = 0; k < AK; ++k) {
                const int u = w + 8 * k;
                pre_cs[k] = load4(p.rope + (size_t)min((half * RH + u % RH) * 16 + lr, rows - 1) * 256 + grp * 16 + 4 * g);
            }
        }
    };
    auto qkv = [&](cFlowP& p, int t, int l, const bf16x8 (&wA)[C::AT][4], const bf16x4 (&pre_cs)[AK]) __attribute__((always_inline)) {
        FLOW_IDS;
        constexpr int NT = C::AT;
        gemm.template operator()<NT, 4>(wA, p.off_x, 32, w * 4, true, DM0 ? (grp >= 8 ? 1 : 9) : 2, false);
        bar();
        if (w < FW) {
#pragma unroll
            for (int k = 0; k < (NT * RH + 7) / 8; ++k) {
                const int u = w + 8 * k;
                if (NT * RH % FW != 0 && u >= NT * RH) continue;
                const int j = u / RH, m = u % RH;
                f32x4 v = tile_sum(lane, NT * RH, u, FW);
                const int row0 = (half * RH + m) * 16;
                if constexpr (DM0) {
                    // products rounded as the reference's QKV buffer; V carries the row's RMS factor.  Q and K leave with norm weight and
                    // rotary embedding but without the row's factors (RMS factor, norm over the head's 128 features), which are scalars
                    // of the logits: for those goes the sum of squares of the tile's 16 features.
                    if (j == 0 || grp < 8) {
                        const int col = (grp & 7) * 16 + 4 * g, row = row0 + lr;
                        const bf16x4 cs = *(const bf16x4*)(rope_lds + row * ROPE_PITCH + col * 2);
                        float ss = 0.f;
#pragma unroll
                        for (int e = 0; e < 4; ++e) { v[e] = round_bf16(v[e]); ss += v[e] * v[e]; v[e] *= bf2f(pre_cs[k][e]); }
                        ss = rows_sum(ss);
                        const float c0 = bf2f(cs[0]), s0 = bf2f(cs[1]), c1 = bf2f(cs[2]), s1 = bf2f(cs[3]);
                        const bf16x4 o = pack4(v[0] * c0 - v[1] * s0, v[1] * c0 + v[0] * s0, v[2] * c1 - v[3] * s1, v[3] * c1 + v[2] * s1);
                        st8(priv, j == 0 ? p.off_q + ft_off((grp >> 3) * RTP * 16 + row, col, KD) : p.off_k + ft_off(row, col, KD), o);
                        if (g == 0) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(ss), priv, p.off_s + (((j == 0 ? grp >> 3 : 2) * RTP * 16 + row) * 8 + (grp & 7)) * 4, 0, 0);
                    }
                    else {
                        const int d = (grp - 8) * 16 + lr, key = row0 + 4 * g;
                        f32x4 o;
#pragma unroll
                        for (int e = 0; e < 4; ++e) o[e] = round_bf16(v[e]) * row_factor(m * 16 + 4 * g + e);
                        st8(priv, p.off_v + (((d >> 4) * 4 + (key >> 5)) * 64 + (d & 15) + 16 * ((key & 15) >> 2)) * 16 + 8 * ((key & 31) >> 4), pack4(o));
                    }
                } else if (j < 2) {
                    v *= row_factor(m * 16 + lr);
                    const int n0 = grp * 16 + 4 * g;
                    if constexpr (PI05) v += *(const f32x4*)(p.bias_qkv + (size_t)(t * p.layers + l) * 2560 + (j == 0 ? x * 256 : 2048) + n0);
                    const bf16x4 cs = pre_cs[k];
                    const float c0 = bf2f(cs[0]), s0 = bf2f(cs[1]), c1 = bf2f(cs[2]), s1 = bf2f(cs[3]);
                    const bf16x4 o = pack4(v[0] * c0 - v[1] * s0, v[1] * c0 + v[0] * s0, v[2] * c1 - v[3] * s1, v[3] * c1 + v[2] * s1);
                    const int row = row0 + lr;
                    st8(priv, (j == 0 ? p.off_q : p.off_k) + ft_off(row, n0, 8), o);
                    // the cache rows behind the prefix, as the reference keeps them after the last step (nothing here reads them back)
                    if (j == 1 && x == 0 && row < rows && t == step1 - 1) store4(p.kcache + (size_t)l * p.kv_stride + ft_index(p.prefix + row, n0, 8), o);
                } else {                                                       // V: lane holds 4 keys of one column
                    const int d = grp * 16 + lr, key = row0 + 4 * g;
                    float b = 0.f;
                    if constexpr (PI05) b = p.bias_qkv[(size_t)(t * p.layers + l) * 2560 + 2304 + d];
                    f32x4 o;
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[e] = v[e] * row_factor(m * 16 + 4 * g + e) + b;
                    const bf16x4 pk = pack4(o);
                    st8(priv, p.off_v + (((d >> 4) * 4 + (key >> 5)) * 64 + (d & 15) + 16 * ((key & 15) >> 2)) * 16 + 8 * ((key & 31) >> 4), pk);
                    if (x == 0 && t == step1 - 1) {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (key + e < rows) p.vcache[(size_t)l * p.kv_stride + vt_index(d, p.prefix + key + e, p.ldvt >> 5)] = pk[e];
                    }
                }
            }
            if constexpr (DM0) {                                               // the row factors, once per row half
                if (grp == 0 && w == FW - 1 && lane < RH * 16) {
                    const float f = row_factor(lane);
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, f), priv, p.off_f + (half * RH * 16 + lane) * 4, 0, 0);
                }
            }
        }
    };

    // DM0: what a row of raw queries (head 0, 1) or keys (2) is scaled by: its RMS factor f, then the RMS norm over the head's 128 features
    auto dm0_scale = [&](cFlowP& p, int which, int row) __attribute__((always_inline)) {
        f32x4 s[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) s[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(priv, p.off_s + ((which * RTP * 16 + row) * 8 + 4 * i) * 4, 0, SC1));
        const float f = ld4(priv, p.off_f + row * 4);
        s[0] += s[1];
        return f * rsqrtf(f * f * (s[0][0] + s[0][1] + s[0][2] + s[0][3]) * (1.0f / 128.0f) + 1e-6f);
    };

    // ---- logits of (query row tile, 16 keys) per wave and their exponentials relative to the row maximum over those 16 keys ----
    // A workgroup takes a 32-key block, a wave one half of it (w & 1) and the row tiles (w >> 1), + 4.  The phase lasts as long as the slowest
    // workgroup: one with keys that this layer made, which it loads behind the barrier beside the queries.  So where workgroups are left over, two of
    // them share a block, half of the row tiles each: all blocks if there are at most 16, else those of the new keys.  Blocks past the 32nd are
    // dealt over the pairs of waves by row tiles, as a second pass.  (Forward with one vision layer, before and after: Pi0 1 view 6 130 ->
    // 6 056 us, 3 views 8 100 -> 8 042, DM0 1 image 8 299 -> 8 165; 33 blocks 9 112 -> 9 104.)
    constexpr int NQ = (QRT + 3) / 4;
    auto first_block = [&](int r, int& tb, int& tc) __attribute__((always_inline)) {           // the block (KB: none) and its row tiles
        tb = 0; tc = QRT;
        int kb = min(r, KB);
        const int whole = 2 * KB <= 32 ? 0 : KBp;                              // blocks that are not shared
        if (whole + 2 * (KB - whole) <= 32 && r >= whole) {
            kb = min(whole + (r - whole) / 2, KB);
            tc = QRT / 2; tb = (r - whole) % 2 * tc;
        }
        return kb;
    };
    auto load_k = [&](cFlowP& p, int lane, int x, int l, int nt, int kb, bf16x8 (&kf)[KD]) __attribute__((always_inline)) {
        const bf16_t* base = p.kcache + (size_t)(DM0 ? l * 8 + x : l) * p.kv_stride;
#pragma unroll
        for (int kd = 0; kd < KD; ++kd) kf[kd] = *(const bf16x8*)(base + ((size_t)((kb * 2 + nt) * KD + kd) * 64 + lane) * 8);
    };
    auto pre_logits = [&](cFlowP& p, int l, bf16x8 (&kf)[KD]) __attribute__((always_inline)) {
        FLOW_IDS;
        int tb, tc;
        const int kb = first_block(r, tb, tc);
        load_k(p, lane, x, l, w & 1, min(kb, KBp - 1), kf);
    };
    auto logits = [&](cFlowP& p, int l, bf16x8 (&kf)[KD]) __attribute__((always_inline)) {
        FLOW_IDS;
        const int nt = w & 1;
        int tb, tc;
        const int kb0 = first_block(r, tb, tc);
        if (kb0 >= KB) return;
        auto new_k = [&](int kb) __attribute__((always_inline)) {
#pragma unroll
            for (int kd = 0; kd < KD; ++kd) kf[kd] = ld16(priv, p.off_k + frag_off((kb - KBp) * 2 + nt, kd, KD, lane));
        };
        auto key_factor = [&](int kb) __attribute__((always_inline)) { return dm0_scale(p, 2, min(((kb - KBp) * 2 + nt) * 16 + lr, RTP * 16 - 1)); };
        auto load_q = [&](int rt, bf16x8 (&q)[KD], float& f) __attribute__((always_inline)) {
#pragma unroll
            for (int kd = 0; kd < KD; ++kd) q[kd] = ld16(priv, p.off_q + frag_off(rt, kd, KD, lane));
            if constexpr (DM0) f = dm0_scale(p, rt / RTP, rt % RTP * 16 + lr);
        };
        auto tile = [&](int kb, int rt, const bf16x8 (&q)[KD], float fq, float fk) __attribute__((always_inline)) {
            // the keys of this lane: 4 g .. 4 g + 3 of the 16; visible are those below `lim` (of the state row, among the new keys, only the first)
            const int key = nt * 16 + 4 * g;
            const int lim = kb < KBp ? vl - kb * 32 : rows - (kb - KBp) * 32;
            const int lim_state = kb < KBp ? lim : KBp == kb ? 1 : 0;
            const int lm = (MODEL == FLOW_PI0 && rt % RTP == 0 && lr == 0) ? lim_state : lim;      // the state token sees the prefix and itself
            f32x4 st = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kd = 0; kd < KD; ++kd) st = mfma16(kf[kd], q[kd], st);
            f32x4 sc = {sc2, sc2, sc2, sc2};
            if constexpr (DM0) {
                if (kb >= KBp)
#pragma unroll
                    for (int e = 0; e < 4; ++e) sc[e] *= __shfl(fk, 4 * g + e, 64);                // (lane lr has the factor of key lr)
                sc *= fq;
            }
            float mx = NEG_BIG;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                st[e] = key + e < lm ? st[e] * sc[e] : NEG_BIG;
                mx = fmaxf(mx, st[e]);
            }
            mx = rows_max(mx);
            float sum = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                st[e] = key + e < lm ? __builtin_amdgcn_exp2f(st[e] - mx) : 0.f;
                sum += st[e];
            }
            sum = rows_sum(sum);
            // this half's four probabilities of the lane's 16-byte piece of the P^T fragment
            st8(priv, p.off_p + ((rt * KB + kb) * 64 + lane) * 16 + nt * 8, pack4(st));
            if (g == 0) __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(mx), __float_as_uint(sum)}, priv, p.off_m + ((rt * KB + kb) * 16 + lr) * 16 + nt * 8, 0, 0);
        };
        // all that the block needs is requested before any of it is used
        bf16x8 qf[NQ][KD];
        float fq[NQ] = {}, fk = 0.f;
#pragma unroll
        for (int i = 0; i < NQ; ++i) load_q(tb + min((w >> 1) + 4 * i, tc - 1), qf[i], fq[i]);     // (by every wave: a branch around the loads costs 1 % of a forward)
        if (kb0 >= KBp) {
            new_k(kb0);
            if constexpr (DM0) fk = key_factor(kb0);
        }
#pragma unroll
        for (int i = 0; i < NQ; ++i)
            if ((w >> 1) + 4 * i < tc) tile(kb0, tb + (w >> 1) + 4 * i, qf[i], fq[i], fk);
        for (int u = r + 32 * (w >> 1); u < (KB - 32) * QRT; u += 128) {
            const int kb = 32 + u / QRT, rt = u % QRT;
            load_q(rt, qf[0], fq[0]);
            if (kb < KBp) load_k(p, lane, x, l, nt, kb, kf);
            else {
                new_k(kb);
                if constexpr (DM0) fk = key_factor(kb);
            }
            tile(kb, rt, qf[0], fq[0], fk);
        }
    };

    // ---- O = P V for one query row tile and NDT 16-wide column tiles; the waves split the key blocks, every 16 keys with their own factor ----
    constexpr int VB = 4;                                                      // blocks of a wave per trip (32 key blocks per workgroup)
    // (a block past the prefix is requested behind the end of the buffer: the hardware returns zero and reads nothing)
    auto load_v = [&](cFlowP& p, int lane, int x, int pdg, int l, int kb, bf16x8 (&v)[NDT]) __attribute__((always_inline)) {
        const rsrc_t rs = make_rsrc(p.vcache + (size_t)(DM0 ? l * 8 + x : l) * p.kv_stride, (unsigned)p.kv_stride * 2u);
#pragma unroll
        for (int d = 0; d < NDT; ++d)
            v[d] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rs, kb < KBp ? (((pdg * NDT + d) * (p.ldvt >> 5) + kb) * 64 + lane) * 16 : 0x7fffff00, 0, 0));
    };
    auto pre_pv = [&](cFlowP& p, int l, bf16x8 (&vf)[VB][NDT]) __attribute__((always_inline)) {
        FLOW_IDS;
        const int pdg = r / QRTP;
#pragma unroll
        for (int i = 0; i < VB; ++i) load_v(p, lane, x, pdg, l, w + FW * i, vf[i]);
    };
    auto pv = [&](cFlowP& p, int l, bf16x8 (&vf)[VB][NDT], auto&& next) __attribute__((always_inline)) {
        FLOW_IDS;
        const int prt = r % QRTP, pdg = r / QRTP;
        if (QRT == QRTP || prt < QRT) {
            f32x4 o[NDT];
#pragma unroll
            for (int d = 0; d < NDT; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
            float M = NEG_BIG, L = 0.f;
            for (int b0 = 0; b0 < KB; b0 += VB * FW) {
                bf16x8 pf[VB];
                f32x4 mo[VB];                                                  // {max, sum} of both halves
#pragma unroll
                for (int i = 0; i < VB; ++i) {
                    const int kb = min(b0 + w + FW * i, KB - 1);
                    mo[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(priv, p.off_m + ((prt * KB + kb) * 16 + lr) * 16, 0, SC1));
                    pf[i] = ld16(priv, p.off_p + ((prt * KB + kb) * 64 + lane) * 16);
                }
#pragma unroll
                for (int i = 0; i < VB; ++i) {
                    const int kb = b0 + w + FW * i;
                    if (kb >= KBp && kb < KB)
#pragma unroll
                        for (int d = 0; d < NDT; ++d) vf[i][d] = ld16(priv, p.off_v + (((pdg * NDT + d) * 4 + kb - KBp) * 64 + lane) * 16);
                    else if (b0 > 0) load_v(p, lane, x, pdg, l, kb, vf[i]);
                }
                float m = M;
#pragma unroll
                for (int i = 0; i < VB; ++i)
                    if (b0 + w + FW * i < KB) m = fmaxf(m, fmaxf(mo[i][0], mo[i][2]));
                if (b0 > 0) {
                    const float f = __builtin_amdgcn_exp2f(M - m);
                    L *= f;
#pragma unroll
                    for (int d = 0; d < NDT; ++d) o[d] *= f;
                }
                M = m;
#pragma unroll
                for (int i = 0; i < VB; ++i) {
                    const bool in = b0 + w + FW * i < KB;
                    const float f0 = in ? __builtin_amdgcn_exp2f(mo[i][0] - M) : 0.f, f1 = in ? __builtin_amdgcn_exp2f(mo[i][2] - M) : 0.f;
                    L += f0 * mo[i][1] + f1 * mo[i][3];
                    if constexpr (ALONE) {
                        // the cache's rows behind the prefix, where a launch that gave up may have left anything: their probabilities are
                        // zero, but 0 x NaN is NaN
                        if (const int kb = b0 + w + FW * i, key0 = kb * 32 + 4 * g; kb < KBp)
#pragma unroll
                            for (int d = 0; d < NDT; ++d)
#pragma unroll
                                for (int j = 0; j < 8; ++j)
                                    if (key0 + (j & 3) + 16 * (j >> 2) >= kernel_args.prefix) vf[i][d][j] = f2bf(0.f);
                    }
#pragma unroll
                    for (int d = 0; d < NDT; ++d) o[d] += f0 * mfma16k16(vf[i][d], pf[i], 0) + f1 * mfma16k16(vf[i][d], pf[i], 1);
                }
            }
#pragma unroll
            for (int d = 0; d < NDT; ++d) red[((size_t)w * NDT + d) * 64 + lane] = o[d];
            if (g == 0) { sq[w * 16 + lr] = M; sq[FW * 16 + w * 16 + lr] = L; }
        }
        next();
        bar();
        if (w < NDT && (QRT == QRTP || prt < QRT)) {
            float mw[FW], M = NEG_BIG, L = 0.f;
#pragma unroll
            for (int ww = 0; ww < FW; ++ww) { mw[ww] = sq[ww * 16 + lr]; M = fmaxf(M, mw[ww]); }
            f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ww = 0; ww < FW; ++ww) {
                const float f = __builtin_amdgcn_exp2f(mw[ww] - M);
                L += f * sq[FW * 16 + ww * 16 + lr];
                v += f * red[((size_t)ww * NDT + w) * 64 + lane];
            }
            v *= L > 0.f ? 1.0f / L : 0.f;
            const int tok = (prt % RTP) * 16 + lr, col = (prt / RTP) * C::HD + (pdg * NDT + w) * 16 + 4 * g;
            st8_flag(priv, p.off_o + ft_off(tok, col, 8), pack4(v));
        }
    };

    // ---- partial sums over this XCD's share of K, exchanged with the CUs r of the other XCDs ----
    // The values are their own flags: a buffer is all ones (a NaN no sum produces) until its values arrive, so a reader polls the data
    // and saves the write acknowledgement, the flag and a second read.  Three buffers take turns: once the partials of exchange e are
    // here, every peer has read exchange e - 1, so that buffer of this workgroup is set to ones again; it is written next in exchange
    // e + 2, which a peer only looks at after it has received this workgroup's exchange e + 1, sent behind a wait for those ones.
    // Tile layout: 64 bytes per row, so that the rows past the last one are neither written nor read.
    int ex = 0;                                                                // exchange number modulo 3
    auto part_off = [&](int buf, int y, int r, int u, int lane) __attribute__((always_inline)) {
        return (((buf * 8 + y) * 32 + r) * (4 * RH) + u) * 1024 + ((lane & 15) * 4 + (lane >> 4)) * 16;
    };
    auto store_part = [&](int waves, f32x4 (&own)[SK]) __attribute__((always_inline)) {
        FLOW_IDS;
#pragma unroll
        for (int k = 0; k < SK; ++k) {
            const int u = w + 8 * k;
            if (4 * RH % FW == 0 || u < 4 * RH) {
                own[k] = tile_sum(lane, 4 * RH, u, waves);
                if ((half * RH + u % RH) * 16 + lr < rows) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, own[k]), part, part_off(ex, x, r, u, lane), 0, SYS);
            }
        }
    };
    // The peers' tiles are requested and what had not arrived is asked for again.  Nothing else may be in flight here: loads return in
    // order, so weights requested between the two would hold up every further look (64 - 96 KB per workgroup, 1.6 - 2.5 us).
    auto sum_residual = [&](cFlowP& p, bool keep, const f32x4 (&own)[SK], const bf16_t* gp) __attribute__((always_inline)) {
        FLOW_IDS;
#pragma unroll
        for (int k = 0; k < SK; ++k) {
            const int u = w + 8 * k, row = (half * RH + u % RH) * 16 + lr, col = (grp * 4 + u / RH) * 16 + 4 * g;
            const bool in = (4 * RH % FW == 0 || u < 4 * RH) && row < rows;
            // (this XCD's own tile is at hand: its request, like those of rows past the end, is moved behind the end of the buffer, where
            // the hardware returns zero and reads nothing)
            auto load = [&](int y) __attribute__((always_inline)) {
                return __builtin_amdgcn_raw_buffer_load_b128(part, in && (ALONE || y != x) ? part_off(ex, y, r, u, lane) : 0x7fffff00, 0, SYS);
            };
            u32x4 v[8];
            const bf16x4 xold = ld8(priv, p.off_x + ft_off(row, col, 32));
            bf16x4 gate = {};
            if constexpr (PI05) gate = load4(gp + col);
#pragma unroll
            for (int y = 0; y < 8; ++y) v[y] = load(y);
            for (;;) {
                bool missing = false;
#pragma unroll
                for (int y = 0; y < 8; ++y)
                    if (__any(v[y][0] == ~0u || v[y][1] == ~0u || v[y][2] == ~0u || v[y][3] == ~0u)) { v[y] = load(y); missing = true; }
                if (!missing || patience.lost || ALONE) break;
                patience.spin(p.sync, p.wait_ticks, lane);
            }
            patience.n = 0;
            if (in) {
                f32x4 sum = {0.f, 0.f, 0.f, 0.f};                              // in the order of the XCDs on each of them
#pragma unroll
                for (int y = 0; y < 8; ++y) sum += !ALONE && y == x ? own[k] : __builtin_bit_cast(f32x4, v[y]);
                if constexpr (PI05) for (int e = 0; e < 4; ++e) sum[e] *= bf2f(gate[e]);
#pragma unroll
                for (int e = 0; e < 4; ++e) sum[e] += bf2f(xold[e]);
                const bf16x4 o = pack4(sum);
                st8(priv, p.off_x + ft_off(row, col, 32), o);
                if (keep && x == 0) store4(p.x + ft_index(row, col, 32), o);
            }
        }
        if constexpr (!ALONE) ex = ex == 2 ? 0 : ex + 1;                       // (ALONE: every partial sum is read before the next ones are made)
    };
    auto reset_part = [&]() __attribute__((always_inline)) {                   // of the exchange before the one just summed; runs behind the next flag
        FLOW_IDS;
        const int last = ex == 2 ? 0 : ex + 1;                                 // two back from the one to come
#pragma unroll
        for (int k = 0; k < SK; ++k) {
            const int u = w + 8 * k;
            if ((4 * RH % FW == 0 || u < 4 * RH) && (half * RH + u % RH) * 16 + lr < rows)
                __builtin_amdgcn_raw_buffer_store_b128(u32x4{~0u, ~0u, ~0u, ~0u}, part, part_off(last, x, r, u, lane), 0, SYS);
        }
    };

    // ---- gate / up ----
    auto mlp_up = [&](cFlowP& p, int t, int l, const bf16x8 (&wE)[2 * C::ET][4]) __attribute__((always_inline)) {
        FLOW_IDS;
        constexpr int NT = 2 * C::ET;
        if (C::EGRP == 16 || grp < C::EGRP) gemm.template operator()<NT, 4>(wE, p.off_x, 32, w * 4, true, 9, false);
        bar();
        if (w < C::ET * RH && (C::EGRP == 16 || grp < C::EGRP)) {
            const int j = w / RH, m = w % RH;
            f32x4 gv = tile_sum(lane, NT * RH, w, FW), uv = tile_sum(lane, NT * RH, C::ET * RH + w, FW);
            const float f = row_factor(m * 16 + lr);
            gv *= f; uv *= f;
            const int hc = (grp * C::ET + j) * 16 + 4 * g;
            if constexpr (PI05) {
                const size_t o = (size_t)(t * p.layers + l) * 4096 + x * C::HID + hc;
                gv += *(const f32x4*)(p.bias_gate + o); uv += *(const f32x4*)(p.bias_up + o);
            }
            f32x4 h;
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = (DM0 ? siluf(gv[e]) : gelu_tanh(gv[e])) * uv[e];
            st8_flag(priv, p.off_h + ft_off((half * RH + m) * 16 + lr, hc, HID32), pack4(h));
        }
    };

    // The attention output and the hidden activations are their own flags: the GEMM that reads them asks until no word is all ones, which
    // saves the acknowledgement of the stores, the flag and the second look (forward of Pi0, 1 view, 6 355 -> 6 273 us, DM0, 3 images, 10 060 ->
    // 9 780; with the residual stream exchanged in the same way, which more CUs look for longer, 6 490).  Behind the flag of the qkv phase everybody has read those
    // of the layer before (the flags of the exchanges lie between), and they are set to ones again, 1 KB pieces dealt over the XCD's waves;
    // the flag of the logits phase, which everybody awaits before looking again, is sent behind a wait for these stores.
    auto reset_values = [&](cFlowP& p) __attribute__((always_inline)) {
        FLOW_IDS;
        constexpr int NO = RTP * 8, N = NO + RTP * HID32;
        static_assert(N <= 256, "one piece per wave");
        const int i = r * FW + w;
        if (i < N) __builtin_amdgcn_raw_buffer_store_b128(u32x4{~0u, ~0u, ~0u, ~0u}, priv, (i < NO ? p.off_o + i * 1024 : p.off_h + (i - NO) * 1024) + lane * 16, 0, 0);
    };

    // ---- start of a flow step: noise -> input projection (+ SiLU, MLP) -> residual stream ----
    const int s0 = MODEL == FLOW_PI0 ? 1 : 0;                                  // action rows follow the state token
    auto action_in = [&](cFlowP& p, int t) __attribute__((always_inline)) {
        FLOW_IDS;
        const bool first = t == step0;
#pragma unroll
        for (int k = 0; k < (2 * RTP + 7) / 8; ++k) {
            const int u = w + 8 * k;
            if (2 * RTP % FW != 0 && u >= 2 * RTP) continue;
            const int ct = 2 * r + (u & 1), rt = u >> 1;
            const int arow = max(0, min(rt * 16 + lr - s0, rows - s0 - 1));
            const bf16x8 nz = first ? *(const bf16x8*)(p.noise + arow * 32 + 8 * g) : ld16(priv, p.off_n + arow * 64 + 16 * g);
            const bf16x8 wi = ldw(p.win, ct, 0, 4, lane);
            const bf16x4 b = load4(p.bin + (PI05 ? 0 : (size_t)t * 1024) + ct * 16 + 4 * g);
            f32x4 v = {bf2f(b[0]), bf2f(b[1]), bf2f(b[2]), bf2f(b[3])};
            v = mfma16(wi, nz, v);
            if constexpr (!PI05) for (int e = 0; e < 4; ++e) v[e] = siluf(v[e]);
            st8(priv, (PI05 ? p.off_x : p.off_xin) + ft_off(rt * 16 + lr, ct * 16 + 4 * g, 32), pack4(v));
        }
    };
    auto pre_mlp_in = [&](cFlowP& p, bf16x8 (&wM)[4][4]) __attribute__((always_inline)) {
        FLOW_IDS;
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) wM[j][i] = ldw(p.wmlp, grp * 4 + j, w * 4 + i, 32, lane);
    };
    auto mlp_in = [&](cFlowP& p, bool keep, const bf16x8 (&wM)[4][4]) __attribute__((always_inline)) {
        FLOW_IDS;
        gemm.template operator()<4, 4>(wM, p.off_xin, 32, w * 4, false, 9, false);
        bar();
        {
#pragma unroll
            for (int k = 0; k < SK; ++k) {
                const int u = w + 8 * k;
                if (4 * RH % FW != 0 && u >= 4 * RH) continue;
                f32x4 v = tile_sum(lane, 4 * RH, u, FW);
                const int row = (half * RH + u % RH) * 16 + lr, col = (grp * 4 + u / RH) * 16 + 4 * g;
                const bf16x4 b = load4(p.bmlp + col);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] += bf2f(b[e]);
                bf16x4 o = pack4(v);
                if (MODEL == FLOW_PI0 && row == 0) o = load4(p.state_x + col);
                st8(priv, p.off_x + ft_off(row, col, 32), o);
                if (keep && x == 0) store4(p.x + ft_index(row, col, 32), o);
            }
        }
    };

    // ---- end of a flow step: final norm, output projection, Euler update of the noise (CU: one 16 x 16 tile) ----
    auto euler = [&](cFlowP& p, int t) __attribute__((always_inline)) {
        FLOW_IDS;
        const int urt = r >> 1, uct = r & 1;
        const bool first = t == step0, last = t == step1 - 1;
        const int row = urt * 16 + lr, arow = row - s0;
        bf16x8 a[4], wU[4];
        if (urt < RTP) {
            float s = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) wU[i] = ldw(p.wout, uct, w * 4 + i, 32, lane);
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = ld16(priv, p.off_x + frag_off(urt, w * 4 + i, 32, lane));
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 8; j += 2) {
                    const bf16x2 v = {a[i][j], a[i][j + 1]};
                    s = __builtin_amdgcn_fdot2_f32_bf16(v, v, s, false);
                }
            s = rows_sum(s);
            if (g == 0) sq[w * (RH * 16) + lr] = s;
        }
        bar();
        if (urt < RTP) {
            if constexpr (PI05) {                                              // adaptive norm: x f (1 + scale) + shift before the product
                const float f = row_factor(lr);
                const bf16_t* st = p.style_final + (size_t)t * 3072;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bf16x8 sc = *(const bf16x8*)(st + (w * 4 + i) * 32 + 8 * g), shf = *(const bf16x8*)(st + 1024 + (w * 4 + i) * 32 + 8 * g);
#pragma unroll
                    for (int j = 0; j < 8; ++j) a[i][j] = f2bf(bf2f(a[i][j]) * f * (1.0f + bf2f(sc[j])) + bf2f(shf[j]));
                }
            }
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 4; ++i) acc = mfma16(wU[i], a[i], acc);
            red[(size_t)w * 64 + lane] = acc;
        }
        bar();
        if (w == 0 && urt < RTP && arow >= 0 && row < rows) {
            const int col = uct * 16 + 4 * g;
            f32x4 v = tile_sum(lane, 1, 0, FW);
            if constexpr (!PI05) v *= row_factor(lr);
            const bf16x4 b = load4(p.bout + col);
            const bf16x4 old = first ? load4(p.noise + arow * 32 + col) : ld8(priv, p.off_n + arow * 64 + col * 2);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = v[e] + bf2f(b[e]) + bf2f(old[e]);
            const bf16x4 o = pack4(v);
            st8(priv, p.off_n + arow * 64 + col * 2, o);
            if (last && x == 0) store4(p.noise_out + arow * 32 + col, o);
        }
    };

    // ---- the program (the waiting wave above walks through the same one) ----
    auto nothing = []() __attribute__((always_inline)) {};
    auto copy_x = [&](bool in) __attribute__((always_inline)) {
        FLOW_IDS;
        cFlowP& p = prm();
        for (int i = r * FW + w; i < RTP * 32; i += 32 * FW) {
            const size_t at = ((size_t)i * 64 + lane) * 8;
            if (in) st16(priv, p.off_x + (i * 64 + lane) * 16, *(const bf16x8*)(p.x_in + at));
            else if (x == 0) *(bf16x8*)(p.x + at) = ld16(priv, p.off_x + (i * 64 + lane) * 16);
        }
    };
    if constexpr (ALONE) {
        // One phase after another, each for all (XCD, number) pairs; between two of them every store has ended and nobody reads LDS.
        // Latency almost throughout (the weights alone would be 0.2 s at the rate of one CU): 0.74 s for Pi0's 180 layers, 0.99 s for DM0's 280.
        auto each = [&](auto&& phase) __attribute__((always_inline)) {
            for (x_ = 0; x_ < 8; ++x_) {
                priv = make_rsrc(kernel_args.priv + (size_t)x_ * kernel_args.priv_stride, (unsigned)kernel_args.priv_stride);
                for (r_ = 0; r_ < 32; ++r_) {
                    phase();
                    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
                }
            }
        };
        // pieces of 8 columns of a row; XCD x holds query head x (DM0: heads 2 x, 2 x + 1), their output, and its share of the hidden columns
        auto publish = [&](int i0, int n) __attribute__((always_inline)) {
            cFlowP& p = prm();
            if (layer0 < layer1) {
                for (int i = i0; i < rows * 256; i += n) {
                    const int c = (i & 31) * 8, y = (i >> 5) & 7, row = i >> 8;
                    const char* src = p.priv + (size_t)y * p.priv_stride;
                    *(bf16x8*)(p.out_attn + ft_index(row, y * 256 + c, 64)) = *(const bf16x8*)(src + p.off_o + ft_off(row, c, 8));
                    if (!DM0) *(bf16x8*)(p.out_q + ft_index(row * 8 + y, c, 8)) = *(const bf16x8*)(src + p.off_q + ft_off(row, c, 8));
                }
                for (int i = i0; i < rows * C::HID; i += n) {
                    const int c = i % (C::HID / 8) * 8, y = i / (C::HID / 8) % 8, row = i / C::HID;
                    *(bf16x8*)(p.out_hidden + ft_index(row, y * C::HID + c, p.hidden_cols32)) = *(const bf16x8*)(p.priv + (size_t)y * p.priv_stride + p.off_h + ft_off(row, c, HID32));
                }
            }
            if (begin && !PI05)
                for (int i = i0; i < (rows - s0) * 128; i += n)
                    *(bf16x8*)(p.out_xin + ft_index(i >> 7, (i & 127) * 8, 32)) = *(const bf16x8*)(p.priv + p.off_xin + ft_off((i >> 7) + s0, (i & 127) * 8, 32));
        };
        if (gate == GATE_DONE) { publish(blockIdx.x * (FW * 64) + tid, gridDim.x * (FW * 64)); return; }
        load_rope();
        __syncthreads();
        f32x4 own[SK];                                                         // (read back from memory like those of the others)
        if (!begin) each([&]() __attribute__((always_inline)) { copy_x(true); });
        for (int t = step0; t < step1; ++t) {
            if (begin) {
                each([&]() __attribute__((always_inline)) { action_in(prm(), t); });
                if constexpr (!PI05) each([&]() __attribute__((always_inline)) { bf16x8 wM[4][4]; pre_mlp_in(prm(), wM); mlp_in(prm(), keep_in, wM); });
                else if (keep_in) each([&]() __attribute__((always_inline)) { copy_x(false); });
            }
            for (int l = layer0; l < layer1; ++l) {
                const size_t tl = (size_t)t * kernel_args.layers + l;
                each([&]() __attribute__((always_inline)) { bf16x8 wA[C::AT][4]; bf16x4 cs[AK]; pre_qkv(prm(), t, l, wA, cs); qkv(prm(), t, l, wA, cs); });
                each([&]() __attribute__((always_inline)) { bf16x8 kf[KD]; pre_logits(prm(), l, kf); logits(prm(), l, kf); });
                each([&]() __attribute__((always_inline)) { bf16x8 vf[VB][NDT]; pre_pv(prm(), l, vf); pv(prm(), l, vf, nothing); });
                each([&]() __attribute__((always_inline)) {
                    bf16x8 wC[4][1];
                    load_c(prm(), l, wC);
                    gemm.template operator()<4, 1>(wC, prm().off_o, 8, w_, false, 9, true);
                    bar();
                    store_part(FW, own);
                });
                each([&]() __attribute__((always_inline)) { sum_residual(prm(), false, own, PI05 ? prm().style_attn + tl * 3072 + 2048 : nullptr); });
                each([&]() __attribute__((always_inline)) { bf16x8 wE[2 * C::ET][4]; load_e(prm(), t, l, 0, wE); load_e(prm(), t, l, 1, wE); mlp_up(prm(), t, l, wE); });
                each([&]() __attribute__((always_inline)) {
                    bf16x8 wF[4][C::FK];
                    load_f(prm(), l, wF);
                    if (C::FWAVES == FW || w_ < C::FWAVES) gemm.template operator()<4, C::FK>(wF, prm().off_h, HID32, w_ * C::FK, false, 9, true);
                    bar();
                    store_part(C::FWAVES, own);
                });
                each([&]() __attribute__((always_inline)) { sum_residual(prm(), l == layer1 - 1, own, PI05 ? prm().style_ffn + tl * 3072 + 2048 : nullptr); });
            }
            if (end) each([&]() __attribute__((always_inline)) { euler(prm(), t); });
        }
        publish(tid, FW * 64);
        if (tid == 0 && kernel_args.alone) __hip_atomic_store(kernel_args.alone, __hip_atomic_load(kernel_args.alone, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        return;
    }
    bf16x8 wA[C::AT][4];
    bf16x4 cs[AK];
    if (!begin) {                                                              // a single stage: the stream comes from the caller's buffer
        copy_x(true);
        sync([&]() __attribute__((always_inline)) { pre_qkv(prm(), step0, layer0 < layer1 ? layer0 : 0, wA, cs); });
    }
    for (int t = step0; t < step1; ++t) {
        if (begin) {
            action_in(prm(), t);
            if constexpr (PI05) {
                sync([&]() __attribute__((always_inline)) { pre_qkv(prm(), t, layer0, wA, cs); });
                if (keep_in) copy_x(false);
            } else {
                bf16x8 wM[4][4];
                sync([&]() __attribute__((always_inline)) { pre_mlp_in(prm(), wM); });
                mlp_in(prm(), keep_in, wM);
                if (!keep_in) sync([&]() __attribute__((always_inline)) { pre_qkv(prm(), t, layer0, wA, cs); });
            }
        }
        for (int l = layer0; l < layer1; ++l) {
            const bool lastl = l == layer1 - 1;
            qkv(prm(), t, l, wA, cs);
            {
                bf16x8 kf[KD];
                sync([&]() __attribute__((always_inline)) { pre_logits(prm(), l, kf); reset_values(prm()); });
                logits(prm(), l, kf);
            }
            bf16x8 wC[4][1];
            {
                bf16x8 vf[VB][NDT];
                sync([&]() __attribute__((always_inline)) { pre_pv(prm(), l, vf); });
                pv(prm(), l, vf, [&]() __attribute__((always_inline)) { load_c(prm(), l, wC); });
            }
            {
                bf16x8 wE[2 * C::ET][4];
                f32x4 own[SK];
                load_e(prm(), t, l, 0, wE);
                bar();                                                         // (LDS: the sums of P V have been read)
                gemm.template operator()<4, 1>(wC, prm().off_o, 8, w_, false, 9, true);
                bar();
                store_part(FW, own);
                cFlowP& p = prm();
                sum_residual(p, false, own, PI05 ? p.style_attn + ((size_t)t * p.layers + l) * 3072 + 2048 : nullptr);
                sync([&]() __attribute__((always_inline)) { reset_part(); load_e(prm(), t, l, 1, wE); });
                mlp_up(prm(), t, l, wE);
            }
            {
                f32x4 own[SK];
                {
                    bf16x8 wF[4][C::FK];
                    load_f(prm(), l, wF);
                    bar();
                    if (C::FWAVES == FW || w_ < C::FWAVES) gemm.template operator()<4, C::FK>(wF, prm().off_h, HID32, w_ * C::FK, false, 9, true);
                }
                bar();
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");               // (the ones of reset_part have arrived; nothing else is under way)
                store_part(C::FWAVES, own);
                cFlowP& p = prm();
                sum_residual(p, lastl, own, PI05 ? p.style_ffn + ((size_t)t * p.layers + l) * 3072 + 2048 : nullptr);
            }
            sync([&]() __attribute__((always_inline)) { reset_part(); pre_qkv(prm(), t, lastl ? l : l + 1, wA, cs); });      // (after the last layer for nothing)
        }
        if (end) {
            euler(prm(), t);
            if (t + 1 < step1) sync(nothing);
        }
    }
}

// zeroes the flags, sets the exchange buffers to ones, copies what the program starts from and, for Pi0, projects the state token (row 0 of the residual stream, the same in every flow step)
__global__ __launch_bounds__(256) void flow_init_kernel(FlowSync* sync, uint4* part, int part16, FlowStart start, const bf16_t* state, const bf16_t* w, const bf16_t* b, bf16_t* out) {
    const int i = blockIdx.x * 256 + threadIdx.x, n = gridDim.x * 256;
    unsigned* s = (unsigned*)sync;
    for (int k = i; k < (int)(sizeof(FlowSync) / 4); k += n) s[k] = 0;
    for (int k = i; k < part16; k += n) part[k] = uint4{~0u, ~0u, ~0u, ~0u};
    for (int k = i; k < start.noise16; k += n) start.noise_copy[k] = start.noise[k];
    for (int k = i; k < start.x16; k += n) start.x_copy[k] = start.x[k];
    if (state && i < 1024) {
        float acc = bf2f(b[i]);
        bf16_t wc[32];
#pragma unroll
        for (int k = 0; k < 32; ++k) wc[k] = w[(size_t)k * 1024 + i];
#pragma unroll
        for (int k = 0; k < 32; ++k) acc += bf2f(state[k]) * bf2f(wc[k]);
        out[i] = f2bf(acc);
    }
}

template <int MODEL, int RH>
int launch_inst(const FlowP& p, hipStream_t s) {
    const size_t need = (size_t)FW * 4 * RH * 1024 + SQ_BYTES + 320 + (MODEL == FLOW_DM0 ? 2 * RH * 16 * ROPE_PITCH : 0);
    const size_t smem = std::max(need, (size_t)96 * 1024);                     // more than half a CU's LDS: one workgroup per CU
    auto kern = flow_kernel<MODEL, RH, false>;
    auto alone = flow_kernel<MODEL, RH, true>;
    static std::atomic<uint64_t> done{0}, done_alone{0};
    if (int rc = ensure_dynamic_lds((const void*)kern, smem, done)) return rc;
    if (int rc = ensure_dynamic_lds((const void*)alone, need, done_alone)) return rc;
    FlowP q = p;
    for (q.attempt = 0; q.attempt < FLOW_ATTEMPTS; ++q.attempt) {
        q.gate_ticks = p.gate_limits[q.attempt];
        hipLaunchKernelGGL(kern, dim3(256), dim3(FLOW_THREADS), smem, s, q);
        if (hipGetLastError() != hipSuccess) return 5;
    }
    hipLaunchKernelGGL(alone, dim3(64), dim3(FW * 64), need, s, q);
    return hipGetLastError() == hipSuccess ? 0 : 5;
}

}  // namespace

int flow_row_pairs(int rows) { return (rows + 31) / 32; }

size_t flow_layout(FlowP* p, int qtiles, int blocks, int hidden) {
    size_t at = 0;
    auto take = [&](size_t bytes) { const int o = (int)at; at += (bytes + 255) & ~(size_t)255; return o; };
    p->off_x = take(128 * 1024 * 2); p->off_xin = take(128 * 1024 * 2);
    p->off_q = take((size_t)std::max(qtiles, 8) * 16 * 256 * 2); p->off_k = take(128 * 256 * 2); p->off_v = take(256 * 128 * 2);
    p->off_o = take(128 * 256 * 2); p->off_h = take((size_t)128 * hidden * 2); p->off_n = take(128 * 32 * 2); p->off_f = take(128 * 4); p->off_s = take(3 * 128 * 8 * 4);
    p->off_m = take((size_t)qtiles * blocks * 16 * 16); p->off_p = take((size_t)qtiles * blocks * 1024);
    return (at + 4095) & ~(size_t)4095;
}

void launch_flow_init(FlowSync* sync, float* part, unsigned part_bytes, const FlowStart& start, const bf16_t* state, const bf16_t* w, const bf16_t* b, bf16_t* out, hipStream_t s) {
    hipLaunchKernelGGL(flow_init_kernel, dim3(512), dim3(256), 0, s, sync, (uint4*)part, (int)(part_bytes / 16), start, state, w, b, out);
}

int launch_flow(const FlowP& p, int model, hipStream_t s) {
    if (p.rows < 1 || p.rows > (model == FLOW_DM0 ? 64 : 128) || p.prefix < 1 || (p.ldvt & 31) || p.ldvt < p.prefix + p.rows) return 1;
    if (p.step0 < 0 || p.step1 <= p.step0 || p.layer0 < 0 || p.layer1 < p.layer0 || p.layer1 > p.layers) return 1;
    if (p.begin && !p.end && p.step1 != p.step0 + 1) return 1;
    const int rh = flow_row_pairs(p.rows);
    if (model == FLOW_PI0) {
        switch (rh) { case 1: return launch_inst<FLOW_PI0, 1>(p, s); case 2: return launch_inst<FLOW_PI0, 2>(p, s); case 3: return launch_inst<FLOW_PI0, 3>(p, s); case 4: return launch_inst<FLOW_PI0, 4>(p, s); }
    } else if (model == FLOW_PI05) {
        switch (rh) { case 1: return launch_inst<FLOW_PI05, 1>(p, s); case 2: return launch_inst<FLOW_PI05, 2>(p, s); case 3: return launch_inst<FLOW_PI05, 3>(p, s); case 4: return launch_inst<FLOW_PI05, 4>(p, s); }
    } else if (model == FLOW_DM0) {
        switch (rh) { case 1: return launch_inst<FLOW_DM0, 1>(p, s); case 2: return launch_inst<FLOW_DM0, 2>(p, s); }
    }
    return 2;
}

// Whether the current device has the 256 CUs the flow kernel splits its work over (a partitioned one has fewer).  Whether this process and
// stream may use them all, and whether they are free, the gate finds out at each launch.
bool flow_supported() {
    int dev = 0, cus = 0;
    return hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && cus == 256;
}
