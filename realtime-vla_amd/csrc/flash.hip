// Softmax attention for long query AND key sequences on v_mfma_f32_32x32x16_bf16, flash style: DM0's ViT attention,
// 2705 tokens per (image, head), head width 64 (/root/reference/dm0_infer.py:589-598), 3 x 16 independent heads.
//
// One workgroup = 4 waves = 128 consecutive query rows of one K/V head; each wave owns 32 query rows and walks ALL keys,
// so there is no merge at the end.  K and V^T tiles of 64 keys go from global memory straight into LDS (global_load_lds,
// three stages, one barrier per tile) and are shared by the four waves: the L2 port of a CU carries each tile once per
// 128 query rows instead of once per wave.  The tiles keep the byte layout they have in memory (MFMA fragments of 1 KB:
// Q and K fragment-tiled [rows][HD], V^T in the permuted-key layout), so staging is a plain copy of 1 KB pieces and every
// operand read is a conflict-free ds_read_b128.
//
// Per 32-key block the wave computes S^T = K Q^T (32 keys x 32 queries): lane (h = lane / 32, n = lane % 32) holds the 16
// logits of query n for keys 8 j + 4 h + v.  The softmax statistics are therefore per-lane scalars shared with ONE other
// lane, the running sum is kept per lane and combined once at the end, and the accumulator is only rescaled when some
// row's maximum grew by more than 2^8 (a wave-uniform branch, taken a few times per row).  The probabilities of
// accumulator groups j = q and j = q + 2 are, packed to bf16, exactly the B operand of O^T += V^T P^T for the q-th 16-key
// step in the key order of the stored V^T: no shuffles between the two products.  The loop is software-pipelined over the
// 32-key blocks (see flash_kernel).
//
// Measured on MI355X, 16 / 32 / 48 heads x 2 705 tokens, in a ViT layer: 40 / 70 / 105 us.  Steps to there: softmax of every second block kept beside its MFMAs (see the end
// of `step`) and waits for single LDS reads 49.6 / 75.5 / 119.9 -> 44.8 / 69.7 / 111.7; stages that K enters a tile earlier, requested by buffer loads whose addresses are
// scalar, 43.2 / 68.9 / 108.1; last row blocks at the end of the grid, where the waves past the last row only stage, 42.1 / 68.7 / 105.5; the two kinds of MFMA in turn 40.0 / 69.6 / 104.9.
// What the rest is spent on, left out one at a time of 111: staging 11, LDS reads 13, v_dot2_f32_bf16 of the row sums 6 (it does not run beside MFMAs: 8 of those take 145 ns a
// wave, with 16 v_exp, 32 v_max3 or 32 v_cvt_pk between them as long, with 32 v_dot2 212), maxima and their branch 5, the barrier 1; without all of these 73.
#include "kernels.h"
#include <type_traits>

namespace {

constexpr float NEG_BIG = -1.0e30f;

RTVLA_DEVICE f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }

RTVLA_DEVICE bf16x8 pack8(const f32x16& s, int a, int b) {
    bf16x8 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) { v[i] = (bf16_t)s[4 * a + i]; v[4 + i] = (bf16_t)s[4 * b + i]; }
    return v;
}

RTVLA_DEVICE bf16_t* flash_out_ptr(const AttnP& p, int batch, int row, int d, int hd) {
    const int tok = row / p.group, sub = row - tok * p.group;
    if (p.out_tiled) return p.out + ft_index(tok, batch * p.out_bcol + sub * hd + d, p.out_cols32);
    const int bo = batch / p.batch_inner, bi = batch - bo * p.batch_inner;
    return p.out + (size_t)bo * p.out_ostride + (size_t)bi * p.out_istride + (size_t)tok * p.ld_tok + sub * hd + d;
}

// Threshold (in bits of the exponent) below which a grown row maximum does not trigger a rescale: the probabilities of later
// keys are then at most 2^8 instead of 1 until the next rescale, which fp32 sums and the bf16 rounding (relative) do not
// mind, and the accumulator is touched a few times per row instead of in most blocks.
constexpr float RESCALE_BITS = 8.0f;
constexpr int FLASH_STAGES = 3;

// All but this wave's newest N loads have landed, its LDS reads are back, and so for every wave of the workgroup
template <int N> RTVLA_DEVICE void wait_and_meet() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(N | 7 << 4);             // vmcnt(N) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// The key loop is software-pipelined over 32-key blocks so that every MFMA has independent VALU work to run under: while
// the softmax of block g is computed (VALU), the matrix pipe takes S^T of block g+1 and O^T += V^T P^T of block g-1.
// A block needs 8 MFMAs (256 cycles) and ~65 VALU instructions of one wave; issued back to back by one wave, or by
// several waves in turn, the two streams mostly add up on a SIMD, interleaved one MFMA to a handful of VALU
// instructions they overlap.  Three LDS stages: tile T+2 is requested when tile T-1 has been read by every wave.
// SCALED: the queries carry scale * log2(e), and S^T starts from minus the running maximum instead of zero, so that the logits leave the MFMAs
// as exponents of 2: 16 multiply-adds per block less, of about 70 vector instructions beside 8 MFMAs that hardly overlap them (busy 59 + 37 % of
// the time).  The rows' maxima are exchanged between the lane halves only where one has grown.  16 / 48 x 2 705 tokens, when this was introduced: 57.1 / 143 us
// without, 53.9 / 134 with.
// The forward takes it: its queries are rounded to bf16 once, behind the scale.  The instance without is for callers whose queries are bf16 already
// (rtvla_attention): rounded again behind the scale, their outputs' error against 64 bits would go from 2.3e-3 to 3.0e-3, in sharp rows (logits of
// standard deviation 6) from 1.7e-3 to 4.8e-3.
template <int HD, bool SCALED>
__global__ __launch_bounds__(256, 3)
void flash_kernel(AttnP p, int items_per_batch, int batches_per_xcd) {
    static_assert(HD == 64, "fragment bookkeeping below is written out for a head width of 64");
    constexpr int KD = HD / 32;                         // 32-wide chunks of the head dimension in the fragment layouts
    constexpr int DS = HD / 16;                         // 16-wide steps of the Q K^T contraction
    constexpr int DT2 = HD / 32;                        // 32-wide tiles of the output's head dimension
    constexpr int KBYTES = 64 * HD * 2;                 // one K tile (64 keys); a V^T tile is as large
    constexpr int NPT = KBYTES / 16 / 256;              // 16-byte pieces per thread and operand
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];   // FLASH_STAGES x { K tile | V^T tile }

    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int h = lane >> 5, n = lane & 31;
    // Workgroup ids are dealt round-robin over the 8 XCDs: decode the id so that all row blocks of one K/V head run on
    // one XCD and its K / V^T are fetched into one L2.
    int batch, item;
    if (batches_per_xcd > 0) {
        // (the last row blocks of the heads, which may have few rows, come last: 48 heads x 2 705 rows are 1 008 whole blocks on 768 places, and 48 of 17 rows)
        const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3, whole = batches_per_xcd * (items_per_batch - 1);
        batch = xcd * batches_per_xcd + (idx < whole ? idx / (items_per_batch - 1) : idx - whole);
        item = idx < whole ? idx % (items_per_batch - 1) : items_per_batch - 1;
    } else { batch = blockIdx.x / items_per_batch; item = blockIdx.x % items_per_batch; }
    const bf16_t* const qbase = p.q + (size_t)batch * p.q_bstride;
    const uint4* const kbase = (const uint4*)(p.k + (size_t)batch * p.k_bstride);
    const uint4* const vbase = (const uint4*)(p.vt + (size_t)batch * p.vt_bstride);
    const int row0 = (item * 4 + w) * 32;
    const bool active = __builtin_amdgcn_readfirstlane(row0) < p.rows;         // a wave past the last row still stages tiles and meets the barriers

    bf16x8 qf[DS];
#pragma unroll
    for (int s4 = 0; s4 < DS; ++s4) {
        const size_t piece = ((size_t)((row0 >> 4) + (n >> 4)) * KD + (s4 >> 1)) * 64 + (2 * (s4 & 1) + h) * 16 + (n & 15);
        qf[s4] = active ? *(const bf16x8*)(qbase + piece * 8) : bf16x8{};
    }
    f32x16 o[DT2];
#pragma unroll
    for (int t = 0; t < DT2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[t][e] = 0.f;
    float m = NEG_BIG, l = 0.f;
    const float c = SCALED ? 1.0f : p.scale * 1.4426950408889634f;
    const float slack = RESCALE_BITS / c;               // the same threshold in units of the raw logits
    f32x16 start;                                       // what S^T starts from: - m (SCALED), 0
#pragma unroll
    for (int e = 0; e < 16; ++e) start[e] = 0.f;

    const int keys32 = (p.keys + 31) >> 5, ldvt32 = p.ldvt >> 5;
    int ntiles = (p.keys + 63) >> 6;
    if (p.causal) ntiles = min(ntiles, ((min(item * 128 + 128, p.rows) - 1) / p.group >> 6) + 1);

    // Staging: each wave copies whole 1 KB pieces (64 lanes x 16 bytes, contiguous on both sides) from global memory straight
    // into LDS; no staging registers and no LDS write instructions.  Stage T % 3 holds what tile T reads: V^T of tile T and K of tile T + 1 (step g takes
    // S^T of block g + 1, and reads the K fragments of g + 2).  It is requested when tile T - 3 has been read by every wave and awaited two tiles later: with K and V^T of one
    // tile in a stage, K of a tile is dead when the tile runs, and the requests had one tile's time.  Only the last tile can reach past the allocated rows (an odd number of
    // 32-key blocks): its second block is then replaced by the first (finite data; those keys are masked below).  A request past the last tile repeats
    // the last tile (for nobody).
    typedef __attribute__((address_space(3))) void* lptr_t;
    const int wu = __builtin_amdgcn_readfirstlane(w);                           // wave-uniform copy: everything but the lane's offset stays scalar
    unsigned koff[NPT], voff[NPT];                                              // this lane's byte offsets inside a tile
#pragma unroll
    for (int cc = 0; cc < NPT; ++cc) {
        const int i0 = wu * 64 + 256 * cc;                                      // first piece of this wave's 1 KB
        koff[cc] = (unsigned)(i0 + lane) * 16u;
        voff[cc] = (unsigned)(((i0 >> 7) * ldvt32 + ((i0 & 127) >> 6)) * 64 + lane) * 16u;
    }
    const int half_tile = (keys32 & 1) ? (keys32 >> 1) : -1;                    // the tile that holds a single 32-key block
    auto request = [&](const void* base, unsigned off, int at) __attribute__((always_inline)) {
#ifdef __HIP_DEVICE_COMPILE__                                                  // (the host pass does not know the LDS load's size)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)base, 0, -1, 0x00027000), (lptr_t)(smem + at), 16, (int)off, 0, 0, 0);
#endif
    };
    auto stage_k = [&](int t, unsigned stage_off) __attribute__((always_inline)) {
        t = min(t, ntiles - 1);
#pragma unroll
        for (int cc = 0; cc < NPT; ++cc) {
            const int i0 = wu * 64 + 256 * cc;
            const bool second = ((i0 / (KD * 128)) & 1) != 0;                   // pieces of keys 32..63 of the tile
            request((const unsigned char*)kbase + (size_t)t * KBYTES - (t == half_tile && second ? KD * 128 * 16 : 0), koff[cc], stage_off + i0 * 16);
        }
    };
    auto stage_v = [&](int t, unsigned stage_off) __attribute__((always_inline)) {
        t = min(t, ntiles - 1);
#pragma unroll
        for (int cc = 0; cc < NPT; ++cc) {
            const int i0 = wu * 64 + 256 * cc;
            request((const unsigned char*)vbase + (size_t)t * (128 * 16) - (t == half_tile && ((i0 & 127) >> 6) ? 64 * 16 : 0), voff[cc], stage_off + KBYTES + i0 * 16);
        }
    };

    // fragment reads of a 32-key block: the lane-dependent part of the address is shared by all of them, the stage is a
    // scalar byte offset that rotates once per tile
    const int lane_piece = ((n >> 4) * KD * 64 + h * 16 + (n & 15)) * 16;
    const int lane_piece_v = ((n >> 4) * 2 * 64 + h * 16 + (n & 15)) * 16 + KBYTES;
    auto piece_k = [&](unsigned stage_off, int b, int s4) __attribute__((always_inline)) {
        return *(const bf16x8*)(smem + stage_off + lane_piece + ((2 * b * KD + (s4 >> 1)) * 64 + 2 * (s4 & 1) * 16) * 16);
    };
    auto read_k = [&](unsigned stage_off, int b, bf16x8 (&kf)[DS]) __attribute__((always_inline)) {
#pragma unroll
        for (int s4 = 0; s4 < DS; ++s4) kf[s4] = piece_k(stage_off, b, s4);
    };
    auto piece_v = [&](unsigned stage_off, int b, int q, int t) __attribute__((always_inline)) {
        return *(const bf16x8*)(smem + stage_off + lane_piece_v + ((2 * t * 2 + b) * 64 + 2 * q * 16) * 16);
    };
    const bf16x2 ones = {(bf16_t)1.0f, (bf16_t)1.0f};
    // masks of block g: keys past the end, and (causal) keys after the row's own token
    auto mask = [&](int g, f32x16& st) __attribute__((always_inline)) {
        const int last = p.causal ? min(p.keys - 1, (row0 + n) / p.group) : p.keys - 1;
#pragma unroll
        for (int e = 0; e < 16; ++e)
            if (g * 32 + 8 * (e >> 2) + 4 * h + (e & 3) > last) st[e] = NEG_BIG;
    };
    auto lane_max = [&](const f32x16& st) __attribute__((always_inline)) {
        const auto max3 = [](float a, float b, float c) { return fmaxf(fmaxf(a, b), c); };
        const float mx0 = max3(max3(max3(st[0], st[1], st[2]), st[3], st[4]), st[5], st[6]), mx1 = max3(max3(max3(st[8], st[9], st[10]), st[11], st[12]), st[13], st[14]);
        return max3(mx0, mx1, fmaxf(st[7], st[15]));
    };
    // One pipeline step for block g = 2 T + b.  On entry: s_cur = S^T(g), kf = K fragments of block g+1, vf = V^T fragments and
    // p_prev = probabilities of block g-1.  On exit: s_next = S^T(g+1), kf = K fragments of g+2, vf / p_cur those of block g.
    // `off` is the stage of tile T, which holds block g's half of V^T and, as the same half of K, block g+2.
    auto step = [&](auto edge_tag, int g, int b, unsigned off, f32x16& s_cur, f32x16& s_next, bf16x8 (&kf)[DS],
                    bf16x8 (&vf)[2][DT2], bf16x8 (&p_prev)[2], bf16x8 (&p_cur)[2]) __attribute__((always_inline)) {
        constexpr bool EDGE = decltype(edge_tag)::value;
        if (EDGE) mask(g, s_cur);
        const float mx = SCALED ? lane_max(s_cur) : halves_max(lane_max(s_cur));
        if (__builtin_expect(__any(mx > (SCALED ? slack : m + slack)), 0)) {
            // rare: the accumulator and the pending probabilities of block g-1 (still in the old scale) move to the new one
            const float mnew = SCALED ? m + fmaxf(halves_max(mx), 0.f) : fmaxf(m, mx);
            const float alpha = __builtin_amdgcn_exp2f((m - mnew) * c);
            if constexpr (SCALED) {
#pragma unroll
                for (int e = 0; e < 16; ++e) { s_cur[e] += m - mnew; start[e] += m - mnew; }
            }
            l *= alpha;
#pragma unroll
            for (int t = 0; t < DT2; ++t)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[t][e] *= alpha;
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int j = 0; j < 8; ++j) p_prev[q][j] = (bf16_t)((float)p_prev[q][j] * alpha);
            m = mnew;
        }
        // ---- the straight-line part: 8 MFMAs, the softmax of block g, 8 fragment reads ----
        static_assert(DS == 2 * DT2, "MFMAs in pairs");
        s_next = start;
#pragma unroll
        for (int i = 0; i < DS; ++i) {                   // (in turn: the four of S^T are a chain)
            const int q = i / DT2, t = i % DT2;
            o[t] = mfma32(vf[q][t], p_prev[q], o[t]);
            s_next = mfma32(kf[i], qf[i], s_next);
            vf[q][t] = piece_v(off, b, q, t);
            kf[i] = piece_k(off, b, i);
        }
        const float mc = m * c;
#pragma unroll
        for (int e = 0; e < 16; ++e) s_cur[e] = __builtin_amdgcn_exp2f(SCALED ? s_cur[e] : s_cur[e] * c - mc);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            p_cur[q] = pack8(s_cur, q, q + 2);
            // the row sum takes the rounded probabilities, two per instruction (v_dot2_f32_bf16)
#pragma unroll
            for (int j = 0; j < 8; j += 2) l = __builtin_amdgcn_fdot2_f32_bf16(bf16x2{p_cur[q][j], p_cur[q][j + 1]}, ones, l, false);
        }
        // issue order: one MFMA to every six (SCALED: four) VALU instructions of the softmax; the fragment reads of the next step go into
        // the registers that the pair of MFMAs before them has consumed
        constexpr int PER = SCALED ? 4 : 6;
#pragma unroll
        for (int i = 0; i < DS; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x402, PER, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x402, PER, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        // the probabilities are made here: their first use is behind the barrier of the tile, and left to itself the compiler moves the softmax of
        // every second block there, away from the MFMAs that it is to run beside
        asm volatile("" :: "v"(p_cur[0]), "v"(p_cur[1]), "v"(l));
    };

    constexpr unsigned STAGE = 2 * KBYTES;
    stage_k(0, 2 * STAGE);
    stage_v(0, 0); stage_k(1, 0);
    stage_v(1, STAGE); stage_k(2, STAGE);
    wait_and_meet<2 * NPT>();                           // all but the last stage are in LDS

    f32x16 sA, sB;
    bf16x8 kf[DS], vf[2][DT2], pP[2], pC[2];
    read_k(2 * STAGE, 0, kf);
#pragma unroll
    for (int e = 0; e < 16; ++e) sA[e] = 0.f;
#pragma unroll
    for (int s4 = 0; s4 < DS; ++s4) sA = mfma32(kf[s4], qf[s4], sA);
    if constexpr (SCALED) {                             // the first block's maxima
        mask(0, sA);
        m = halves_max(lane_max(sA));
#pragma unroll
        for (int e = 0; e < 16; ++e) { sA[e] -= m; start[e] = -m; }
    }
    read_k(2 * STAGE, 1, kf);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        pP[q] = bf16x8{};                               // "block -1": zero probabilities, any finite V^T
#pragma unroll
        for (int t = 0; t < DT2; ++t) vf[q][t] = bf16x8{};
    }
    unsigned off = 0, off_next2 = 2 * STAGE;            // stages of tile T and of tile T+2
    wait_and_meet<2 * NPT>();                           // everybody has read K of tile 0 (and with no scalar load under way the loop's waits are for single LDS reads)
    auto tile = [&](auto edge_tag, int T) __attribute__((always_inline)) {
        stage_v(T + 2, off_next2);
        stage_k(T + 3, off_next2);
        if (active) {
            step(edge_tag, 2 * T, 0, off, sA, sB, kf, vf, pP, pC);
            step(edge_tag, 2 * T + 1, 1, off, sB, sA, kf, vf, pC, pP);        // (K past the last tile: that one's again, never used)
        }
        off_next2 = off;
        off = off == (FLASH_STAGES - 1) * STAGE ? 0 : off + STAGE;
        wait_and_meet<2 * NPT>();                       // stage T+1 has landed, stage T has been read
    };
    // only the last tile of a non-causal pass has keys to mask
    const int plain_tiles = p.causal ? 0 : ntiles - 1;
    for (int T = 0; T < plain_tiles; ++T) tile(std::false_type{}, T);
    for (int T = plain_tiles; T < ntiles; ++T) tile(std::true_type{}, T);
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int t = 0; t < DT2; ++t) o[t] = mfma32(vf[q][t], pP[q], o[t]);

    __builtin_amdgcn_s_waitcnt(0x0f70);                 // vmcnt(0): nothing may land in LDS after the workgroup has ended
    l = halves_sum(l);
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    const int row = row0 + n;
    if (row < p.rows) {
#pragma unroll
        for (int t = 0; t < DT2; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                store4(flash_out_ptr(p, batch, row, 32 * t + 8 * j + 4 * h, HD),
                       pack4(o[t][4 * j] * inv, o[t][4 * j + 1] * inv, o[t][4 * j + 2] * inv, o[t][4 * j + 3] * inv));
    }
}

}  // namespace

// p as for launch_mqa_attention, without the prefix / state masks and without a key split.  Q must be allocated in whole
// 32-row blocks up to the last valid row, K up to keys rounded up to 32 rows, V^T with p.ldvt >= that many key columns.
int launch_flash_attention(const AttnP& p0, int hd, hipStream_t s) {
    AttnP p = p0;
    if (p.rows <= 0 || p.keys <= 0 || (p.ldvt & 31) || p.ldvt < ((p.keys + 31) / 32) * 32 || p.group < 1) return 1;
    if (p.valid_len || p.state_rows || p.prefix_alloc < p.keys || p.nsplit > 1) return 1;
    if (p.batch < 1) p.batch = 1;
    if (p.batch_inner < 1) p.batch_inner = 1;
    const int items = (p.rows + 127) / 128;
    const int bpx = (p.batch % 8 == 0) ? p.batch / 8 : 0;
    if (hd != 64) return 2;
    if (p.q_scaled) hipLaunchKernelGGL((flash_kernel<64, true>), dim3(items * p.batch), dim3(256), FLASH_STAGES * 2 * 64 * 64 * 2, s, p, items, bpx);
    else hipLaunchKernelGGL((flash_kernel<64, false>), dim3(items * p.batch), dim3(256), FLASH_STAGES * 2 * 64 * 64 * 2, s, p, items, bpx);
    return hipGetLastError() == hipSuccess ? 0 : 5;
}
