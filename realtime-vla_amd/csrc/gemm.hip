// Large-M bf16 GEMM on MFMA for the SigLIP and Gemma-prefix layers
// (replaces the Triton GEMM family of /root/reference/pi0_infer.py:5-346, :664-691, :777-810).
//
// out[M][N] = epilogue(A[M][K] * W[K][N]) with v_mfma_f32_32x32x16_bf16: measured on MI355X this
// instruction sustains ~2.1 PFLOP/s with a single wave per SIMD, while streams of independent
// 16x16x32 MFMAs issue at half that rate.  The activations A are staged through LDS in MFMA
// operand-fragment order (each wave reads whole 1 KB fragments with ds_read_b128, conflict free) and
// are shared by all waves of the workgroup; the weights are read straight from their pre-tiled layout
// in HBM into registers (one coalesced 1 KB load per fragment, no LDS round trip), each wave owning
// its own column tiles.  The product is computed transposed (weights as the MFMA A operand) so that
// every lane ends up with 4 groups of 4 consecutive output columns of one row: 8-byte packed stores,
// and RoPE pairs / GeGLU partners sit in the same lane.
#include "kernels.h"
#include "gemm_scatter.h"
#include <algorithm>
#include <type_traits>

namespace {

template <int EPI> struct EpiTraits { static constexpr bool dual = (EPI == EPI_GEGLU || EPI == EPI_SWIGLU); };

RTVLA_DEVICE f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }

// MT, NT: 32-row tiles per workgroup and 32-column tiles per wave.  Small tiles are compiled to fit two
// workgroups per CU so that one workgroup's MFMAs run under the other's memory latency.
// One block tile of MT 32-row tiles starting at row m0: K loop and epilogue.
// V: a tile of V columns, whose product is taken as activations x weights (gemm_scatter.h)
// KG: one group of WN waves, or two that share a block tile and split its K stages, each with stage buffers of its own.  For launches of few workgroups, where
// the waves of a CU wait for their loads: two groups have twice as much on the way and half as many stages one after another.  us of a whole layer with one / two
// groups, weights cold: DM0's prefix QKV, K = 2 048, 206 rows (64 x 128) 75.8 / 74.0, 398 90.9 / 89.1, 607 (96 x 128) 105.9 / 105.0, Gemma's, 968 rows 235.4 / 232.6, ViT
// down projection, K = 4 096, 2 720 rows 161.4 / 159.2.  With two groups a tile of 64 x 64 has eight 32 x 32 products a stage for four waves, which on its own would be two waves
// to a CU; it doubles the workgroups where 64 x 128 leaves half of the chip idle: Gemma QKV, 256 rows, 80 workgroups of 64 x 128 105.6, 160 of 64 x 64 99.9; SigLIP QKV 256 rows 53.8 /
// 51.7.  Where the chip is full it gives nothing (SigLIP up, 768 rows, 128 x 128 69.1 / 69.1) or less (dual tiles of 64 x 256: GeGLU, 256 rows 105.6 / 117.8), and neither do three or four
// groups.
template <int WN, int MT, int NT, int EPI, int KG = 1>
struct GemmLds {
    static constexpr bool f32 = EPI == EPI_PARTIAL || EPI == EPI_RESIDUAL;
    static constexpr int stages = 3 * MT * 32 * 128;                                   // of one group
    static constexpr int out_tile = 32 * (WN * (EpiTraits<EPI>::dual ? NT / 2 : NT) * 32 * (f32 ? 4 : 2) + 16);
    static constexpr int group = stages > out_tile ? stages : out_tile;                // a group's own memory
    static constexpr int sums = KG == 2 ? MT * WN * NT * 4096 : 0;                     // the tiles the groups hand each other
    static constexpr int bytes = KG * group > sums ? KG * group : sums;
};
template <int WN, int MT, int NT, int EPI, bool V = false, int KG = 1>
RTVLA_DEVICE void gemm_block(const GemmP& pk, unsigned char* smem_all, int m0_wg, int n_blk, int split, int stages_total, int stages_per_split) {
    constexpr int NTH = WN * 64;
    using Lds = GemmLds<WN, MT, NT, EPI, KG>;
    constexpr int BM = MT * 32;
    constexpr int A_CHUNKS = BM * 8;                       // 16-byte chunks per 64-wide K stage
    constexpr int AIT = (A_CHUNKS + NTH - 1) / NTH;
    constexpr int STAGE_ELEMS = BM * 64;
    const int kg = KG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / NTH) : 0;
    unsigned char* const smem_raw = smem_all + kg * Lds::group;
    bf16_t* lds = (bf16_t*)smem_raw;

    const int tid = threadIdx.x - kg * NTH, lane = tid & 63, wn = tid >> 6;
    const int h = lane >> 5, r = lane & 31;
    int m0 = m0_wg;
    std::conditional_t<KG == 1, const GemmP&, GemmP> p = pk;
    const int s_begin = split * stages_per_split + kg * (stages_per_split / KG);
    const int s_end = min(s_begin + stages_per_split / KG, stages_total);

    // 32-column tiles of this wave
    constexpr int HALF = EpiTraits<EPI>::dual ? NT / 2 : NT;
    int tile_of[NT];
    const bf16_t* bptr[NT];
    const int n32 = (p.N16 + 1) >> 1;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int t = (n_blk * WN + wn) * HALF + (j % HALF);
        tile_of[j] = t;
        const bf16_t* base = (EpiTraits<EPI>::dual && j >= HALF) ? p.B1 : p.B0;
        const int G = p.bgroup;
        const int tc = min(t, ((n32 + G - 1) / G) * G - 1);
        bptr[j] = base + ((size_t)(tc / G) * (p.K32p * 2) * G + (tc % G)) * 512 + lane * 8;
    }

    const size_t bstep = (size_t)p.bgroup * 512;          // distance between consecutive k16 blocks of one column tile
    f32x16 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    bf16x8 areg0[AIT], areg1[AIT];
    bf16x8 breg0[NT][4], breg1[NT][4];

    // LDS stage layout: fragment (row tile i, k16 step ks) is 1 KB = 64 slots of 16 bytes; the chunk of row r
    // (0..31) and k half hh sits at slot 8 ((r >> 3) + 4 hh) + ((r + 2 ks + hh) & 7).  The low three bits pick
    // the 128-byte bank group: any 8 consecutive lanes of a fragment read (8 rows, one hh) and any 8
    // consecutive lanes of a staging write (one row, 8 chunks = 4 ks x 2 hh) land in 8 different bank
    // groups, so neither side conflicts.
    auto load_a = [&](int s, bf16x8 (&ar)[AIT]) __attribute__((always_inline)) {
#pragma unroll
        for (int it = 0; it < AIT; ++it) {
            // a ragged last round re-reads the final chunk instead of branching
            const int c = min(it * NTH + tid, A_CHUNKS - 1);
            const int row = c >> 3, kc = c & 7;
            const int gr = min(m0 + row, p.a_rows - 1);
            ar[it] = *(const bf16x8*)(p.A + (size_t)gr * p.lda + s * 64 + kc * 8);
        }
    };
    auto store_a = [&](bf16_t* buf, bf16x8 (&ar)[AIT]) __attribute__((always_inline)) {
#pragma unroll
        for (int it = 0; it < AIT; ++it) {
            const int c = min(it * NTH + tid, A_CHUNKS - 1);      // duplicates write identical data
            const int row = c >> 3, kc = c & 7, ks = kc >> 1, hh = kc & 1;
            const int rr = row & 31;
            const int off = ((((row >> 5) * 4 + ks) * 64) + 8 * ((rr >> 3) + 4 * hh) + ((rr + 2 * ks + hh) & 7)) * 8;
            *(bf16x8*)(buf + off) = ar[it];
        }
    };
    auto load_b_half = [&](int s, bf16x8 (&br)[NT][4], int kk) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int q = 0; q < 2; ++q) br[j][2 * kk + q] = *(const bf16x8*)(bptr[j] + (size_t)(s * 4 + 2 * kk + q) * bstep);
    };
    int lane_off[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) lane_off[ks] = (8 * ((r >> 3) + 4 * h) + ((r + 2 * ks + h) & 7)) * 8;
    // One K stage, software-pipelined so that nothing but MFMAs sits on the critical path:
    //  * LDS holds THREE stage buffers.  Stage t reads buffer `rd`; in its first half it also writes the
    //    activations of stage t+1 into `wr`, and the single barrier of the stage sits in the MIDDLE, between
    //    the two k halves, with MFMAs queued on both sides.  A wave that runs ahead into stage t+1 writes the
    //    third buffer, which everybody finished reading before that barrier, so one barrier per stage is
    //    enough, and the first fragments of stage t+1 are read before stage t ends (carried in `afn`).
    //  * global loads run two stages ahead: the activations of stage t+2 go to the register set that was
    //    stored to LDS during stage t-1, and each half of the weight registers is re-loaded with stage t+2 as
    //    soon as the MFMAs of stage t have consumed it, so no third register set is needed.
    //  * the scheduler is given the instruction order explicitly: fragment reads run PRE ahead of the MFMAs
    //    that use them and loads / LDS writes are spread one per MFMA group.
    constexpr int PRE = MT >= 3 ? 3 : MT;
    constexpr int HR = 2 * MT;                                          // fragment reads per k half
    static_assert(HR >= 2 * NT && AIT <= HR, "not enough MFMA groups to spread the loads over");
    bf16x8 afn[PRE];                                                    // first fragments of the coming stage
    auto frag = [&](const bf16_t* base, int f) __attribute__((always_inline)) {     // f = ks * MT + i
        const int ks = f / MT, i = f - ks * MT;
        return *(const bf16x8*)(base + (i * 4 + ks) * 512 + lane_off[ks]);
    };
    auto stage = [&](const bf16_t* rd, bf16_t* wr, int s_next, bf16x8 (&br)[NT][4], bf16x8 (&ar_next)[AIT], bf16x8 (&ar_store)[AIT]) __attribute__((always_inline)) {
        // ---- first k half ----
        load_a(s_next, ar_next);
        bf16x8 af[4 * MT];
#pragma unroll
        for (int f = 0; f < PRE; ++f) af[f] = afn[f];
#pragma unroll
        for (int f = PRE; f < HR + PRE; ++f) af[f] = frag(rd, f);      // includes the first PRE fragments of the second half
#pragma unroll
        for (int f = 0; f < HR; ++f)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[f % MT][j] = V ? mfma32(af[f], br[j][f / MT], acc[f % MT][j]) : mfma32(br[j][f / MT], af[f], acc[f % MT][j]);
        store_a(wr, ar_store);
#pragma unroll
        for (int t = 0; t < HR; ++t) {
            __builtin_amdgcn_sched_group_barrier(0x008, NT, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            if (t < AIT) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);                        // activation loads of stage t+2
            if (t >= HR - AIT) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);                  // LDS writes of stage t+1
        }
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        // ---- second k half ----
        load_b_half(s_next, br, 0);
#pragma unroll
        for (int f = HR + PRE; f < 2 * HR; ++f) af[f] = frag(rd, f);
#pragma unroll
        for (int f = 0; f < PRE; ++f) afn[f] = frag(wr, f);            // written before the barrier above
#pragma unroll
        for (int f = HR; f < 2 * HR; ++f)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[f % MT][j] = V ? mfma32(af[f], br[j][f / MT], acc[f % MT][j]) : mfma32(br[j][f / MT], af[f], acc[f % MT][j]);
        load_b_half(s_next, br, 1);
#pragma unroll
        for (int t = 0; t < HR; ++t) {
            __builtin_amdgcn_sched_group_barrier(0x008, NT, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            if (t < 2 * NT) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);                     // weight loads, k half 0 of stage t+2
        }
        __builtin_amdgcn_sched_group_barrier(0x020, 2 * NT, 0);                                    // weight loads, k half 1
        __builtin_amdgcn_sched_barrier(0);
    };

    // K loop, two stages per trip so the register sets alternate without a runtime index and the body has a
    // single exit; for the tiles of at most 128 rows an odd stage count ends in one peeled stage (the larger ones
    // need an even count).  The LDS buffers rotate through three
    // pointers.  Past the end the prefetch re-reads the last stage instead of branching.
    const int n_st = s_end - s_begin;
    if (n_st > 0) {
        const int last = s_end - 1;
        bf16_t* b0 = lds; bf16_t* b1 = lds + STAGE_ELEMS; bf16_t* b2 = lds + 2 * STAGE_ELEMS;
        load_a(s_begin, areg0);
        load_b_half(s_begin, breg0, 0); load_b_half(s_begin, breg0, 1);
        load_a(min(s_begin + 1, last), areg1);
        load_b_half(min(s_begin + 1, last), breg1, 0); load_b_half(min(s_begin + 1, last), breg1, 1);
        store_a(b0, areg0);
        __syncthreads();
#pragma unroll
        for (int f = 0; f < PRE; ++f) afn[f] = frag(b0, f);
        int s = s_begin;
        for (; s + 1 < s_end; s += 2) {
            stage(b0, b1, min(s + 2, last), breg0, areg0, areg1);
            stage(b1, b2, min(s + 3, last), breg1, areg1, areg0);
            bf16_t* t0 = b0; b0 = b2; b2 = b1; b1 = t0;     // (b0, b1, b2) <- (b2, b0, b1)
        }
        if constexpr (MT <= 4) {                            // (the large tiles have no registers to spare for a third copy of the stage)
            if (s < s_end) stage(b0, b1, last, breg0, areg0, areg1);
        }
    }
    // Each group keeps MTO of the row tiles and gets the other's sums of them for its own; from here on m0 and p.M are those of its rows.
    constexpr int MTO = (MT + KG - 1) / KG;
    f32x16 own[MTO][NT];
    if constexpr (KG == 1) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) own[i][j] = acc[i][j];
    } else {
        f32x4* const sums = (f32x4*)smem_all;
        static_assert(KG == 2, "each tile has one other sum");
        auto at = [&](int i, int j) __attribute__((always_inline)) { return sums + ((i * WN + wn) * NT + j) * 256 + lane; };
        __syncthreads();
#pragma unroll
        for (int i = 0; i < MT; ++i)
            if (i / MTO != kg)
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) at(i, j)[e * 64] = f32x4{acc[i][j][4 * e], acc[i][j][4 * e + 1], acc[i][j][4 * e + 2], acc[i][j][4 * e + 3]};
        __syncthreads();
#pragma unroll
        for (int g = 0; g < KG; ++g) {
            if (g != kg) continue;
#pragma unroll
            for (int k = 0; k < MTO; ++k) {
                const int i = g * MTO + k;
                if (i >= MT) continue;
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    f32x16 v = acc[i][j];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const f32x4 o = at(i, j)[e * 64];
#pragma unroll
                        for (int q = 0; q < 4; ++q) v[4 * e + q] += o[q];
                    }
                    own[k][j] = v;
                }
            }
        }
        m0 += kg * MTO * 32;
        p.M = min(p.M, m0_wg + min((kg + 1) * MTO, MT) * 32);
    }
    // the bias of this wave's columns, asked for as one: a load per group of four columns is a branch and a trip to the cache for each
    // (768 x 1 152 x 4 304 with GELU, in a trace: 17.4 -> 15.9 us)
    constexpr bool BIAS = EPI == EPI_BIAS || EPI == EPI_BIAS_GELU || EPI == EPI_PATCH || EPI == EPI_RESIDUAL;
    f32x4 bias[BIAS ? HALF : 1][4];
    if constexpr (BIAS) {
        auto col = [&](int j, int grp) { return min((n_blk * (WN * HALF) + wn * HALF + j) * 32 + 8 * grp + 4 * h, p.N16 * 16 - 4); };      // clamped: columns past the end are never copied out
        if (p.bias_f32) {
#pragma unroll
            for (int j = 0; j < HALF; ++j)
#pragma unroll
                for (int grp = 0; grp < 4; ++grp) bias[j][grp] = *(const f32x4*)(p.bias_f32 + col(j, grp));
        } else {
            bf16x4 b[HALF][4];
#pragma unroll
            for (int j = 0; j < HALF; ++j)
#pragma unroll
                for (int grp = 0; grp < 4; ++grp) b[j][grp] = load4(p.bias + col(j, grp));
#pragma unroll
            for (int j = 0; j < HALF; ++j)
#pragma unroll
                for (int grp = 0; grp < 4; ++grp)
#pragma unroll
                    for (int e = 0; e < 4; ++e) bias[j][grp][e] = bf2f(b[j][grp][e]);
        }
    }
    float factor[EPI == EPI_SWIGLU ? MTO : 1];
    if constexpr (EPI == EPI_SWIGLU)
#pragma unroll
        for (int i = 0; i < MTO; ++i) factor[i] = p.rowscale[min(m0 + i * 32 + r, p.M - 1)];
    __syncthreads();                                        // the epilogue reuses the stage buffers

    // ---- epilogue: lane (h, r) holds rows m = m0 + 32 i + r, columns n = 32 tile + 8 grp + 4 h + e ----
    // Row-major outputs go through LDS one 32-row tile at a time so that the global stores are whole
    // 16-byte chunks of contiguous row segments (256 B - 1 KB per row) instead of 8-byte pieces of 32 rows.
    constexpr bool ROWMAJOR = (EPI == EPI_BIAS || EPI == EPI_BIAS_GELU || EPI == EPI_PATCH || EPI == EPI_GEGLU || EPI == EPI_SWIGLU || EPI == EPI_PARTIAL ||
                              EPI == EPI_RESIDUAL);
    if constexpr (ROWMAJOR) {
        constexpr bool RES = EPI == EPI_RESIDUAL;                  // staged as fp32: the residual joins on the way out, where a row's chunks are contiguous
        constexpr int ESZ = (EPI == EPI_PARTIAL || RES) ? 4 : 2;
        constexpr int OUTW = WN * HALF * 32;                       // output columns of the workgroup
        constexpr int ROWB = OUTW * ESZ + 16;                      // padded LDS row pitch in bytes
        constexpr int COLS = EPI == EPI_PARTIAL ? 4 : 8;           // columns of a 16-byte output chunk
        constexpr int CPR = OUTW / COLS;                           // chunks per row
        constexpr int RPP = NTH / CPR;                             // rows per copy pass
        static_assert(NTH % CPR == 0 && 32 % RPP == 0, "copy-out mapping");
        unsigned char* obuf = smem_raw;
        const int nbase = n_blk * OUTW;
        const int ncols = p.N16 * 16;
        // As many 32-row tiles as fit into the stage buffers are converted and staged back to back, then copied out
        // back to back: one barrier pair per group instead of one per tile, and the stores of a group stream.
        constexpr int TILE_B = 32 * ROWB;
        constexpr int GROUP = Lds::group / TILE_B >= MTO ? MTO : (Lds::group / TILE_B < 1 ? 1 : Lds::group / TILE_B);
#pragma unroll
        for (int g0 = 0; g0 < MTO; g0 += GROUP) {
          bf16x8 res[RES ? GROUP * (32 / RPP) : 1];
          if constexpr (RES) {
#pragma unroll
            for (int k = 0; k < GROUP * (32 / RPP); ++k) {
                const int mm = min(m0 + (g0 + k / (32 / RPP)) * 32 + (k % (32 / RPP)) * RPP + tid / CPR, p.M - 1), n = min(nbase + (tid % CPR) * COLS, ncols - COLS);
                res[k] = *(const bf16x8*)(p.res + (size_t)mm * p.ldr + n);
            }
          }
#pragma unroll
          for (int i = g0; i < (g0 + GROUP < MTO ? g0 + GROUP : MTO); ++i) {
            if (m0 + i * 32 >= p.M) continue;                                     // a row tile past the end (uniform)
            const int m = m0 + i * 32 + r;
            unsigned char* const tbuf = obuf + (i - g0) * TILE_B;
#pragma unroll
            for (int j = 0; j < HALF; ++j) {
#pragma unroll
                for (int grp = 0; grp < 4; ++grp) {
                    const int cl = (wn * HALF + j) * 32 + 8 * grp + 4 * h;        // column inside the workgroup tile
                    const int n0 = min(nbase + cl, ncols - 4);                    // clamped: out-of-range columns are never copied out
                    f32x4 v = {own[i][j][4 * grp], own[i][j][4 * grp + 1], own[i][j][4 * grp + 2], own[i][j][4 * grp + 3]};
                    unsigned char* dst = tbuf + r * ROWB + cl * ESZ;
                    if constexpr (EPI == EPI_PARTIAL) {
                        *(f32x4*)dst = v;
                    } else if constexpr (EPI == EPI_GEGLU) {
                        const f32x4 u = {own[i][j + HALF][4 * grp], own[i][j + HALF][4 * grp + 1], own[i][j + HALF][4 * grp + 2], own[i][j + HALF][4 * grp + 3]};
                        *(bf16x4*)dst = pack4(gelu_tanh(v[0]) * u[0], gelu_tanh(v[1]) * u[1], gelu_tanh(v[2]) * u[2], gelu_tanh(v[3]) * u[3]);
                    } else if constexpr (EPI == EPI_SWIGLU) {
                        const float f = factor[i];
                        f32x4 u = {own[i][j + HALF][4 * grp], own[i][j + HALF][4 * grp + 1], own[i][j + HALF][4 * grp + 2], own[i][j + HALF][4 * grp + 3]};
                        v *= f; u *= f;
                        *(bf16x4*)dst = pack4(siluf(v[0]) * u[0], siluf(v[1]) * u[1], siluf(v[2]) * u[2], siluf(v[3]) * u[3]);
                    } else {
                        v += bias[j][grp];
                        if constexpr (EPI == EPI_PATCH) {
                            const bf16x4 rs = load4(p.res + (size_t)(min(m, p.M - 1) % p.res_mod) * p.ldr + n0);
#pragma unroll
                            for (int e = 0; e < 4; ++e) v[e] += bf2f(rs[e]);
                        }
                        if constexpr (EPI == EPI_BIAS_GELU) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) v[e] = gelu_tanh(v[e]);
                        }
                        if constexpr (RES) *(f32x4*)dst = v;
                        else *(bf16x4*)dst = pack4(v);
                    }
                }
            }
          }
          __syncthreads();
#pragma unroll
          for (int i = g0; i < (g0 + GROUP < MTO ? g0 + GROUP : MTO); ++i) {
            const unsigned char* const tbuf = obuf + (i - g0) * TILE_B;
#pragma unroll
            for (int ps = 0; ps < 32 / RPP; ++ps) {
                const int row = ps * RPP + tid / CPR, ch = tid % CPR;
                const int mm = m0 + i * 32 + row;
                const int n = nbase + ch * COLS;
                if (mm < p.M && n < ncols) {
                    if constexpr (RES) {
                        f32x4 lo = *(const f32x4*)(tbuf + row * ROWB + ch * 32), hi = *(const f32x4*)(tbuf + row * ROWB + ch * 32 + 16);
                        const bf16x8 rs = res[(i - g0) * (32 / RPP) + ps];
#pragma unroll
                        for (int e = 0; e < 4; ++e) { lo[e] += bf2f(rs[e]); hi[e] += bf2f(rs[4 + e]); }
                        const bf16x4 a = pack4(lo), b = pack4(hi);
                        *(uint4*)(p.out + (size_t)mm * p.ldo + n) = uint4{((const uint2*)&a)->x, ((const uint2*)&a)->y, ((const uint2*)&b)->x, ((const uint2*)&b)->y};
                        continue;                                  // (no streaming hint: the normalising pass reads it next)
                    }
                    const uint4 val = *(const uint4*)(tbuf + row * ROWB + ch * 16);
                    // (streaming hint: the output is read once by the next launch and should not displace the operand tiles in L2)
                    if constexpr (EPI == EPI_PARTIAL) __builtin_nontemporal_store(*(const f32x4*)&val, (f32x4*)(p.partial + (size_t)split * p.pstride + (size_t)mm * p.ldp + n));
                    else __builtin_nontemporal_store(*(const f32x4*)&val, (f32x4*)(p.out + (size_t)mm * p.ldo + n));
                }
            }
          }
          if (g0 + GROUP < MTO) __syncthreads();
        }
    } else {
        static_assert(epi_scatters(EPI), "every epilogue is one of the two kinds");
        if constexpr (EPI == EPI_GQA_QKV) {
            static_assert(WN == 4 && NT == 1, "a head is 128 columns");
            scatter_head<MTO, V>(p, own, (float*)smem_raw, m0, tile_of[0] * 32, wn, lane);
            return;
        }
        else scatter_tiles<EPI, V>(p, own, MTO, m0, tile_of, lane);
    }
}

// Workgroup -> block tile.  Row blocks come in two sizes when MIXED: the first n_big blocks have MT 32-row tiles, the
// others MT - 1, so that M rows are covered with ceil(M / 32) tiles instead of a multiple of MT (788 rows: 7 + 6 + 6 + 6 =
// 25 tiles where four 7-tile blocks would compute 28).
template <int WN, int MT, int NT, int EPI, bool MIXED, int KG = 1>
__global__ __launch_bounds__(WN * 64 * KG, (MT <= 2 && WN == 4 && KG == 1 ? 2 : 1))
void gemm_mfma_kernel(GemmP p, int m_blocks, int n_blocks, int stages_total, int stages_per_split, int n_big) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int total = m_blocks * n_blocks * p.nsplit;
    const int lid = xcd_remap(blockIdx.x, total);
    const int split = lid / (m_blocks * n_blocks);
    const int rem = lid - split * (m_blocks * n_blocks);
    const int n_blk = rem / m_blocks;
    const int m_blk = rem - n_blk * m_blocks;
    auto block = [&](auto v) __attribute__((always_inline)) {
        if constexpr (MIXED) {
            if (m_blk < n_big) gemm_block<WN, MT, NT, EPI, v.value>(p, smem_raw, m_blk * (MT * 32), n_blk, split, stages_total, stages_per_split);
            else gemm_block<WN, MT - 1, NT, EPI, v.value>(p, smem_raw, n_big * (MT * 32) + (m_blk - n_big) * ((MT - 1) * 32), n_blk, split, stages_total, stages_per_split);
        } else {
            gemm_block<WN, MT, NT, EPI, v.value, KG>(p, smem_raw, m_blk * (MT * 32), n_blk, split, stages_total, stages_per_split);
        }
    };
    if constexpr (epi_scatters(EPI)) {
        if (n_blk * (WN * NT * 32) >= epi_first_v(EPI)) { block(std::true_type{}); return; }
    }
    block(std::false_type{});
}

template <int WN, int MT, int NT, int EPI, bool MIXED, int KG = 1>
int launch_cfg(const GemmP& p, hipStream_t s) {
    constexpr int HALF = EpiTraits<EPI>::dual ? NT / 2 : NT;
    const int tiles = (p.M + 31) / 32;
    int m_blocks = (tiles + MT - 1) / MT, n_big = m_blocks;
    if (MIXED) {
        n_big = tiles - m_blocks * (MT - 1);               // blocks that need the MT-th tile
        if (n_big < 0) n_big = 0;
    }
    const int n_blocks = ((p.N16 + 1) / 2 + WN * HALF - 1) / (WN * HALF);
    const int stages_total = p.K32p / 2;
    const int nsplit = p.nsplit < 1 ? 1 : p.nsplit;
    const int sps = (stages_total + nsplit - 1) / nsplit;
    if ((nsplit - 1) * sps >= stages_total) return 3;      // an empty split would leave its partial unwritten
    if (MT > 4 && ((sps & 1) || (stages_total & 1))) return 3;              // the large tiles consume K stages in pairs
    if constexpr (KG > 1)                                  // the groups meet at every barrier, so they have as many stages each (a caller's own split need not give them that)
        if (sps % KG || stages_total % sps) return launch_cfg<4, MT, NT, EPI, MIXED>(p, s);
    GemmP q = p; q.nsplit = nsplit;
    // three K-stage buffers; the row-major epilogues stage 32-row output tiles in the same memory
    constexpr size_t smem = GemmLds<WN, MT, NT, EPI, KG>::bytes;
    static_assert(smem <= 160 * 1024, "LDS");
    auto kern = gemm_mfma_kernel<WN, MT, NT, EPI, MIXED, KG>;
    if (smem > 65536) {
        static std::atomic<uint64_t> done{0};
        if (int rc = ensure_dynamic_lds((const void*)kern, smem, done)) return rc;
    }
    hipLaunchKernelGGL(kern, dim3(m_blocks * n_blocks * nsplit), dim3(WN * 64 * KG), smem, s, q, m_blocks, n_blocks, stages_total, sps, n_big);
    return hipGetLastError() == hipSuccess ? 0 : 5;
}

template <int EPI>
int launch_epi(const GemmP& p, int tile, hipStream_t s) {
    switch (tile) {
        case TILE_224x256: if constexpr (EPI != EPI_GQA_QKV) return launch_cfg<4, 7, 2, EPI, true>(p, s); else return 2;
        case TILE_192x256: if constexpr (EPI != EPI_GQA_QKV) return launch_cfg<4, 6, 2, EPI, true>(p, s); else return 2;
        case TILE_160x256: if constexpr (EPI != EPI_GQA_QKV) return launch_cfg<4, 5, 2, EPI, true>(p, s); else return 2;
        case TILE_128x256: if constexpr (EPI != EPI_GQA_QKV) return launch_cfg<4, 4, 2, EPI, true>(p, s); else return 2;
        case TILE_64x256:  if constexpr (EPI != EPI_GQA_QKV) return launch_cfg<4, 2, 2, EPI, false>(p, s); else return 2;
        case TILE_64x128:  if constexpr (!EpiTraits<EPI>::dual) return launch_cfg<4, 2, 1, EPI, false>(p, s); else return 2;
        case TILE_128x128: if constexpr (!EpiTraits<EPI>::dual) return launch_cfg<4, 4, 1, EPI, false>(p, s); else return 2;
        case TILE_96x128:  if constexpr (!EpiTraits<EPI>::dual) return launch_cfg<4, 3, 1, EPI, false>(p, s); else return 2;
        case TILE2_64x64:  if constexpr (!EpiTraits<EPI>::dual && EPI != EPI_GQA_QKV) return launch_cfg<2, 2, 1, EPI, false, 2>(p, s); else return 2;
        case TILE2_64x128: if constexpr (!EpiTraits<EPI>::dual) return launch_cfg<4, 2, 1, EPI, false, 2>(p, s); else return 2;
        case TILE2_96x128: if constexpr (!EpiTraits<EPI>::dual) return launch_cfg<4, 3, 1, EPI, false, 2>(p, s); else return 2;
    }
    return 2;
}

}  // namespace

int gemm_tile_bm(int tile) { static const int v[TILE_END] = {224, 192, 160, 128, 64, 64, 128, 256, 224, 192, 128, 96, 160, 64, 64, 96}; return v[tile]; }
int gemm_tile_bn(int tile) { return tile == TILE2_64x64 ? 64 : (tile == TILE_64x128 || tile == TILE_128x128 || tile == TILE_96x128 || gemm_tile_two_k_groups(tile)) ? 128 : 256; }

int launch_gemm(const GemmP& p, int epi, int tile, hipStream_t s) {
    if (p.M <= 0 || p.N16 <= 0 || p.K32p <= 0 || (p.K32p & 1) || p.a_rows <= 0 || p.bgroup < 1) return 1;
    if (epi != EPI_PARTIAL && p.nsplit > 1) return 1;
    if (gemm_tile_eight_waves(tile)) return launch_gemm8(p, epi, tile, s);
    switch (epi) {
        case EPI_BIAS:      return launch_epi<EPI_BIAS>(p, tile, s);
        case EPI_BIAS_GELU: return launch_epi<EPI_BIAS_GELU>(p, tile, s);
        case EPI_PATCH:     return launch_epi<EPI_PATCH>(p, tile, s);
        case EPI_GEGLU:     return launch_epi<EPI_GEGLU>(p, tile, s);
        case EPI_PARTIAL:   return launch_epi<EPI_PARTIAL>(p, tile, s);
        case EPI_RESIDUAL:  return launch_epi<EPI_RESIDUAL>(p, tile, s);
        case EPI_QKV_ROPE:  return launch_epi<EPI_QKV_ROPE>(p, tile, s);
        case EPI_VIS_QKV:   return launch_epi<EPI_VIS_QKV>(p, tile, s);
        case EPI_SWIGLU:    return launch_epi<EPI_SWIGLU>(p, tile, s);
        case EPI_GQA_QKV:   return launch_epi<EPI_GQA_QKV>(p, tile, s);
    }
    return 2;
}
