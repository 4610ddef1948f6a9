// Eight-wave bf16 GEMM for many rows (csrc/gemm.hip has the four-wave tiles): MT 32-row tiles x 256 columns per workgroup, wave (wm, wn) of
// 2 x 4 owning the upper or lower half of the row tiles and 64 columns (at most 128 accumulator registers, two waves per SIMD), with the same
// pre-tiled weights, v_mfma_f32_32x32x16_bf16 and order of K as the four-wave kernel: the same bits.
//
// Both operands go through LDS by DMA (buffer_load ... lds, 16 bytes per lane, no staging registers) in K stages of 32, a ring of 4 - 6 of them.
// With the weights read straight into registers the two waves of a column slice each pulled them through the CU's load path: 96 KB per 64 of K
// for the 256 x 256 tile, 48 of the 64 bytes per clock that the path gives under full MFMAs; through LDS it is 64 KB, and nothing but LDS reads and
// MFMAs waits.  us on MI355X, weights cold, registers -> LDS: 8 160 x 1 024 x 4 096 with bias + GELU 85 -> 73, 8 160 x 1 024 x 3 072 65 -> 54,
// 2 720 x 1 024 x 4 096 43 (four waves, 128 rows) -> 28, 8 160 x 4 096 x 1 024 66 (four waves) -> 59, 788 x 2 048 x 2 * 16 384 with GeGLU 109 (four waves) -> 102.
// The longest of them computes at 1.16 PFLOP/s by itself.  Counters inside a layer: 65 us, the matrix pipe busy in 60 % of the cycles (K = 1 024 with GELU 55, QKV 49 %) at
// 1.65 GHz.  A loop of nothing but MFMAs on such values reaches 1.5 - 1.8 PFLOP/s, so the clock is a part of the distance and the cycles without products the rest: two
// rounds of a 256 x 256 tile with K = 1 024 spend 2 x 10 us on first loads and epilogue.
//
// LDS of a stage: the activation rows at a pitch of 64 bytes, the 16-byte chunk c (8 of K) of row r in place c ^ ((r >> 2) & 3): 16 consecutive lanes of a
// fragment read (16 rows, one chunk) touch each of the 64 banks once.  A DMA instruction writes 16 rows in lane order, so the permutation is
// applied to the address a lane reads from.  Behind them the weights in fragment order as they lie in memory, 1 KB per instruction.
//
// A stage is two halves of 16 of K.  In each, the MFMAs of one half run while the fragments of the next are read, one read between two MFMAs, so the
// order in the source is kept (sched_barrier).  The one barrier of a stage stands in its middle: behind it all have read stage s - 1, whose memory the
// loads of stage s + RING - 1 may overwrite, half of them issued in the second half of stage s, the rest in the first half of s + 1: issued together they
// hold up the wave's MFMAs while the load path takes them in (8 160 x 4 096 x 1 024 with 128 rows: 61 -> 59 us).  And in front of it every wave has waited for its own loads of stage s + 1.
#include "kernels.h"
#include "gemm_scatter.h"
#include <algorithm>

namespace {

template <int EPI> struct Epi8 { static constexpr bool dual = (EPI == EPI_GEGLU || EPI == EPI_SWIGLU); };

RTVLA_DEVICE f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }

typedef __amdgpu_buffer_rsrc_t rsrc_t;
typedef __attribute__((address_space(3))) void* lptr_t;

constexpr int ring_of(int mt) { return mt >= 8 ? 4 : mt >= 6 ? 5 : 6; }               // K stages in LDS: 128 - 156 of 160 KB
constexpr int stage_bytes(int mt) { return mt * 2048 + 16384; }

// all but the newest N vector loads of this wave have landed, its LDS reads are back, and so for every wave of the workgroup
template <int N> RTVLA_DEVICE void wait_and_meet() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((N & 15) | (N >> 4 << 14) | (7 << 4));                 // vmcnt(N) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// The K loop of one wave: MTW of the workgroup's MT row tiles, from i0 on, and its 64 columns (two column tiles; DUAL: one of each weight).
template <int MT, int MTW, int RING, bool DUAL, bool V, int MTA>
RTVLA_DEVICE void gemm8_loop(const GemmP& p, unsigned char* smem, int m0, int n_blk, int i0, int s_begin, int s_end, f32x16 (&acc)[MTA][2]) {
#ifdef __HIP_DEVICE_COMPILE__                                                          // (the host pass knows neither the LDS load's size nor the waits)
    constexpr int NT = 2, A_B = MT * 2048, STAGE_B = stage_bytes(MT);
    constexpr int NA = MT * 2, NDMA = (NA + 16 + 7) / 8, ND1 = NDMA / 2;              // 1 KB instructions of a stage: A, per wave, and of those in its second half
    constexpr int G = DUAL ? 4 : 8;                                                    // a weight's column tiles in this workgroup, contiguous per 16 of K
    static_assert(RING * STAGE_B <= 160 * 1024 && (RING - 3) * NDMA + ND1 < 64, "LDS, vmcnt");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave & 3, h = lane >> 5, r = lane & 31;
    // rows from m0 on (the last valid one again for those past the end) and this workgroup's column tiles
    const rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)(p.A + (size_t)m0 * p.lda), 0, -1, 0x00027000);
    const size_t wblock = (size_t)n_blk * (p.K32p * 2) * G * 512;
    const rsrc_t rb0 = __builtin_amdgcn_make_buffer_rsrc((void*)(p.B0 + wblock), 0, -1, 0x00027000);
    const rsrc_t rb1 = __builtin_amdgcn_make_buffer_rsrc((void*)((DUAL ? p.B1 : p.B0) + wblock), 0, -1, 0x00027000);
    int voff[NDMA], lds_at[NDMA];
#pragma unroll
    for (int k = 0; k < NDMA; ++k) {
        if (k < 2) {                                                                   // weights: half k of the stage, column tile `wave` (DUAL: gate 0-3, up 0-3)
            voff[k] = k * G * 1024 + (DUAL ? wn : wave) * 1024 + lane * 16;
            lds_at[k] = A_B + (k * 8 + (DUAL ? wn * 2 + (wave >> 2) : wave)) * 1024;
        } else {                                                                       // a ragged last round loads the last rows again
            const int q = min(wave + 8 * (k - 2), NA - 1), row = q * 16 + (lane >> 2);
            voff[k] = min(row, p.a_rows - 1 - m0) * p.lda * 2 + (((lane & 3) ^ ((row >> 2) & 3)) * 16);
            lds_at[k] = q * 1024;
        }
    }
    auto dma = [&](int k, int s, int buf) __attribute__((always_inline)) {
        unsigned char* const dst = smem + buf * STAGE_B + lds_at[k];
        if (k >= 2) __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lptr_t)dst, 16, voff[k], s * 64, 0, 0);
        else __builtin_amdgcn_raw_ptr_buffer_load_lds(DUAL && wave >= 4 ? rb1 : rb0, (lptr_t)dst, 16, voff[k], s * (2 * G * 1024), 0, 0);
    };
    int a_off[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) a_off[ks] = i0 * 2048 + r * 64 + (((2 * ks + h) ^ ((r >> 2) & 3)) * 16);
    const int b_off = A_B + wn * 2048 + lane * 16;
    bf16x8 af[2][MTW], bf[2][NT];
    auto read = [&](int ks, int q, int buf) __attribute__((always_inline)) {
        if (q < NT) bf[ks][q] = *(const bf16x8*)(smem + buf * STAGE_B + b_off + ks * 8192 + q * 1024);
        else af[ks][q - NT] = *(const bf16x8*)(smem + buf * STAGE_B + a_off[ks] + (q - NT) * 2048);
    };
    // the products of half `ks`, between them the fragments of the other one (of stage buffer rbuf) and the DMA instructions [d0, d1) of stage ds
    auto half = [&](int ks, int rbuf, int d0, int d1, int ds, int dbuf) __attribute__((always_inline)) {
        constexpr int TOT = MTW * NT, NR = MTW + NT;
#pragma unroll
        for (int i = 0; i < MTW; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const int at = i * NT + j;
                acc[i][j] = V ? mfma32(af[ks][i], bf[ks][j], acc[i][j]) : mfma32(bf[ks][j], af[ks][i], acc[i][j]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int q = 0; q < NR; ++q)
                    if (q * TOT / NR == at) read(ks ^ 1, q, rbuf);
#pragma unroll
                for (int q = 0; q < NDMA; ++q)
                    if (q >= d0 && q < d1 && (q - d0) * TOT / (d1 - d0) + TOT / (2 * (d1 - d0)) == at) dma(q, ds, dbuf);
                __builtin_amdgcn_sched_barrier(0);
            }
    };
    // past the end the loads take the last stage again
    const int last = s_end - 1;
#pragma unroll
    for (int k = 0; k < RING - 2; ++k)
#pragma unroll
        for (int q = 0; q < NDMA; ++q) dma(q, min(s_begin + k, last), k);
#pragma unroll
    for (int q = 0; q < ND1; ++q) dma(q, min(s_begin + RING - 2, last), RING - 2);
    wait_and_meet<(RING - 3) * NDMA + ND1>();
#pragma unroll
    for (int q = 0; q < MTW + NT; ++q) read(0, q, 0);
    int buf = 0;
    for (int s = s_begin; s < s_end; ++s) {
        const int next = buf + 1 == RING ? 0 : buf + 1, before = buf == 0 ? RING - 1 : buf - 1, before2 = before == 0 ? RING - 1 : before - 1;
        half(0, buf, ND1, NDMA, min(s + RING - 2, last), before2);
        wait_and_meet<(RING - 3) * NDMA>();
        half(1, next, 0, ND1, min(s + RING - 1, last), before);
        buf = next;
    }
    wait_and_meet<0>();                                                                // the epilogue reuses the ring
#endif
}

template <int MT, int RING, int EPI, bool V>
RTVLA_DEVICE void gemm8_block(const GemmP& p, unsigned char* smem_raw, int m0, int n_blk, int split, int s_begin, int s_end) {
    constexpr int WN = 4, NT = 2, NTH = 512;
    constexpr int MTW = (MT + 1) / 2;                      // row tiles of the upper wave; the lower one has MT / 2
    constexpr bool DUAL = Epi8<EPI>::dual;
    constexpr int HALF = DUAL ? 1 : 2;

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave & 3, wm = wave >> 2;               // waves w and w + 4 share a SIMD: the two halves of one column slice
    const int h = lane >> 5, r = lane & 31;
    const int i0 = wm ? MTW : 0, mtw = wm ? MT / 2 : MTW;

    int tile_of[HALF];
#pragma unroll
    for (int j = 0; j < HALF; ++j) tile_of[j] = (n_blk * WN + wn) * HALF + j;

    f32x16 acc[MTW][NT];
#pragma unroll
    for (int i = 0; i < MTW; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    // the bias of this wave's columns, asked for ahead of the loop (bf16: in the lower half of the registers until the loop has ended).
    // Per group of four columns in the epilogue: 8 160 x 1 024 x 4 096 with GELU 76.3 us in a trace, this 73.5
    constexpr bool BIAS = EPI == EPI_BIAS || EPI == EPI_BIAS_GELU || EPI == EPI_RESIDUAL;
    f32x4 bias[BIAS ? HALF : 1][4];
    if constexpr (BIAS) {
#pragma unroll
        for (int j = 0; j < HALF; ++j)
#pragma unroll
            for (int grp = 0; grp < 4; ++grp) {
                const int n0 = min(tile_of[j] * 32 + 8 * grp + 4 * h, p.N16 * 16 - 4);        // clamped: columns past the end are never copied out
                if (p.bias_f32) bias[j][grp] = *(const f32x4*)(p.bias_f32 + n0);
                else *(bf16x4*)&bias[j][grp] = load4(p.bias + n0);
            }
    }
    float factor[EPI == EPI_SWIGLU ? MTW : 1];
    if constexpr (EPI == EPI_SWIGLU)
#pragma unroll
        for (int k = 0; k < MTW; ++k) factor[k] = p.rowscale[min(m0 + (i0 + k) * 32 + r, p.M - 1)];
    if (MT % 2 == 0 || wm == 0) gemm8_loop<MT, MTW, RING, DUAL, V>(p, smem_raw, m0, n_blk, i0, s_begin, s_end, acc);
    else gemm8_loop<MT, MT / 2, RING, DUAL, V>(p, smem_raw, m0, n_blk, i0, s_begin, s_end, acc);

    if constexpr (BIAS) {
        if (!p.bias_f32)
#pragma unroll
            for (int j = 0; j < HALF; ++j)
#pragma unroll
                for (int grp = 0; grp < 4; ++grp) {
                    const bf16x4 b = *(const bf16x4*)&bias[j][grp];
#pragma unroll
                    for (int e = 0; e < 4; ++e) bias[j][grp][e] = bf2f(b[e]);
                }
    }
    if constexpr (epi_scatters(EPI)) {
        scatter_tiles<EPI, V>(p, acc, mtw, m0 + 32 * i0, tile_of, lane);
        return;
    }
    // ---- epilogue: lane (h, r) holds rows m0 + 32 (i0 + i) + r, columns 32 tile + 8 grp + 4 h + e.  The k-th row tiles of
    // the two wave halves are converted into two LDS tiles and copied out together as 16-byte chunks of row segments.
    constexpr bool RES = EPI == EPI_RESIDUAL;              // staged as fp32: the residual joins on the way out, as in the four-wave kernel
    constexpr int ESZ = (EPI == EPI_PARTIAL || RES) ? 4 : 2;
    constexpr int OUTW = WN * HALF * 32;
    constexpr int ROWB = OUTW * ESZ + 16;
    constexpr int COLS = EPI == EPI_PARTIAL ? 4 : 8;       // columns of a 16-byte piece of the output
    constexpr int CPR = OUTW / COLS;
    constexpr int TILE_B = 32 * ROWB;
    constexpr int CIT = 2 * 32 * CPR / NTH;
    static_assert((2 * 32 * CPR) % NTH == 0, "copy-out mapping");
    unsigned char* obuf = smem_raw;
    const int nbase = n_blk * OUTW;
    const int ncols = p.N16 * 16;
#pragma unroll
    for (int k = 0; k < MTW; ++k) {
        const int i = i0 + k;
        bf16x8 res[RES ? CIT : 1];
        if constexpr (RES) {
#pragma unroll
            for (int it = 0; it < CIT; ++it) {
                const int idx = it * NTH + tid, half = idx / (32 * CPR), rem = idx - half * (32 * CPR), row = rem / CPR, ch = rem - row * CPR;
                const int mm = min(m0 + ((half ? MTW : 0) + k) * 32 + row, p.M - 1), n = min(nbase + ch * COLS, ncols - COLS);
                res[it] = *(const bf16x8*)(p.res + (size_t)mm * p.ldr + n);
            }
        }
        if (k < mtw && m0 + i * 32 < p.M) {
            unsigned char* const tbuf = obuf + wm * TILE_B;
#pragma unroll
            for (int j = 0; j < HALF; ++j) {
#pragma unroll
                for (int grp = 0; grp < 4; ++grp) {
                    const int cl = (wn * HALF + j) * 32 + 8 * grp + 4 * h;
                    f32x4 v = {acc[k][j][4 * grp], acc[k][j][4 * grp + 1], acc[k][j][4 * grp + 2], acc[k][j][4 * grp + 3]};
                    unsigned char* dst = tbuf + r * ROWB + cl * ESZ;
                    if constexpr (EPI == EPI_PARTIAL) {
                        *(f32x4*)dst = v;
                    } else if constexpr (EPI == EPI_GEGLU) {
                        const f32x4 u = {acc[k][j + HALF][4 * grp], acc[k][j + HALF][4 * grp + 1], acc[k][j + HALF][4 * grp + 2], acc[k][j + HALF][4 * grp + 3]};
                        *(bf16x4*)dst = pack4(gelu_tanh(v[0]) * u[0], gelu_tanh(v[1]) * u[1], gelu_tanh(v[2]) * u[2], gelu_tanh(v[3]) * u[3]);
                    } else if constexpr (EPI == EPI_SWIGLU) {
                        const float f = factor[k];
                        f32x4 u = {acc[k][j + HALF][4 * grp], acc[k][j + HALF][4 * grp + 1], acc[k][j + HALF][4 * grp + 2], acc[k][j + HALF][4 * grp + 3]};
                        v *= f; u *= f;
                        *(bf16x4*)dst = pack4(siluf(v[0]) * u[0], siluf(v[1]) * u[1], siluf(v[2]) * u[2], siluf(v[3]) * u[3]);
                    } else {
                        v += bias[j][grp];
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
        for (int it = 0; it < CIT; ++it) {
            const int idx = it * NTH + tid;
            const int half = idx / (32 * CPR), rem = idx - half * (32 * CPR);
            const int row = rem / CPR, ch = rem - row * CPR;
            const int ii = (half ? MTW : 0) + k;
            const int mm = m0 + ii * 32 + row;
            const int n = nbase + ch * COLS;
            if (k < (half ? MT / 2 : MTW) && mm < p.M && n < ncols) {
                const unsigned char* const src = obuf + half * TILE_B + row * ROWB + ch * COLS * ESZ;
                if constexpr (RES) {
                    f32x4 lo = *(const f32x4*)src, hi = *(const f32x4*)(src + 16);
                    const bf16x8 rs = res[it];
#pragma unroll
                    for (int e = 0; e < 4; ++e) { lo[e] += bf2f(rs[e]); hi[e] += bf2f(rs[4 + e]); }
                    const bf16x4 a = pack4(lo), b = pack4(hi);
                    *(uint4*)(p.out + (size_t)mm * p.ldo + n) = uint4{((const uint2*)&a)->x, ((const uint2*)&a)->y, ((const uint2*)&b)->x, ((const uint2*)&b)->y};
                    continue;                              // (no streaming hint: the normalising pass reads it next)
                }
                const f32x4 val = *(const f32x4*)src;
                if constexpr (EPI == EPI_PARTIAL) __builtin_nontemporal_store(val, (f32x4*)(p.partial + (size_t)split * p.pstride + (size_t)mm * p.ldp + n));
                else __builtin_nontemporal_store(val, (f32x4*)(p.out + (size_t)mm * p.ldo + n));
            }
        }
        if (k + 1 < MTW) __syncthreads();
    }
}

// Workgroup -> block tile.  Row blocks come in two sizes as in csrc/gemm.hip.  Consecutive workgroups share an XCD, so groups of eight row blocks
// take all their column blocks before the next eight rows: the 32 workgroups of an XCD then read 8 row and 4 column blocks instead of 32 and one
// (8 160 x 1 024 x 4 096: 79 -> 75 us, four rows to a group the same).
template <int MT, int EPI>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm8_kernel(GemmP p, int m_blocks, int n_blocks, int stages_total, int stages_per_split, int n_big) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    constexpr int RING = ring_of(MT), ROWS = 8;
    const int total = m_blocks * n_blocks * p.nsplit;
    const int lid = xcd_remap(blockIdx.x, total);
    const int split = lid / (m_blocks * n_blocks);
    const int rem = lid - split * (m_blocks * n_blocks);
    const int group = rem / (ROWS * n_blocks), in_group = rem - group * (ROWS * n_blocks);
    const int rows = min(ROWS, m_blocks - group * ROWS);
    const int n_blk = in_group / rows, m_blk = group * ROWS + in_group % rows;
    const int s_begin = split * stages_per_split, s_end = min(s_begin + stages_per_split, stages_total);
    auto block = [&](auto v) __attribute__((always_inline)) {
        if (m_blk < n_big) gemm8_block<MT, RING, EPI, v.value>(p, smem_raw, m_blk * (MT * 32), n_blk, split, s_begin, s_end);
        else gemm8_block<MT - 1, RING, EPI, v.value>(p, smem_raw, n_big * (MT * 32) + (m_blk - n_big) * ((MT - 1) * 32), n_blk, split, s_begin, s_end);
    };
    if constexpr (epi_scatters(EPI)) {
        if (n_blk * 256 >= epi_first_v(EPI)) { block(std::true_type{}); return; }
    }
    block(std::false_type{});
}

template <int MT, int EPI>
int launch8_cfg(const GemmP& p, hipStream_t s) {
    constexpr int HALF = Epi8<EPI>::dual ? 1 : 2;
    constexpr int ESZ = (EPI == EPI_PARTIAL || EPI == EPI_RESIDUAL) ? 4 : 2;
    const int tiles = (p.M + 31) / 32;
    const int n_blocks = ((p.N16 + 1) / 2 + 4 * HALF - 1) / (4 * HALF);
    const int m_blocks = gemm8_row_blocks(tiles, MT, n_blocks);
    int n_big = tiles - m_blocks * (MT - 1);
    if (n_big < 0) n_big = 0;
    const int pairs = p.K32p / 2;                          // K is split in pairs of stages, as the four-wave kernel's stages of 64
    const int nsplit = p.nsplit < 1 ? 1 : p.nsplit;
    const int sps = (pairs + nsplit - 1) / nsplit;
    if ((nsplit - 1) * sps >= pairs) return 3;
    GemmP q = p; q.nsplit = nsplit;
    constexpr size_t smem = std::max((size_t)ring_of(MT) * stage_bytes(MT), (size_t)2 * 32 * (4 * HALF * 32 * ESZ + 16));
    auto kern = gemm8_kernel<MT, EPI>;
    static std::atomic<uint64_t> done{0};
    if (int rc = ensure_dynamic_lds((const void*)kern, smem, done)) return rc;
    hipLaunchKernelGGL(kern, dim3(m_blocks * n_blocks * nsplit), dim3(512), smem, s, q, m_blocks, n_blocks, p.K32p, sps * 2, n_big);
    return hipGetLastError() == hipSuccess ? 0 : 5;
}

template <int EPI>
int launch8_epi(const GemmP& p, int tile, hipStream_t s) {
    switch (tile) {
        case TILE8_256x256: return launch8_cfg<8, EPI>(p, s);
        case TILE8_224x256: return launch8_cfg<7, EPI>(p, s);
        case TILE8_192x256: return launch8_cfg<6, EPI>(p, s);
        case TILE8_160x256: return launch8_cfg<5, EPI>(p, s);
        case TILE8_128x256: return launch8_cfg<4, EPI>(p, s);
    }
    return 2;
}

}  // namespace

// As many row blocks as the last round of 256 workgroups has room for: 8 160 rows by 3 072 columns in blocks of at most 224 rows are
// 37 x 12 = 444 workgroups, two rounds whose second leaves 68 CUs idle; as 42 x 12 = 504 nearly all CUs get two smaller ones.
int gemm8_row_blocks(int row_tiles, int mt, int n_blocks) {
    const int least = (row_tiles + mt - 1) / mt, room = (least * n_blocks + 255) / 256 * 256 / n_blocks;
    return std::max(least, std::min(room, row_tiles / (mt - 1)));
}

int launch_gemm8(const GemmP& p, int epi, int tile, hipStream_t s) {
    if (p.M <= 0 || p.N16 <= 0 || p.K32p <= 0 || (p.K32p & 1) || p.a_rows <= 0 || p.bgroup < 1) return 1;
    if (epi != EPI_PARTIAL && p.nsplit > 1) return 1;
    // the loads' offsets have 32 bits and count from the workgroup's first row and column: the four-wave kernel takes what they cannot reach (it has no
    // EPI_VIT_QKV_ROPE, whose rows are 1 024 wide)
    if (p.a_rows < p.M || p.lda > 1 << 21 || p.K32p > 1 << 16 || p.bgroup != (epi == EPI_GEGLU || epi == EPI_SWIGLU ? 4 : 8)) return launch_gemm(p, epi, TILE_128x256, s);
    switch (epi) {
        case EPI_BIAS:      return launch8_epi<EPI_BIAS>(p, tile, s);
        case EPI_BIAS_GELU: return launch8_epi<EPI_BIAS_GELU>(p, tile, s);
        case EPI_GEGLU:     return launch8_epi<EPI_GEGLU>(p, tile, s);
        case EPI_PARTIAL:   return launch8_epi<EPI_PARTIAL>(p, tile, s);
        case EPI_RESIDUAL:  return launch8_epi<EPI_RESIDUAL>(p, tile, s);
        case EPI_SWIGLU:    return launch8_epi<EPI_SWIGLU>(p, tile, s);
        case EPI_VIT_QKV_ROPE: return launch8_epi<EPI_VIT_QKV_ROPE>(p, tile, s);
    }
    return 2;
}
