// Epilogue of the QKV GEMMs: one 32 x 32 tile of accumulators into the fragment order the attention kernels read.  Everything leaves as whole 16-byte
// pieces.  A Q / K tile is the product weights x activations: lanes h = 0 / 1 of a row hold the two halves of every 8 columns and swap registers, which
// goes for the rotary table as well.  A V tile is taken the other way round, activations x weights, so that a lane holds four consecutive keys of one
// column: two 16-byte pieces of V^T as they are.  What it replaces stored Q / K in 8-byte and V^T in 2-byte pieces (DM0: through LDS) and read the
// tables 8 bytes at a time; us, before and after: SigLIP 256 rows x 3 456 10.4 and 8.7, 768 14.0 and 11.7, Gemma 256 x 2 560 14.8 and 13.3, 788 20.2 and 18.4.
#pragma once
#include "kernels.h"

constexpr bool epi_scatters(int epi) { return epi == EPI_QKV_ROPE || epi == EPI_VIS_QKV || epi == EPI_VIT_QKV_ROPE || epi == EPI_GQA_QKV; }
// first V column: a multiple of 256, so no workgroup tile holds both kinds
constexpr int epi_first_v(int epi) { return epi == EPI_GQA_QKV ? 3072 : epi == EPI_VIT_QKV_ROPE ? 2048 : 2304; }

// lanes h = 0 / 1: {x0 (h = 0), x0 (h = 1)} / {x1 (h = 0), x1 (h = 1)}
RTVLA_DEVICE uint4 swap_halves(uint2 x0, uint2 x1) {
    const rtvla_u2 a = __builtin_amdgcn_permlane32_swap(x0.x, x1.x, false, false), b = __builtin_amdgcn_permlane32_swap(x0.y, x1.y, false, false);
    return uint4{a[0], b[0], a[1], b[1]};
}

// What a tile needs besides its accumulators.  Asked for ahead where scatter_tiles says so: behind the stores of the tile before, which the compiler may not
// move loads across, each is a trip to the cache of its own.  us in a trace: SigLIP 768 rows x 3 456 13.9 -> 12.9, Gemma 788 x 2 560 22.2 -> 21.6, DM0's prefix 607 x 4 096
// 22.0 -> 21.0.
struct ScatterBias { f32x4 v[4]; float b; };               // Q, K: columns nt0 + 8 g + 4 h + e; V: column nt0 + r
struct ScatterTable { uint4 v[2]; };

template <int EPI, bool V>
RTVLA_DEVICE ScatterBias scatter_bias(const GemmP& p, int nt0, int lane) {
    ScatterBias o = {};
    const int h = lane >> 5, r = lane & 31, last = p.N16 * 16 - 4;                     // clamped: columns past the end are not stored
    if constexpr (V) {
        if constexpr (EPI == EPI_VIS_QKV) o.b = bf2f(p.bias[min(nt0 + r, last + 3)]);
        if constexpr (EPI == EPI_VIT_QKV_ROPE) o.b = p.bias_f32[min(nt0 + r, last + 3)];
    } else {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int n0 = min(nt0 + 8 * g + 4 * h, last);
            if constexpr (EPI == EPI_VIT_QKV_ROPE) o.v[g] = *(const f32x4*)(p.bias_f32 + n0);
            if constexpr (EPI == EPI_VIS_QKV) {
                const bf16x4 b = load4(p.bias + n0);
#pragma unroll
                for (int e = 0; e < 4; ++e) o.v[g][e] = bf2f(b[e]);
            }
        }
    }
    return o;
}
template <int EPI, bool V>
RTVLA_DEVICE ScatterTable scatter_table(const GemmP& p, int mt0, int nt0, int lane) {
    ScatterTable o = {};
    if constexpr (!V) {
        const int h = lane >> 5, mc = min(mt0 + (lane & 31), p.M - 1);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            if constexpr (EPI == EPI_QKV_ROPE) o.v[q] = *(const uint4*)(p.rope + (size_t)mc * 256 + (nt0 & 255) + 16 * q + 8 * h);
            if constexpr (EPI == EPI_VIT_QKV_ROPE) o.v[q] = *(const uint4*)(p.rope + (size_t)min(mc - mt0 / p.seq_pad * p.seq_pad, p.seq - 1) * 64 + (nt0 & 63) + 16 * q + 8 * h);
        }
    }
    return o;
}

// rows mt0 .. mt0 + 31, columns nt0 .. nt0 + 31 (multiples of 32), mt0 < p.M
template <int EPI, bool V, bool AHEAD>
RTVLA_DEVICE void scatter_tile(const GemmP& p, const f32x16& acc, const ScatterBias& bias, const ScatterTable& tab, int mt0, int nt0, int lane) {
    const int h = lane >> 5, r = lane & 31;
    if constexpr (V) {
        const int n = nt0 + r;                             // rows mt0 + 8 grp + 4 h + e
        const float b = bias.b;
        bf16x4 pk[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) pk[g] = pack4(acc[4 * g] + b, acc[4 * g + 1] + b, acc[4 * g + 2] + b, acc[4 * g + 3] + b);
        bf16_t* base;
        int d, key0, keys32;
        if constexpr (EPI == EPI_QKV_ROPE) { base = p.vt; d = n - 2304; key0 = mt0; keys32 = p.ldvt >> 5; }
        else if constexpr (EPI == EPI_VIS_QKV) {
            const int c = n - 2304, head = c / 72;
            base = p.vt + (size_t)((mt0 >> 8) * 16 + head) * (80 * 256); d = c - head * 72; key0 = mt0 & 255; keys32 = 8;
        } else {
            const int c = n - 2048, img = mt0 / p.seq_pad;
            base = p.vt + (size_t)(img * 16 + (c >> 6)) * ((size_t)64 * p.seq_pad); d = c & 63; key0 = mt0 - img * p.seq_pad; keys32 = p.seq_pad >> 5;
        }
        if (EPI != EPI_QKV_ROPE || mt0 + 32 <= p.M) {      // (the others' rows are whole tiles)
#pragma unroll
            for (int q = 0; q < 2; ++q) {                  // keys 8 q + 4 h + e and 16 more
                const uint2 lo = *(const uint2*)&pk[q], hi = *(const uint2*)&pk[q + 2];
                *(uint4*)(base + vt_index(d, key0 + 8 * q + 4 * h, keys32)) = uint4{lo.x, lo.y, hi.x, hi.y};
            }
        } else {
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (mt0 + 8 * g + 4 * h + e < p.M) base[vt_index(d, key0 + 8 * g + 4 * h + e, keys32)] = pk[g][e];
        }
    } else {
        const int m = mt0 + r, mc = min(m, p.M - 1);       // columns nt0 + 8 grp + 4 h + e
        int tok = mc, img = 0;
        if constexpr (EPI == EPI_VIS_QKV) { img = mc >> 8; tok = mc & 255; }
        if constexpr (EPI == EPI_VIT_QKV_ROPE) { img = mt0 / p.seq_pad; tok = mc - img * p.seq_pad; }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            bf16x4 pk[2];
            uint4 cs4 = {};
            if constexpr (EPI != EPI_VIS_QKV) cs4 = swap_halves(uint2{tab.v[q].x, tab.v[q].y}, uint2{tab.v[q].z, tab.v[q].w});       // this lane's halves of the two groups
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int g = 2 * q + k;
                f32x4 v = {acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
                if constexpr (EPI == EPI_VIS_QKV) {
                    v += bias.v[g];
                } else {
                    // rounded to bf16 before the rotation, as the reference's QKV buffers are (pi0_infer.py:793; dm0_infer.py:589-598)
                    if constexpr (EPI == EPI_VIT_QKV_ROPE) v += AHEAD ? bias.v[g] : *(const f32x4*)(p.bias_f32 + nt0 + 8 * g + 4 * h);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = round_bf16(v[e]);
                    const uint2 raw = k ? uint2{cs4.z, cs4.w} : uint2{cs4.x, cs4.y};
                    const bf16x4 cs = *(const bf16x4*)&raw;
                    const float c0 = bf2f(cs[0]), s0 = bf2f(cs[1]), c1 = bf2f(cs[2]), s1 = bf2f(cs[3]);
                    const f32x4 w = v;
                    v[0] = w[0] * c0 - w[1] * s0; v[1] = w[1] * c0 + w[0] * s0;
                    v[2] = w[2] * c1 - w[3] * s1; v[3] = w[3] * c1 + w[2] * s1;
                    if constexpr (EPI == EPI_VIT_QKV_ROPE) v *= nt0 < 1024 ? p.qscale : 1.0f;
                }
                pk[k] = pack4(v);
            }
            const uint4 piece = swap_halves(*(const uint2*)&pk[0], *(const uint2*)&pk[1]);
            const int n8 = nt0 + 16 * q + 8 * h;           // whole 8 columns now
            if (m >= p.M) continue;
            if constexpr (EPI == EPI_QKV_ROPE) {
                // Q rows are token * 8 + head
                if (n8 < 2048) *(uint4*)(p.q + ft_index(m * 8 + (n8 >> 8), n8 & 255, 8)) = piece;
                else *(uint4*)(p.k + ft_index(m, n8 - 2048, 8)) = piece;
            } else if constexpr (EPI == EPI_VIS_QKV) {
                // per (view, head): [256 tokens][96], 72 of them used
                const int which = n8 >= 1152, c = n8 - which * 1152, head = c / 72;
                *(uint4*)((which ? p.k : p.q) + (size_t)(img * 16 + head) * (256 * 96) + ft_index(tok, c - head * 72, 3)) = piece;
            } else {
                const int which = n8 >> 10, head = (n8 & 1023) >> 6;
                *(uint4*)((which ? p.k : p.q) + (size_t)(img * 16 + head) * ((size_t)p.seq_pad * 64) + ft_index(tok, n8 & 63, 2)) = piece;
            }
        }
    }
}

// The first cnt of a wave's row tiles, from row mt0 on, and its NT column tiles.  One column tile (four waves a CU): four row tiles ahead.  Two column tiles are
// those of the eight-wave kernel, whose other wave on the SIMD covers the loads of a tile (8 160 x 1 024 x 3 072: 63.5 us, 65.0 with all ahead, 64.4 with a
// tile's).
template <int EPI, bool V, int MT, int NT>
RTVLA_DEVICE void scatter_tiles(const GemmP& p, const f32x16 (&acc)[MT][NT], int cnt, int mt0, const int (&tile_of)[NT], int lane) {
    if constexpr (NT > 1) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            if (i >= cnt || mt0 + 32 * i >= p.M) continue;
#pragma unroll
            for (int j = 0; j < NT; ++j)
                if (tile_of[j] * 32 < p.N16 * 16)
                    scatter_tile<EPI, V, false>(p, acc[i][j], scatter_bias<EPI, V>(p, tile_of[j] * 32, lane), scatter_table<EPI, V>(p, mt0 + 32 * i, tile_of[j] * 32, lane),
                                                mt0 + 32 * i, tile_of[j] * 32, lane);
        }
    } else {
        static_assert(MT <= 4, "the tables of a wave's rows are in registers at once");
        if (tile_of[0] * 32 >= p.N16 * 16) return;
        const ScatterBias bias = scatter_bias<EPI, V>(p, tile_of[0] * 32, lane);
        ScatterTable tab[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) tab[i] = scatter_table<EPI, V>(p, min(mt0 + 32 * i, (p.M - 1) & ~31), tile_of[0] * 32, lane);
#pragma unroll
        for (int i = 0; i < MT; ++i)
            if (i < cnt && mt0 + 32 * i < p.M) scatter_tile<EPI, V, true>(p, acc[i][0], bias, tab[i], mt0 + 32 * i, tile_of[0] * 32, lane);
    }
}

// DM0's prefix (dm0_infer.py:853-878; EPI_GQA_QKV): the MT x 1 tiles of a wave whose workgroup's four waves hold the 128 columns of one head.  The product of the raw stream is
// rounded to bf16 and takes its row's RMS factor; queries and keys are then normalised over their head's features and rotated (interleaved pairs).  As a
// launch of its own behind the GEMM this read the products back and stored 2 and 4 bytes at a time, 8.3 us at 607 rows, 3.8 at 206; a forward
// with 3 images and 100 tokens took 17 991 us with it and takes 17 727, with 1 and 37 12 064 and 11 922.  Only 128-column tiles qualify (choose_tile): a head's
// sum of squares then stays in the workgroup.  With p.out the products themselves are left there as well, row-major (callers that look at a layer: one
// layer of a forward).
template <int MT, bool V>
RTVLA_DEVICE void scatter_head(const GemmP& p, f32x16 (&acc)[MT][1], float* lds, int m0, int nt0, int wn, int lane) {
    const int h = lane >> 5, r = lane & 31;
    if (p.out) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const bf16x4 v = pack4(acc[i][0][4 * g], acc[i][0][4 * g + 1], acc[i][0][4 * g + 2], acc[i][0][4 * g + 3]);
                if constexpr (V) {                         // rows m0 + 32 i + 8 g + 4 h + e, column nt0 + r
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int m = m0 + 32 * i + 8 * g + 4 * h + e;
                        if (m < p.M) p.out[(size_t)m * p.ldo + nt0 + r] = v[e];
                    }
                } else if (m0 + 32 * i + r < p.M) {
                    store4(p.out + (size_t)(m0 + 32 * i + r) * p.ldo + nt0 + 8 * g + 4 * h, v);
                }
            }
    }
    if constexpr (V) {
        const int c = nt0 - 3072 + r;
        bf16_t* const base = p.vt + (size_t)(c >> 7) * p.vt_bstride;
        f32x4 f[MT][4];
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int e = 0; e < 4; ++e) f[i][g][e] = p.rowscale[min(m0 + 32 * i + 8 * g + 4 * h + e, p.M - 1)];
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const int mt0 = m0 + 32 * i;                   // rows mt0 + 8 g + 4 h + e
            if (mt0 >= p.M) continue;
            bf16x4 pk[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                f32x4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = round_bf16(acc[i][0][4 * g + e]) * f[i][g][e];
                pk[g] = pack4(v);
            }
            if (mt0 + 32 <= p.M) {
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const uint2 lo = *(const uint2*)&pk[q], hi = *(const uint2*)&pk[q + 2];
                    *(uint4*)(base + vt_index(c & 127, mt0 + 8 * q + 4 * h, p.ldvt >> 5)) = uint4{lo.x, lo.y, hi.x, hi.y};
                }
            } else {
#pragma unroll
                for (int g = 0; g < 4; ++g)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (mt0 + 8 * g + 4 * h + e < p.M) base[vt_index(c & 127, mt0 + 8 * g + 4 * h + e, p.ldvt >> 5)] = pk[g][e];
            }
        }
    } else {
        const int head = nt0 >> 7, d0 = nt0 & 127;         // 16 query heads, 8 of keys
        float f[MT];
        uint4 table[MT][2];
        bf16x4 nw[4];
#pragma unroll
        for (int i = 0; i < MT; ++i) f[i] = p.rowscale[min(m0 + 32 * i + r, p.M - 1)];
#pragma unroll
        for (int g = 0; g < 4; ++g) nw[g] = load4((head < 16 ? p.qnorm : p.knorm) + d0 + 8 * g + 4 * h);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < 2; ++q) table[i][q] = *(const uint4*)(p.rope + (size_t)min(m0 + 32 * i + r, p.M - 1) * 128 + d0 + 16 * q + 8 * h);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            float ss = 0.f;
#pragma unroll
            for (int e = 0; e < 16; ++e) { const float v = round_bf16(acc[i][0][e]) * f[i]; acc[i][0][e] = v; ss += v * v; }
            ss = halves_sum(ss);
            if (h == 0) lds[wn * (MT * 32) + 32 * i + r] = ss;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const int m = m0 + 32 * i + r;
            float ss = 0.f;
#pragma unroll
            for (int k = 0; k < 4; ++k) ss += lds[k * (MT * 32) + 32 * i + r];
            const float inv = rsqrtf(ss * (1.0f / 128.0f) + 1e-6f);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const uint4 cs4 = swap_halves(uint2{table[i][q].x, table[i][q].y}, uint2{table[i][q].z, table[i][q].w});
                bf16x4 pk[2];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const int g = 2 * q + k;
                    const bf16x4 w = nw[g];
                    f32x4 v;
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = acc[i][0][4 * g + e] * inv * bf2f(w[e]);
                    const uint2 raw = k ? uint2{cs4.z, cs4.w} : uint2{cs4.x, cs4.y};
                    const bf16x4 cs = *(const bf16x4*)&raw;
                    const float c0 = bf2f(cs[0]), s0 = bf2f(cs[1]), c1 = bf2f(cs[2]), s1 = bf2f(cs[3]);
                    pk[k] = pack4(v[0] * c0 - v[1] * s0, v[1] * c0 + v[0] * s0, v[2] * c1 - v[3] * s1, v[3] * c1 + v[2] * s1);
                }
                const uint4 piece = swap_halves(*(const uint2*)&pk[0], *(const uint2*)&pk[1]);
                const int d = d0 + 16 * q + 8 * h;
                if (m >= p.M) continue;
                if (head < 16) *(uint4*)(p.q + (size_t)(head >> 1) * p.q_bstride + ft_index(m * 2 + (head & 1), d, 4)) = piece;
                else *(uint4*)(p.k + (size_t)(head - 16) * p.k_bstride + ft_index(m, d, 4)) = piece;
            }
        }
    }
}
