// The prefix passes for many rows, on v_mfma_f32_32x32x16_bf16; query rows = token * G + head.  HD = 256: Gemma's (/root/reference/pi0_infer.py:819-824, pi05_infer.py:335-360), one K/V
// head.  HD = 128, CAUSAL: DM0's (/root/reference/dm0_infer.py:913-918), where a token sees the keys up to its own; 8 K/V heads, each on one XCD.
//
// A workgroup takes 32 query rows, its four waves every fourth block of 32 keys, and they merge through LDS.  As in csrc/flash.hip the loop runs a block behind and a
// block ahead: while the softmax of block i is computed, the matrix pipe takes O^T += V^T P^T of block i - 1 and S^T of block i + 1, in turn, and between two products stands one
// load of the fragments that the next trip needs, asked for where its registers have been consumed.  K and V^T go straight into registers: the keys are split between the
// waves, so there is nothing that two of them would share in LDS.
//
// What bounds it: a CU's load path.  788 tokens are 197 workgroups that pull 807 KB each, 6.2 us at 64 bytes per clock; with the launch (1.7), the first loads (2) and the merge
// (2) that is 12 of the 13.0 us.  The kernel of csrc/attention.hip with two row tiles per workgroup, which it replaces here, took 64 products of 22 cycles, two softmaxes and two bursts
// of 16 loads a block one after another, and waited for all its loads before the first product, because it asked for them behind a branch.  us with that / with this, weights
// cold, both in turn on one machine: 683 tokens 16.3 / 11.9, 768 16.0 / 12.4, 788 17.9 / 13.0, 968 19.7 / 15.6, 1 540 50.7 / 37.8, 2 048 60.1 / 50.5 (one row tile: csrc/kernels.h).
// CAUSAL: 38 row blocks of 607 tokens are 304 workgroups of one to nineteen key blocks, two to a CU; those with the most start first.  The work itself is small (2.4 us of products and 1.5 of
// loads if it were even): most of the 7.6 us are the launch, the first loads and the longest workgroups' five trips.  It replaces 16x16x32 products with one row tile, three workgroups
// to a CU (two row tiles at 2 107 tokens): 269 / 438 / 607 / 2 107 tokens 6.3 / 7.9 / 11.1 / 46.9 -> 5.4 / 6.4 / 7.6 / 30.4.
// (Built with the MFMA results in ordinary registers: 788 tokens 23 us otherwise, of copies and spills.)
#include "kernels.h"
#include <atomic>

namespace {

constexpr float HIDDEN = -__builtin_inff(), LOWEST = -3.402823466e38f;

RTVLA_DEVICE bf16x8 cat44(bf16x4 lo, bf16x4 hi) {
    bf16x8 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) { v[j] = lo[j]; v[4 + j] = hi[j]; }
    return v;
}
RTVLA_DEVICE f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }

// SUFFIX: keys past the prefix, all of them for rows past the state's, which see the first only.  An instance of its own, without which a launch
// of the others takes 0.1 - 0.2 us more.  us of rtvla_attention, its passes over the operands included, with a suffix of a tenth of the keys, one row tile / this: Gemma 1 000 tokens 37.4 / 30.6,
// 2 048 95.8 / 73.8, 5 120 453 / 320; causal 607 24.4 / 19.9, 2 107 84.6 / 64.5.
template <int HD, bool CAUSAL, bool SUFFIX>
__global__ __launch_bounds__(256, HD == 256 ? 1 : 2)
void prefix_attn_kernel(AttnP p) {
    constexpr int WAVES = 4, KD = HD / 32, DS = HD / 16, DT2 = HD / 32;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    f32x4* const obuf = (f32x4*)smem_raw;               // [wave][d tile][4][64]
    float* const ms = (float*)(smem_raw + (size_t)WAVES * DT2 * 4 * 64 * 16);          // [wave][32], then the sums
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, n = lane & 31;
    // CAUSAL: K/V heads dealt over the XCDs, the rows with the most keys first
    const int batch = CAUSAL ? blockIdx.x % p.batch : 0;
    const int row0 = CAUSAL ? ((int)(gridDim.x / p.batch) - 1 - (int)(blockIdx.x / p.batch)) * 32 : blockIdx.x * 32;
    const int prefix = min(p.keys, p.prefix_alloc);
    int vis = prefix;                                   // keys that every row sees, causal aside
    if (p.valid_len) vis = max(0, min(*p.valid_len, prefix));
    const int all = CAUSAL ? min(vis, row0 / p.group + 1) : vis;                       // that all rows of this workgroup see
    // hidden from this lane's row are the keys from `lim` on, and `hole` of them behind the valid ones
    int end = SUFFIX ? p.keys : vis;
    int lim = SUFFIX && row0 + n < p.state_rows ? prefix + 1 : end;
    const unsigned hole = SUFFIX ? prefix - vis : 0;
    if (CAUSAL) {
        lim = min(lim, (row0 + n) / p.group + 1);
        end = min(end, (row0 + 31) / p.group + 1);      // that some row sees
    }
    const float c = p.scale * 1.4426950408889634f;
    const int blocks = (end + 31) >> 5, keys32 = p.ldvt >> 5;

    // A block past the last one is a buffer of no bytes, from which the hardware returns zeros and reads nothing: behind a branch the compiler could not tell how many loads
    // are under way and would wait for all of them.
    auto rows_of = [&](const bf16_t* base, size_t at, int kb, unsigned bytes) __attribute__((always_inline)) {
        return __builtin_amdgcn_make_buffer_rsrc((void*)(base + at), 0, kb < blocks ? (int)bytes : 0, 0x00027000);
    };
    auto k_block = [&](int kb) __attribute__((always_inline)) { return rows_of(p.k, (size_t)batch * p.k_bstride + (size_t)kb * (2 * KD * 512), kb, 2 * KD * 1024); };
    auto v_block = [&](int kb) __attribute__((always_inline)) { return rows_of(p.vt, (size_t)batch * p.vt_bstride + (size_t)kb * 512, kb, (unsigned)(HD / 16 * keys32) * 1024u); };
    const int k_lane = ((n >> 4) * KD * 64 + h * 16 + (n & 15)) * 16, v_lane = (n >> 4) * keys32 * 1024 + (h * 16 + (n & 15)) * 16;
    auto piece = [&](__amdgpu_buffer_rsrc_t rs, int off, int uniform) __attribute__((always_inline)) { return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rs, off, uniform, 0)); };
    auto piece_k = [&](__amdgpu_buffer_rsrc_t rs, int s) __attribute__((always_inline)) { return piece(rs, k_lane + (s >> 1) * 1024 + (s & 1) * 512, 0); };
    auto piece_v = [&](__amdgpu_buffer_rsrc_t rs, int q, int t) __attribute__((always_inline)) { return piece(rs, v_lane + q * 512, 2 * t * keys32 * 1024); };

    bf16x8 qf[DS], kf[DS], vf[2][DT2], pP[2], pC[2];
    {
        const auto kr = k_block(w);
#pragma unroll
        for (int s = 0; s < DS; ++s) kf[s] = piece_k(kr, s);
        const bf16_t* const q0 = p.q + (size_t)batch * p.q_bstride + ((size_t)((row0 >> 4) + (n >> 4)) * KD * 64 + h * 16 + (n & 15)) * 8;
#pragma unroll
        for (int s = 0; s < DS; ++s) qf[s] = *(const bf16x8*)(q0 + (s >> 1) * 512 + (s & 1) * 256);
    }
    f32x16 o[DT2], sA, sB;
#pragma unroll
    for (int t = 0; t < DT2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[t][e] = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) sA[e] = 0.f;
    auto mask = [&](int kb, f32x16& st) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int key = kb * 32 + 8 * (e >> 2) + 4 * h + (e & 3);
            if (key >= lim || (SUFFIX && (unsigned)(key - vis) < hole)) st[e] = HIDDEN;
        }
    };
    auto lane_max = [&](const f32x16& st) __attribute__((always_inline)) {
        const auto max3 = [](float a, float b, float c) { return fmaxf(fmaxf(a, b), c); };
        const float m0 = max3(max3(max3(st[0], st[1], st[2]), st[3], st[4]), st[5], st[6]), m1 = max3(max3(max3(st[8], st[9], st[10]), st[11], st[12]), st[13], st[14]);
        return max3(m0, m1, fmaxf(st[7], st[15]));
    };
    __builtin_amdgcn_sched_barrier(0);
    const auto k1 = k_block(w + WAVES);
#pragma unroll
    for (int s = 0; s < DS; ++s) {
        sA = mfma32(kf[s], qf[s], sA);
        kf[s] = piece_k(k1, s);
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        pP[q] = bf16x8{};                               // "block -1": zero probabilities, any finite V^T
#pragma unroll
        for (int t = 0; t < DT2; ++t) vf[q][t] = bf16x8{};
    }
    __builtin_amdgcn_sched_barrier(0);
    if (w * 32 + 32 > all) mask(w, sA);
    // a row's maximum is finite, so that a key it does not see (minus infinity) has no weight at any scale, also where it sees nothing of the block
    float m = fmaxf(LOWEST, w < blocks ? halves_max(lane_max(sA)) : HIDDEN), l = 0.f;

    // block kb: on entry s_cur = S^T(kb), kf = K of kb + 4 (under way), vf = V^T and p_prev = probabilities of kb - 4; on exit the same for the next
    auto step = [&](int kb, f32x16& s_cur, f32x16& s_next, bf16x8 (&p_prev)[2], bf16x8 (&p_cur)[2]) __attribute__((always_inline)) {
        const auto kr = k_block(kb + 2 * WAVES), vr = v_block(kb);
        const bool edge = kb * 32 + 32 > all;
        if (edge) mask(kb, s_cur);
        // The largest probability of a row so far is exactly 1, and each is rounded to bf16 once: the maximum follows every block, and the accumulators are scaled behind the
        // products of block kb - 4, whose probabilities are relative to the maximum before.  (Scaled ahead of them, with those probabilities, and only where the maximum has grown by
        // 8 bits, the error against 64 bits was 1.08 times as large, in rows of sharp logits 1.18 times; it was 0.5 us faster at 788 tokens and 0.2 at DM0's 607.)
        const float m_old = m;
        m = fmaxf(m, halves_max(lane_max(s_cur)));
        const float alpha = __builtin_amdgcn_exp2f((m_old - m) * c);
        l *= alpha;
#pragma unroll
        for (int e = 0; e < 16; ++e) s_next[e] = 0.f;
#pragma unroll
        for (int i = 0; i < DS; ++i) {
            const int q = i / DT2, t = i % DT2;
            o[t] = mfma32(vf[q][t], p_prev[q], o[t]);
            s_next = mfma32(kf[i], qf[i], s_next);
            vf[q][t] = piece_v(vr, q, t);
            kf[i] = piece_k(kr, i);
        }
        float sum[2] = {0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 16; ++e) { s_cur[e] = __builtin_amdgcn_exp2f((s_cur[e] - m) * c); sum[e & 1] += s_cur[e]; }       // (a difference first: of equal logits it is 0, however large they are)
        l += sum[0] + sum[1];
#pragma unroll
        for (int q = 0; q < 2; ++q) p_cur[q] = cat44(pack4(s_cur[4 * q], s_cur[4 * q + 1], s_cur[4 * q + 2], s_cur[4 * q + 3]),
                                                     pack4(s_cur[4 * q + 8], s_cur[4 * q + 9], s_cur[4 * q + 10], s_cur[4 * q + 11]));
#pragma unroll
        for (int i = 0; i < 2 * DS; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x402, HD == 256 ? 3 : 5, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" :: "v"(p_cur[0]), "v"(p_cur[1]), "v"(l));               // (made here, beside the MFMAs)
        if (__any(m > m_old))
#pragma unroll
            for (int t = 0; t < DT2; ++t)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[t][e] *= alpha;
    };
    int kb = w;
    for (; kb + WAVES < blocks; kb += 2 * WAVES) {
        step(kb, sA, sB, pP, pC);
        step(kb + WAVES, sB, sA, pC, pP);
    }
    if (kb < blocks) {
        step(kb, sA, sB, pP, pC);
        pP[0] = pC[0]; pP[1] = pC[1];
    }
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int t = 0; t < DT2; ++t) o[t] = mfma32(vf[q][t], pP[q], o[t]);

    // ---- merge: wave w finishes d tiles 2 w, 2 w + 1 ----
    l = halves_sum(l);
    if (h == 0) ms[w * 32 + n] = m;
    __syncthreads();
    float M = LOWEST;
#pragma unroll
    for (int ww = 0; ww < WAVES; ++ww) M = fmaxf(M, ms[ww * 32 + n]);
    const float f = __builtin_amdgcn_exp2f((m - M) * c);
    if (h == 0) ms[(WAVES + w) * 32 + n] = l * f;
#pragma unroll
    for (int t = 0; t < DT2; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) obuf[((w * DT2 + t) * 4 + j) * 64 + lane] = f32x4{o[t][4 * j], o[t][4 * j + 1], o[t][4 * j + 2], o[t][4 * j + 3]} * f;
    __syncthreads();
    float L = 0.f;
#pragma unroll
    for (int ww = 0; ww < WAVES; ++ww) L += ms[(WAVES + ww) * 32 + n];
    const float inv = L > 0.f ? 1.0f / L : 0.f;
    const int row = row0 + n;
    if (row >= p.rows) return;
    const int tok = row / p.group;
    bf16_t* const out = p.out + (size_t)(batch / p.batch_inner) * p.out_ostride + (size_t)(batch % p.batch_inner) * p.out_istride + (size_t)tok * p.ld_tok + (row - tok * p.group) * HD;
#pragma unroll
    for (int k = 0; k < DT2 / WAVES; ++k) {
        const int t = w * (DT2 / WAVES) + k;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ww = 0; ww < WAVES; ++ww) v += obuf[((ww * DT2 + t) * 4 + j) * 64 + lane];
            store4(out + 32 * t + 8 * j + 4 * h, pack4(v * inv));
        }
    }
}

}  // namespace

bool prefix_attention_takes(const AttnP& p, int variant) {
    const bool form = variant == ATTN_PREFIX ? !p.causal && p.batch <= 1 : variant == ATTN_GQA128_PREFIX && p.causal;
    return form && attn_two_row_tiles(variant, p.rows, p.batch) && p.nsplit <= 1 && !p.out_tiled && p.scale > 0.f;
}
template <int HD, bool CAUSAL, bool SUFFIX>
int launch_prefix_inst(const AttnP& p, hipStream_t s) {
    constexpr size_t smem = 4 * (HD / 32) * 4 * 64 * 16 + 2 * 4 * 32 * 4;
    auto kern = prefix_attn_kernel<HD, CAUSAL, SUFFIX>;
    static std::atomic<uint64_t> done{0};
    if (int rc = ensure_dynamic_lds((const void*)kern, smem, done)) return rc;
    hipLaunchKernelGGL(kern, dim3((p.rows + 31) / 32 * (CAUSAL ? p.batch : 1)), dim3(256), smem, s, p);
    return hipGetLastError() == hipSuccess ? 0 : 5;
}
int launch_prefix_attention(const AttnP& p, hipStream_t s) {
    if (p.prefix_alloc < p.keys) return p.causal ? launch_prefix_inst<128, true, true>(p, s) : launch_prefix_inst<256, false, true>(p, s);
    return p.causal ? launch_prefix_inst<128, true, false>(p, s) : launch_prefix_inst<256, false, false>(p, s);
}
