// sp_sqfree_attn.hip -- fused decode attention over sqfree+spinor records (the
// sqfree cache's K and V arrays) for the shipping geometry: head_dim 128 padded to
// 154, skeleton 77 or 115 (K bands 5/4/4/4/5; V 5/4/4/4/5, or one 3-bit band at
// skeleton 115), 3-bit residuals, spinor sheet on.
//
// The read path (sp_cuda_sqfree_read_one, shannon_prime_sqfree.cu:857-950) rebuilds
// the pad coefficients c~ (skeleton values from the bands; residual coefficient r as
// (sheet_r ? -pred_r : pred_r) + (level_r - centre) * step, pred = the Knight CSR over
// the dequantized skeleton) and returns V(c~)[0, hd), V the length-154 Vilenkin
// transform, which is symmetric and its own inverse. So nothing is reconstructed:
//   * with q~ = kq_scale * V(q zero-padded to 154) (once per query head),
//     q . K~_t = q~ . c~_t, a dot product in the coefficient domain;
//   * sum_t p_t V~_t = V(sum_t p_t c~_t)[0, hd): the weighted coefficient sums are
//     finished by one transform per query head.
//
// Three launches per layer: the hier attention's query preparation and merge
// kernels (sp_hier_attn.hip) with no predictor (W = 0: skeleton slots = the Knight
// skeleton, target slots = the residual coefficients), and the split kernel below:
// block (KV head, run) is one wave walking the run's 64-position tiles, lane =
// position, the record decoded into the lane's registers exactly as the read path
// decodes it (compile-time Knight CSR and record fields), the scores as dot products
// with the prepared queries, an online softmax across the run's tiles, and the
// weighted coefficient sums through LDS (the wave's coefficients transposed so that
// each lane sums one coefficient over the tile's 64 positions); both products in fp32, on
// the matrix cores or (one or two query heads, on_matrix_cores()) on the vector unit.
#include <cstdlib>
#include <utility>

#include "sp_sqfree_lane.h"

namespace {

constexpr int PAD = 154;
constexpr int RBITS = 3;

// The record's pad coefficients in [skeleton slot s | residual r] order: the same
// arithmetic, in the same order, as k_sqfree_decode_lane before its transform.
template <int SK, class SL, int DW>
__device__ __forceinline__ void sq_coefficients(const uint32_t (&rec)[DW], float (&e)[PAD]) {
    using G = SqRec<PAD, SK, RBITS, true, SL>;
    constexpr int NR = PAD - SK;
    float sk[SK];
    dequant_bands<SL, false, true>(rec, SL::nb, sk);
#pragma unroll
    for (int s = 0; s < SK; s++) e[s] = sk[s];
    const float mag = __uint_as_float(rec_get32(rec, G::mag_byte));
    constexpr int L = 1 << RBITS;
    const float center = 0.5f * (float)(L - 1);
    const float sat = mag * (float)RBITS;
    const float step = sp_div(2.0f * sat, (float)(L - 1));
#pragma unroll
    for (int r = 0; r < NR; r++) {
        float p = csr_predict<PAD, SK>(sk, r);
        if (rec_extract(rec, G::sheet_bit + r, 1)) p = -p;
        const float d = ((float)rec_extract(rec, G::res_bit + r * RBITS, RBITS) - center) * step;
        e[SK + r] = p + d;
    }
}

// wave reductions on DPP and the row swaps (every lane active at each call)
__device__ __forceinline__ float wave_max(float v) { return sp_wave_max_dpp(v); }
__device__ __forceinline__ float wave_add(float v) { return sp_wave_sum_dpp(v); }
// a value that every lane holds, in a scalar register
__device__ __forceinline__ float wave_uniform(float v) {
    return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v)));
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Sixteen 4x4x1 fp32 products in one matrix instruction, each of the sixteen 4-lane
// blocks taking its A rows from block AB of its group of 2^CB blocks: with CB = 4,
// c[i](lane) += a(lane 4*AB + i) * b(lane) for i < 4. An fp32 fused multiply-add of
// four query heads' factors with a value per lane, at twice the vector unit's rate
// and without the factors in scalar registers.
template <int CB, int AB>
__device__ __forceinline__ f32x4 fma_heads(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, CB, AB, 0);
}

// The vector unit's score factors of one query head in chunks of at most 16: the skeleton
// part (SK factors) then the residual part (PAD - SK), a chunk never spanning both.
template <int SK>
struct QChunks {
    static constexpr int NS = (SK + 15) / 16, NR = (PAD - SK + 15) / 16, N = NS + NR;
    // coefficient index of chunk k's first factor, and the chunk's factor count
    static constexpr int first(int k) { return k < NS ? 16 * k : SK + 16 * (k - NS); }
    static constexpr int size(int k) {
        return k < NS ? (SK - 16 * k < 16 ? SK - 16 * k : 16) : (PAD - SK - 16 * (k - NS) < 16 ? PAD - SK - 16 * (k - NS) : 16);
    }
};

constexpr int NQ = (PAD + 15) / 16;  // registers of one head group's factors, 16 coefficients each

// scores: s[g][C % 3][i](position) += q~[4g + i][C] * e[C](position), every C of the pack
template <int NG, int C>
__device__ __forceinline__ void score_step(const float (&q)[NG][NQ], const float (&e)[PAD], f32x4 (&s)[NG][3]) {
#pragma unroll
    for (int g = 0; g < NG; g++) s[g][C % 3] = fma_heads<4, C % 16>(q[g][C / 16], e[C], s[g][C % 3]);
}
template <int NG, int... C>
__device__ __forceinline__ void score_all(const float (&q)[NG][NQ], const float (&e)[PAD], f32x4 (&s)[NG][3],
                                          std::integer_sequence<int, C...>) {
    (score_step<NG, C>(q, e, s), ...);
}

// weighted sums: acc[g][i](coefficient) += p[4g + i][position] * E[coefficient][position]
// for the four positions 4*K .. 4*K + 3 of the row ei (PER positions per weight register)
template <int NG, int PER, int CB, int K, int NP>
__device__ __forceinline__ void sum_step(const float (&pw)[NG][NP], const f32x4 &ei, f32x4 (&acc)[NG]) {
#pragma unroll
    for (int g = 0; g < NG; g++) {
        acc[g] = fma_heads<CB, (4 * K + 0) % PER>(pw[g][4 * K / PER], ei[0], acc[g]);
        acc[g] = fma_heads<CB, (4 * K + 1) % PER>(pw[g][4 * K / PER], ei[1], acc[g]);
        acc[g] = fma_heads<CB, (4 * K + 2) % PER>(pw[g][4 * K / PER], ei[2], acc[g]);
        acc[g] = fma_heads<CB, (4 * K + 3) % PER>(pw[g][4 * K / PER], ei[3], acc[g]);
    }
}
// all of a row's positions, sixteen at a time: the next sixteen are read while these
// multiply, and no more (the barriers keep the rest of the reads behind)
template <int NG, int PER, int CB, int N16, int J, int NP>
__device__ __forceinline__ void sum_16(const float (&pw)[NG][NP], const float *row, const f32x4 (&ei)[4],
                                       f32x4 (&acc)[NG]) {
    f32x4 en[4];
    if constexpr (J + 1 < N16) {
#pragma unroll
        for (int k = 0; k < 4; k++) en[k] = *reinterpret_cast<const f32x4 *>(row + 16 * (J + 1) + 4 * k);
    }
    sum_step<NG, PER, CB, 4 * J + 0>(pw, ei[0], acc);
    sum_step<NG, PER, CB, 4 * J + 1>(pw, ei[1], acc);
    sum_step<NG, PER, CB, 4 * J + 2>(pw, ei[2], acc);
    sum_step<NG, PER, CB, 4 * J + 3>(pw, ei[3], acc);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (J + 1 < N16) sum_16<NG, PER, CB, N16, J + 1>(pw, row, en, acc);
}
template <int NG, int PER, int CB, int N16, int NP>
__device__ __forceinline__ void sum_all(const float (&pw)[NG][NP], const float *row, f32x4 (&acc)[NG]) {
    f32x4 ei[4];
#pragma unroll
    for (int k = 0; k < 4; k++) ei[k] = *reinterpret_cast<const f32x4 *>(row + 4 * k);
    sum_16<NG, PER, CB, N16, 0>(pw, row, ei, acc);
}

// LDS row pitch (floats) of the transposed coefficient chunk: 16-byte rows, eight lanes'
// 16-byte pieces on distinct banks; for the vector unit's 4-byte reads, lanes on distinct banks
constexpr int row_pitch(bool mx) { return mx ? 68 : 65; }

// Scores, online softmax and the V records' weighted coefficient sums. Block
// (kvh, run) takes tiles run, run + n_runs, ... of KV head kvh (64 positions each).
// prep: the G query heads of KV head kvh at prep + (kvh * G + h) * ps:
// [q~ at the skeleton slots (r4(SK)) | q~ at the residual coefficients | ...], qo the
// residual part's offset. Partial per (query head, run) at part + ((h0 + h) * n_runs
// + run) * pp: [m, l, 0, 0, sum p c~ (PAD coefficients, skeleton then residuals)].
// OUT = false: scores only.
//
// Both contractions run on the matrix cores in fp32 (fma_heads), four query heads at a
// time: the scores with the prepared queries in registers (lane 4b + i of register j:
// head i of the group, coefficient 16j + b) against the lane's own coefficients, in three
// chains of sums; the weighted sums with the tile's weights (lane 4b + i of register j:
// head i, position 16j + b) against the transposed chunk (lane = coefficient, four
// positions per 16-byte LDS read). MX = false (one or two heads) takes the same sums on the
// vector unit: the factors by scalar loads, the weights by LDS broadcasts.
//
// Bound by the decode of the two records (2400 vector instructions a tile beside 628
// matrix instructions) and by latency at two waves per SIMD, which the 154 coefficients a
// lane holds allow at most. Four sequences of 16384 over 4 KV heads and 8 query heads
// each: 71 us with the products on the vector unit (4900 instructions a tile), 48 us here. Two chains of sums took 45 us and
// four 50; the mean error against 64-bit results over 126 shapes was 4.6e-7 with two,
// 3.9e-7 with three, 3.6e-7 with four, and 4.5e-7 before.
template <int SK, class SLK, class SLV, int GM, bool MX, bool OUT>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
k_sqfree_attn_split(const unsigned char *__restrict__ kc0, const unsigned char *__restrict__ vc0, long long k_slot,
                    long long v_slot, const SpSeqTab T, int G, int hs, const float *__restrict__ prep0, int ps, int qo,
                    float *__restrict__ scores0, float *__restrict__ part0, int pp, int n_runs) {
    using GK = SqRec<PAD, SK, RBITS, true, SLK>;
    using GV = SqRec<PAD, SK, RBITS, true, SLV>;
    constexpr int NCK = RecTile<GK>::NCK > RecTile<GV>::NCK ? RecTile<GK>::NCK : RecTile<GV>::NCK;
    constexpr int C2 = PAD - 128;  // coefficients of the third 64-coefficient chunk
    constexpr int EP = row_pitch(MX);
    constexpr int NG = (GM + 3) / 4;  // groups of four query heads
    constexpr int PP = MX ? 4 * NG : GM;  // weights per position
    static_assert(C2 > 0 && C2 <= 32, "two whole chunks, and one of at most 32 coefficients");
    // the record stage and the transposed coefficient chunks share their memory: in
    // this one-wave block the stage's last reads (the V records) come before the first
    // chunk's writes, and the next tile's K records are staged after the last chunk's
    // barrier; the smaller block fits 8 per CU (two waves per SIMD) instead of 6
    __shared__ __attribute__((aligned(16))) float E[OUT ? 64 * EP : (NCK * 1024 + 16 + 3) / 4];
    static_assert(NCK * 1024 + 16 <= 64 * EP * 4, "the record stage fits the chunk memory");
    unsigned char *const stage = reinterpret_cast<unsigned char *>(E);
    // At skeleton 77 the matrix instances stage a tile's V records beside its K records: held in
    // registers through the K half they spilled there (52 to 63 dwords a lane, each load waited
    // for and stored at once). 8 KV heads x 30000 positions, 4 query heads: 59.6 us against 52.0,
    // 55.7 on the vector unit. At skeleton 115 (13 dwords) the registers are faster, 47.9 / 50.0.
    constexpr bool V_STAGED = MX && SK == 77 && OUT;
    unsigned char *const stage_v = V_STAGED ? stage + NCK * 1024 + 16 : stage;
    static_assert(!V_STAGED || 2 * (NCK * 1024 + 16) <= 64 * EP * 4, "both sides' records fit the chunk memory");
    __shared__ __attribute__((aligned(16))) float Pw[OUT ? 64 * PP : 4];  // [position][head]
    // block x: head group x (query heads x G .. x G + G - 1) of KV head x / hs
    const int hb = blockIdx.x, kvh = hb / hs, run = blockIdx.y, lane = threadIdx.x;
    // sequence blockIdx.z: its positions, prepared queries, score rows and partials
    const int seq = blockIdx.z, n_q = (int)gridDim.x * G, n_kv = T.len[seq];
    const unsigned char *__restrict__ kc = kc0 + (long long)T.start[seq] * GK::total;
    const unsigned char *__restrict__ vc = vc0 + (long long)T.start[seq] * GV::total;
    const long long s_stride = T.len[seq];
    float *__restrict__ scores = scores0 ? scores0 + T.soff[seq] : nullptr;
    const float *__restrict__ prep = prep0 + (long long)seq * n_q * ps;
    float *__restrict__ part = part0 + (long long)seq * n_q * n_runs * pp;
    const int h0 = hb * G;
    const int tpo = (n_kv + 63) / 64;
    const int n_tiles = ((int)gridDim.x / hs) * tpo;
    const TileMap M{tpo, n_kv};
    const float *__restrict__ pq = prep + (long long)h0 * ps;

    const int lb = lane / 4, li = lane % 4;
    const f32x4 z4 = {0.0f, 0.0f, 0.0f, 0.0f};
    float m_run[GM], l_run[GM];
    f32x4 acc0[NG], acc1[NG], acc2[NG];
#pragma unroll
    for (int h = 0; h < GM; h++) {
        m_run[h] = -INFINITY;
        l_run[h] = 0.0f;
    }
#pragma unroll
    for (int g = 0; g < NG; g++) acc0[g] = acc1[g] = acc2[g] = z4;
    float va0[GM], va1[GM], va2 = 0.0f;  // the vector unit's
#pragma unroll
    for (int h = 0; h < GM; h++) va0[h] = va1[h] = 0.0f;
    // third chunk: lane = coefficient 128 + c2i, positions 32 * half .. 32 * half + 31
    // (the two halves are added at the end). On the vector unit lane = coefficient 128 + vi of
    // head vh, every position.
    const int vi = lane % C2, vh = lane / C2;
    const bool v_on = vh < GM;
    static_assert(MX || GM <= 2, "a lane per head and coefficient of the third chunk");
    const int half = lane / 32, c2i = lane % 32 < C2 ? lane % 32 : C2 - 1;

    // a tile's K and V records load at the tile's start (holding the next tile's K records
    // through a tile took the registers that keep the full instances from spilling at two
    // waves per SIMD; the other wave hides the load)
    for (int c = run; c < tpo; c += n_runs) {
        const int t = kvh * tpo + c;
        // with the V records staged: an opaque copy of the lane index a tile, so that LDS
        // addresses are not held through the loop either
        int ln = lane;
        if (V_STAGED) __asm__ volatile("" : "+v"(ln));
        RecTile<GK> Rk;
        rec_tile_load<GK>(Rk, kc, k_slot, M, t, n_tiles, ln);
        RecTile<GV> Rv;
        if (OUT) rec_tile_load<GV>(Rv, vc, v_slot, M, t, n_tiles, ln);
        // the head groups' factors, again for each tile (cache hits beside the records' loads):
        // held across the V half they cost the registers that keep it from spilling
        float q[NG][NQ];
        int zero = 0;
        if constexpr (MX) __asm__ volatile("" : "+v"(zero));  // no hoisting out of the tile loop
#pragma unroll
        for (int g = 0; g < (MX ? NG : 0); g++) {
            // heads past the group's and coefficients past the pad repeat the last: their
            // products are never read
            const int h = 4 * g + li < G ? 4 * g + li : G - 1, o = h * ps + lb + zero;
#pragma unroll
            for (int j = 0; j < NQ; j++) {
                const int k = 16 * j;  // coefficients k + lb
                if (k + 16 <= SK) q[g][j] = pq[o + k];
                else if (k >= SK && k + 16 <= PAD) q[g][j] = pq[o + k + (qo - SK)];
                else if (k < SK) q[g][j] = pq[o + k + (k + lb < SK ? 0 : qo - SK)];
                else q[g][j] = pq[o + (k + lb < PAD ? k : PAD - 1 - lb) + (qo - SK)];
            }
        }
        __syncthreads();  // the previous tile is done with the stage
        rec_tile_stage<GK>(Rk, stage, M, t, ln);
        if (V_STAGED) rec_tile_stage<GV>(Rv, stage_v, M, t, ln);
        __syncthreads();
        uint32_t rk[GK::dwords];
        rec_from_lds<GK>(rk, stage, ln);
        float e[PAD];
        sq_coefficients<SK, SLK>(rk, e);
        const int pos = c * 64 + lane;
        const bool live = pos < n_kv;
        f32x4 s3[NG][3];
#pragma unroll
        for (int g = 0; g < NG; g++) s3[g][0] = s3[g][1] = s3[g][2] = z4;
        if constexpr (MX) score_all<NG>(q, e, s3, std::make_integer_sequence<int, PAD>{});
        float s[GM];
#pragma unroll
        for (int h = 0; h < GM; h++) {
            s[h] = -INFINITY;
            if constexpr (MX) {
                if (h < G && live) {
                    const f32x4(&v)[3] = s3[h / 4];
                    s[h] = (v[0][h % 4] + v[1][h % 4]) + v[2][h % 4];
                    if (scores) scores[(long long)(h0 + h) * s_stride + pos] = s[h];
                }
            } else if (h < G) {
                // the matrix path's sums bit for bit (three chains, coefficient k in chain k % 3)
                // on the vector unit. The head's factors are wave-uniform and arrive by scalar
                // loads, 16 at a time. With an output chunk k + 1 is loaded after the first product
                // of chunk k (a scalar-load wait covers every scalar load in flight, so the next
                // chunk cannot go out before the wait for the current one): 2% faster there; the
                // scores-only instances measured 4% slower with it and keep the compiler's
                // placement. (In a function of its own this spilled 130 scalar registers.)
                const float *__restrict__ qh = pq + h * ps;
                using QC = QChunks<SK>;
                float qa[16], qb[16];
#pragma unroll
                for (int i = 0; i < QC::size(0); i++) qa[i] = qh[i];
                float a[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int k = 0; k < QC::N; k++) {
                    float(&qc)[16] = (k & 1) ? qb : qa;
                    float(&qn)[16] = (k & 1) ? qa : qb;
                    const int e0 = QC::first(k);
                    a[e0 % 3] = fmaf(qc[0], e[e0], a[e0 % 3]);
                    if (k + 1 < QC::N) {
                        const float *__restrict__ qs = qh + (k + 1 < QC::NS ? 16 * (k + 1) : qo + 16 * (k + 1 - QC::NS));
                        if constexpr (OUT) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int i = 0; i < QC::size(k + 1); i++) qn[i] = qs[i];
                        if constexpr (OUT) __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int i = 1; i < QC::size(k); i++) a[(e0 + i) % 3] = fmaf(qc[i], e[e0 + i], a[(e0 + i) % 3]);
                }
                const float v = (a[0] + a[1]) + a[2];
                if (live) {
                    s[h] = v;
                    if (scores) scores[(long long)(h0 + h) * s_stride + pos] = v;
                }
            }
        }
        if (!OUT) continue;
        // ---- online softmax over the tile (wave-wide per head) ----
        float alpha[GM];
        f32x4 pr[NG];
#pragma unroll
        for (int g = 0; g < NG; g++) pr[g] = z4;
#pragma unroll
        for (int h = 0; h < GM; h++) {
            alpha[h] = 1.0f;
            if (h < G) {
                const float mn = fmaxf(m_run[h], wave_max(s[h]));
                alpha[h] = wave_uniform(__expf(m_run[h] - mn));
                const float p = live ? __expf(s[h] - mn) : 0.0f;
                l_run[h] = wave_uniform(fmaf(l_run[h], alpha[h], wave_add(p)));
                m_run[h] = wave_uniform(mn);
                pr[h / 4][h % 4] = p;
            }
        }
        if constexpr (MX) {
#pragma unroll
            for (int g = 0; g < NG; g++) *reinterpret_cast<f32x4 *>(Pw + ln * PP + 4 * g) = pr[g];
        } else {
#pragma unroll
            for (int h = 0; h < GM; h++) Pw[ln * PP + h] = pr[0][h];
        }
        // ---- V records of the tile, then their coefficients ----
        __syncthreads();  // every lane has read its K record from the stage
        if (!V_STAGED) {
            rec_tile_stage<GV>(Rv, stage, M, t, ln);
            __syncthreads();
        }
        uint32_t rv[GV::dwords];
        rec_from_lds<GV>(rv, stage_v, ln);
        float ev[PAD];
        sq_coefficients<SK, SLV>(rv, ev);
#pragma unroll
        for (int h = 0; h < GM; h++) {
            acc0[h / 4][h % 4] *= alpha[h];
            acc1[h / 4][h % 4] *= alpha[h];
            acc2[h / 4][h % 4] *= alpha[h];
            va0[h] *= alpha[h];
            va1[h] *= alpha[h];
            if (h == vh) va2 *= alpha[h];
        }
        // ---- weighted coefficient sums: chunk of 64 coefficients transposed through
        // LDS (row = coefficient, column = position), lane = coefficient ----
        float pw[NG][4];  // lane 4b + i, register j: head i, position 16j + b
        if constexpr (MX) {
#pragma unroll
            for (int g = 0; g < NG; g++)
#pragma unroll
                for (int j = 0; j < 4; j++) pw[g][j] = Pw[(16 * j + lb) * PP + 4 * g + li];
        }
#pragma unroll
        for (int ch = 0; ch < 3; ch++) {
            const int i0 = 64 * ch, n_i = ch < 2 ? 64 : C2;
#pragma unroll
            for (int i = 0; i < 64; i++)
                if (i < n_i) E[i * EP + ln] = ev[i0 + i];
            __syncthreads();
            if constexpr (!MX) {
                if (ch < 2) {
                    float(&va)[GM] = ch == 0 ? va0 : va1;
#pragma unroll 4
                    for (int p = 0; p < 64; p++) {
                        const float ei = E[ln * EP + p];
#pragma unroll
                        for (int h = 0; h < GM; h++) va[h] = fmaf(Pw[p * PP + h], ei, va[h]);
                    }
                } else if (v_on) {
#pragma unroll 4
                    for (int p = 0; p < 64; p++) va2 = fmaf(Pw[p * PP + vh], E[vi * EP + p], va2);
                }
            } else if (ch == 0) {
                sum_all<NG, 16, 4, 4>(pw, E + ln * EP, acc0);
            } else if (ch == 1) {
                sum_all<NG, 16, 4, 4>(pw, E + ln * EP, acc1);
            } else {
                // half h of the wave: head i, position 32h + 8j + b of its eight blocks b
#pragma unroll
                for (int g = 0; g < NG; g++)
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        pw[g][j] = Pw[(32 * half + 8 * j + lb % 8) * PP + 4 * g + li];
                sum_all<NG, 8, 3, 2>(pw, E + c2i * EP + 32 * half, acc2);
            }
            __syncthreads();
        }
    }
    if (!OUT) return;
    // ---- the run's partial per query head ----
#pragma unroll
    for (int h = 0; h < GM; h++) {
        float a2 = 0.0f;
        if constexpr (MX) a2 = acc2[h / 4][h % 4] + __shfl_xor(acc2[h / 4][h % 4], 32);
        if (h >= G) continue;
        float *dst = part + ((long long)(h0 + h) * n_runs + run) * pp;
        if (lane == 0) {
            dst[0] = m_run[h];
            dst[1] = l_run[h];
            dst[2] = 0.0f;
            dst[3] = 0.0f;
        }
        dst[4 + lane] = MX ? acc0[h / 4][h % 4] : va0[h];
        dst[4 + 64 + lane] = MX ? acc1[h / 4][h % 4] : va1[h];
        if (MX && lane < C2) dst[4 + 128 + lane] = a2;
        if (!MX && h == vh) dst[4 + 128 + vi] = va2;
    }
}

using SkelL77 = Layout<77, 5, 4, 4, 4, 5>;
using SkelL115 = Layout<115, 5, 4, 4, 4, 5>;
using SkelL115V3 = Layout<115, 3>;

// compute units of the current device (256 when the runtime cannot say)
int device_cus() {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        n <= 0)
        n = 256;
    return n;
}

// Whether a launch over `tiles` tiles (all sequences, KV heads and head groups) for g query heads
// a block takes its products on the matrix cores. A matrix instruction serves four heads
// whatever the number used, in the time of two vector instructions, and needs no factors from
// scalar loads: the better one for three heads and more, and for one or two while a SIMD has
// few waves to hide those loads (one wave a SIMD for one head, two for two). Measured on
// 256 CUs, 8 KV heads, skeleton 115, us, vector / matrix: one head, 30000 positions (3752 tiles)
// 38.3 / 46.2, 16 sequences of up to 1500 (about 2000) 35.8 / 39.2, 4 of up to 4000 (1300) 28.2 /
// 31.1, 2 KV heads at 30000 (938) 31.2 / 29.9; two heads, 43.2 / 47.0, 40.9 / 40.4, 32.7 / 31.9;
// four heads at 30000 52.9 / 48.1. Both give the same scores bit for bit.
bool on_matrix_cores(int g, long long tiles) { return g > 2 || tiles <= 4LL * g * device_cus(); }

// hs head groups per KV head (1 or 2): block x takes the query heads of group x.
template <int SK, class SLK, class SLV, int GM, bool MX>
void launch_split(const SpSqAttnArgs &A, const SpSeqTab &T, const float *prep, float *part, int n_runs, int hs,
                  hipStream_t s) {
    const dim3 grid(A.n_kvh * hs, n_runs, T.n_seq), block(64);
    const int G = A.n_q / A.n_kvh / hs;
    if (A.out)
        hipLaunchKernelGGL((k_sqfree_attn_split<SK, SLK, SLV, GM, MX, true>), grid, block, 0, s, A.kcache, A.vcache,
                           A.k_slot_bytes, A.v_slot_bytes, T, G, hs, prep, A.ps, A.qo, A.scores, part, A.pp, n_runs);
    else
        hipLaunchKernelGGL((k_sqfree_attn_split<SK, SLK, SLV, GM, MX, false>), grid, block, 0, s, A.kcache, A.vcache,
                           A.k_slot_bytes, A.v_slot_bytes, T, G, hs, prep, A.ps, A.qo, A.scores, part, A.pp, n_runs);
}

template <int SK, class SLK, class SLV>
void launch_split_g(const SpSqAttnArgs &A, const SpSeqTab &T, const float *prep, float *part, int n_runs, int hs,
                    hipStream_t s) {
    const int G = A.n_q / A.n_kvh / hs;
    long long tiles = 0;
    for (int i = 0; i < T.n_seq; i++) tiles += (long long)A.n_kvh * hs * ((T.len[i] + 63) / 64);
    const bool mx = on_matrix_cores(G, tiles);
    if (G <= 1 && !mx) launch_split<SK, SLK, SLV, 1, false>(A, T, prep, part, n_runs, hs, s);
    else if (G <= 2 && !mx) launch_split<SK, SLK, SLV, 2, false>(A, T, prep, part, n_runs, hs, s);
    else if (G <= 2) launch_split<SK, SLK, SLV, 2, true>(A, T, prep, part, n_runs, hs, s);
    else if (G <= 4) launch_split<SK, SLK, SLV, 4, true>(A, T, prep, part, n_runs, hs, s);
    else launch_split<SK, SLK, SLV, 8, true>(A, T, prep, part, n_runs, hs, s);
}

template <class SL>
bool bands_are(const SpPlan &P) {
    if (P.n_bands != SL::nb || P.total_bytes != SL::total) return false;
    for (int b = 0; b < SL::nb; b++)
        if (P.band_bits[b] != SL::bits[b] || P.band_off[b] != SL::off(b) || P.band_sz[b] != SL::sz(b)) return false;
    return true;
}

}  // namespace

// Which split kernel serves this cache geometry (0: none).
int sp_sqfree_attn_kind(const SpPlan &KP, const SpPlan &VP, const SpSqGeo &G) {
    if (!G.default_tables || G.hd != 128 || G.pad != PAD || G.rbits != RBITS || !G.spinor) return 0;
    if (G.sk_k == 77 && bands_are<SkelL77>(KP) && bands_are<SkelL77>(VP)) return 1;
    if (G.sk_k == 115 && bands_are<SkelL115>(KP) && bands_are<SkelL115>(VP)) return 2;
    if (G.sk_k == 115 && bands_are<SkelL115>(KP) && bands_are<SkelL115V3>(VP)) return 3;
    return 0;
}

namespace {
// One-wave blocks of the split kernel instance for this call that are resident on a CU
// at once (its registers and LDS decide; 4 when the runtime cannot say).
template <int SK, class SLK, class SLV, int GM>
int resident_per_cu(bool out) {
    int nb = 0;
    const hipError_t e =
        out ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_sqfree_attn_split<SK, SLK, SLV, GM, (GM > 2), true>, 64, 0)
            : hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_sqfree_attn_split<SK, SLK, SLV, GM, (GM > 2), false>, 64, 0);
    return e == hipSuccess && nb > 0 ? nb : 4;
}
template <int SK, class SLK, class SLV>
int resident_per_cu_g(int G, bool out) {
    if (G <= 1) return resident_per_cu<SK, SLK, SLV, 1>(out);
    if (G <= 2) return resident_per_cu<SK, SLK, SLV, 2>(out);
    if (G <= 4) return resident_per_cu<SK, SLK, SLV, 4>(out);
    return resident_per_cu<SK, SLK, SLV, 8>(out);
}
}  // namespace

// Runs per KV head and sequence: the blocks that are resident at once (the split
// kernel instance's occupancy) spread over the sequences' KV heads, so the launch runs
// in one round, every run getting at least one tile.
int sp_sqfree_attn_runs(const SpPlan &KP, const SpPlan &VP, const SpSqGeo &G, int n_q, int n_kvh, int n_kv, int cus,
                        int n_seq, bool out) {
    const int kind = sp_sqfree_attn_kind(KP, VP, G);
    if (!kind || n_kvh <= 0 || n_q % n_kvh) return 1;
    const int g = n_q / n_kvh;
    const int per_cu = kind == 1   ? resident_per_cu_g<77, SkelL77, SkelL77>(g, out)
                       : kind == 2 ? resident_per_cu_g<115, SkelL115, SkelL115>(g, out)
                                   : resident_per_cu_g<115, SkelL115, SkelL115V3>(g, out);
    const int tpo = (n_kv + 63) / 64;
    const int per_head = std::max(1, (per_cu * cus) / std::max(1, n_kvh * n_seq));
    return std::max(1, std::min(std::min(tpo, per_head), 1024));
}

hipError_t sp_launch_sqfree_attn(const SpPlan &KP, const SpPlan &VP, const SpSqGeo &G, const SpHierAttnArgs &HA,
                                 const SpSqAttnArgs &A, const SpSeqTab &T, float *ws, size_t ws_floats, int n_runs,
                                 hipStream_t s) {
    const int kind = sp_sqfree_attn_kind(KP, VP, G);
    if (!kind || A.n_kv <= 0 || A.n_q <= 0 || A.n_kvh <= 0 || A.n_q % A.n_kvh || A.n_q / A.n_kvh > 8 ||
        n_runs <= 0 || n_runs > 1024 || A.pp < 4 + PAD || A.ps != HA.ps || A.pp != HA.pp || T.n_seq < 1 ||
        T.n_seq > SP_ATTN_MAX_SEQ)
        return hipErrorInvalidValue;
    if (sp_hier_attn_workspace_floats(HA, n_runs, T.n_seq) > ws_floats) return hipErrorInvalidValue;
    float *prep = ws;
    float *part = ws + (size_t)T.n_seq * A.n_q * A.ps;
    hipError_t e = sp_launch_hier_attn_prep(KP, HA, T.n_seq, prep, s);
    if (e != hipSuccess) return e;
    // Two head groups per KV head when twice the blocks still run in one resident round
    // (a single sequence leaves half the wave slots empty otherwise): each tile's records
    // are then decoded twice, for half the heads each.
    int hs = 1;
    const int gq = A.n_q / A.n_kvh;
    if (gq % 2 == 0) {
        const bool out = A.out != nullptr;
        const int per_cu = kind == 1   ? resident_per_cu_g<77, SkelL77, SkelL77>(gq / 2, out)
                           : kind == 2 ? resident_per_cu_g<115, SkelL115, SkelL115>(gq / 2, out)
                                       : resident_per_cu_g<115, SkelL115, SkelL115V3>(gq / 2, out);
        if (2LL * A.n_kvh * n_runs * T.n_seq <= (long long)per_cu * device_cus()) hs = 2;
        // SP_HIP_SQFREE_ATTN_GROUPS=1 (read at each call) keeps one group (tests cover both)
        const char *eg = getenv("SP_HIP_SQFREE_ATTN_GROUPS");
        if (eg && eg[0] == '1') hs = 1;
    }
    if (kind == 1) launch_split_g<77, SkelL77, SkelL77>(A, T, prep, part, n_runs, hs, s);
    else if (kind == 2) launch_split_g<115, SkelL115, SkelL115>(A, T, prep, part, n_runs, hs, s);
    else launch_split_g<115, SkelL115, SkelL115V3>(A, T, prep, part, n_runs, hs, s);
    e = hipGetLastError();
    if (e != hipSuccess || !A.out) return e;
    return sp_launch_hier_attn_merge(KP, HA, T.n_seq, part, n_runs, s);
}
