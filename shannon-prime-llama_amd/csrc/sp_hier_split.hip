// sp_hier_split.hip -- the hierarchical codec at the default geometry (head_dim 256, pad
// 330 = 2*3*5*11, skeleton 30 in two 5-bit bands, 300 targets at 2 bits) with the work on
// a 64-vector tile split over the eight waves of a block.
//
// The arithmetic and its order are those of k_hier_encode / k_hier_decode
// (sp_cuda_hier_write_one / read_one, shannon_prime_hier.cu:399-571). Lane = vector, as in
// the one-wave kernels (sp_hier_lane.hip), which keep a whole vector in one lane's
// registers and so take one tile's serial time, 65 us, for any call of up to one tile per
// SIMD. Here the coefficients sit in LDS as [index][lane] and each wave takes a part:
//   * the transform's stages p = 2, 3, 5 act within 11 blocks of 30 coefficients, its
//     stage p = 11 across 30 columns of 11: blocks, then columns, by wave;
//   * the 9000-term prediction by target triples (the slot's rows through scalar loads, one
//     triple ahead);
//   * the tree sum of the deviations by the eight classes of target mod 8, which its first
//     five levels (strides 128 .. 8) never mix;
//   * the levels by record dwords.
// Bound by VALU issue (about 34k instructions a tile over four SIMDs) at two waves a SIMD.
#include "sp_hier_codec.h"

namespace {

constexpr int HD = 256, PAD = 330, NS = 30, NT = PAD - NS, NW = 8, THREADS = 64 * NW;
constexpr int RW = NS / 2;       // dwords of a predictor row
constexpr int TRIPLES = NT / 3;
using SkL = Layout<NS, 5, 5>;
using Rec = HierRec<NT, 2, SkL>;
static_assert(Rec::total == 103 && Rec::mag_byte == 24 && Rec::res_bit == 224, "record fields on the bytes assumed below");
constexpr int RES_BYTE = Rec::res_bit / 8, RES_DW = (NT * 2 + 31) / 32;
constexpr int STAGE = (64 * Rec::total + 16 + 16 + 15) & ~15;  // records at byte (address & 15)

// order[p]: the coefficient at place p of the squarefree-first order (skeleton, then
// targets); place[i]: the inverse.
struct HierOrder {
    int order[PAD], place[PAD];
    constexpr HierOrder() : order(), place() {
        const MobOrder<PAD> mo{};
        for (int p = 0; p < PAD; p++) order[p] = mo.v[p], place[mo.v[p]] = p;
    }
};
__constant__ const HierOrder kOrd{};

// Two block-stage parts of the transform on 30 consecutive coefficients: p = 3 and 5 (after
// p = 2).
__device__ __forceinline__ void block_stages_35(float (&x)[30], const XfConst &K) {
    vil_stage<30, 3, 2>(x, K);
    vil_stage<30, 5, 6>(x, K);
}

// Predictions of target triples w, w + 8, ...: f(triple, p0, p1, p2) for each. The next
// triple's rows load behind the current one's products (the last loads its own again).
template <class F>
__device__ __forceinline__ void predict_triples(wptr_t w32, int w, const float (&sk)[NS], F f) {
    uint32_t wa[3 * RW], wb[3 * RW];
    int i = w;
#pragma unroll
    for (int k = 0; k < 3 * RW; k++) wa[k] = w32[i * 3 * RW + k];
    for (;;) {
        float p0, p1, p2;
        int nx = min(i + NW, TRIPLES - 1);
        hier_predict3<NS, true>(wa, wb, w32 + nx * 3 * RW, sk, sk[0], p0, p1, p2);
        f(i, p0, p1, p2);
        i += NW;
        if (i >= TRIPLES) break;
        nx = min(i + NW, TRIPLES - 1);
        hier_predict3<NS, true>(wb, wa, w32 + nx * 3 * RW, sk, sk[0], p0, p1, p2);
        f(i, p0, p1, p2);
        i += NW;
        if (i >= TRIPLES) break;
    }
}

// One side of a call (K or V): rows at src + (o*so + i*si) elements, records at dst + o*dout.
struct EncSide {
    const void *src;
    unsigned char *dst;
};
struct DecSide {
    const unsigned char *src;
    void *dst;
};

template <int DT>
__global__ void __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(2)))
k_hier_encode_split(const EncSide s0, const EncSide s1, long long so, long long si, long long dout,
                    int n_inner, int tiles_per_outer, int n_tiles, const XfConst K, const uint16_t *__restrict__ W, long long w_outer) {
    constexpr int ES = DT == SP_DT_F16 ? 2 : 4, RB = HD * ES, RP = RB + 16, CPR = RB / 16;
    __shared__ __attribute__((aligned(16))) unsigned char rows[64 * RP];  // input rows
    __shared__ float C[PAD * 64];                                         // coefficients, then deviations: [place][lane]
    __shared__ __attribute__((aligned(16))) unsigned char stage[STAGE];
    __shared__ float part[NW * 64];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const TileMap M{tiles_per_outer, n_inner};
    const bool second = (int)blockIdx.x >= n_tiles;
    const void *src = second ? s1.src : s0.src;
    unsigned char *dst = second ? s1.dst : s0.dst;
    int o, i0, nv;
    M.at(second ? (int)blockIdx.x - n_tiles : (int)blockIdx.x, o, i0, nv);

    // ---- rows into LDS (a row past the last is the last again) ----
    {
        const unsigned char *g = reinterpret_cast<const unsigned char *>(src) + ((long long)o * so + (long long)i0 * si) * ES;
        u32x4 v[64 * CPR / THREADS];
#pragma unroll
        for (int j = 0; j < 64 * CPR / THREADS; j++) {
            const int q = tid + j * THREADS, r = min(q / CPR, nv - 1);
            v[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(g + (long long)r * si * ES + (q % CPR) * 16));
        }
#pragma unroll
        for (int j = 0; j < 64 * CPR / THREADS; j++) {
            const int q = tid + j * THREADS;
            *reinterpret_cast<u32x4 *>(rows + (q / CPR) * RP + (q % CPR) * 16) = v[j];
        }
    }
    __syncthreads();

    // ---- stages 2, 3, 5: waves 0-3 two blocks of 30 each (coefficients 60w ..), wave 4 the
    // block the pad mean starts in, wave 5 the blocks that are all mean (equal) ----
    const unsigned char *row = rows + lane * RP;
    float mx = 0.0f;
    if (w < 4) {
        float x[2][30];
        if (DT == SP_DT_F16) {
#pragma unroll
            for (int q = 0; q < 15; q++) {
                const uint2 a = *reinterpret_cast<const uint2 *>(row + 120 * w + 8 * q);
                const uint32_t wd[2] = {a.x, a.y};
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    const int e = 4 * q + 2 * k;
                    vil_first_f16_pair(wd[k], K.isp[0], x[e / 30][e % 30], x[e / 30][e % 30 + 1]);
                }
            }
        } else {
#pragma unroll
            for (int q = 0; q < 15; q++) {
                const float4 a = *reinterpret_cast<const float4 *>(row + 240 * w + 16 * q);
                const float f[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
                for (int k = 0; k < 4; k++) x[(4 * q + k) / 30][(4 * q + k) % 30] = f[k];
            }
#pragma unroll
            for (int b = 0; b < 2; b++) vil_stage<30, 2, 1>(x[b], K);
        }
#pragma unroll
        for (int b = 0; b < 2; b++) {
            block_stages_35(x[b], K);
#pragma unroll
            for (int k = 0; k < 30; k++) C[(60 * w + 30 * b + k) * 64 + lane] = x[b][k];
        }
    } else if (w < 6) {
        // pad mean: the 256-slot tree over the row, x[i] + x[i + 128] first
        float l1[HD / 2];
        if (DT == SP_DT_F16) {
#pragma unroll
            for (int q = 0; q < HD / 16; q++) {
                const uint4 a = *reinterpret_cast<const uint4 *>(row + q * 16);
                const uint4 b = *reinterpret_cast<const uint4 *>(row + HD + q * 16);
                const uint32_t wa[4] = {a.x, a.y, a.z, a.w}, wb[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    l1[q * 8 + 2 * k] = add_f16_halves<0>(wa[k], wb[k]);
                    l1[q * 8 + 2 * k + 1] = add_f16_halves<1>(wa[k], wb[k]);
                }
            }
        } else {
#pragma unroll
            for (int q = 0; q < HD / 8; q++) {
                const float4 a = *reinterpret_cast<const float4 *>(row + q * 16);
                const float4 b = *reinterpret_cast<const float4 *>(row + 2 * HD + q * 16);
                const float fa[4] = {a.x, a.y, a.z, a.w}, fb[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    l1[q * 4 + k] = fa[k] + fb[k];
                    mx = fmaxf(mx, fmaxf(fabsf(fa[k]), fabsf(fb[k])));
                }
                if (q % 4 == 3) __asm__ volatile("" ::: "memory");  // no more than eight pieces in flight
            }
        }
#pragma unroll
        for (int s = HD / 4; s > 0; s >>= 1) {
#pragma unroll
            for (int i = 0; i < s; i++) l1[i] = l1[i] + l1[i + s];
        }
        const float mean = sp_div(l1[0] + 0.0f, (float)HD);
        float x[30];
#pragma unroll
        for (int k = 0; k < 30; k++) x[k] = mean;
        if (w == 4) {  // coefficients 240 .. 255 of the row, then the mean
#pragma unroll
            for (int k = 0; k < 16; k++) x[k] = sp_load1<DT>(row, 240 + k);
        }
        vil_stage<30, 2, 1>(x, K);
        block_stages_35(x, K);
        const int at = w == 4 ? 240 : 270;
#pragma unroll
        for (int k = 0; k < 30; k++) C[(at + k) * 64 + lane] = x[k];
        if (w == 5) {
#pragma unroll
            for (int k = 0; k < 30; k++) C[(300 + k) * 64 + lane] = x[k];
        }
    }
    __syncthreads();

    // ---- stage 11: columns w, w + 8, ...; the results go to their places in the order
    // (skeleton, then targets), so every column is read before any is written ----
    {
        float x[4][11];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int c = min(w + NW * j, 29);
#pragma unroll
            for (int k = 0; k < 11; k++) x[j][k] = C[(c + 30 * k) * 64 + lane];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int c = w + NW * j;
            if (c >= 30) break;
            vil_stage<11, 11, 1>(x[j], K);
#pragma unroll
            for (int k = 0; k < 11; k++) C[kOrd.place[c + 30 * k] * 64 + lane] = x[j][k];
        }
    }
    __syncthreads();

    // ---- the skeleton (every wave), its bands (wave 5, which knows the largest input), and
    // the deviations of the targets from the prediction of the unquantized skeleton ----
    float sk[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) sk[s] = C[s * 64 + lane];
    const int nbytes = nv * Rec::total;
    unsigned char *const gdst = dst + (long long)o * dout + (long long)i0 * Rec::total;
    const int sh = (int)((uintptr_t)gdst & 15);
    unsigned char *const myrec = stage + sh + lane * Rec::total;
    if (w == 5) {
        // growth is at most sqrt(2p) per stage: fp16 inputs stay finite, fp32
        // inputs below 2^100 too; inf/NaN inputs reach the DC coefficient
        const bool fastv = (DT == SP_DT_F16 || mx < 1.2676506e30f) && __builtin_isfinite(sk[0]);
        uint32_t rec[SkL::dwords];
#pragma unroll
        for (int d = 0; d < SkL::dwords; d++) rec[d] = 0u;
        quant_bands<SkL, false>(sk, fastv, rec);
#pragma unroll
        for (int b = 0; b < SkL::total; b++) myrec[b] = (unsigned char)(rec[b / 4] >> (8 * (b % 4)));
    }
    const wptr_t w32 = (wptr_t)(W + (long long)__builtin_amdgcn_readfirstlane(o) * w_outer);
    predict_triples(w32, w, sk, [&](int i, float p0, float p1, float p2) {
        float *c = C + (NS + 3 * i) * 64 + lane;
        c[0] = c[0] - p0;
        c[64] = c[64] - p1;
        c[128] = c[128] - p2;
    });
    __syncthreads();

    // ---- residual magnitude: class w of the 256-slot tree (slots w + 8i), then the classes ----
    {
        float s[32];
#pragma unroll
        for (int i = 0; i < 32; i++) s[i] = C[(NS + w + 8 * i) * 64 + lane];
#pragma unroll
        for (int i = 0; i < 32; i++) s[i] = fabsf(s[i]);
#pragma unroll
        for (int i = 0; 8 * i < NT - 256; i++)
            if (w + 8 * i + 256 < NT) s[i] = s[i] + fabsf(C[(NS + w + 8 * i + 256) * 64 + lane]);
#pragma unroll
        for (int h = 16; h > 0; h >>= 1) {
#pragma unroll
            for (int i = 0; i < h; i++) s[i] = s[i] + s[i + h];
        }
        part[w * 64 + lane] = s[0];
    }
    __syncthreads();
    float q[NW];
#pragma unroll
    for (int j = 0; j < NW; j++) q[j] = part[j * 64 + lane];
#pragma unroll
    for (int h = NW / 2; h > 0; h >>= 1) {
#pragma unroll
        for (int j = 0; j < h; j++) q[j] = q[j] + q[j + h];
    }
    float mag = sp_div(q[0], (float)NT);
    mag = mag < 1e-12f ? 1e-12f : mag;
    // levels rint(dev * inv_step + center) clamped to [0, 3] with step = 2*mag/3
    // (shannon_prime_hier.cu:151-171); clamping before the rounding gives the same level
    // for every value, NaN (-> 0) included
    const float step = sp_div(2.0f * mag, 3.0f);
    const float inv_step = (step > 0.0f) ? sp_div(1.0f, step) : 0.0f;
    for (int d = w; d < RES_DW; d += NW) {
        uint32_t word = 0;
        const float *c = C + (NS + 16 * d) * 64 + lane;
        const int n = d == RES_DW - 1 ? NT - 16 * (RES_DW - 1) : 16;
#pragma unroll
        for (int e = 0; e < 16; e++) {
            if (e >= NT - 16 * (RES_DW - 1) && e >= n) break;  // the last dword holds 12
            const float v = c[e * 64] * inv_step + 1.5f;
            const float cl = fminf(fmaxf(v, 0.0f), 3.0f);
            // cl + 1.5 * 2^23 rounds cl to the nearest integer, ties to even
            word |= (__float_as_uint(cl + 12582912.0f) & 3u) << (2 * e);
        }
        unsigned char *p = myrec + RES_BYTE + 4 * d;
        p[0] = (unsigned char)word;
        p[1] = (unsigned char)(word >> 8);
        p[2] = (unsigned char)(word >> 16);
        if (n == 16) p[3] = (unsigned char)(word >> 24);
    }
    if (w == NW - 1) {
        const uint32_t mb = __float_as_uint(mag);
#pragma unroll
        for (int b = 0; b < 4; b++) myrec[Rec::mag_byte + b] = (unsigned char)(mb >> (8 * b));
    }
    __syncthreads();

    // ---- records out: the stage mirrors the destination's 16-byte alignment; whole pieces as
    // such, the first and the last by bytes ----
    {
        unsigned char *g0 = gdst - sh;
        const int b0 = 16 * tid, end = sh + nbytes;
        if (b0 >= sh && b0 + 16 <= end) {
            *reinterpret_cast<u32x4 *>(g0 + b0) = *reinterpret_cast<const u32x4 *>(stage + b0);
        } else if (b0 < end && b0 + 16 > sh) {
            for (int b = max(b0, sh); b < min(b0 + 16, end); b++) g0[b] = stage[b];
        }
    }
}

// The 32 bits at byte `at` of the LDS records.
__device__ __forceinline__ uint32_t stage_u32(const unsigned char *stage, int at) {
    const uint32_t *p = reinterpret_cast<const uint32_t *>(stage + (at & ~3));
    return __builtin_amdgcn_alignbit(p[1], p[0], 8u * (uint32_t)(at & 3));
}

template <int DT>
__global__ void __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(2)))
k_hier_decode_split(const DecSide s0, const DecSide s1, long long so, long long dout, long long din,
                    int n_inner, int tiles_per_outer, int n_tiles, const XfConst K, const uint16_t *__restrict__ W, long long w_outer) {
    constexpr int ES = DT == SP_DT_F16 ? 2 : 4, RB = HD * ES, CPR = RB / 16;
    constexpr int RP = RB + 4;  // an odd number of dwords: lanes' element writes fall in distinct banks
    __shared__ float C[PAD * 64];  // coefficients [index][lane]
    __shared__ __attribute__((aligned(16))) unsigned char stage[STAGE];
    __shared__ __attribute__((aligned(16))) unsigned char rows[64 * RP];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const TileMap M{tiles_per_outer, n_inner};
    const bool second = (int)blockIdx.x >= n_tiles;
    const unsigned char *src = second ? s1.src : s0.src;
    void *dst = second ? s1.dst : s0.dst;
    int o, i0, nv;
    M.at(second ? (int)blockIdx.x - n_tiles : (int)blockIdx.x, o, i0, nv);

    // ---- the tile's records as the 16-byte pieces that cover them (the caches begin on such a
    // boundary and carry slack past their last record) ----
    const unsigned char *g = src + (long long)o * so + (long long)i0 * Rec::total;
    const int sh = (int)((uintptr_t)g & 15);
    if (16 * tid < sh + nv * Rec::total)
        *reinterpret_cast<u32x4 *>(stage + 16 * tid) = *reinterpret_cast<const u32x4 *>(g - sh + 16 * tid);
    __syncthreads();

    // ---- skeleton (every wave) and targets: prediction plus (level - 1.5) * step ----
    const int rb = sh + lane * Rec::total;
    float sk[NS];
    float step;
    {
        uint32_t rec[7];
#pragma unroll
        for (int d = 0; d < 7; d++) rec[d] = stage_u32(stage, rb + 4 * d);
        dequant_bands<SkL, false, true>(rec, SkL::nb, sk);
        step = sp_div(2.0f * __uint_as_float(rec[6]), 3.0f);
    }
    if (w == NW - 1) {  // (a wave with 12 triples)
#pragma unroll
        for (int s = 0; s < NS; s++) C[kHier<PAD, NS>.skel[s] * 64 + lane] = sk[s];
    }
    const wptr_t w32 = (wptr_t)(W + (long long)__builtin_amdgcn_readfirstlane(o) * w_outer);
    predict_triples(w32, w, sk, [&](int i, float p0, float p1, float p2) {
        const int at = rb + RES_BYTE + (6 * i) / 8;
        const uint32_t lv = ((uint32_t)stage[at] | ((uint32_t)stage[at + 1] << 8)) >> ((6 * i) % 8);
        C[kOrd.order[NS + 3 * i] * 64 + lane] = p0 + ((float)(lv & 3u) - 1.5f) * step;
        C[kOrd.order[NS + 3 * i + 1] * 64 + lane] = p1 + ((float)((lv >> 2) & 3u) - 1.5f) * step;
        C[kOrd.order[NS + 3 * i + 2] * 64 + lane] = p2 + ((float)((lv >> 4) & 3u) - 1.5f) * step;
    });
    __syncthreads();

    // ---- stages 2, 3, 5 on blocks of 30, in place ----
    for (int b = w; b < 11; b += NW) {
        float x[30];
#pragma unroll
        for (int k = 0; k < 30; k++) x[k] = C[(30 * b + k) * 64 + lane];
        vil_stage<30, 2, 1>(x, K);
        block_stages_35(x, K);
#pragma unroll
        for (int k = 0; k < 30; k++) C[(30 * b + k) * 64 + lane] = x[k];
    }
    __syncthreads();

    // ---- stage 11 on columns, the first 256 elements to the rows ----
    for (int c = w; c < 30; c += NW) {
        float x[11];
#pragma unroll
        for (int k = 0; k < 11; k++) x[k] = C[(c + 30 * k) * 64 + lane];
        vil_stage<11, 11, 1>(x, K);
#pragma unroll
        for (int k = 0; k < 9; k++)
            if (c + 30 * k < HD) sp_store1<DT>(rows + lane * RP, c + 30 * k, x[k]);
    }
    __syncthreads();

    // ---- rows out ----
    unsigned char *gd = reinterpret_cast<unsigned char *>(dst) + ((long long)o * dout + (long long)i0 * din) * ES;
#pragma unroll
    for (int j = 0; j < 64 * CPR / THREADS; j++) {
        const int q = tid + j * THREADS, r = q / CPR;
        if (r < nv) {
            const uint32_t *p = reinterpret_cast<const uint32_t *>(rows + r * RP + (q % CPR) * 16);
            const u32x4 v = {p[0], p[1], p[2], p[3]};
            __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(gd + (long long)r * din * ES + (q % CPR) * 16));
        }
    }
}

bool geometry_matches(const SpPlan &P, const SpHierGeo &G) {
    return G.default_geo && G.hd == HD && G.pad == PAD && G.n_skel == NS && G.n_target == NT && G.rbits == 2 &&
           G.bytes == Rec::total && layout_matches<SkL>(P) && vil_consts_exact(P) && ((uintptr_t)G.W % 4) == 0 &&
           (G.w_outer % 2) == 0;
}

}  // namespace

// A CU takes a tile in 20.5 us (encode; decode 18.3) here, one tile at a time, and in 65 us as
// four one-wave tiles side by side in the lane kernels (`launches` of them). So fp16 calls
// compare whole rounds of each: 8 heads, K and V, 2048 positions (512 tiles) 42 us encode and 40
// decode against 66 and 126, 6144 positions 121 and 107 against 137 and 131, 16384 positions 312
// and 282 against 282 and 268 (the lane kernels). fp32 rows always pay: the lane kernels' second
// row register set halves them (32768 positions 690 and 586 us against 1084 and 1026).
bool sp_hier_split_pays(int dtype, long long tiles, int launches) {
    if (dtype != SP_DT_F16) return true;
    const long long cus = device_cu_count(), per = (tiles + launches - 1) / launches;
    return 5 * ((tiles + cus - 1) / cus) <= 16 * launches * ((per + 4 * cus - 1) / (4 * cus));
}

hipError_t sp_launch_hier_encode_split(const SpPlan &P, const SpHierGeo &G, const void *src, int dtype, long long so,
                                       long long si, unsigned char *dst, long long dout, int n_outer, int n_inner,
                                       hipStream_t s, const void *src2, unsigned char *dst2) {
    const int esz = dtype == SP_DT_F16 ? 2 : 4;
    if (((uintptr_t)src % 16) || ((so * esz) % 16) || ((si * esz) % 16) || si < HD || (src2 && ((uintptr_t)src2 % 16 || !dst2)))
        return hipErrorNotSupported;
    if (!geometry_matches(P, G)) return hipErrorNotSupported;
    const int tpo = (n_inner + 63) / 64;
    const long long n_tiles = (long long)n_outer * tpo, blocks = n_tiles * (src2 ? 2 : 1);
    if (n_tiles <= 0 || blocks > 0x7fffffffLL) return hipErrorNotSupported;
    const EncSide a{src, dst}, b{src2, dst2};
    if (dtype == SP_DT_F16)
        hipLaunchKernelGGL((k_hier_encode_split<SP_DT_F16>), dim3((unsigned)blocks), dim3(THREADS), 0, s, a, b, so, si, dout,
                           n_inner, tpo, (int)n_tiles, xf_const(P), G.W, G.w_outer);
    else
        hipLaunchKernelGGL((k_hier_encode_split<SP_DT_F32>), dim3((unsigned)blocks), dim3(THREADS), 0, s, a, b, so, si, dout,
                           n_inner, tpo, (int)n_tiles, xf_const(P), G.W, G.w_outer);
    return hipGetLastError();
}

hipError_t sp_launch_hier_decode_split(const SpPlan &P, const SpHierGeo &G, const unsigned char *src, long long so, void *dst,
                                       int dtype, long long dout, long long din, int n_outer, int n_inner, hipStream_t s,
                                       const unsigned char *src2, void *dst2) {
    const int esz = dtype == SP_DT_F16 ? 2 : 4;
    if (((uintptr_t)dst % 16) || ((dout * esz) % 16) || ((din * esz) % 16) || din < HD || (src2 && ((uintptr_t)dst2 % 16 || !dst2)))
        return hipErrorNotSupported;
    if (!geometry_matches(P, G)) return hipErrorNotSupported;
    const int tpo = (n_inner + 63) / 64;
    const long long n_tiles = (long long)n_outer * tpo, blocks = n_tiles * (src2 ? 2 : 1);
    if (n_tiles <= 0 || blocks > 0x7fffffffLL) return hipErrorNotSupported;
    const DecSide a{src, dst}, b{src2, dst2};
    if (dtype == SP_DT_F16)
        hipLaunchKernelGGL((k_hier_decode_split<SP_DT_F16>), dim3((unsigned)blocks), dim3(THREADS), 0, s, a, b, so, dout, din,
                           n_inner, tpo, (int)n_tiles, xf_const(P), G.W, G.w_outer);
    else
        hipLaunchKernelGGL((k_hier_decode_split<SP_DT_F32>), dim3((unsigned)blocks), dim3(THREADS), 0, s, a, b, so, dout, din,
                           n_inner, tpo, (int)n_tiles, xf_const(P), G.W, G.w_outer);
    return hipGetLastError();
}
