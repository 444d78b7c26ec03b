// sp_attn_wave.h -- the matrix-core decode-attention kernel over ship records: one
// template, instantiated per record layout in sp_attn_wave*.hip.
//
// Same algebra as the general kernel (sp_attn.hip), replacing the CPU op
// llama_sp_kq_compute (src/engine/llama_sp_fused_kq.cpp:83-165) and the ggml
// softmax . V after it: with q~ = kq_scale * reorder(transform(q)),
//   score_t = sum_b scale_b[t] * sum_{k in b} q~[k] (u_k - m_b),
//   sum_t p_t V~_t = transform(sum_t p_t dq(V_t)).
//
// Block = NW waves, one sequence, one KV head, a run of consecutive 64-position tiles;
// each wave works its own tiles with no block barrier:
//   * the tile's K and V records arrive as 16-byte buffer loads (range-checked,
//     so a partial tile reads zeros) and are staged in the wave's LDS region;
//     lane t then holds record t of the K tile in registers. Records may start 2 bytes
//     off a dword (a sequence at an odd cell of a layout whose records are 2 mod 4
//     bytes): the tile is loaded from the dword below.
//   * scores on v_mfma_f32_4x4x4_16b_f16 (16 blocks of 4 x 4 x 4): block b's
//     rows are positions 4b .. 4b+3 (A: lane 4b + i gives 4 codes of its own
//     record as fp16, see "score slots" below), its columns 4 query heads
//     (B: the query's fp16 hi and lo parts from LDS, two MFMAs into the same
//     accumulator), K = 4 coefficients of one band, one accumulator per band.
//     Every code field sits at a compile-time bit of the record. Lane 4b + j
//     ends with head j's scores for positions 4b .. 4b+3; band scales come from
//     the quad's records by DPP broadcast.
//   * softmax over the tile in that layout (4 positions of one head per lane);
//     the weights w = p * scale_v, scaled per head by a power of two, go to LDS
//     as fp16 hi + lo rows.
//   * values on v_mfma_f32_16x16x32_f16, A = weights, B = V codes: a lane's
//     column n covers EPC = head_dim / 16 consecutive elements (one or two 32-bit
//     windows of the record) and its two K slots per dword are two positions, so a
//     permute puts both positions' codes of an element in one dword; a shift and an
//     and-or land each at the top of an fp16 mantissa (2^BITS + u), and a packed
//     subtract centres it (u - m, exact).
//   * the block's waves merge their (m, l, o~) in LDS. A sequence and KV head that is one
//     block is finished there; otherwise each block writes one spectral-domain partial
//     [m, l, o~[head_dim]] per query head with agent-scope atomic stores, waits for them
//     to complete and counts itself on its KV head's counter; the block that arrives
//     last reads the partials back with agent-scope atomic loads, merges them and
//     applies one inverse transform per head.
//
// What bounds it: a few tiles per SIMD are a chain of latencies (the launch, the query,
// the records, the merge across blocks); many are VALU issue (about 740 instructions per
// 64-position tile at head_dim 96, 660 at 128, of which unpacking codes to fp16 is half).
// Measured per layer, 8 KV heads unless said (before: the general kernel of sp_attn.hip;
// at head_dim 96 a lane-per-position kernel; at 128 this kernel once per sequence):
//   head_dim 64, K 5/4/4 V 5, GQA 4: 4096 positions 100 -> 7.3 us, 131072 455 -> 25 us
//   head_dim 96, 32 KV heads, 16 x 4096 positions: 86 -> 55 us (4.6 TB/s of records)
//   head_dim 128, GQA 4: 12 sequences of 1100-4500 positions 157 -> 22 us; one of 8192
//     13.9 -> 10.5 us, of 131072 63.5 -> 42 us
//   head_dim 256, GQA 2: 8191 positions 147 -> 13.4 us, 131072 1414 -> 62 us
#pragma once

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <type_traits>
#include <utility>

#include "sp_internal.h"
#include "sp_mfma_codes.h"

namespace {

typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef float float4_t __attribute__((ext_vector_type(4)));

constexpr int TILE = 64;                     // positions per wave and tile
constexpr uint32_t BUF_WORD3 = 0x00020000u;  // raw buffer resource, dword data (gfx9 family)
constexpr int BUF_NT = 2;                    // non-temporal load policy

struct SpNoTab {};  // a single sequence needs no table

constexpr int c_r16(int n) { return (n + 15) & ~15; }

// Score slots. A band's codes are fed to the MFMAs in pairs, one dword of two fp16
// (pair p: slots 2p, 2p + 1; a step takes two pairs). A pair built with one shift and
// one masked OR needs its two codes about 16 bits apart:
//   5-bit bands: codes i and i + 3 of a span of 6 are 15 bits apart: the first code
//     lands at mantissa bits 5..9 (2^5 + c), the second at bits 4..8 of the high half
//     (2^5 + c/2: half gain, so its query slot holds 2q~);
//   3-bit bands: likewise codes i and i + 5 of a span of 10;
//   4-bit bands: codes i and i + 4 of a span of 8 are 16 bits apart (both 2^4 + c).
// Codes past the last whole span pair with their neighbour (both 2^BITS + c); slots past
// the band's codes hold a zero query.
constexpr int c_half(int bits) { return bits == 5 ? 3 : bits == 4 ? 4 : 5; }

template <int HD_, int VBITS_, bool CENTRE_, int... KBITS>
struct WaveLayout {
    static constexpr int HD = HD_, NB = sizeof...(KBITS), VBITS = VBITS_;
    // CENTRE: K codes are centred (u - m, exact) before the MFMA. Otherwise the
    // accumulator starts at -(offset + m) * sum(q~), one VALU instruction per pair
    // cheaper, at about twice the rounding error of the fp32 dot product.
    static constexpr bool CENTRE = CENTRE_;
    static constexpr int bits[NB] = {KBITS...};
    static constexpr int off(int b) { return b * (HD / NB); }
    static constexpr int sz(int b) { return b == NB - 1 ? HD - off(b) : HD / NB; }
    static constexpr int kbyte(int b) {
        int o = 0;
        for (int i = 0; i < b; i++) o += 2 + (sz(i) * bits[i] + 7) / 8;
        return o;
    }
    static constexpr int KB = kbyte(NB), VB = 2 + HD * VBITS / 8;
    static_assert(KB % 2 == 0 && VB % 2 == 0 && HD % 16 == 0, "records of whole 16-bit words");
    static constexpr int spans(int b) { return sz(b) / (2 * c_half(bits[b])); }
    static constexpr int rest(int b) { return sz(b) - spans(b) * 2 * c_half(bits[b]); }
    static constexpr int pairs(int b) { return spans(b) * c_half(bits[b]) + (rest(b) + 1) / 2; }
    static constexpr int steps(int b) { return (pairs(b) + 1) / 2; }
    static constexpr int slot0(int b) {
        int o = 0;
        for (int i = 0; i < b; i++) o += 4 * steps(i);
        return o;
    }
    static constexpr int SLOTS = slot0(NB);
    static constexpr int max_steps() {
        int m = 0;
        for (int i = 0; i < NB; i++) m = steps(i) > m ? steps(i) : m;
        return m;
    }
    // V columns: EPC consecutive elements per MFMA column, in NWIN 32-bit windows
    static constexpr int EPC = HD / 16, NWIN = EPC * VBITS > 32 ? 2 : 1, EPW = EPC / NWIN;
    static_assert(EPW * VBITS <= 32, "a window holds its codes");
    // transforms in registers: lane l holds elements (l % EL) + EL * e, e < NE
    static constexpr int EL = HD == 96 ? 32 : 64, NE = HD / EL;
    static constexpr int HP = (HD + 63) & ~63;  // threads per head in the merges (whole waves)
    static constexpr int KDW = (KB + 3) / 4;
    static constexpr int K_LOADS = (TILE * KB + 2 + 1023) / 1024, V_LOADS = (TILE * VB + 2 + 1023) / 1024;  // 16 B per lane
    // Per-wave LDS region (bytes). Once every lane holds its K record in registers the K
    // area carries the weight rows and the per-head softmax state; before the records
    // land it is the scratch of the query's reorder.
    static constexpr int WT_STRIDE = 72;  // fp16 per weight row: 64 slots + 8 (bank shift)
    static constexpr int R_ST = 16 * WT_STRIDE * 2;  // per head [m, l, 1/f, -] f32
    static constexpr int R_V = c_r16(TILE * KB + 16);
    static constexpr int R_SIZE = R_V + c_r16(2 + TILE * VB + 14);
    static_assert(R_ST + 8 * 16 <= R_V && HD * 4 <= R_V, "K area holds the weights and state, and a query");
    static constexpr int QS_STRIDE = SLOTS + 4;  // fp16 per (part, head) query row: the 4 heads of a read fall in distinct banks
    static constexpr int MB_STRIDE = HD + 4;     // floats per (wave, head) in the in-block merge: m, l, -, -, o~[HD]
};

// Block-shared LDS after the wave regions.
template <class LY, int NW>
struct WaveLds {
    static constexpr int WAVES = NW * (LY::R_SIZE > 8 * LY::MB_STRIDE * 4 ? LY::R_SIZE : 8 * LY::MB_STRIDE * 4);
    static constexpr int QS = WAVES;                              // query operand [part][head 8][QS_STRIDE] fp16
    static constexpr int CB = c_r16(QS + 2 * 8 * LY::QS_STRIDE * 2);  // accumulator starts [head 8][band 4] f32
    static constexpr int FU = CB + 8 * 4 * 4;                     // inverse query scale [head 8] f32
    static constexpr int FLAG = FU + 8 * 4;  // [0] the block arrived last for its KV head, [1] query operand ready
    static constexpr int BYTES = FLAG + 16;
    static_assert(BYTES <= 160 * 1024, "LDS of one CU");
    // the final merge's o~ of two halves and (M, L) of the second
    static_assert((2 * 8 * LY::HP + 16) * 4 <= WAVES, "merge scratch fits the wave regions");
};

// Where record coefficient r goes: its slot (bits 0..7), half gain (bit 8), band (bits 9..).
// A table: the query's preparation loads its entries beside the query row.
template <class LY>
struct SlotTable {
    unsigned short v[LY::HD];
    constexpr SlotTable() : v() {
        for (int b = 0; b < LY::NB; b++) {
            const int half = c_half(LY::bits[b]), span = 2 * half, n = LY::spans(b);
            for (int c = 0; c < LY::sz(b); c++) {
                const int g = c / span, i = c % span;
                int slot = 0, gain = 0;
                if (c >= n * span) slot = 2 * n * half + (c - n * span);
                else if (i < half) slot = 2 * (half * g + i);
                else slot = 2 * (half * g + i - half) + 1, gain = LY::bits[b] != 4;
                v[LY::off(b) + c] = (unsigned short)((LY::slot0(b) + slot) | (gain << 8) | (b << 9));
            }
        }
    }
};
template <class LY>
__device__ constexpr SlotTable<LY> kSlots{};

// The 32 record bits starting at bit p (p compile-time after unrolling; bits past
// the record's dwords read from the zero dword r[DW]).
template <int N>
__device__ __forceinline__ uint32_t rec_window(const uint32_t (&r)[N], int p) {
    const int d = p >> 5, o = p & 31;
    return o == 0 ? r[d] : __builtin_amdgcn_alignbit(r[d + 1], r[d], o);
}

// Bits [p, p + w) of a K record (p, w compile-time after unrolling).
template <int N>
__device__ __forceinline__ uint32_t rec_bits(const uint32_t (&r)[N], int p, int w) {
    const int d = p >> 5, o = p & 31;
    if (o + w <= 32) return __builtin_amdgcn_ubfe(r[d], o, w);
    return __builtin_amdgcn_ubfe(__builtin_amdgcn_alignbit(r[d + 1], r[d], o), 0, w);
}

// v -> (hi, lo) fp16 bit patterns with hi + lo ~= v to ~22 bits.
__device__ __forceinline__ void split_hl(float v, uint32_t &hi, uint32_t &lo) {
    const _Float16 h = (_Float16)v;
    hi = (uint32_t)__builtin_bit_cast(unsigned short, h);
    const _Float16 l = (_Float16)(v - (float)h);
    lo = (uint32_t)__builtin_bit_cast(unsigned short, l);
}

// Power of two p with amax * p in [2^11, 2^12), and its reciprocal (both exact). An amax below
// 2^-113, zero too, takes the p of 2^-113: p and 1/p, also with the weights' 2^-6 on them, stay
// normal numbers (an infinite p would make a NaN of every zero), what it scales still has its
// fp32 precision down to about 2^-126, and a wave that has seen no weight yet keeps the largest
// p there is, so the first one sets its own. An infinite amax takes the largest number's p.
// (The clamp is one v_med3, but for two head sets at head_dim 256: there it had the register
// allocator spill eight more, 16 sequences of up to 2000 positions 42.4 us against 40.8.
// With fminf and fmaxf at head_dim 96 it spilled eight: 16 x 4096 positions 54.7 -> 59.)
template <class LY, int NH>
__device__ __forceinline__ float pow2_norm(float amax, float &inv) {
    constexpr float lo = 0x1p-113f, hi = 0x1.fffffep127f;
    const float a = LY::HD == 256 && NH == 2 ? fminf(fmaxf(amax, lo), hi) : __builtin_amdgcn_fmed3f(amax, lo, hi);
    const uint32_t E = __float_as_uint(a) & 0x7f800000u;  // a = f * 2^e, f in [0.5, 1): e + 126 in place
    inv = __uint_as_float(E - (11u << 23));               // 2^(e - 12)
    return __uint_as_float((265u << 23) - E);             // 2^(12 - e)
}

// fp16 scale bits -> float; a non-finite scale dequantizes to 0.
__device__ __forceinline__ float scale_of(uint32_t h) {
    const float f = (float)__builtin_bit_cast(_Float16, (unsigned short)h);
    return ((h & 0x7c00u) == 0x7c00u) ? 0.0f : f;
}

// Value of lane (lane ^ M) for M a power of two below 64, all on the VALU (no
// LDS crossbar round trip): quad permutes and row shifts / rotates via DPP,
// 16 and 32 via the gfx950 row swaps (permlane16/32_swap(x, x) leave lane l
// with lane l ^ 16 (^ 32) in one result or the other, by that lane bit).
template <int M>
__device__ __forceinline__ float lane_xor(float v) {
    const int x = __float_as_int(v);
    const int lane = (int)__lane_id();
    int r;
    if (M == 1) r = __builtin_amdgcn_mov_dpp(x, 0xB1, 0xF, 0xF, true);        // quad_perm [1,0,3,2]
    else if (M == 2) r = __builtin_amdgcn_mov_dpp(x, 0x4E, 0xF, 0xF, true);   // quad_perm [2,3,0,1]
    else if (M == 4) {                                                        // row_shr:4 / row_shl:4
        const int dn = __builtin_amdgcn_mov_dpp(x, 0x114, 0xF, 0xF, true), up = __builtin_amdgcn_mov_dpp(x, 0x104, 0xF, 0xF, true);
        r = (lane & 4) ? dn : up;
    } else if (M == 8) r = __builtin_amdgcn_mov_dpp(x, 0x128, 0xF, 0xF, true);  // row_ror:8 (xor 8 in a row of 16)
    else if (M == 16) {
        const u32x2 t = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)x, false, false);
        r = (int)((lane & 16) ? t[0] : t[1]);
    } else {
        const u32x2 t = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)x, false, false);
        r = (int)((lane & 32) ? t[0] : t[1]);
    }
    return __int_as_float(r);
}

// Value of lane I of this lane's quad (DPP quad_perm [I, I, I, I]).
template <int I>
__device__ __forceinline__ float quad_bcast(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), I * 0x55, 0xF, 0xF, true));
}

// One Sylvester stage across lane bit M: x' = x + p (bit clear) or p - x (bit set).
template <int M>
__device__ __forceinline__ float lane_butterfly(float x, int lane) {
    const float p = lane_xor<M>(x);
    return fmaf(x, (lane & M) ? -1.0f : 1.0f, p);
}

// max(a, b) of finite or infinite values as one v_med3 (fmaxf would first quiet
// the exchanged operand, an extra instruction per step)
__device__ __forceinline__ float max_ninf(float a, float b) { return __builtin_amdgcn_fmed3f(a, b, INFINITY); }

template <int M>
__device__ __forceinline__ float wave_max_step(float v) { return max_ninf(v, lane_xor<M>(v)); }
template <int M>
__device__ __forceinline__ float wave_sum_step(float v) { return v + lane_xor<M>(v); }

// Max / sum over the 16 lanes with the same lane & 3 (one head's quads).
__device__ __forceinline__ float head_max(float v) {
    v = wave_max_step<4>(v);
    v = wave_max_step<8>(v);
    v = wave_max_step<16>(v);
    return wave_max_step<32>(v);
}
__device__ __forceinline__ float head_sum(float v) {
    v = wave_sum_step<4>(v);
    v = wave_sum_step<8>(v);
    v = wave_sum_step<16>(v);
    return wave_sum_step<32>(v);
}


// Two adjacent BITS-bit codes y = c0 | c1 << BITS -> fp16 pair (2^BITS + c0, 2^BITS + c1)
// (the multiply-and-mask of sp_mfma_codes.h on a field already extracted).
template <int BITS>
__device__ __forceinline__ uint32_t pair_fp16(uint32_t y, uint32_t kmask, uint32_t kbias) {
    return __builtin_amdgcn_bitop3_b32(y * ((1u << (10 - BITS)) + (1u << (26 - 2 * BITS))), kmask, kbias, 0xEA);
}

constexpr uint32_t c_f16(int v) {  // fp16 bits of an integer or half-integer v / 2, 0 < v < 2048
    int e = 0;
    while ((v >> e) > 1) e++;
    return (uint32_t)((14 + e) << 10) | (uint32_t)((v << (10 - e)) & 0x3ff);
}

// Masks, exponent bits and centres of the pairs of a BITS-bit band.
template <int BITS>
struct PairConst {
    static constexpr uint32_t NEAR = (((1u << BITS) - 1u) << (10 - BITS)) * 0x10001u;  // neighbours, and 4-bit spans
    static constexpr uint32_t SPAN =
        BITS == 4 ? NEAR : ((((1u << BITS) - 1u) << (10 - BITS)) | (((1u << BITS) - 1u) << (25 - BITS)));
    static constexpr int M = (1 << (BITS - 1)) - 1;
    // 2^BITS + m; a half-gain half holds 2^BITS + c/2, so its centre is 2^BITS + m/2
    static constexpr uint32_t C_FULL = c_f16(2 * ((1 << BITS) + M)), C_HALF = c_f16(2 * (1 << BITS) + M);
    static constexpr uint32_t C_NEAR = C_FULL * 0x10001u, C_SPAN = BITS == 4 ? C_NEAR : C_FULL | (C_HALF << 16);
};

// The masks and exponents the score codes need, held in registers for bitop3.
struct CodeRegs {
    uint32_t bias[6], near[6], span[6];  // by BITS (3, 4, 5)
};

// Pair p of band B as one dword of two fp16.
template <class LY, int B>
__device__ __forceinline__ uint32_t band_pair(const uint32_t (&r)[LY::KDW + 1], int p, const CodeRegs &C) {
    constexpr int BITS = LY::bits[B], half = c_half(BITS), b0 = 8 * (LY::kbyte(B) + 2), n = LY::spans(B);
    if (p >= LY::pairs(B)) return 0u;
    const bool spanned = p < n * half;
    uint32_t x;
    if (spanned) {
        const int a = 2 * half * (p / half) + p % half;  // first code of the pair
        // the first code lands at mantissa bits 10-BITS .. 9, the second 15 or 16 bits above it
        x = __builtin_amdgcn_bitop3_b32(rec_window(r, b0 + BITS * a - (10 - BITS)), C.span[BITS], C.bias[BITS], 0xEA);
    } else {
        const int a = 2 * half * n + 2 * (p - n * half);
        x = pair_fp16<BITS>(rec_bits(r, b0 + BITS * a, 2 * BITS), C.near[BITS], C.bias[BITS]);
    }
    if (LY::CENTRE)
        x = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, x) -
                                             __builtin_bit_cast(half2_t, spanned ? PairConst<BITS>::C_SPAN : PairConst<BITS>::C_NEAR));
    return x;
}

// The 32 bits at bit `sh` past the dword-aligned p (a V window's codes).
__device__ __forceinline__ uint32_t v_window(const unsigned char *p, uint32_t sh) {
    const uint32_t *d = reinterpret_cast<const uint32_t *>(p);
    return __builtin_amdgcn_alignbit(d[1], d[0], sh);
}

// Code J of two positions' windows as two fp16 u - m (exact): a shift and an and-or put
// each code at the top of an fp16 mantissa under the exponent of 2^VBITS, one packed
// subtract centres it. pl, pm, ph = 16 bits of both windows from bits 0, 8 and 16.
// (Centring here rather than subtracting offset * sum(w) after the MFMA keeps the
// offset's rounding out of the sums: that rounding would be the same for every
// coefficient and the inverse transform would gather it into output element 0.)
template <int VBITS, int J>
__device__ __forceinline__ uint32_t v_pair(uint32_t pl, uint32_t pm, uint32_t ph, uint32_t vmask, uint32_t vbias) {
    constexpr int lo = VBITS * J, hi = lo + VBITS - 1;
    constexpr int from = hi <= 15 ? 0 : hi <= 23 ? 8 : 16;
    constexpr int up = (10 - VBITS) - (lo - from);  // left shift that lands the code at bits 10-VBITS .. 9
    uint32_t x = from == 0 ? pl : from == 8 ? pm : ph;
    if constexpr (up > 0) x <<= up;
    else if constexpr (up < 0) x >>= -up;
    const half2_t c = __builtin_bit_cast(half2_t, __builtin_amdgcn_bitop3_b32(x, vmask, vbias, 0xEA)) -
                      __builtin_bit_cast(half2_t, PairConst<VBITS>::C_NEAR);
    return __builtin_bit_cast(uint32_t, c);
}

// Records of one tile in registers: 16-byte buffer loads, out-of-range dwords
// read as 0. Each stream starts `shift` (0 or 2) bytes before its first record.
template <class LY>
struct TileRegs {
    u32x4 k[LY::K_LOADS];
    u32x4 v[LY::V_LOADS];
};

template <class LY, bool WANT_V>
__device__ __forceinline__ void load_tile(const unsigned char *kseq, const unsigned char *vseq, int c0, int n_chunk,
                                          int kshift, int vshift, int lane, TileRegs<LY> &r) {
    // whole dwords up to the last record's end: the caches carry slack past their last record
    const unsigned char *kg = kseq + (long long)c0 * LY::KB - kshift;
    const int kbytes = n_chunk > 0 ? (n_chunk * LY::KB + kshift + 3) & ~3 : 0;
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc((void *)kg, (short)0, kbytes, BUF_WORD3);
#pragma unroll
    for (int i = 0; i < LY::K_LOADS; i++) r.k[i] = __builtin_amdgcn_raw_buffer_load_b128(rk, 16 * lane, 1024 * i, BUF_NT);
    if (WANT_V) {
        const unsigned char *vg = vseq + (long long)c0 * LY::VB - vshift;
        const int vbytes = n_chunk > 0 ? (n_chunk * LY::VB + vshift + 3) & ~3 : 0;
        const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc((void *)vg, (short)0, vbytes, BUF_WORD3);
#pragma unroll
        for (int i = 0; i < LY::V_LOADS; i++) r.v[i] = __builtin_amdgcn_raw_buffer_load_b128(rv, 16 * lane, 1024 * i, BUF_NT);
    }
}

template <class LY, bool WANT_V>
__device__ __forceinline__ void stage_tile(unsigned char *wl, const TileRegs<LY> &r, int lane) {
#pragma unroll
    for (int i = 0; i < LY::K_LOADS; i++) {
        const int off = 16 * lane + 1024 * i;
        if (off < LY::R_V) *reinterpret_cast<u32x4 *>(wl + off) = r.k[i];
    }
    if (WANT_V) {
#pragma unroll
        for (int i = 0; i < LY::V_LOADS; i++) {
            const int off = 16 * lane + 1024 * i;
            if (off < LY::R_SIZE - LY::R_V) *reinterpret_cast<u32x4 *>(wl + LY::R_V + off) = r.v[i];
        }
    }
}

// The transform of a vector held as elements (lane % EL) + EL * e, scaled by `scale`
// (which carries the 1/sqrt(HD)): p = 2 stages over the lane bits, then over the
// registers (2 or 4 of them: p = 2 again; 3: the cas block of p = 3, without its
// 1/sqrt(3)). Symmetric and its own inverse.
template <class LY>
__device__ __forceinline__ void transform_reg(float (&x)[LY::NE], float scale, int lane) {
#pragma unroll
    for (int e = 0; e < LY::NE; e++) {
        x[e] = lane_butterfly<1>(x[e], lane);
        x[e] = lane_butterfly<2>(x[e], lane);
        x[e] = lane_butterfly<4>(x[e], lane);
        x[e] = lane_butterfly<8>(x[e], lane);
        x[e] = lane_butterfly<16>(x[e], lane);
        if (LY::EL == 64) x[e] = lane_butterfly<32>(x[e], lane);
    }
    if constexpr (LY::NE == 1) {
        x[0] *= scale;
    } else if constexpr (LY::NE == 2) {
        const float a = x[0], b = x[1];
        x[0] = (a + b) * scale;
        x[1] = (a - b) * scale;
    } else if constexpr (LY::NE == 3) {
        constexpr float c1 = 0.36602540378443864676f, c2 = -1.36602540378443864676f;  // cas(2 pi m / 3), m = 1, 2
        const float a = x[0], b = x[1], c = x[2];
        x[0] = (a + b + c) * scale;
        x[1] = (a + c1 * b + c2 * c) * scale;
        x[2] = (a + c2 * b + c1 * c) * scale;
    } else {
        static_assert(LY::NE == 4, "head_dim 64, 96, 128 or 256");
        const float a = x[0] + x[1], b = x[0] - x[1], c = x[2] + x[3], d = x[2] - x[3];
        x[0] = (a + c) * scale;
        x[1] = (b + d) * scale;
        x[2] = (a - c) * scale;
        x[3] = (b - d) * scale;
    }
}
constexpr float c_inv_sqrt(int hd) {
    return hd == 64 ? 0.125f : hd == 96 ? 0.10206207261596575409f : hd == 128 ? 0.08838834764831844055f : 0.0625f;
}

template <class LY, int... BS>
__device__ __forceinline__ void score_step(const uint32_t (&r)[LY::KDW + 1], int s, const CodeRegs &C, half4_t (&a)[LY::NB],
                                           std::integer_sequence<int, BS...>) {
    ((a[BS] = s < LY::steps(BS) ? __builtin_bit_cast(half4_t, u32x2{band_pair<LY, BS>(r, 2 * s, C), band_pair<LY, BS>(r, 2 * s + 1, C)})
                                : half4_t{}),
     ...);
}

template <class LY, int... JS>
__device__ __forceinline__ void value_step(float4_t (&vacc)[LY::EPC], half8_t a, int w, const uint32_t (&pl)[4],
                                           const uint32_t (&pm)[4], const uint32_t (&ph)[4], uint32_t vmask, uint32_t vbias,
                                           std::integer_sequence<int, JS...>) {
    ((vacc[w * LY::EPW + JS] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
          a,
          as_half8(v_pair<LY::VBITS, JS>(pl[0], pm[0], ph[0], vmask, vbias),
                   v_pair<LY::VBITS, JS>(pl[1], pm[1], ph[1], vmask, vbias),
                   v_pair<LY::VBITS, JS>(pl[2], pm[2], ph[2], vmask, vbias),
                   v_pair<LY::VBITS, JS>(pl[3], pm[3], ph[3], vmask, vbias)),
          vacc[w * LY::EPW + JS], 0, 0, 0)),
     ...);
}

// Waves resident on a SIMD (the registers an instance may use): head_dim 256 needs 256
// of them; several tiles per wave at head_dim 128, or with 8 heads below it, spill at 128
// and fit at 168.
constexpr int wave_waves_per_simd(int hd, int nh, bool multi) {
    return hd == 256 ? 2 : multi && (hd == 128 || nh == 2) ? 3 : 4;
}
// The launch shapes that exist: blocks of 4, 8 or 16 waves at one tile per wave; several
// tiles per wave in blocks of up to that many waves (0: none; 5 to 8 heads at head_dim 128, us
// at one tile per wave in blocks of 16 / the best with several: 8 KV heads x 60000 positions
// 38.8 / 66.5, x 131000 77.5 / 122.7), and in blocks of 16 for the scores alone of one
// sequence at head_dim 128.
constexpr int wave_max_nw(int hd) { return hd == 256 ? 8 : 16; }
constexpr int wave_multi_nw(int hd, int nh) {
    return hd == 256 ? 8 : hd == 128 ? (nh == 1 ? 4 : 0) : nh == 1 ? 16 : 4;
}

// Grid (KV head, block of tiles, sequence). Wave w of block b works tiles
// (b * NW + w) * tpw .. + tpw - 1 of its sequence; a block past the sequence's last tile
// ends at once. Partials go to part[((seq * n_q + query head) * part_rows + block)] as
// [m, l, o~[HD]]. NH = 1 serves up to 4 query heads per KV head, NH = 2 up to 8 (a
// second set of columns). MULTI = false: one tile per wave (tpw = 1), so no running
// state is carried.
// Band limits: K bands b >= kbands and the V band when vbands == 0 take a zero
// scale (a finite sum times 0 adds exactly nothing, so the scores and outputs
// equal those with the bands read as 0, at the cost of the all-band loop).
template <class LY, int NW, bool WANT_OUT, int NH, bool MULTI, bool SEQS>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(wave_waves_per_simd(LY::HD, NH, MULTI && NW < 16))))
k_attn_wave(const SpAttnArgs A, const int *__restrict__ order, float *__restrict__ part, int part_rows, int tpw, int kbands,
            int vbands, int *__restrict__ counters, const std::conditional_t<SEQS, SpSeqTab, SpNoTab> T) {
    using L = WaveLds<LY, NW>;
    constexpr int HD = LY::HD, NB = LY::NB, NT = 64 * NW, NE = LY::NE, EL = LY::EL, HP = LY::HP, EPC = LY::EPC;
    constexpr int QS_STRIDE = LY::QS_STRIDE, WT_STRIDE = LY::WT_STRIDE, MB_STRIDE = LY::MB_STRIDE;
    __shared__ __attribute__((aligned(16))) unsigned char smem[L::BYTES];
    const int kvh = blockIdx.x, blk = blockIdx.y, seq = SEQS ? blockIdx.z : 0, tid = threadIdx.x;
    int n_kv = A.n_kv, start = A.start, n_parts = part_rows;  // part_rows: blocks per KV head
    long long soff = 0;
    if constexpr (SEQS) {
        n_kv = T.len[seq];
        start = T.start[seq];
        soff = T.soff[seq];
        n_parts = (n_kv + TILE * NW * tpw - 1) / (TILE * NW * tpw);  // this sequence's
        if (blk >= n_parts) return;                                  // block-uniform, before any barrier
    }
    // the wave index is wave-uniform: a scalar, so the buffer resources and LDS bases built from it are too
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, q4 = lane >> 4, c16 = lane & 15;
    const int el = lane & (EL - 1);
    const int G = A.n_q / A.n_kvh, h0 = kvh * G;
    unsigned char *wl = smem + w * LY::R_SIZE;
    unsigned short *qs = reinterpret_cast<unsigned short *>(smem + L::QS);  // [part][head][slot] fp16
    float *cb = reinterpret_cast<float *>(smem + L::CB);                    // [head][4]
    float *fu = reinterpret_cast<float *>(smem + L::FU);                    // [head]

    // ---- 1. wave w prepares heads w, w + NW: their query rows and the order and slot
    // entries of the lane's record coefficients are the first loads, every wave's first
    // tile of records the next ----
    int *ready = reinterpret_cast<int *>(smem + L::FLAG + 4);  // query heads prepared
    if (tid == 0) *ready = 0;
    __syncthreads();
    const unsigned char *kseq = A.kpack + (long long)kvh * A.k_head_stride + (long long)start * LY::KB;
    const unsigned char *vseq = A.vpack + (long long)kvh * A.v_head_stride + (long long)start * LY::VB;
    const int kshift = LY::KB % 4 ? (int)((uintptr_t)kseq & 3) : 0;
    const int vshift = WANT_OUT && LY::VB % 4 ? (int)((uintptr_t)vseq & 3) : 0;
    const float *__restrict__ qseq = A.q + ((long long)seq * A.n_q + h0) * HD;
    const int tile0 = (blk * NW + w) * tpw;  // tile index of the wave's first tile within the sequence
    const int c00 = tile0 * TILE;
    const int n_chunk0 = c00 < n_kv ? min(TILE, n_kv - c00) : 0;
    TileRegs<LY> regs;

    // ---- 2. q~ = kq_scale * reorder(transform(q)) per head, in registers, scaled by a
    // power of two f so its largest entry lies in [2^11, 2^12) and split into fp16 hi +
    // lo, stored in the score MFMA's slot order. Without CENTRE, per band,
    // -(2^BITS + m_b) * sum(hi + lo over the band): the accumulator start. ----
    float y[NE];
    int ord[NE], where[NE];
    if (w < G) {
        // Without an order table, read (and ignore) in-bounds words of q: both
        // candidates are kernel-argument pointers, so these stay global loads.
        const int *op = order ? order : reinterpret_cast<const int *>(A.q);
#pragma unroll
        for (int e = 0; e < NE; e++) {
            y[e] = qseq[w * HD + el + EL * e];
            ord[e] = op[el + EL * e];
            where[e] = kSlots<LY>.v[el + EL * e];
        }
#pragma unroll
        for (int e = 0; e < NE; e++) ord[e] = order ? ord[e] : el + EL * e;
    }
    load_tile<LY, WANT_OUT>(kseq, vseq, c00, n_chunk0, kshift, vshift, lane, regs);
    // (eight waves or more: one head each)
    for (int h = w; h < (NW < 8 ? G : min(G, w + 1)); h += NW) {
        if (NW < 8 && h != w) {
#pragma unroll
            for (int e = 0; e < NE; e++) y[e] = qseq[h * HD + el + EL * e];
        }
        transform_reg<LY>(y, A.kq_scale * c_inv_sqrt(HD), lane);
        float amax = fabsf(y[0]);
#pragma unroll
        for (int e = 1; e < NE; e++) amax = fmaxf(amax, fabsf(y[e]));
        amax = wave_max_step<1>(amax);
        amax = wave_max_step<2>(amax);
        amax = wave_max_step<4>(amax);
        amax = wave_max_step<8>(amax);
        amax = wave_max_step<16>(amax);
        amax = wave_max_step<32>(amax);
        float finv;
        const float f = pow2_norm<LY, NH>(amax, finv);
        // reorder through the wave's (not yet used) record area; clear the row's pad slots
        float *qx = reinterpret_cast<float *>(wl);
#pragma unroll
        for (int e = 0; e < NE; e++) qx[el + EL * e] = y[e];
        if (LY::SLOTS != HD) {
            for (int s = lane; s < 2 * LY::SLOTS; s += 64)
                qs[((s >= LY::SLOTS ? 8 : 0) + h) * QS_STRIDE + (s >= LY::SLOTS ? s - LY::SLOTS : s)] = 0;
        }
        __asm__ volatile("" ::: "memory");
#pragma unroll
        for (int e = 0; e < NE; e++) {
            const float v = qx[ord[e]] * f;
            uint32_t hi, lo;
            split_hl(v, hi, lo);
            const int slot = where[e] & 0xff, band = where[e] >> 9;
            const float gain = (where[e] & 0x100) ? 2.0f : 1.0f;
            const float fh = (float)__builtin_bit_cast(_Float16, (unsigned short)hi);
            const float fl = (float)__builtin_bit_cast(_Float16, (unsigned short)lo);
            // a half-gain slot (its code stored as 2^BITS + c/2) holds 2q~: exact in fp16
            qs[h * QS_STRIDE + slot] = __builtin_bit_cast(unsigned short, (_Float16)(fh * gain));
            qs[(8 + h) * QS_STRIDE + slot] = __builtin_bit_cast(unsigned short, (_Float16)(fl * gain));
            if (!LY::CENTRE) {
                // the slot's fp16 value is offset + code / gain with offset 2^BITS, against gain *
                // q~; lanes 0-31 and 32-63 of a register are one band each (32 coefficients)
                static_assert(LY::CENTRE || (LY::HD == 128 && LY::NB == 4), "bands of 32 coefficients");
                const int bits = band < 2 ? LY::bits[0] : band == 2 ? LY::bits[LY::NB > 2 ? 2 : 0] : LY::bits[LY::NB - 1];
                float t = (fh + fl) * (gain * (float)(1 << bits) + (float)((1 << (bits - 1)) - 1));
                t = wave_sum_step<1>(t);
                t = wave_sum_step<2>(t);
                t = wave_sum_step<4>(t);
                t = wave_sum_step<8>(t);
                t = wave_sum_step<16>(t);
                if ((lane & 31) == 0) cb[h * 4 + band] = -t;
            }
        }
        if (lane == 0) fu[h] = finv;
        // publish: this wave's LDS writes are complete before it counts the head
        __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (lane == 0) __hip_atomic_fetch_add(ready, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }

    // score rows 16-byte aligned at every tile: one 16-byte non-temporal store per lane
    float *__restrict__ scores = A.scores ? A.scores + soff : nullptr;
    const bool sc_vec = ((uintptr_t)scores & 15) == 0 && (n_kv & 3) == 0;

    // code-slot masks and the fp16 2^BITS exponent bits, kept in registers for bitop3
    CodeRegs C;
    C.bias[5] = __builtin_amdgcn_readfirstlane(code_bias<5>());
    C.bias[4] = __builtin_amdgcn_readfirstlane(code_bias<4>());
    C.bias[3] = __builtin_amdgcn_readfirstlane(code_bias<3>());
    const uint32_t vbias = __builtin_amdgcn_readfirstlane(code_bias<LY::VBITS>());
    uint32_t near5 = PairConst<5>::NEAR, near4 = PairConst<4>::NEAR, near3 = PairConst<3>::NEAR;
    uint32_t span5 = PairConst<5>::SPAN, span3 = PairConst<3>::SPAN, vmask = PairConst<LY::VBITS>::NEAR;
    __asm__("" : "+v"(near5), "+v"(near4), "+v"(near3), "+v"(vmask), "+v"(span5), "+v"(span3));
    C.near[5] = near5; C.near[4] = near4; C.near[3] = near3;
    C.span[5] = span5; C.span[4] = near4; C.span[3] = span3;

    // running state over the wave's tiles: per score column (head 4*st + hj) the softmax
    // reference m, the weights' power of two f and this lane's part of the sum of p; the
    // value accumulators (lane (c16, q4): rows 4*q4 + i, i.e. head 2*q4 + (i >> 1)) hold
    // sums of weights scaled by f
    float m_run[NH], f_run[NH], fi_run[NH], l_run[NH];
#pragma unroll
    for (int st = 0; st < NH; st++) m_run[st] = -INFINITY, f_run[st] = fi_run[st] = 1.0f, l_run[st] = 0.0f;
    float4_t vacc[EPC];
#pragma unroll
    for (int j = 0; j < EPC; j++) vacc[j] = float4_t{0.f, 0.f, 0.f, 0.f};

    for (int it = 0; it < (MULTI ? tpw : 1); it++) {
        const int c0 = (tile0 + it) * TILE;
        if (c0 >= n_kv) break;  // wave-uniform
        const int n_chunk = min(TILE, n_kv - c0);
        // LDS addresses below derive from an opaque per-tile copy of the lane
        // index: loop-invariant, they would otherwise be hoisted out of the tile
        // loop and held (or spilled) through it.
        int ln = lane;
        __asm__ volatile("" : "+v"(ln));
        const int c16i = ln & 15, q4i = ln >> 4, hj = ln & 3, qd = ln >> 2;
        __asm__ volatile("" ::: "memory");  // the previous tile's LDS reads are issued before the new records land
        stage_tile<LY, WANT_OUT>(wl, regs, lane);
        __asm__ volatile("" ::: "memory");
        // ---- lane t takes record t of the K tile into registers, and the scale of its V record ----
        uint32_t r[LY::KDW + 1];
        if (LY::KB % 4 == 0) {
            const uint32_t *kr = reinterpret_cast<const uint32_t *>(wl + ln * LY::KB);
#pragma unroll
            for (int m = 0; m < LY::KDW; m++) r[m] = kr[m];
        } else {
            // records at 2 mod 4 bytes: the covering dwords, funnel-shifted
            const int at = kshift + ln * LY::KB;
            const uint32_t *kr = reinterpret_cast<const uint32_t *>(wl + (at & ~3));
            const uint32_t sh = (uint32_t)(at & 3) * 8u;
            uint32_t x[LY::KDW + 1];
#pragma unroll
            for (int m = 0; m <= LY::KDW; m++) x[m] = kr[m];
#pragma unroll
            for (int m = 0; m < LY::KDW; m++) r[m] = __builtin_amdgcn_alignbit(x[m + 1], x[m], sh);
        }
        r[LY::KDW] = 0;
        float sv_own = 0.0f;
        if (WANT_OUT)
            // (a lane past the tile's end takes whatever scale lies there: its weight is p = 0)
            sv_own = vbands > 0
                         ? scale_of(*reinterpret_cast<const unsigned short *>(wl + LY::R_V + vshift + ln * LY::VB))
                         : 0.0f;
        __asm__ volatile("" ::: "memory");  // every lane has read its record before the K area is reused

        // ---- the query operand is in LDS once the G heads are counted (each is counted
        // once, unconditionally, by a wave that waits for nothing before it, so this ends) ----
        if (it == 0) {
            while (__hip_atomic_load(ready, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < G) __builtin_amdgcn_s_sleep(1);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        }
        // ---- scores: accumulator (set, band), without CENTRE started at the band's centring ----
        float4_t acc[NH][NB];
#pragma unroll
        for (int st = 0; st < NH; st++) {
#pragma unroll
            for (int b = 0; b < NB; b++) acc[st][b] = float4_t{0.f, 0.f, 0.f, 0.f};
            if (!LY::CENTRE) {
                const float4 c4 = *reinterpret_cast<const float4 *>(cb + (4 * st + hj) * 4);
                const float cv[4] = {c4.x, c4.y, c4.z, c4.w};
#pragma unroll
                for (int b = 0; b < NB; b++) acc[st][b] = float4_t{cv[b], cv[b], cv[b], cv[b]};
            }
        }
#pragma unroll
        for (int s = 0; s < LY::max_steps(); s++) {  // step s of every band: its slots 4s .. 4s+3
            half4_t a[NB];
            score_step<LY>(r, s, C, a, std::make_integer_sequence<int, NB>{});
#pragma unroll
            for (int st = 0; st < NH; st++)
#pragma unroll
                for (int hl = 0; hl < 2; hl++)
#pragma unroll
                    for (int b = 0; b < NB; b++) {
                        if (s >= LY::steps(b)) continue;
                        const half4_t qv = __builtin_bit_cast(
                            half4_t, *reinterpret_cast<const u32x2 *>(qs + (hl * 8 + 4 * st + hj) * QS_STRIDE + LY::slot0(b) + 4 * s));
                        acc[st][b] = __builtin_amdgcn_mfma_f32_4x4x4f16(a[b], qv, acc[st][b], 0, 0, 0);
                    }
        }
        // band scales of the lane's own record; position 4*qd + i's come from quad lane i
        float ks[NB];
#pragma unroll
        for (int b = 0; b < NB; b++)
            ks[b] = b < kbands ? scale_of(rec_bits(r, 8 * LY::kbyte(b), 16)) : 0.0f;
        float sc[NH][4];
#pragma unroll
        for (int st = 0; st < NH; st++) {
            const float un = fu[4 * st + hj];
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const float s0 = quad_bcast<0>(ks[b]), s1 = quad_bcast<1>(ks[b]);
                const float s2 = quad_bcast<2>(ks[b]), s3 = quad_bcast<3>(ks[b]);
                if (b == 0) {
                    sc[st][0] = s0 * acc[st][b][0];
                    sc[st][1] = s1 * acc[st][b][1];
                    sc[st][2] = s2 * acc[st][b][2];
                    sc[st][3] = s3 * acc[st][b][3];
                } else {
                    sc[st][0] = fmaf(s0, acc[st][b][0], sc[st][0]);
                    sc[st][1] = fmaf(s1, acc[st][b][1], sc[st][1]);
                    sc[st][2] = fmaf(s2, acc[st][b][2], sc[st][2]);
                    sc[st][3] = fmaf(s3, acc[st][b][3], sc[st][3]);
                }
            }
#pragma unroll
            for (int i = 0; i < 4; i++) sc[st][i] *= un;
            if (scores && 4 * st + hj < G) {
                float *dst = scores + (long long)(h0 + 4 * st + hj) * n_kv + c0 + 4 * qd;
                if (n_chunk == TILE && sc_vec) {
                    __builtin_nontemporal_store(float4_t{sc[st][0], sc[st][1], sc[st][2], sc[st][3]}, reinterpret_cast<float4_t *>(dst));
                } else {
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (4 * qd + i < n_chunk) dst[i] = sc[st][i];
                }
            }
        }
        if (!WANT_OUT) {
            if (MULTI && it + 1 < tpw)
                load_tile<LY, WANT_OUT>(kseq, vseq, c0 + TILE, min(TILE, max(0, n_kv - c0 - TILE)), kshift, vshift, lane, regs);
            continue;
        }

        // ---- softmax weights, lane (quad qd, head hj) holding positions 4*qd + i; w =
        // p * scale_v * f as fp16 hi / lo rows 2h / 2h + 1 (slot = position). m and f are the
        // first tile's (largest weight in [2^5, 2^6)) and stay while every weight stays within
        // 2^15 and every p within 2^60, so a usual tile needs no reduction across lanes and no
        // rescaling; the lo parts still resolve 2^-35. A head that outgrows them takes the
        // tile's maximum as its m and rescales its sums; so does one whose tiles had zero V
        // records only, at its first weight (f is the largest there is until then). (p has a
        // bound of its own for positions whose V record is zero: its weight stays 0, or is
        // inf * 0, however far its score is above m.) ----
        unsigned short *wt = reinterpret_cast<unsigned short *>(wl);
        float *stt = reinterpret_cast<float *>(wl + LY::R_ST);
        const float sv[4] = {quad_bcast<0>(sv_own), quad_bcast<1>(sv_own), quad_bcast<2>(sv_own), quad_bcast<3>(sv_own)};
        float v[NH][4], pr[NH][4], wx[NH][4];
        bool grown[NH], any_grown = false;
#pragma unroll
        for (int st = 0; st < NH; st++) {
#pragma unroll
            for (int i = 0; i < 4; i++) v[st][i] = 4 * qd + i < n_chunk ? sc[st][i] : -INFINITY;  // past the tile's end: no weight
            grown[st] = false;
            if (MULTI) {
                float wm = 0.0f, pm = 0.0f;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    pr[st][i] = __expf(v[st][i] - m_run[st]);
                    wx[st][i] = pr[st][i] * sv[i] * f_run[st];
                    wm = fmaxf(wm, wx[st][i]);
                    pm = fmaxf(pm, pr[st][i]);
                }
                // both bounds in one: 2^60 * 2^-45 is 2^15 (and an infinite p passes it)
                grown[st] = 4 * st + hj < G && !(fmaf(pm, 0x1p-45f, wm) <= 32768.0f);
                any_grown = any_grown || grown[st];
            }
        }
        if (!MULTI || it == 0 || __any(any_grown)) {
#pragma unroll
            for (int st = 0; st < NH; st++) {
                const bool head_grown = !MULTI || it == 0 || head_max(grown[st] ? 1.0f : 0.0f) > 0.0f;
                const float m = max_ninf(head_max(fmaxf(fmaxf(v[st][0], v[st][1]), fmaxf(v[st][2], v[st][3]))), m_run[st]);
                float p[4], wm = 0.0f;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    p[i] = __expf(v[st][i] - m);
                    wm = fmaxf(wm, p[i] * sv[i]);
                }
                float fi;
                const float f = pow2_norm<LY, NH>(head_max(wm), fi) * 0.015625f;
                fi *= 64.0f;
                const float alpha = !MULTI || it == 0 ? 0.0f : __expf(m_run[st] - m);
                // what the head's value sums are multiplied by
                if (MULTI && qd == 0) stt[4 * st + hj] = head_grown ? alpha * f * fi_run[st] : 1.0f;
                if (head_grown) {
                    l_run[st] *= alpha;
                    m_run[st] = m;
                    f_run[st] = f;
                    fi_run[st] = fi;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        pr[st][i] = p[i];
                        wx[st][i] = p[i] * sv[i] * f;
                    }
                }
            }
            __asm__ volatile("" ::: "memory");
            if (MULTI && it > 0) {
                const float2 sc2 = *reinterpret_cast<const float2 *>(stt + 2 * q4i);  // NH = 1: rows past 7 are not used
#pragma unroll
                for (int j = 0; j < EPC; j++) {
                    vacc[j][0] *= sc2.x;
                    vacc[j][1] *= sc2.x;
                    vacc[j][2] *= sc2.y;
                    vacc[j][3] *= sc2.y;
                }
            }
            __asm__ volatile("" ::: "memory");
        }
#pragma unroll
        for (int st = 0; st < NH; st++) {
            l_run[st] += (pr[st][0] + pr[st][1]) + (pr[st][2] + pr[st][3]);
            uint32_t hi[4], lo[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                // lo part scaled by 2^11 (exact) so it stays a normal fp16 value
                const float x = wx[st][i];
                const _Float16 hv = (_Float16)x;
                hi[i] = (uint32_t)__builtin_bit_cast(unsigned short, hv);
                lo[i] = (uint32_t)__builtin_bit_cast(unsigned short, (_Float16)((x - (float)hv) * 2048.0f));
            }
            const int row = 2 * (4 * st + hj);
            *reinterpret_cast<u32x2 *>(wt + row * WT_STRIDE + 4 * qd) = u32x2{hi[0] | (hi[1] << 16), hi[2] | (hi[3] << 16)};
            *reinterpret_cast<u32x2 *>(wt + (row + 1) * WT_STRIDE + 4 * qd) = u32x2{lo[0] | (lo[1] << 16), lo[2] | (lo[3] << 16)};
        }
        __asm__ volatile("" ::: "memory");

        // the next tile's records load while this tile's values are summed
        if (MULTI && it + 1 < tpw)
            load_tile<LY, WANT_OUT>(kseq, vseq, c0 + TILE, min(TILE, max(0, n_kv - c0 - TILE)), kshift, vshift, lane, regs);
        // ---- values: D[(h, part)][n] over K slots 32k + 8*q4 + e (positions
        // 32k + 8*q4 + e); B column n = element EPC*n + j of MFMA j ----
        // lane (c16, q4)'s first code of position t sits at bit 8 * (vshift + VB * t + 2) +
        // VBITS * EPC * c16 of the V region; its positions 32k + 8*q4 + e keep one dword
        // alignment for even e and one for odd e (steps of 2 VB and 32 VB bytes, both
        // whole dwords), so each has a dword-aligned base and a shift
        const int xw0 = 8 * (vshift + 8 * q4i * LY::VB + 2) + LY::VBITS * EPC * c16i, xw1 = xw0 + 8 * LY::VB;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const half8_t a =
                __builtin_bit_cast(half8_t, *reinterpret_cast<const u32x4 *>(wt + c16i * WT_STRIDE + 32 * k + 8 * q4i));
#pragma unroll
            for (int wn = 0; wn < LY::NWIN; wn++) {
                const int y0 = xw0 + wn * LY::EPW * LY::VBITS, y1 = xw1 + wn * LY::EPW * LY::VBITS;
                const unsigned char *vb0 = wl + LY::R_V + ((y0 >> 5) << 2), *vb1 = wl + LY::R_V + ((y1 >> 5) << 2);
                const uint32_t vsh0 = (uint32_t)y0 & 31u, vsh1 = (uint32_t)y1 & 31u;
                // K slot pair p (slots 2p, 2p + 1): both positions' bits from 0, 8 and 16
                uint32_t pl[4], pm[4], ph[4];
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    const uint32_t we = v_window(vb0 + 32 * k * LY::VB + 2 * p * LY::VB, vsh0);
                    const uint32_t wo = v_window(vb1 + 32 * k * LY::VB + 2 * p * LY::VB, vsh1);
                    pl[p] = __builtin_amdgcn_perm(wo, we, 0x05040100u);
                    pm[p] = __builtin_amdgcn_perm(wo, we, 0x06050201u);
                    ph[p] = __builtin_amdgcn_perm(wo, we, 0x07060302u);
                }
                value_step<LY>(vacc, a, wn, pl, pm, ph, vmask, vbias, std::make_integer_sequence<int, LY::EPW>{});
            }
        }
        __asm__ volatile("" ::: "memory");  // this tile's LDS reads are issued before the next tile is staged
    }
    if (!WANT_OUT) return;

    // ---- the wave's sums: [m, l, 1/f] per head by LDS to the value lanes; o~ = rows 2h
    // (hi) and 2h + 1 (lo, scaled by 2^11) ----
    float om[2], ol[2], oo[2][EPC];
    {
        float *stt = reinterpret_cast<float *>(wl + LY::R_ST);
        __asm__ volatile("" ::: "memory");
#pragma unroll
        for (int st = 0; st < NH; st++) {
            const float l = head_sum(l_run[st]);
            if (lane < 4) *reinterpret_cast<float4 *>(stt + 4 * (4 * st + lane)) = float4{m_run[st], l, fi_run[st], 0.0f};
        }
        __asm__ volatile("" ::: "memory");
#pragma unroll
        for (int hh = 0; hh < 2; hh++) {
            const float4 t4 = *reinterpret_cast<const float4 *>(stt + 4 * (2 * q4 + hh));
            om[hh] = t4.x;
            ol[hh] = t4.y;
#pragma unroll
            for (int j = 0; j < EPC; j++) oo[hh][j] = fmaf(vacc[j][2 * hh + 1], 1.0f / 2048.0f, vacc[j][2 * hh]) * t4.z;
        }
    }
    // ---- merge the block's waves: record (wave, head) = [m, l, -, -, o~[HD]] ----
    __syncthreads();  // every wave is done with its LDS region
    float *mb = reinterpret_cast<float *>(smem);
#pragma unroll
    for (int hh = 0; hh < 2; hh++) {
        const int h = 2 * q4 + hh;
        if (h < G) {
            float *rec = mb + (w * 8 + h) * MB_STRIDE;
            if constexpr (EPC % 4 == 0) {
#pragma unroll
                for (int j = 0; j < EPC; j += 4)
                    *reinterpret_cast<float4 *>(rec + 4 + EPC * c16 + j) = float4{oo[hh][j], oo[hh][j + 1], oo[hh][j + 2], oo[hh][j + 3]};
            } else {
#pragma unroll
                for (int j = 0; j < EPC; j += 2) *reinterpret_cast<float2 *>(rec + 4 + EPC * c16 + j) = float2{oo[hh][j], oo[hh][j + 1]};
            }
            if (c16 == 0) {
                rec[0] = om[hh];
                rec[1] = ol[hh];
            }
        }
    }
    __syncthreads();
    // thread (head, element): HP threads a head (whole waves), in rounds of the block
    constexpr int ROUNDS = (8 * HP + NT - 1) / NT;  // up to 8 heads
    float bo[ROUNDS];  // the block's o~ / l of the thread's elements, for a head that is one block
#pragma unroll
    for (int rd = 0; rd < ROUNDS; rd++) {
        bo[rd] = 0.0f;
        const int at = rd * NT + tid, h = at / HP, i = at % HP;
        if (h >= G || i >= HD) continue;
        float M = -INFINITY;
#pragma unroll
        for (int v = 0; v < NW; v++) M = fmaxf(M, mb[(v * 8 + h) * MB_STRIDE]);
        float Ls = 0.0f, O = 0.0f;
#pragma unroll
        for (int v = 0; v < NW; v++) {
            const float *rec = mb + (v * 8 + h) * MB_STRIDE;
            const float e = __expf(rec[0] - M);  // a wave without tiles: m = -inf, e = 0
            Ls = fmaf(rec[1], e, Ls);
            O = fmaf(rec[4 + i], e, O);
        }
        if (n_parts == 1) {
            bo[rd] = O / Ls;
        } else {
            // agent-scope atomic stores: written through to where every CU's
            // agent-scope loads read, with no cache writeback needed before the count
            float *dst = part + (((long long)seq * A.n_q + h0 + h) * part_rows + blk) * (HD + 2);
            __hip_atomic_store(dst + 2 + i, O, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (i == 0) {
                __hip_atomic_store(dst, M, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(dst + 1, Ls, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
    float *vec = reinterpret_cast<float *>(smem);  // [G][HP] merged o~ / l
    if (n_parts == 1) {
        __syncthreads();  // every thread has read the records
#pragma unroll
        for (int rd = 0; rd < ROUNDS; rd++) {
            const int at = rd * NT + tid;
            if (at < G * HP) vec[at] = bo[rd];
        }
    } else {
        // ---- the last block of the KV head to arrive merges every block's partial:
        // each block's stores have completed before it counts itself ----
        __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        int *flag = reinterpret_cast<int *>(smem + L::FLAG);
        if (tid == 0) {
            int *cnt = counters + ((long long)seq * A.n_kvh + kvh) * SP_ATTN_COUNTER_STRIDE;
            const int arrived = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const int last = arrived == n_parts - 1;
            if (last) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // ready for the next call
            *flag = last;
        }
        __syncthreads();
        if (!*flag) return;
        // Two halves of the block (when the heads fit half of it) take half the partials
        // each: thread (half, h, i) loads o~[i] of its partials, and lane k of each
        // 16-lane row the m and l of partial p0 + k, shared across the wave (one m, l load
        // per partial and lane instead of one per element)
        const int GH = G * HP, halves = 2 * GH <= NT ? 2 : 1;
        float *xo = vec + 8 * HP;  // second half's o~ [G][HP]
        float *xml = xo + 8 * HP;  // second half's (M, L) [G][2]
        for (int r0 = 0; r0 < GH; r0 += NT) {  // one round when halves == 2
            const int half = halves == 2 && tid >= GH ? 1 : 0, rr = r0 + tid - half * GH;
            const int h = rr / HP, i = rr % HP;
            const int per = (n_parts + halves - 1) / halves, pb = half * per, pe = min(n_parts, pb + per);
            float M = -INFINITY, Ls = 0.0f, O = 0.0f;
            if (rr < GH) {  // wave-uniform: GH and HP are whole waves
                const float *src = part + ((long long)seq * A.n_q + h0 + h) * part_rows * (HD + 2);
                const int ii = min(i, HD - 1);
                for (int p0 = pb; p0 < pe; p0 += 16) {
                    const int pk = min(p0 + (lane & 15), pe - 1);
                    const float mk0 = __hip_atomic_load(src + (long long)pk * (HD + 2), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    const float lk = __hip_atomic_load(src + (long long)pk * (HD + 2) + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    float po[16];
#pragma unroll
                    for (int k = 0; k < 16; k++)
                        po[k] = __hip_atomic_load(src + (long long)min(p0 + k, pe - 1) * (HD + 2) + 2 + ii, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT);
                    const float mk = p0 + (lane & 15) < pe ? mk0 : -INFINITY;  // a repeated last partial counts once
                    float cm = mk;
                    cm = wave_max_step<1>(cm);
                    cm = wave_max_step<2>(cm);
                    cm = wave_max_step<4>(cm);
                    cm = wave_max_step<8>(cm);
                    cm = fmaxf(cm, M);
                    const float ek = mk == -INFINITY ? 0.0f : __expf(mk - cm);
                    float ls = lk * ek;
                    ls = wave_sum_step<1>(ls);
                    ls = wave_sum_step<2>(ls);
                    ls = wave_sum_step<4>(ls);
                    ls = wave_sum_step<8>(ls);
                    const float sa = M == -INFINITY ? 0.0f : __expf(M - cm);  // rescale of the running sums
                    Ls = fmaf(Ls, sa, ls);
                    O *= sa;
#pragma unroll
                    for (int k = 0; k < 16; k++)
                        O = fmaf(po[k], __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ek), k)), O);
                    M = cm;
                }
            }
            if (halves == 2) {
                if (half == 1 && rr < GH) {
                    xo[rr] = O;
                    if (i == 0) {
                        xml[2 * h] = M;
                        xml[2 * h + 1] = Ls;
                    }
                }
                __syncthreads();
                if (half == 0 && rr < GH) {
                    const float m2 = xml[2 * h], l2 = xml[2 * h + 1], o2 = xo[rr];
                    const float cm = fmaxf(M, m2);
                    const float a = M == -INFINITY ? 0.0f : __expf(M - cm), b = m2 == -INFINITY ? 0.0f : __expf(m2 - cm);
                    Ls = fmaf(Ls, a, l2 * b);
                    O = fmaf(O, a, o2 * b);
                }
            }
            if (half == 0 && rr < GH) vec[rr] = O / Ls;
        }
    }
    __syncthreads();
    // ---- one inverse transform per query head: lane holds elements el + EL * e ----
    for (int h = w; h < G; h += NW) {
        float x[NE];
#pragma unroll
        for (int e = 0; e < NE; e++) x[e] = vec[h * HP + el + EL * e];
        transform_reg<LY>(x, c_inv_sqrt(HD), lane);
        float *o = A.out + ((long long)seq * A.n_q + h0 + h) * HD;
#pragma unroll
        for (int e = 0; e < NE; e++)
            if (lane < EL) o[el + EL * e] = x[e];
    }
}

template <class LY, int NW, int NH, bool MULTI, bool SEQS>
hipError_t launch_wave(const SpAttnArgs &A, const SpSeqTab &T, const int *order, float *part, int nb, int tpw, int kb_lim,
                 int vb_lim, int *cnt, hipStream_t s) {
    const dim3 grid(A.n_kvh, nb, T.n_seq), block(64 * NW);
    std::conditional_t<SEQS, SpSeqTab, SpNoTab> tab{};
    if constexpr (SEQS) tab = T;
    if constexpr (!MULTI || NW <= wave_multi_nw(LY::HD, NH)) {
        if (A.out) {
            hipLaunchKernelGGL((k_attn_wave<LY, NW, true, NH, MULTI, SEQS>), grid, block, 0, s, A, order, part, nb, tpw, kb_lim,
                               vb_lim, cnt, tab);
            return hipGetLastError();
        }
    } else if (A.out) {
        return hipErrorInvalidValue;
    }
    hipLaunchKernelGGL((k_attn_wave<LY, NW, false, NH, MULTI, SEQS>), grid, block, 0, s, A, order, part, nb, tpw, kb_lim,
                       vb_lim, cnt, tab);
    return hipGetLastError();
}

// Whether the K and V plans are the layout's records.
template <class LY>
bool wave_layout_is(const SpPlan &KP, const SpPlan &VP) {
    if (KP.hd != LY::HD || VP.hd != LY::HD || KP.skip_transform || VP.skip_transform || KP.total_bytes != LY::KB ||
        VP.total_bytes != LY::VB || KP.n_bands != LY::NB || VP.n_bands != 1 || VP.band_bits[0] != LY::VBITS)
        return false;
    for (int b = 0; b < LY::NB; b++)
        if (KP.band_bits[b] != LY::bits[b] || KP.band_off[b] != LY::off(b) || KP.band_sz[b] != LY::sz(b) ||
            KP.band_byte_off[b] != LY::kbyte(b))
            return false;
    return true;
}

}  // namespace

// One launch over T's sequences with nb blocks of nw waves per (KV head, sequence), tpw
// tiles per wave; each layout's file instantiates it.
struct SpWaveLaunch {
    const SpAttnArgs &A;
    const SpSeqTab &T;
    const int *order;
    float *part;
    int nb, nw, tpw, kbands, vbands;
    int *counters;
    hipStream_t s;
};

hipError_t sp_wave_hd64_bridge(const SpWaveLaunch &W);
hipError_t sp_wave_hd64_ship(const SpWaveLaunch &W);
hipError_t sp_wave_hd96(const SpWaveLaunch &W);
hipError_t sp_wave_hd128(const SpWaveLaunch &W);
hipError_t sp_wave_hd256(const SpWaveLaunch &W);

namespace {

// The record layouts served: the bridge's default bands at head_dim 64 and 96 (K 5/4/4,
// V 5) and 128 and 256 (K 5/5/4/3, V 3), and the latter at head_dim 64.
using WaveHd64Bridge = WaveLayout<64, 5, true, 5, 4, 4>;
using WaveHd64Ship = WaveLayout<64, 3, true, 5, 5, 4, 3>;
using WaveHd96 = WaveLayout<96, 5, true, 5, 4, 4>;
using WaveHd128 = WaveLayout<128, 3, false, 5, 5, 4, 3>;
using WaveHd256 = WaveLayout<256, 3, true, 5, 5, 4, 3>;

template <class LY, int NW, int NH, bool MULTI>
hipError_t launch_wave_seqs(const SpWaveLaunch &W) {
    if (W.T.n_seq > 1)
        return launch_wave<LY, NW, NH, MULTI, true>(W.A, W.T, W.order, W.part, W.nb, W.tpw, W.kbands, W.vbands, W.counters, W.s);
    return launch_wave<LY, NW, NH, MULTI, false>(W.A, W.T, W.order, W.part, W.nb, W.tpw, W.kbands, W.vbands, W.counters, W.s);
}
template <class LY, int NW, int NH>
hipError_t wave_launch_nw(const SpWaveLaunch &W) {
    if (W.tpw == 1) return launch_wave_seqs<LY, NW, NH, false>(W);
    if constexpr (NW <= wave_multi_nw(LY::HD, NH)) return launch_wave_seqs<LY, NW, NH, true>(W);
    else if constexpr (LY::HD == 128 && NW == 16) {  // scores of one sequence
        if (W.T.n_seq == 1)
            return launch_wave<LY, NW, NH, true, false>(W.A, W.T, W.order, W.part, W.nb, W.tpw, W.kbands, W.vbands, W.counters, W.s);
    }
    return hipErrorInvalidValue;
}
template <class LY, int NH>
hipError_t wave_launch_nh(const SpWaveLaunch &W) {
    if (W.nw == 4) return wave_launch_nw<LY, 4, NH>(W);
    if (W.nw == 8) return wave_launch_nw<LY, 8, NH>(W);
    if constexpr (wave_max_nw(LY::HD) == 16) return wave_launch_nw<LY, 16, NH>(W);
    return hipErrorInvalidValue;
}
template <class LY>
hipError_t wave_launch(const SpWaveLaunch &W) {
    return W.A.n_q / W.A.n_kvh <= 4 ? wave_launch_nh<LY, 1>(W) : wave_launch_nh<LY, 2>(W);
}

}  // namespace
