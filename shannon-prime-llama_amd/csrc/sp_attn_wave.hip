// sp_attn_wave.hip -- the matrix-core decode-attention kernel (sp_attn_wave.h): the
// dispatch over record layouts and launch shapes, and the instances for head_dim 128,
// K 5/5/4/3 and V 3.
#include "sp_attn_wave.h"

hipError_t sp_wave_hd128(const SpWaveLaunch &W) { return wave_launch<WaveHd128>(W); }

// Compute units of the current device (cached per device).
static int wave_device_cus() {
    static int cus[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (cus[dev] <= 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cus[dev] = n;
    }
    return cus[dev];
}

// Waves per block and tiles per wave of a launch over `tiles` tiles (all KV heads and
// sequences), the longest sequence `longest` tiles. Measured per layer on 256 CUs (8 KV
// heads, GQA 4, unless said):
//   * fewer tiles than resident waves: one tile per wave. Small blocks spread a short
//     sequence over more CUs, large ones leave fewer partials to the last block's merge
//     (head_dim 128, blocks of 4 / 8 / 16 waves: 4096 positions 9.3 / 10.2 / 13.7 us, 16384
//     15.5 / 11.9 / 14.4, 32768 24.1 / 17.8 / 15.9).
//   * more: several tiles per wave, so a wave's next records load behind its values and
//     one merge serves them all (head_dim 96, 32 KV heads, 65536 tiles: 1 tile 134-157 us, 16
//     tiles 101 us), in the smallest block that covers the sequence, which then merges inside
//     the block alone.
//   * where several tiles per wave need 168 registers (3 waves a SIMD, blocks of 4), from 1.5
//     times the wave slots on, aimed at two blocks a CU (more only add partials) and at most 8
//     tiles (head_dim 128: 8192 tiles 26.5 us against 29.0 at one tile per wave, 16384 tiles
//     39.1 against 54.1, 4096 tiles 18.7 against 16.3). One sequence's scores alone, with no
//     partials to merge, go in blocks of 16 over one round there, from 9/8 of the slots on (60000
//     positions 9.3 us against 11.5, 131000 17.8 against 20.6, 40000 9.0 against 10.6, 33000, below the
//     line, 9.0 against 8.5; 8 query heads 15.0 against 16.5, 31.3 against 33.5).
// The block sizes' lines were measured at head_dim 128; at 64, 96 and 256, 1 to 8 query heads and
// one sequence of 250 to 40000 positions they are within 10% of the best of the three sizes but
// for 5000 tiles at one tile per wave (8 waves would be 15-25% faster than 16). Batches of
// short sequences with 5 to 8 heads per KV head would be up to twice as fast in blocks of 16
// (12 of up to 600 positions: 25.9 us, 12.2): a last block of 4 merges eight heads in four rounds.
struct WaveShape {
    int nw, tpw;
};
static WaveShape wave_shape(int hd, int nh, int cus, long long tiles, long long longest, int n_seq, bool out) {
    const int most = wave_max_nw(hd), multi = wave_multi_nw(hd, nh);
    const long long slots = (long long)cus * 4 * wave_waves_per_simd(hd, nh, false);
    // (5 to 8 tiles: one block of 8 has no partials to merge, 7.8 us against 9.2 at 333 positions)
    WaveShape s = {longest <= 4 ? 4 : longest <= 8 ? 8 : longest <= 64 ? 4 : longest <= 256 ? 8 : most, 1};
    if (hd == 128 && !out && n_seq == 1 && 8 * tiles >= 9 * slots) {
        s.nw = 16;
        s.tpw = (int)((tiles + slots - 1) / slots);
    } else if (multi == 4 && 2 * tiles >= 3 * slots) {
        s.nw = 4;
        s.tpw = (int)std::min({8LL, (tiles + slots / 2 - 1) / (slots / 2), (longest + 3) / 4});
    } else if (multi > 4 && tiles >= slots) {
        s.tpw = (int)((tiles + slots - 1) / slots);
        for (s.nw = 4; s.nw < multi && (long long)s.nw * s.tpw < longest;) s.nw *= 2;
        s.tpw = (int)std::min<long long>(s.tpw, (longest + s.nw - 1) / s.nw);  // no wave without a tile
    }
    return s;
}

hipError_t sp_launch_attn_wave(const SpPlan &KP, const SpPlan &VP, const int *order, const SpAttnArgs &A, const SpSeqTab &T,
                               float *part, size_t part_floats, int *counters, hipStream_t s) {
    const char *off = getenv("SP_HIP_NO_MFMA_ATTN");
    if (off && off[0] == '1') return hipErrorNotSupported;
    hipError_t (*run)(const SpWaveLaunch &) = nullptr;
    if (wave_layout_is<WaveHd128>(KP, VP)) run = sp_wave_hd128;
    else if (wave_layout_is<WaveHd96>(KP, VP)) run = sp_wave_hd96;
    else if (wave_layout_is<WaveHd64Bridge>(KP, VP)) run = sp_wave_hd64_bridge;
    else if (wave_layout_is<WaveHd64Ship>(KP, VP)) run = sp_wave_hd64_ship;
    else if (wave_layout_is<WaveHd256>(KP, VP)) run = sp_wave_hd256;
    if (!run || A.hd != KP.hd || A.kB != KP.total_bytes || A.vB != VP.total_bytes) return hipErrorNotSupported;
    if (A.n_q % A.n_kvh || A.n_q / A.n_kvh > 8 || A.n_kvh > SP_ATTN_MAX_KVH) return hipErrorNotSupported;
    // record bases on whole 16-bit words; K records of whole dwords stay on dwords
    const uintptr_t kal = A.kB % 4 ? 1 : 3;
    if (((uintptr_t)A.kpack & kal) || ((uintptr_t)A.vpack & 1) || ((uintptr_t)A.k_head_stride & kal) || (A.v_head_stride & 1))
        return hipErrorNotSupported;
    if (T.n_seq < 1 || T.n_seq > SP_ATTN_MAX_SEQ) return hipErrorInvalidValue;

    // Launches of consecutive sequences: as many as the arrival counters and the
    // partials' workspace hold (nearly always all of them).
    const int cus = wave_device_cus(), nh = A.n_q / A.n_kvh <= 4 ? 1 : 2;
    for (int s0 = 0, n; s0 < T.n_seq; s0 += n) {
        n = T.n_seq - s0;
        int nb = 0;
        WaveShape sh;
        for (;; n = (n + 1) / 2) {
            long long tiles = 0, longest = 0;
            for (int i = s0; i < s0 + n; i++) {
                const long long t = (T.len[i] + TILE - 1) / TILE;
                tiles += A.n_kvh * t;
                longest = std::max(longest, t);
            }
            sh = wave_shape(A.hd, nh, cus, tiles, longest, n, A.out != nullptr);
            nb = (int)((longest + (long long)sh.nw * sh.tpw - 1) / ((long long)sh.nw * sh.tpw));
            if (!A.out || n == 1 || nb == 1 ||
                (n * A.n_kvh <= SP_ATTN_MAX_KVH && (size_t)n * A.n_q * nb * (A.hd + 2) <= part_floats))
                break;
        }
        if (A.out && nb > 1 && (!part || !counters || (size_t)n * A.n_q * nb * (A.hd + 2) > part_floats)) return hipErrorInvalidValue;
        if (nb > 65535) return hipErrorInvalidValue;
        SpAttnArgs B = A;
        B.q += (size_t)s0 * A.n_q * A.hd;
        if (B.out) B.out += (size_t)s0 * A.n_q * A.hd;
        B.start = T.start[s0];
        B.n_kv = T.len[s0];
        if (B.scores && n == 1) B.scores += T.soff[s0];
        SpSeqTab U;
        memset(&U, 0, sizeof(U));
        U.n_seq = n;
        for (int i = 0; i < n; i++) {
            U.start[i] = T.start[s0 + i];
            U.len[i] = T.len[s0 + i];
            U.soff[i] = T.soff[s0 + i];
            U.max_len = std::max(U.max_len, U.len[i]);
        }
        const hipError_t e = run(SpWaveLaunch{B, U, order, part, nb, sh.nw, sh.tpw, KP.max_bands, VP.max_bands, counters, s});
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
