// sp_hier_codec.h -- device building blocks shared by the hierarchical codec kernels for
// the default geometry: the index tables and the predictions from scalar registers.
#pragma once
#include "sp_lane.h"

namespace {

// Default geometry (sp_hier_default_geometry): skeleton = the first NS entries
// of the squarefree-first order over [0, PAD), targets = the rest in order.
template <int PAD, int NS>
struct HierGeoC {
    static constexpr int NT = PAD - NS;
    int skel[NS];
    int tgt[NT];
    constexpr HierGeoC() : skel(), tgt() {
        const MobOrder<PAD> mo{};
        for (int s = 0; s < NS; s++) skel[s] = mo.v[s];
        for (int t = 0; t < NT; t++) tgt[t] = mo.v[NS + t];
    }
};
template <int PAD, int NS>
__device__ constexpr HierGeoC<PAD, NS> kHier{};

// Three predictions at once: ak += wk.lo*x0, then ak += wk.hi*x1 for k = 0..2, each
// step rounded once. v_fma_mix widens the fp16 weight (from a scalar register)
// exactly and rounds w*x + 0 (the + 0 turns a -0 product into +0, which a running
// sum started at +0.0f cannot tell apart: such a sum is never -0), then v_add_f32.
// The three independent chains give each add two free slots after its product; one
// asm block keeps products next to their adds, so the predictions stay serial chains
// in registers.
__device__ __forceinline__ void wmac3x2(float &a0, float &a1, float &a2, uint32_t w0, uint32_t w1, uint32_t w2,
                                        float x0, float x1) {
    float p0, p1, p2;
    __asm__("v_fma_mix_f32 %3, %6, %9, 0 op_sel_hi:[1,0,0]\n\t"
            "v_fma_mix_f32 %4, %7, %9, 0 op_sel_hi:[1,0,0]\n\t"
            "v_fma_mix_f32 %5, %8, %9, 0 op_sel_hi:[1,0,0]\n\t"
            "v_add_f32 %0, %0, %3\n\t"
            "v_add_f32 %1, %1, %4\n\t"
            "v_add_f32 %2, %2, %5\n\t"
            "v_fma_mix_f32 %3, %6, %10, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
            "v_fma_mix_f32 %4, %7, %10, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
            "v_fma_mix_f32 %5, %8, %10, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
            "v_add_f32 %0, %0, %3\n\t"
            "v_add_f32 %1, %1, %4\n\t"
            "v_add_f32 %2, %2, %5"
            : "+v"(a0), "+v"(a1), "+v"(a2), "=&v"(p0), "=&v"(p1), "=&v"(p2)
            : "s"(w0), "s"(w1), "s"(w2), "v"(x0), "v"(x1));
}

// The first step of wmac3x2 for sums started at +0.0f: 0 + w*x rounds to w*x + 0,
// which is what v_fma_mix gives (never -0), so the sums start at the first products
// (no zero moves, no first adds). after: a value the triple is ordered behind (an
// operand the block does not read).
__device__ __forceinline__ void wmac3x2_first(float &a0, float &a1, float &a2, uint32_t w0, uint32_t w1,
                                              uint32_t w2, float x0, float x1, float after) {
    float p0, p1, p2;
    __asm__("v_fma_mix_f32 %0, %6, %9, 0 op_sel_hi:[1,0,0]\n\t"
            "v_fma_mix_f32 %1, %7, %9, 0 op_sel_hi:[1,0,0]\n\t"
            "v_fma_mix_f32 %2, %8, %9, 0 op_sel_hi:[1,0,0]\n\t"
            "v_fma_mix_f32 %3, %6, %10, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
            "v_fma_mix_f32 %4, %7, %10, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
            "v_fma_mix_f32 %5, %8, %10, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
            "v_add_f32 %0, %0, %3\n\t"
            "v_add_f32 %1, %1, %4\n\t"
            "v_add_f32 %2, %2, %5"
            : "=&v"(a0), "=&v"(a1), "=&v"(a2), "=&v"(p0), "=&v"(p1), "=&v"(p2)
            : "s"(w0), "s"(w1), "s"(w2), "v"(x0), "v"(x1), "v"(after));
}

// W is read through the constant address space: the tile-uniform row address
// then always becomes scalar loads (the scalar cache), whatever the compiler
// can prove about the kernel's other stores.
typedef const __attribute__((address_space(4))) uint32_t *wptr_t;

// pred = sum_s (float)W[t][s] * sk[s] from 0.0f, s ascending, separately rounded
// products and adds (kernel_hier_predict, shannon_prime_hier.cu:74-92), for targets
// t, t+1, t+2: w holds their three rows, NS/2 fp16 pairs each, in scalar registers.
// after: a value the triple is ordered behind.
//
// With MORE, the rows of the next triple are loaded into wn after the first
// products: the wait for w (loaded one triple earlier) comes before those products,
// and a scalar-load wait covers every scalar load in flight, so rows loaded before it
// would be waited for there too. The scheduling barriers keep the loads in that
// place, with three targets' products (~180 VALU instructions) in front of the next
// wait. Loaded where their own target pair started, the rows left the wave (one per
// SIMD) waiting ~600 times per tile; one pair ahead, two targets' products covered
// each wait.
template <int NS, bool MORE>
__device__ __forceinline__ void hier_predict3(const uint32_t (&w)[3 * NS / 2], uint32_t (&wn)[3 * NS / 2],
                                              wptr_t next, const float (&sk)[NS], float after, float &r0,
                                              float &r1, float &r2) {
    static_assert(NS % 2 == 0, "rows of fp16 pairs");
    constexpr int RW = NS / 2;
    float a0, a1, a2;
    wmac3x2_first(a0, a1, a2, w[0], w[RW], w[2 * RW], sk[0], sk[1], after);
    if constexpr (MORE) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 3 * RW; i++) wn[i] = next[i];
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int s = 2; s < NS; s += 2) wmac3x2(a0, a1, a2, w[s / 2], w[RW + s / 2], w[2 * RW + s / 2], sk[s], sk[s + 1]);
    r0 = a0, r1 = a1, r2 = a2;
}

// fp16 halves H of a and b: a + b rounded once (exact widening).
template <int H>
__device__ __forceinline__ float add_f16_halves(uint32_t a, uint32_t b) {
    float r;
    if (H)
        __asm__("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[1,0,1] op_sel_hi:[1,0,1]" : "=v"(r) : "v"(a), "v"(b));
    else
        __asm__("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel_hi:[1,0,1]" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

}  // namespace
