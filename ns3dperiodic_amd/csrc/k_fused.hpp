// k_fused.hpp -- the fused pseudo-spectral stage pipeline.
//
// One evaluation of the 2/3-masked nonlinear term (reference
// calculate_convolution_2p3, Source/advection_2_3.cu:480-497) plus the
// projection/diffusion/update epilogue (Source/diffusion.cu:96-365) runs as
// five passes over HBM:
//   P1 x-inverse : w^ (3, FP64 state) -> mask, i kx  -> A (6 fields)
//   P2 y-inverse : A (6)              -> i ky       -> B (9 fields)
//   P3 z         : B (9) -> C2R (+ i kz), (w.grad)w, R2C -> C (3 fields)
//   P4 y-forward : C (3) -> D (3)
//   P5 x-forward : D (3) -> IPQ -> epilogue (update / RHS / Q out)
// Real-space fields never touch HBM.  NF=2 evaluates B(u,v) of the J.v path
// (calculate_convolution_2p3_UV, :500-525) with the same passes.
#pragma once
#include <type_traits>

#include "fft_core.hpp"

namespace ns3d {

template <typename T, int N> struct PtrArr { T* p[N]; };

// Minimum waves per SIMD requested from the register allocator (the passes are
// latency bound: more resident waves hide HBM latency better than ILP).
#ifndef NS3D_WAVES_XY
#define NS3D_WAVES_XY 2
#endif
#ifndef NS3D_WAVES_Z
#define NS3D_WAVES_Z 2
#endif
// Tile order of each pass (1: last tile first).  The 256 MB Infinity Cache
// behind L2 keeps part of what a pass has just written; a pass that reads it
// back in the reverse of the order it was written finds the newest data first.
// The y-inverse -> z -> y-forward passes walk the x-planes in the same
// direction when all run forward, and the x-forward -> x-inverse passes the
// (k, l) columns; reversing the z and x-inverse passes alternates both chains
// (256^3 step: FP64 -0.3%, FP32 modes -0.4 to -0.5%; results bitwise unchanged).
#ifndef NS3D_REV_XINV
#define NS3D_REV_XINV 1
#endif
#ifndef NS3D_REV_YINV
#define NS3D_REV_YINV 0
#endif
#ifndef NS3D_REV_Z
#define NS3D_REV_Z 1
#endif
#ifndef NS3D_REV_YFWD
#define NS3D_REV_YFWD 0
#endif
#ifndef NS3D_REV_XFWD
#define NS3D_REV_XFWD 0
#endif
// The x- and y-inverse passes stage their twiddle table after their first
// global loads are issued (1) or before them (0): the table's own round trip
// and block barrier then overlap the HBM latency of the pencil loads.  The
// other passes stage it first: issuing their loads first made the 512^3 z pass
// 3-4% (FP64) and the FP32 y-forward pass 5% slower, with no gain at 256^3.
#ifndef NS3D_TW_LATE
#define NS3D_TW_LATE 1
#endif
// Runs put(true_type) or put(false_type): the nontemporal and the ordinary form of a store loop.
template <class F> __device__ __forceinline__ void by_nt(int nt, F&& put) {
    if (nt)
        put(std::true_type{});
    else
        put(std::false_type{});
}
template <int REV>
__device__ __forceinline__ int tile_order(int bid, int nb) {
    return REV ? nb - 1 - bid : bid;
}
// Minimum waves per SIMD of the FP32 z pass and of the FP32 x-forward
// epilogue pass (their register budgets: 2 -> 256 VGPRs, 3 -> 168, 4 -> 128).
#ifndef NS3D_WAVES_Z32
#define NS3D_WAVES_Z32 2
#endif
#ifndef NS3D_WAVES_XFWD32
#define NS3D_WAVES_XFWD32 2
#endif
// Minimum waves per SIMD of the FP64 x-forward pass.
#ifndef NS3D_WAVES_XFWD64
#define NS3D_WAVES_XFWD64 2
#endif
// x-forward pass: modes of one component per operand unit, and units in flight
// (k_x_fwd_epi), for FP64 with 4 and 8 points per thread and for FP32.
#ifndef NS3D_XFWD_UM64
#define NS3D_XFWD_UM64 4
#endif
#ifndef NS3D_XFWD_RING64
#define NS3D_XFWD_RING64 2
#endif
#ifndef NS3D_XFWD_RING64_8
#define NS3D_XFWD_RING64_8 1
#endif
#ifndef NS3D_XFWD_UM32
#define NS3D_XFWD_UM32 1
#endif
#ifndef NS3D_XFWD_RING32
#define NS3D_XFWD_RING32 2
#endif
template <typename TB> constexpr int XFWD_UM = sizeof(TB) == 8 ? NS3D_XFWD_UM64 : NS3D_XFWD_UM32;
template <typename TB, int NX, int E>
constexpr int XFWD_RING = sizeof(TB) == 8 ? (E == 8 ? NS3D_XFWD_RING64_8 : NS3D_XFWD_RING64)
                                          : (NX >= 256 ? 1 : NS3D_XFWD_RING32);
template <typename TB, int NX>
constexpr int XFWD_WAVES = sizeof(TB) == 8 ? NS3D_WAVES_XFWD64 : (NX >= 256 ? 4 : NS3D_WAVES_XFWD32);
// x/y-pass plan: E = 8 points per thread (Plan) or 4 (ZPlan); chosen per kernel
// and precision by the host from measurements.
template <int N, int E> struct XYSel { using type = Plan<N>; };
template <int N> struct XYSel<N, 4> { using type = ZPlan<N>; };
template <int N, int E> using XYPlan = typename XYSel<N, E>::type;
// The inverse passes and the y-forward pass handle one field per block
// (blockIdx.y): shorter blocks, more of them in flight.
// Batches: blockIdx.z is the member of a batch of same-size fields advanced
// by one launch; each kernel shifts its per-member pointers by z times the
// member stride it is given (bsc: scratch, bwi: input state; 0 when z is 1).
#define NS3D_FIELD_LOOP(f, n) for (int f = blockIdx.y; f < (int)blockIdx.y + 1; f++)

// Members of a batch that sit out a step (resident requests of one grid that
// need fewer steps than the launch carries): member z takes part in step
// `step` iff step < left[z]; left null: every member does.  The test is
// uniform over a block, so an idle member's blocks return before any barrier.
struct MemberMask {
    const int* left;
    int step;
};
__device__ __forceinline__ bool member_idle(const MemberMask& m) { return m.left && m.step >= m.left[blockIdx.z]; }

// ---------------------------------------------------------------- P1
// x-inverse of M w^_b and of M (i kx w^_b).  Block: one y index k and P
// consecutive z indices l; lanes p-fastest so each row load is contiguous.
// grid.y enumerates the fields; with OS = 1 each block produces one output
// (w_b or dx w_b) and the input is read by two blocks.
// TS: scalar type of the state w (double, or float for the FP32-state RK3 loop).
// VEC = 1 (NF = 2): the second vector field comes from a reduced Krylov vector, vec[c*(N-1)
// + i-1] = Im v^_c[i] over the N modes of the reference layout (k_unpack_reduced's rule).
// ADD = 1: the transformed field is w + w2 (w2 of the same type and layout; the
// FP32-increment RK3 loop's stage value base + increment where no x-forward pass
// leaves P1's output), summed in FP64.
// The plan: XYPlan, or for FP64 where the x-forward pass carries P1 too, the mirror image
// of its plan (XInvPlan), so that both kernels give the same bits.
template <typename TB, int NX> constexpr bool MIRROR_P1 = sizeof(TB) == 8 && NX <= 256;
template <typename TB, int NX, int E>
using XInvPlan = typename std::conditional<MIRROR_P1<TB, NX>, typename SeqRev<typename XYPlan<NX, E>::R>::type,
                                           typename XYPlan<NX, E>::R>::type;
// P1's transforms are pinned (PencilFFT's PIN) wherever the x-forward pass may carry them.
template <typename TB, int NX> constexpr bool PIN_P1 = sizeof(TB) == 8 || NX % 5 != 0;
// i kx w: the products rounded by themselves (the transform's additions must not absorb them).
template <typename TB> __device__ __forceinline__ cplx<TB> ikx(cplx<double> s, double kx) {
    return mk<TB>((TB)mul_rounded(-s.y, kx), (TB)mul_rounded(s.x, kx));
}
template <typename TB, int NX, int P, int NF, int E, int OS, typename TS = double, int ADD = 0, int VEC = 0>
__global__ void __attribute__((amdgpu_waves_per_eu(NS3D_WAVES_XY, 8))) __launch_bounds__((P * XYPlan<NX, E>::TPP))
k_x_inv_grad(PtrArr<const cplx<TS>, 3 * NF> w, cplx<TB>* __restrict__ A, long nc, int Ny, int Mz, int Mw, int Ms,
             int nlt, int nb, SpecTables tab, const cplx<TB>* __restrict__ twg, int nt, long bwi, long bsc,
             MemberMask mm, PtrArr<const cplx<TS>, 3> w2 = {}, const double* __restrict__ vec = nullptr) {
    constexpr int TPP = XYPlan<NX, E>::TPP;
    using F = PencilFFT<TB, NX, TPP, +1, XInvPlan<TB, NX, E>, IndexMajor<P>, false, PIN_P1<TB, NX>>;
    __shared__ cplx<TB> lds[NX * P];
    __shared__ cplx<TB> tw[NX];
    const int bid0 = xcd_tile();
    if (bid0 >= nb || member_idle(mm)) return;
    const int bid = tile_order<NS3D_REV_XINV>(bid0, nb);
    const int tid = threadIdx.x, p = tid % P, t = tid / P;
    const int k = bid / nlt, lt = bid % nlt;
    const int l = lt * P + p;
    const bool lv = l < Mz;
    // a column (k,l) whose every x mode is masked stays unwritten: the y pass skips it
    const bool keep = lv && column_kept(tab, k, l);
    if (!__syncthreads_or(keep)) return;
    if (!NS3D_TW_LATE) stage_twiddles<TB, NX>(tw, twg);
    const long S = (long)Ny * Mw;        // state: row stride Mw (Mz: reference layout)
    const long base = (long)k * Mw + l;
    const long So = (long)Ny * Ms;       // scratch: rows padded to Ms
    const long baseo = (long)k * Ms + l;
    const int f = OS ? (int)blockIdx.y >> 1 : (int)blockIdx.y;
    const int which = OS ? (int)blockIdx.y & 1 : 0;  // OS: 0 -> w_b, 1 -> dx w_b
    const cplx<TS>* __restrict__ src = w.p[f] + (long)blockIdx.z * bwi;
    const cplx<TS>* __restrict__ src2 = ADD ? w2.p[f % 3] : nullptr;
    A += (long)blockIdx.z * bsc;
    cplx<TB> v[F::E], d[OS ? 1 : F::E];
    // the loads first (raw), then the twiddle table, then the arithmetic
    cplx<TS> raw[F::E], raw2[ADD != 0 ? F::E : 1];
#pragma unroll
    for (int q = 0; q < F::B0; q++) {
#pragma unroll
        for (int r = 0; r < F::R0; r++) {
            const int j = F::in_index(t, q, r);
            const int i = q * F::R0 + r;
            raw[i] = mk<TS>(0, 0);
            if constexpr (ADD != 0) raw2[i] = mk<TS>(0, 0);
            if (F::in_active(t, q) && keep && mask_keep(tab, j, k, l)) {
                if (VEC && f >= 3)   // (mode 0 is masked)
                    raw[i].y = (TS)vec[(f - 3) * ((long)NX * Ny * Mz - 1) + base + j * S - 1];
                else
                    raw[i] = src[base + j * S];
                if constexpr (ADD != 0) raw2[i] = src2[base + j * S];
            }
        }
    }
    if (NS3D_TW_LATE) stage_twiddles<TB, NX>(tw, twg);
#pragma unroll
    for (int q = 0; q < F::B0; q++) {
#pragma unroll
        for (int r = 0; r < F::R0; r++) {
            const int j = F::in_index(t, q, r);
            const int i = q * F::R0 + r;
            cplx<double> s = cvt<double>(raw[i]);
            if constexpr (ADD != 0) s = s + cvt<double>(raw2[i]);
            const double kx = F::in_active(t, q) ? tab.kx[j] : 0.0;
            const cplx<TB> dv = ikx<TB>(s, kx);
            if constexpr (OS) {
                v[q * F::R0 + r] = which ? dv : cvt<TB>(s);
            } else {
                v[q * F::R0 + r] = cvt<TB>(s);
                d[q * F::R0 + r] = dv;
            }
        }
    }
    const int s_ = f / 3, b = f % 3;
    cplx<TB>* __restrict__ ow = A + (long)(s_ * 6 + (OS ? 3 * which : 0) + b) * nc;
    cplx<TB>* __restrict__ od = A + (long)(s_ * 6 + 3 + b) * nc;
    F::run(v, lds, tw, t, p);
    if constexpr (!OS) F::run(d, lds, tw, t, p);
    if (keep) by_nt(nt, [&](auto NT) {
#pragma unroll
        for (int q = 0; q < F::BL; q++) {
            if (!F::out_active(t, q)) continue;
#pragma unroll
            for (int r = 0; r < F::RL; r++) {
                const long g = baseo + F::out_index(t, q, r) * So;
                st_cplx<NT.value>(ow + g, v[q * F::RL + r]);
                if constexpr (!OS) st_cplx<NT.value>(od + g, d[q * F::RL + r]);
            }
        }
    });
}

// ---------------------------------------------------------------- P2
// How P2 loads a thread's elements, of which some are masked.  Range
// checked: all at once.  Behind branches: at the lengths with a radix-3 or radix-5 pass, where
// a thread's last elements may not exist, most of the loads wait for the one before, and it is
// the compiler's choice how many.  P2 behind branches and range checked, FP64: 384^3 1.69 and
// 1.18 ms, 192^3 190 and 161 us, 160^3 115 and 81; FP32: 192^3 115 and 102, 320x384x320 735 and
// 518, 128^3 in an RK3 step 29.3 and 27.0.  The branches stay for FP64 powers of two (64^3 in a
// step 10.2 and 10.5 us), FP32 at 512 (512^3 1.65 and 1.82 ms) and at radix 5 (320^3 458 and 493 us).
template <typename TB, int NY>
constexpr bool Y_RANGE_LOADS = sizeof(TB) == 4 ? NY % 5 != 0 && NY < 512 : (NY & (NY - 1)) != 0;
// y-inverse: B(w_b) , B(dx w_b) , B(i ky w_b).  Block: one x index j and P z
// indices.  grid.y enumerates components; with OS = 1 each block produces one
// of the three outputs (A_b is then read by two blocks): a third of the serial
// chain of a block, for grids whose blocks all fit the chip at once (launch_y_inv).
template <typename TB, int NY, int P, int NF, int E, int OS>
__global__ void __attribute__((amdgpu_waves_per_eu(NS3D_WAVES_XY, 8))) __launch_bounds__((P * XYPlan<NY, E>::TPP))
k_y_inv_grad(const cplx<TB>* __restrict__ A, cplx<TB>* __restrict__ B, long nc, int Ny, int Mz, int Ms, int nlt,
             int nb, SpecTables tab, const cplx<TB>* __restrict__ twg, int nt, long bsc, MemberMask mm) {
    constexpr int TPP = XYPlan<NY, E>::TPP;
    using F = PencilFFT<TB, NY, TPP, +1, typename XYPlan<NY, E>::R, IndexMajor<P>, false, sizeof(TB) == 8>;
    __shared__ cplx<TB> lds[NY * P];
    __shared__ cplx<TB> tw[NY];
    const int bid0 = xcd_tile();
    if (bid0 >= nb || member_idle(mm)) return;
    const int bid = tile_order<NS3D_REV_YINV>(bid0, nb);
    const int tid = threadIdx.x, p = tid % P, t = tid / P;
    const int j = bid / nlt, lt = bid % nlt;
    if (lt * P > tab.lmax) return;  // z-planes beyond lmax are zero; the z pass skips them
    A += (long)blockIdx.z * bsc;
    B += (long)blockIdx.z * bsc;
    const int l = lt * P + p;
    const bool lv = l < Mz && l <= tab.lmax;
    if (!NS3D_TW_LATE) stage_twiddles<TB, NY>(tw, twg);
    const long S = Ms;
    const long base = (long)j * Ny * Ms + l;
    const int f = OS ? (int)blockIdx.y / 3 : (int)blockIdx.y;
    const int which = OS ? (int)blockIdx.y % 3 : -1;  // OS: 0 -> w_b, 1 -> dy w_b, 2 -> dx w_b
    const int s_ = f / 3, b = f % 3;
#ifndef NS3D_HOIST
#define NS3D_HOIST 1
#endif
    // A masked element is zero: RANGE: its load is out of a buffer's range, else it is not loaded.
    constexpr bool RANGE = Y_RANGE_LOADS<TB, NY>;
    int off[RANGE ? F::E : 1];   // byte offsets of this thread's elements in a field
    if constexpr (RANGE) {
#pragma unroll
        for (int q = 0; q < F::B0; q++) {
#pragma unroll
            for (int r = 0; r < F::R0; r++) {
                const int kk = F::in_active(t, q) ? F::in_index(t, q, r) : 0;
                const bool on = F::in_active(t, q) && lv && column_kept(tab, kk, lv ? l : 0);
                off[q * F::R0 + r] = on ? (int)((base + kk * S) * (long)sizeof(cplx<TB>)) : BUF_OOB;
            }
        }
    }
    auto load = [&](cplx<TB>* x, int field) __attribute__((always_inline)) {
        const auto src = buf_rsrc(A + (long)field * nc, (int)(nc * (long)sizeof(cplx<TB>)));
#pragma unroll
        for (int e = 0; e < F::B0 * F::R0; e++) x[e] = buf_load<TB>(src, off[RANGE ? e : 0]);
    };
    // x-derivative input, loaded before the first transforms when both are done here
    cplx<TB> v2[(!OS && NS3D_HOIST) ? F::E : 1];
    if constexpr (!OS && NS3D_HOIST && RANGE) {
        load(v2, s_ * 6 + 3 + b);
    } else if constexpr (!OS && NS3D_HOIST) {
        const cplx<TB>* __restrict__ src = A + (long)(s_ * 6 + 3 + b) * nc;
#pragma unroll
        for (int q = 0; q < F::B0; q++) {
#pragma unroll
            for (int r = 0; r < F::R0; r++) {
                const int kk = F::in_index(t, q, r);
                cplx<TB> s = mk<TB>(0, 0);
                if (F::in_active(t, q) && lv && column_kept(tab, kk, l)) s = src[base + kk * S];
                v2[q * F::R0 + r] = s;
            }
        }
    }
    // velocity component: produce w_b and dy w_b
    if (!OS || which < 2) {
        cplx<TB> v[F::E], d[OS ? 1 : F::E];
        if constexpr (RANGE) {
            load(v, s_ * 6 + b);
        } else {
            const cplx<TB>* __restrict__ src = A + (long)(s_ * 6 + b) * nc;
#pragma unroll
            for (int q = 0; q < F::B0; q++) {
#pragma unroll
                for (int r = 0; r < F::R0; r++) {
                    const int kk = F::in_index(t, q, r);
                    cplx<TB> s = mk<TB>(0, 0);
                    if (F::in_active(t, q) && lv && column_kept(tab, kk, l)) s = src[base + kk * S];
                    v[q * F::R0 + r] = s;
                }
            }
        }
        if (NS3D_TW_LATE) stage_twiddles<TB, NY>(tw, twg);
#pragma unroll
        for (int q = 0; q < F::B0; q++) {
#pragma unroll
            for (int r = 0; r < F::R0; r++) {
                const int kk = F::in_index(t, q, r);
                const cplx<TB> s = v[q * F::R0 + r];
                const TB ky = F::in_active(t, q) ? (TB)tab.ky[kk] : (TB)0;
                // (FP64: rounded products and pinned transforms, both forms of the pass give the same bits)
                const cplx<TB> dv = sizeof(TB) == 8 ? mk<TB>(mul_rounded(-s.y, ky), mul_rounded(s.x, ky)) : mk<TB>(-s.y * ky, s.x * ky);
                if constexpr (OS) {
                    v[q * F::R0 + r] = which ? dv : s;
                } else {
                    v[q * F::R0 + r] = s;
                    d[q * F::R0 + r] = dv;
                }
            }
        }
        F::run(v, lds, tw, t, p);
        if constexpr (!OS) F::run(d, lds, tw, t, p);
        cplx<TB>* __restrict__ ow = B + (long)(s_ * 9 + (OS && which == 1 ? 6 : 0) + b) * nc;
        cplx<TB>* __restrict__ od = B + (long)(s_ * 9 + 6 + b) * nc;
        if (lv) by_nt(nt, [&](auto NT) {
#pragma unroll
            for (int q = 0; q < F::BL; q++) {
                if (!F::out_active(t, q)) continue;
#pragma unroll
                for (int r = 0; r < F::RL; r++) {
                    const long g = base + F::out_index(t, q, r) * S;
                    st_cplx<NT.value>(ow + g, v[q * F::RL + r]);
                    if constexpr (!OS) st_cplx<NT.value>(od + g, d[q * F::RL + r]);
                }
            }
        });
    }
    // x-derivative component: plain y-inverse
    if (!OS || which == 2) {
        cplx<TB> v[F::E];
        if constexpr (!OS && NS3D_HOIST) {
#pragma unroll
            for (int e = 0; e < F::E; e++) v[e] = v2[e];
        } else if constexpr (RANGE) {
            load(v, s_ * 6 + 3 + b);
        } else {
            const cplx<TB>* __restrict__ src = A + (long)(s_ * 6 + 3 + b) * nc;
#pragma unroll
            for (int q = 0; q < F::B0; q++) {
#pragma unroll
                for (int r = 0; r < F::R0; r++) {
                    const int kk = F::in_index(t, q, r);
                    cplx<TB> s = mk<TB>(0, 0);
                    if (F::in_active(t, q) && lv && column_kept(tab, kk, l)) s = src[base + kk * S];
                    v[q * F::R0 + r] = s;
                }
            }
        }
        // with OS these blocks skip the velocity branch, where the table is staged otherwise
        if (NS3D_TW_LATE && OS) stage_twiddles<TB, NY>(tw, twg);
        F::run(v, lds, tw, t, p);
        cplx<TB>* __restrict__ ow = B + (long)(s_ * 9 + 3 + b) * nc;
        if (lv) by_nt(nt, [&](auto NT) {
#pragma unroll
            for (int q = 0; q < F::BL; q++) {
                if (!F::out_active(t, q)) continue;
#pragma unroll
                for (int r = 0; r < F::RL; r++) st_cplx<NT.value>(ow + (base + F::out_index(t, q, r) * S), v[q * F::RL + r]);
            }
        });
    }
}

// ---------------------------------------------------------------- P3
// z pass on one (x,y) pencil: paired C2R transforms (two real fields per
// complex FFT), the advective product, and paired R2C transforms.
// C2R convention: x,y passes already done; only Re of l=0 and l=Nz/2 is used.
template <typename TB, int NZ, int P, bool TRUNC = false, int NF = 1>
struct ZPencil {
    static constexpr int TPP = ZTPP<TB, NZ>;
    static constexpr int PAD = (sizeof(TB) == 8) ? 1 : 2;
#ifndef NS3D_ZSWZ
#define NS3D_ZSWZ 8
#endif
#ifndef NS3D_ZSWZ32
#define NS3D_ZSWZ32 16
#endif
    // LDS swizzle group in elements (0: none); measured gains: FP64 with the 4-point
    // plan, FP32 with the 8-point plan
#ifndef NS3D_R3_ZSWZ
#define NS3D_R3_ZSWZ 0
#endif
    static constexpr int SWG = sizeof(TB) == 8 ? (NZ % 3 == 0 && NZ >= 192 ? NS3D_R3_ZSWZ : NS3D_ZSWZ) : NS3D_ZSWZ32;
    using LA = typename std::conditional<SWG == 0, PencilMajor<NZ, PAD>, PencilMajorSw<NZ, PAD, (SWG == 0 ? 1 : SWG)>>::type;
    // Each pencil's LDS region is private to its TPP threads; when TPP divides
    // the wavefront size, those threads lie in one wavefront and every exchange
    // is ordered within the wave (exch_sync<true>) instead of by a block barrier.
#ifndef NS3D_ZWAVE
#define NS3D_ZWAVE 1
#endif
    static constexpr bool WAVE = NS3D_ZWAVE != 0 && TPP <= 64 && 64 % TPP == 0;
    // The first exchange by lane swaps, FP64 at power-of-two lengths: z pass at 512^3 3.40 ->
    // 3.10 ms, 256^3 0.324 -> 0.309, 128^3 49.3 -> 47.6 us, bilinear 86.6 -> 80.4; at 64 the
    // bilinear step gains (J.v 48.0 -> 47.3 us), the other does not (65 fields 280 -> 282 us).
    static constexpr bool SWAP = sizeof(TB) == 8 && (NZ & (NZ - 1)) == 0 && NZ >= (NF == 2 ? 64 : 128);
    static_assert(!SWAP || P * TPP % 64 == 0, "whole waves");
    using FI = PencilFFT<TB, NZ, TPP, +1, typename ZPlanT<TB, NZ>::R, LA, WAVE, false, SWAP>;
    using FF = PencilFFT<TB, NZ, TPP, -1, typename SeqRev<typename ZPlanT<TB, NZ>::R>::type, LA, WAVE, false, SWAP>;
    __device__ __forceinline__ static void lanes(int tid, int& t, int& p) {
        if constexpr (SWAP) {
            SwapLanes<TPP>::map(tid, t, p);
        } else {
            t = tid % TPP;
            p = tid / TPP;
        }
    }
    static_assert(FI::RL == FF::R0 && FI::BL == FF::B0, "mirror plans must share the product layout");
    static constexpr int E = FI::E > FF::E ? FI::E : FF::E;
    static constexpr int NPT = FI::BL * FI::RL;  // physical points per thread

    // Load the Hermitian extension of (X1 + i X2); dk selects i*kz multiplication.
    __device__ __forceinline__ static void load_pair(cplx<TB>* v, const cplx<TB>* __restrict__ s1, bool d1,
                                                     const cplx<TB>* __restrict__ s2, bool d2, bool valid,
                                                     const SpecTables& tab, int t) {
#pragma unroll
        for (int q = 0; q < FI::B0; q++) {
#pragma unroll
            for (int r = 0; r < FI::R0; r++) {
                const int n = FI::in_index(t, q, r);
                const int sl = n <= NZ / 2 ? n : NZ - n;
                cplx<TB> a = mk<TB>(0, 0), b = mk<TB>(0, 0);
                TB kz = 0;
                if (FI::in_active(t, q)) {
                    kz = (TB)tab.kz[sl];
                    if (valid && (!TRUNC || sl <= tab.lmax)) {
                        a = s1[sl];
                        b = s2[sl];
                    }
                }
                if (d1) a = mk<TB>(-a.y * kz, a.x * kz);
                if (d2) b = mk<TB>(-b.y * kz, b.x * kz);
                if (n == 0 || n == NZ / 2) {
                    a.y = 0;
                    b.y = 0;
                } else if (n > NZ / 2) {
                    a.y = -a.y;
                    b.y = -b.y;
                }
                v[q * FI::R0 + r] = mk<TB>(a.x - b.y, a.y + b.x);
            }
        }
    }

    // Split form of load_pair for software pipelining.  fetch_pair issues the
    // global loads of a pair's first-pass inputs (zeros where inactive,
    // invalid or truncated); finish_pair forms the Hermitian-extended
    // (X1 + i X2) from them.  kz_regs holds kz of each input slot (the same
    // for every pair).
    static constexpr int NIN = FI::B0 * FI::R0;
    __device__ __forceinline__ static void kz_regs(TB* kz, const SpecTables& tab, int t) {
#pragma unroll
        for (int q = 0; q < FI::B0; q++) {
#pragma unroll
            for (int r = 0; r < FI::R0; r++) {
                const int n = FI::in_index(t, q, r);
                const int sl = n <= NZ / 2 ? n : NZ - n;
                kz[q * FI::R0 + r] = FI::in_active(t, q) ? (TB)tab.kz[sl] : (TB)0;
            }
        }
    }
    __device__ __forceinline__ static void fetch_pair(cplx<TB>* r1, cplx<TB>* r2, const cplx<TB>* __restrict__ s1,
                                                      const cplx<TB>* __restrict__ s2, bool valid,
                                                      const SpecTables& tab, int t) {
#pragma unroll
        for (int q = 0; q < FI::B0; q++) {
#pragma unroll
            for (int r = 0; r < FI::R0; r++) {
                const int n = FI::in_index(t, q, r);
                const int sl = n <= NZ / 2 ? n : NZ - n;
                cplx<TB> a = mk<TB>(0, 0), b = mk<TB>(0, 0);
                // masked and truncated elements stay zero without a load (a branch-free
                // variant that loaded a clamped in-bounds element and zeroed it instead
                // made the 256^3 z pass 3.4x slower in FP64, 1.6x in FP32)
                if (FI::in_active(t, q) && valid && (!TRUNC || sl <= tab.lmax)) {
                    a = s1[sl];
                    b = s2[sl];
                }
                r1[q * FI::R0 + r] = a;
                r2[q * FI::R0 + r] = b;
            }
        }
    }
    // fetch_pair through buffer resources b1, b2 over the block's valid pencils:
    // prow = this pencil's first element in them (p * row stride); masked and
    // truncated elements and padding pencils fall outside the range and read 0.
    __device__ __forceinline__ static void fetch_pair_buf(cplx<TB>* r1, cplx<TB>* r2, __amdgpu_buffer_rsrc_t b1,
                                                          __amdgpu_buffer_rsrc_t b2, int prow, const SpecTables& tab,
                                                          int t) {
#pragma unroll
        for (int q = 0; q < FI::B0; q++) {
#pragma unroll
            for (int r = 0; r < FI::R0; r++) {
                const int n = FI::in_index(t, q, r);
                const int sl = n <= NZ / 2 ? n : NZ - n;
                const bool on = FI::in_active(t, q) && (!TRUNC || sl <= tab.lmax);
                const int o = on ? (prow + sl) * (int)sizeof(cplx<TB>) : BUF_OOB;
                r1[q * FI::R0 + r] = buf_load<TB>(b1, o);
                r2[q * FI::R0 + r] = buf_load<TB>(b2, o);
            }
        }
    }
    __device__ __forceinline__ static void finish_pair(cplx<TB>* v, const cplx<TB>* r1, bool d1, const cplx<TB>* r2,
                                                       bool d2, const TB* kz, int t) {
#pragma unroll
        for (int q = 0; q < FI::B0; q++) {
#pragma unroll
            for (int r = 0; r < FI::R0; r++) {
                const int i = q * FI::R0 + r;
                const int n = FI::in_index(t, q, r);
                cplx<TB> a = r1[i], b = r2[i];
                if (d1) a = mk<TB>(-a.y * kz[i], a.x * kz[i]);
                if (d2) b = mk<TB>(-b.y * kz[i], b.x * kz[i]);
                if (n == 0 || n == NZ / 2) {
                    a.y = 0;
                    b.y = 0;
                } else if (n > NZ / 2) {
                    a.y = -a.y;
                    b.y = -b.y;
                }
                v[i] = mk<TB>(a.x - b.y, a.y + b.x);
            }
        }
    }

    // load_pair through buffer resources over the block's valid pencils (as
    // fetch_pair_buf): out-of-range elements read as zero.
    __device__ __forceinline__ static void load_pair_buf(cplx<TB>* v, __amdgpu_buffer_rsrc_t b1, bool d1,
                                                         __amdgpu_buffer_rsrc_t b2, bool d2, int prow,
                                                         const SpecTables& tab, int t) {
#pragma unroll
        for (int q = 0; q < FI::B0; q++) {
#pragma unroll
            for (int r = 0; r < FI::R0; r++) {
                const int n = FI::in_index(t, q, r);
                const int sl = n <= NZ / 2 ? n : NZ - n;
                const bool on = FI::in_active(t, q) && (!TRUNC || sl <= tab.lmax);
                const int o = on ? (prow + sl) * (int)sizeof(cplx<TB>) : BUF_OOB;
                cplx<TB> a = buf_load<TB>(b1, o), b = buf_load<TB>(b2, o);
                const TB kz = FI::in_active(t, q) ? (TB)tab.kz[sl] : (TB)0;
                if (d1) a = mk<TB>(-a.y * kz, a.x * kz);
                if (d2) b = mk<TB>(-b.y * kz, b.x * kz);
                if (n == 0 || n == NZ / 2) {
                    a.y = 0;
                    b.y = 0;
                } else if (n > NZ / 2) {
                    a.y = -a.y;
                    b.y = -b.y;
                }
                v[q * FI::R0 + r] = mk<TB>(a.x - b.y, a.y + b.x);
            }
        }
    }
    __device__ __forceinline__ static void c2r_pair_buf(TB* x1, TB* x2, __amdgpu_buffer_rsrc_t b1, bool d1,
                                                        __amdgpu_buffer_rsrc_t b2, bool d2, int prow,
                                                        const SpecTables& tab, cplx<TB>* lds, const cplx<TB>* tw,
                                                        int t, int p, TB scale) {
        cplx<TB> v[E];
        load_pair_buf(v, b1, d1, b2, d2, prow, tab, t);
        FI::run(v, lds, tw, t, p);
#pragma unroll
        for (int e = 0; e < NPT; e++) {
            x1[e] = v[e].x * scale;
            x2[e] = v[e].y * scale;
        }
    }

    // Inverse-transform a pair; x1/x2 receive the scaled real fields.
    __device__ __forceinline__ static void c2r_pair(TB* x1, TB* x2, const cplx<TB>* s1, bool d1, const cplx<TB>* s2, bool d2,
                                                    bool valid, const SpecTables& tab, cplx<TB>* lds,
                                                    const cplx<TB>* tw, int t, int p, TB scale) {
        cplx<TB> v[E];
        load_pair(v, s1, d1, s2, d2, valid, tab, t);
        FI::run(v, lds, tw, t, p);
#pragma unroll
        for (int e = 0; e < NPT; e++) {
            x1[e] = v[e].x * scale;
            x2[e] = v[e].y * scale;
        }
    }

    // Forward-transform (q1 + i q2) and q3 at once (two exchange buffers) and
    // store the three half spectra: the results of r2c_pair(q1, q2) and
    // r2c_pair(q3, null), with one barrier per exchange for both.
    // With twr (the inverse plan's register twiddles; FI and FF must share
    // their radix sequence, as the palindromic power-of-two z plans do) the
    // forward transforms read their twiddles from registers too.
    static constexpr bool SAME_PLAN = std::is_same<typename ZPlanT<TB, NZ>::R,
                                                   typename SeqRev<typename ZPlanT<TB, NZ>::R>::type>::value;
    template <bool TWR>
    __device__ __forceinline__ static void r2c_two(const TB* q1, const TB* q2, const TB* q3, cplx<TB>* __restrict__ o1,
                                                   cplx<TB>* __restrict__ o2, cplx<TB>* __restrict__ o3, bool valid,
                                                   cplx<TB>* la, cplx<TB>* lb, const cplx<TB>* tw, int t, int p,
                                                   const typename FI::TwReg& twr, int nt) {
        cplx<TB> va[E], vb[E];
#pragma unroll
        for (int e = 0; e < NPT; e++) {
            va[e] = mk<TB>(q1[e], q2[e]);
            vb[e] = mk<TB>(q3[e], (TB)0);
        }
        if constexpr (TWR && SAME_PLAN)
            FF::run2_r(va, vb, la, lb, twr, t, p);
        else
            FF::run2(va, vb, la, lb, tw, t, p);
#pragma unroll
        for (int q = 0; q < FF::BL; q++) {
            if (!FF::out_active(t, q)) continue;
#pragma unroll
            for (int r = 0; r < FF::RL; r++) {
                la[LA::at(p, FF::out_index(t, q, r))] = va[q * FF::RL + r];
                lb[LA::at(p, FF::out_index(t, q, r))] = vb[q * FF::RL + r];
            }
        }
        exch_sync<WAVE>();
        if (valid) by_nt(nt, [&](auto NT) {
            for (int n = t; n <= NZ / 2; n += TPP) {
                const cplx<TB> zn = la[LA::at(p, n)];
                const cplx<TB> zm = la[LA::at(p, (NZ - n) % NZ)];
                st_cplx<NT.value>(o1 + n, mk<TB>((TB)0.5 * (zn.x + zm.x), (TB)0.5 * (zn.y - zm.y)));
                st_cplx<NT.value>(o2 + n, mk<TB>((TB)0.5 * (zn.y + zm.y), (TB)0.5 * (zm.x - zn.x)));
                st_cplx<NT.value>(o3 + n, lb[LA::at(p, n)]);
            }
        });
        exch_sync<WAVE>();
    }

    // Forward-transform (q1 + i q2) and store the two half spectra (q2 may be null).
    __device__ __forceinline__ static void r2c_pair(const TB* q1, const TB* q2, cplx<TB>* __restrict__ o1,
                                                    cplx<TB>* __restrict__ o2, bool valid, cplx<TB>* lds,
                                                    const cplx<TB>* tw, int t, int p, int nt = 0) {
        cplx<TB> v[E];
#pragma unroll
        for (int e = 0; e < NPT; e++) v[e] = mk<TB>(q1[e], q2 ? q2[e] : (TB)0);
        FF::run(v, lds, tw, t, p);
#pragma unroll
        for (int q = 0; q < FF::BL; q++) {
            if (!FF::out_active(t, q)) continue;
#pragma unroll
            for (int r = 0; r < FF::RL; r++) lds[LA::at(p, FF::out_index(t, q, r))] = v[q * FF::RL + r];
        }
        exch_sync<WAVE>();
        if (valid) by_nt(nt, [&](auto NT) {
            for (int n = t; n <= NZ / 2; n += TPP) {
                const cplx<TB> zn = lds[LA::at(p, n)];
                if (q2) {
                    const cplx<TB> zm = lds[LA::at(p, (NZ - n) % NZ)];
                    st_cplx<NT.value>(o1 + n, mk<TB>((TB)0.5 * (zn.x + zm.x), (TB)0.5 * (zn.y - zm.y)));
                    st_cplx<NT.value>(o2 + n, mk<TB>((TB)0.5 * (zn.y + zm.y), (TB)0.5 * (zm.x - zn.x)));
                } else {
                    st_cplx<NT.value>(o1 + n, zn);
                }
            }
        });
        exch_sync<WAVE>();
    }
};

template <typename TB, int NZ, int P, int NF>
// The bilinear z pass (24 real fields per point): with its inputs through
// buffer loads the FP32 pass fits 2 waves/SIMD in 240 VGPRs whatever the
// bound; FP64 fits 2 waves/SIMD in 252, or spills there at the lengths that
// run one pair at a time, which still beats 1 wave with the overflow in AGPRs.
#ifndef NS3D_WAVES_Z2
#define NS3D_WAVES_Z2 2
#endif
#ifndef NS3D_WAVES_Z2_32
#define NS3D_WAVES_Z2_32 1
#endif
__global__ void __attribute__((amdgpu_waves_per_eu(NF == 1 ? (sizeof(TB) == 4 ? NS3D_WAVES_Z32 : NS3D_WAVES_Z)
                                                          : (sizeof(TB) == 4 ? NS3D_WAVES_Z2_32 : NS3D_WAVES_Z2), 8)))
__launch_bounds__((P * ZTPP<TB, NZ>))
k_z_product(const cplx<TB>* __restrict__ Bf, cplx<TB>* __restrict__ C, long nc, long npen, int Mz, int nb,
            SpecTables tab, const cplx<TB>* __restrict__ twg, TB scale, TB* __restrict__ uphys, long nr, int nt, long bsc,
            MemberMask mm) {
    // B is zero on z-planes l > lmax (never written by the y pass): TRUNC skips them
    using Z = ZPencil<TB, NZ, P, true, NF>;
    constexpr int TPP = Z::TPP, NPT = Z::NPT;
#ifndef NS3D_ZILP
#define NS3D_ZILP 1
#endif
#ifndef NS3D_ZILP32
#define NS3D_ZILP32 0
#endif
    // Two paired transforms at once (two exchange buffers): FP64 at power-of-two
    // lengths (256^3: z pass 0.458 -> 0.406 ms) and at the radix-3 lengths whose pencils
    // lie within a wave (192^3: 0.193 -> 0.178 ms; the others spill).  Measured no gain in FP32.
    constexpr bool ILP = NF == 1 && ((NZ & (NZ - 1)) == 0 || (NZ % 3 == 0 && Z::WAVE)) && (sizeof(TB) == 8 ? NS3D_ZILP != 0 : NS3D_ZILP32 != 0);
#ifndef NS3D_ZTWREG
#define NS3D_ZTWREG 1
#endif
#ifndef NS3D_ZTWREG32
#define NS3D_ZTWREG32 0
#endif
    // The inverse transforms' twiddles in registers, read from the table once
    // (NZ >= 32; below, the extra registers cost a wave per SIMD).  FP64 at
    // 256^3: z pass 0.375 -> 0.352 ms, at 512^3 3.68 -> 3.54 ms (+42 and +24
    // VGPRs, no spills); FP32 measured 1% slower and stays on the LDS table.
    constexpr bool TWR = NF == 1 && NZ >= 32 && (sizeof(TB) == 8 ? NS3D_ZTWREG != 0 : NS3D_ZTWREG32 != 0);
#ifndef NS3D_ZTWFWD
#define NS3D_ZTWFWD 1
#endif
    // The bilinear pass in FP64 at the same lengths, its pairs two at a time as well: 128^3
    // 0.119 -> 0.096 ms, 256^3 0.95 -> 0.71 (where one pair at a time spilled 92 B a lane and
    // waited for its loads); at the other lengths two pairs spill more (160^3 0.49 -> 0.64).
    constexpr bool ILP2 = NF == 2 && sizeof(TB) == 8 && ((NZ & (NZ - 1)) == 0 || (NZ % 3 == 0 && Z::WAVE));
    __shared__ cplx<TB> lds[(ILP || ILP2 ? 2 : 1) * P * (NZ + Z::PAD)];
    __shared__ cplx<TB> tw[NZ];
    const int bid0 = xcd_tile();
    if (bid0 >= nb || member_idle(mm)) return;
    const int bid = tile_order<NS3D_REV_Z>(bid0, nb);
    stage_twiddles<TB, NZ>(tw, twg);
    const int tid = threadIdx.x;
    int t, p;
    Z::lanes(tid, t, p);
    const long pen = (long)bid * P + p;
    const bool valid = pen < npen;
    const long off = valid ? pen * Mz : 0;
    Bf += (long)blockIdx.z * bsc;
    C += (long)blockIdx.z * bsc;
    auto fld = [&](int f) { return Bf + (long)f * nc + off; };
#ifndef NS3D_ZBUF
#define NS3D_ZBUF 1
#endif
    // the first-pass inputs of fields fa and fb (the pipelined paths): with
    // NS3D_ZBUF through buffer resources over the block's valid pencils
    // (branch-free, no zero fill), else by predicated global loads
    const long pen0 = (long)bid * P;
    const int rbytes = (int)((npen - pen0 < P ? npen - pen0 : P) * Mz * (long)sizeof(cplx<TB>));
    auto rsrc = [&](int f) { return buf_rsrc(Bf + pen0 * Mz + (long)f * nc, rbytes); };
    auto fetch = [&](cplx<TB>* ra, cplx<TB>* rb, int fa, int fb) {
        if constexpr (NS3D_ZBUF != 0)
            Z::fetch_pair_buf(ra, rb, rsrc(fa), rsrc(fb), p * Mz, tab, t);
        else
            Z::fetch_pair(ra, rb, fld(fa), fld(fb), valid, tab, t);
    };
    // the bilinear path's paired inverse transform of fields fa, fb (d: times i kz)
    auto c2r = [&](TB* x1, TB* x2, int fa, bool d1, int fb, bool d2) {
        if constexpr (NS3D_ZBUF != 0)
            Z::c2r_pair_buf(x1, x2, rsrc(fa), d1, rsrc(fb), d2, p * Mz, tab, lds, tw, t, p, scale);
        else
            Z::c2r_pair(x1, x2, fld(fa), d1, fld(fb), d2, valid, tab, lds, tw, t, p, scale);
    };
    typename Z::FI::TwReg twi;
    if constexpr (TWR) Z::FI::load_tw(twi, tw, t);
    // field ids: s*9 + {0..2: w_b, 3..5: dx w_b, 6..8: dy w_b}
    TB Q[3][NPT];
    if constexpr (ILP) {
        // Two paired transforms at a time, the inputs of the next two loaded
        // before the current ones run; the same pairs and products as below.
        cplx<TB>* lb = lds + P * (NZ + Z::PAD);
        TB w[3][NPT], g0[NPT], g1[NPT], g2[NPT], g3[NPT], g4[NPT];
        TB kz[Z::NIN];
        cplx<TB> r1[Z::NIN], r2[Z::NIN], r3[Z::NIN], r4[Z::NIN];
        Z::kz_regs(kz, tab, t);
        fetch(r1, r2, 0, 1);
        fetch(r3, r4, 2, 3);
        // n1..n4: the fields of the next two pairs (-1: none)
        auto run_two = [&](TB* x1, TB* x2, bool d1, bool d2, TB* x3, TB* x4, bool d3, bool d4, int n1, int n2, int n3,
                           int n4) {
            cplx<TB> va[Z::E], vb[Z::E];
            Z::finish_pair(va, r1, d1, r2, d2, kz, t);
            Z::finish_pair(vb, r3, d3, r4, d4, kz, t);
            if (n1 >= 0) {
                fetch(r1, r2, n1, n2);
                fetch(r3, r4, n3, n4);
            }
            if constexpr (TWR)
                Z::FI::run2_r(va, vb, lds, lb, twi, t, p);
            else
                Z::FI::run2(va, vb, lds, lb, tw, t, p);
#pragma unroll
            for (int e = 0; e < NPT; e++) {
                x1[e] = va[e].x * scale;
                x2[e] = va[e].y * scale;
                x3[e] = vb[e].x * scale;
                x4[e] = vb[e].y * scale;
            }
        };
        // (w_x, w_y), (w_z, dx w_x)
        run_two(w[0], w[1], false, false, w[2], g0, false, false, 6, 0, 4, 7);
        if (uphys && valid) {
#pragma unroll
            for (int e = 0; e < NPT; e++) {
                if (!Z::FI::out_active(t, e / Z::FI::RL)) continue;
                const long g = pen * NZ + Z::FI::out_index(t, e / Z::FI::RL, e % Z::FI::RL);
                uphys[g] = w[0][e];
                uphys[nr + g] = w[1][e];
                uphys[2 * nr + g] = w[2][e];
            }
        }
        // (dy w_x, dz w_x), (dx w_y, dy w_y)
        run_two(g1, g2, false, true, g3, g4, false, false, 1, 5, 8, 2);
#pragma unroll
        for (int e = 0; e < NPT; e++) Q[0][e] = w[0][e] * g0[e] + w[1][e] * g1[e] + w[2][e] * g2[e];
        // (dz w_y, dx w_z), (dy w_z, dz w_z)
        run_two(g0, Q[2], true, false, g1, g2, false, true, -1, -1, -1, -1);
#pragma unroll
        for (int e = 0; e < NPT; e++) {
            Q[1][e] = w[0][e] * g3[e] + w[1][e] * g4[e] + w[2][e] * g0[e];
            Q[2][e] = w[0][e] * Q[2][e] + w[1][e] * g1[e] + w[2][e] * g2[e];
        }
    } else if constexpr (NF == 1) {
        // Software-pipelined: the loads of pair i+1 are issued before the
        // transform of pair i, so HBM latency overlaps the LDS passes.
        TB w[3][NPT], a[NPT], b[NPT], keep[NPT];
        TB kz[Z::NIN];
        cplx<TB> r1[Z::NIN], r2[Z::NIN];
        Z::kz_regs(kz, tab, t);
        fetch(r1, r2, 0, 1);
        auto run_pair = [&](TB* x1, TB* x2, bool d1, bool d2, int n1, int n2) {   // n1, n2: next pair (-1: none)
            cplx<TB> v[Z::E];
            Z::finish_pair(v, r1, d1, r2, d2, kz, t);
            if (n1 >= 0) fetch(r1, r2, n1, n2);
            if constexpr (TWR)
                Z::FI::run_r(v, lds, twi, t, p);
            else
                Z::FI::run(v, lds, tw, t, p);
#pragma unroll
            for (int e = 0; e < NPT; e++) {
                x1[e] = v[e].x * scale;
                x2[e] = v[e].y * scale;
            }
        };
        run_pair(w[0], w[1], false, false, 2, 3);   // w_x, w_y
        run_pair(w[2], keep, false, false, 6, 0);   // w_z, dx w_x
        if (uphys && valid) {
#pragma unroll
            for (int e = 0; e < NPT; e++) {
                if (!Z::FI::out_active(t, e / Z::FI::RL)) continue;
                const long g = pen * NZ + Z::FI::out_index(t, e / Z::FI::RL, e % Z::FI::RL);
                uphys[g] = w[0][e];
                uphys[nr + g] = w[1][e];
                uphys[2 * nr + g] = w[2][e];
            }
        }
        run_pair(a, b, false, true, 4, 7);          // dy w_x, dz w_x
#pragma unroll
        for (int e = 0; e < NPT; e++) Q[0][e] = w[0][e] * keep[e] + w[1][e] * a[e] + w[2][e] * b[e];
        run_pair(keep, a, false, false, 1, 5);      // dx w_y, dy w_y
        run_pair(b, Q[2], true, false, 8, 2);       // dz w_y, dx w_z
#pragma unroll
        for (int e = 0; e < NPT; e++) Q[1][e] = w[0][e] * keep[e] + w[1][e] * a[e] + w[2][e] * b[e];
        run_pair(a, b, false, true, -1, -1);        // dy w_z, dz w_z
#pragma unroll
        for (int e = 0; e < NPT; e++) Q[2][e] = w[0][e] * Q[2][e] + w[1][e] * a[e] + w[2][e] * b[e];
    } else if constexpr (ILP2) {
        // As the last branch below, two paired transforms at a time with the inputs of the
        // next two in flight (one u-derived, one v-derived pair).
        cplx<TB>* lb = lds + P * (NZ + Z::PAD);
        TB u[3][NPT], vv[3][NPT], a[NPT], b[NPT], c[NPT], d[NPT];
        TB kz[Z::NIN];
        cplx<TB> r1[Z::NIN], r2[Z::NIN], r3[Z::NIN], r4[Z::NIN];
        Z::kz_regs(kz, tab, t);
        fetch(r1, r2, 0, 1);
        fetch(r3, r4, 9, 10);
        auto run_two = [&](TB* x1, TB* x2, bool d1, bool d2, TB* x3, TB* x4, int n1, int n2, int n3, int n4) {
            cplx<TB> va[Z::E], vb[Z::E];
            Z::finish_pair(va, r1, d1, r2, d2, kz, t);
            Z::finish_pair(vb, r3, d1, r4, d2, kz, t);
            if (n1 >= 0) {
                fetch(r1, r2, n1, n2);
                fetch(r3, r4, n3, n4);
            }
            Z::FI::run2(va, vb, lds, lb, tw, t, p);
#pragma unroll
            for (int e = 0; e < NPT; e++) {
                x1[e] = va[e].x * scale;
                x2[e] = va[e].y * scale;
                x3[e] = vb[e].x * scale;
                x4[e] = vb[e].y * scale;
            }
        };
        run_two(u[0], u[1], false, false, vv[0], vv[1], 2, 3, 11, 12);
        run_two(u[2], a, false, false, vv[2], c, 6, 0, 15, 9);        // u_z, dx u_x; v_z, dx v_x
#pragma unroll
        for (int e = 0; e < NPT; e++) Q[0][e] = vv[0][e] * a[e] + u[0][e] * c[e];
        run_two(a, b, false, true, c, d, 4, 7, 13, 16);               // dy, dz of u_x; of v_x
#pragma unroll
        for (int e = 0; e < NPT; e++) {
            Q[0][e] += vv[1][e] * a[e] + vv[2][e] * b[e];
            Q[0][e] += u[1][e] * c[e] + u[2][e] * d[e];
        }
        run_two(a, b, false, false, c, d, 1, 5, 10, 14);              // dx, dy of u_y; of v_y
#pragma unroll
        for (int e = 0; e < NPT; e++) {
            Q[1][e] = vv[0][e] * a[e] + vv[1][e] * b[e];
            Q[1][e] += u[0][e] * c[e] + u[1][e] * d[e];
        }
        run_two(a, b, true, false, c, d, 8, 2, 17, 11);               // dz u_y, dx u_z; dz v_y, dx v_z
#pragma unroll
        for (int e = 0; e < NPT; e++) {
            Q[1][e] += vv[2][e] * a[e] + u[2][e] * c[e];
            Q[2][e] = vv[0][e] * b[e] + u[0][e] * d[e];
        }
        run_two(a, b, false, true, c, d, -1, -1, -1, -1);             // dy, dz of u_z; of v_z
#pragma unroll
        for (int e = 0; e < NPT; e++) {
            Q[2][e] += vv[1][e] * a[e] + vv[2][e] * b[e];
            Q[2][e] += u[1][e] * c[e] + u[2][e] * d[e];
        }
    } else {
        // Q_c = (v.grad) u_c + (u.grad) v_c  (convolute_2p3_UV, Source/advection_2_3.cu:401-475).
        // Each paired transform holds two u-derived or two v-derived fields,
        // never one of each: v (a Krylov vector) can be orders of magnitude
        // smaller than u, and a shared transform's rounding is relative to
        // the larger of its two fields.
        // ids: u_b = b, dx u_b = 3+b, dy u_b = 6+b; v_b = 9+b, dx v_b = 12+b, dy v_b = 15+b
        TB u[3][NPT], vv[3][NPT], a[NPT], b[NPT];
        c2r(u[0], u[1], 0, false, 1, false);
        c2r(vv[0], vv[1], 9, false, 10, false);
        c2r(u[2], a, 2, false, 3, false);      // u_z, dx u_x
        c2r(vv[2], b, 11, false, 12, false);   // v_z, dx v_x
#pragma unroll
        for (int e = 0; e < NPT; e++) Q[0][e] = vv[0][e] * a[e] + u[0][e] * b[e];
        c2r(a, b, 6, false, 0, true);          // dy u_x, dz u_x
#pragma unroll
        for (int e = 0; e < NPT; e++) Q[0][e] += vv[1][e] * a[e] + vv[2][e] * b[e];
        c2r(a, b, 15, false, 9, true);         // dy v_x, dz v_x
#pragma unroll
        for (int e = 0; e < NPT; e++) Q[0][e] += u[1][e] * a[e] + u[2][e] * b[e];
        c2r(a, b, 4, false, 7, false);         // dx u_y, dy u_y
#pragma unroll
        for (int e = 0; e < NPT; e++) Q[1][e] = vv[0][e] * a[e] + vv[1][e] * b[e];
        c2r(a, b, 1, true, 5, false);          // dz u_y, dx u_z
#pragma unroll
        for (int e = 0; e < NPT; e++) {
            Q[1][e] += vv[2][e] * a[e];
            Q[2][e] = vv[0][e] * b[e];
        }
        c2r(a, b, 13, false, 16, false);       // dx v_y, dy v_y
#pragma unroll
        for (int e = 0; e < NPT; e++) Q[1][e] += u[0][e] * a[e] + u[1][e] * b[e];
        c2r(a, b, 10, true, 14, false);        // dz v_y, dx v_z
#pragma unroll
        for (int e = 0; e < NPT; e++) {
            Q[1][e] += u[2][e] * a[e];
            Q[2][e] += u[0][e] * b[e];
        }
        c2r(a, b, 8, false, 2, true);          // dy u_z, dz u_z
#pragma unroll
        for (int e = 0; e < NPT; e++) Q[2][e] += vv[1][e] * a[e] + vv[2][e] * b[e];
        c2r(a, b, 17, false, 11, true);        // dy v_z, dz v_z
#pragma unroll
        for (int e = 0; e < NPT; e++) Q[2][e] += u[1][e] * a[e] + u[2][e] * b[e];
    }
    cplx<TB>* o0 = C + off;
    cplx<TB>* o1 = C + nc + off;
    cplx<TB>* o2 = C + 2 * nc + off;
    if constexpr (ILP) {
        Z::template r2c_two<TWR && NS3D_ZTWFWD != 0>(Q[0], Q[1], Q[2], o0, o1, o2, valid, lds, lds + P * (NZ + Z::PAD),
                                                     tw, t, p, twi, nt);
    } else {
        Z::r2c_pair(Q[0], Q[1], o0, o1, valid, lds, tw, t, p, nt);
        Z::r2c_pair(Q[2], nullptr, o2, nullptr, valid, lds, tw, t, p, nt);
    }
}

// ---------------------------------------------------------------- P4 / generic
// C2C transform along x (AXIS 0) or y (AXIS 1) of nf spectral fields, out of
// place or in place (each block reads its pencils completely before writing).
template <typename TB, int NA, int P, int DIR, int AXIS, int E>
__global__ void __attribute__((amdgpu_waves_per_eu(NS3D_WAVES_XY, 8))) __launch_bounds__((P * XYPlan<NA, E>::TPP))
k_axis_c2c(const cplx<TB>* in, cplx<TB>* out, int nf, long nc, int Ny, int Mz, int Ms, int nlt, int nb,
           const cplx<TB>* __restrict__ twg, int nt = 0, long bsc = 0, MemberMask mm = {}) {
    constexpr int TPP = XYPlan<NA, E>::TPP;
    using F = PencilFFT<TB, NA, TPP, DIR, typename XYPlan<NA, E>::R, IndexMajor<P>>;
    __shared__ cplx<TB> lds[NA * P];
    __shared__ cplx<TB> tw[NA];
    const int bid0 = xcd_tile();
    if (bid0 >= nb || member_idle(mm)) return;
    const int bid = tile_order<NS3D_REV_YFWD>(bid0, nb);
    stage_twiddles<TB, NA>(tw, twg);
    const int tid = threadIdx.x, p = tid % P, t = tid / P;
    const int o = bid / nlt, lt = bid % nlt;
    const int l = lt * P + p;
    const bool lv = l < Mz;
    const long S = AXIS == 0 ? (long)Ny * Ms : (long)Ms;
    const long base = AXIS == 0 ? (long)o * Ms + l : (long)o * Ny * Ms + l;
    in += (long)blockIdx.z * bsc;
    out += (long)blockIdx.z * bsc;
#pragma unroll 1
    NS3D_FIELD_LOOP(f, nf) {
        const cplx<TB>* src = in + (long)f * nc;
        cplx<TB>* dst = out + (long)f * nc;
        cplx<TB> v[F::E];
#pragma unroll
        for (int q = 0; q < F::B0; q++) {
#pragma unroll
            for (int r = 0; r < F::R0; r++) {
                cplx<TB> s = mk<TB>(0, 0);
                if (F::in_active(t, q) && lv) s = src[base + F::in_index(t, q, r) * S];
                v[q * F::R0 + r] = s;
            }
        }
        __syncthreads();  // in-place use: every pencil element is read before any is written
        F::run(v, lds, tw, t, p);
        if (lv) by_nt(nt, [&](auto NT) {
#pragma unroll
            for (int q = 0; q < F::BL; q++) {
                if (!F::out_active(t, q)) continue;
#pragma unroll
                for (int r = 0; r < F::RL; r++) st_cplx<NT.value>(dst + (base + F::out_index(t, q, r) * S), v[q * F::RL + r]);
            }
        });
    }
}

// ---------------------------------------------------------------- P5 epilogues
// EPI_STAGE32: EPI_STAGE with w, u0 and out in FP32 (the FP32-state RK3 loop);
// the arithmetic and the forcing stay FP64.
// EPI_UV_VEC: EPI_UV_RHS with v read from a reduced Krylov vector (vin, k_unpack_reduced's
// rule) and Im(r) - shift*Im(v) written to another (vout, k_pack_reduced's rule).
// EPI_INC / EPI_INC_FINAL: the SSP stages in increment form over a base state
// u^n held as a pair of FP32 fields, u^n = hi + lo (the FP32-increment RK3
// loop).  With w = base + d (d: the previous stage's FP32 increment, u0; null
// in the first stage):
//   EPI_INC        out = a1*(d + dt*L(w)),  base = hi (w)            out FP32
//   EPI_INC_FINAL  r = base + a1*(d + dt*L(w)),  base = hi + lo (w, out32):
//                  hi = fp32(r) written to w, lo = fp32(r - hi) to out32
// which is RK3_SSP's u1 = u + dt L(u), u2 = 3/4 u + 1/4 (u1 + dt L(u1)),
// u = 1/3 u + 2/3 (u2 + dt L(u2)) with a1 = 1, 1/4, 2/3 and the stage values
// u1 = u + d1, u2 = u + d2.  out may alias u0 (each mode is read, then written,
// by one thread).
enum EpiMode {
    EPI_Q = 0, EPI_STAGE = 1, EPI_RHS = 2, EPI_UV = 3, EPI_UV_RHS = 4, EPI_IUV = 5, EPI_STAGE32 = 6,
    EPI_INC = 7, EPI_INC_FINAL = 8, EPI_UV_VEC = 9
};

struct EpiArgs {
    cplx<double>* w[3];          // state (read; written in place for UV/UV_RHS/IUV); cplx<float> for EPI_STAGE32
    const cplx<double>* u0[3];   // SSP combination base (EPI_STAGE, may be null); cplx<float> for EPI_STAGE32
    const cplx<double>* f[3];    // forcing (EPI_STAGE / EPI_RHS, may be null)
    cplx<double>* out[3];        // output (EPI_Q, EPI_STAGE, EPI_RHS); cplx<float> for EPI_STAGE32
    double dt, Re, a0, a1;       // EPI_STAGE: out = a0*u0 + a1*E(w)
    double nu, dtnu;             // 1/Re and dt/Re (formed once on the host)
    // per-member dt and Re of a batch (device arrays indexed by blockIdx.z; null: dt, Re above)
    const double* dtv;
    const double* rev;
    int ipq;                     // reference IPQ rule (Q1)
    // mode (j,k,l) of w / u0 / out / f sits at (j*ny + k)*m + l: m = Mz for the
    // reference layout, a padded row stride for the library's own stage buffers
    int ny, mw, mu0, mo, mf;
    // batch member strides (elements) of w, u0 and out; f is shared by the members
    long bw, bu0, bo;
    // sticky non-finite flag: set to 1 by any lane that writes a NaN or Inf (may be null)
    int* nf;
    // EPI_INC_FINAL: the lo half of the state (read and written), rows of stride mw
    cplx<float>* out32[3];
    // EPI_UV_VEC (may be one vector)
    const double* vin;
    double* vout;
    double shift;
};

// Non-finite flag of the fused epilogues and the scalar stage: every lane that
// produced a NaN or Inf stores 1 (a plain vector store; all writers store the
// same value).  The flag is read and cleared by the host.
__device__ __forceinline__ void flag_nonfinite(int* nf, bool bad) {
    if (bad && nf) *(volatile int*)nf = 1;
}
template <typename T> __device__ __forceinline__ bool finite2(cplx<T> a) { return isfinite(a.x) && isfinite(a.y); }

// Projection/diffusion/update at one mode (Source/diffusion.cu:96-365), k_update's.
template <int MODE>
__device__ __forceinline__ void epilogue(const EpiArgs& ea, const SpecTables& tab, int j, int k, int l,
                                         cplx<double> Qx, cplx<double> Qy, cplx<double> Qz) {
    const long row = (long)j * ea.ny + k;
    const long gw = row * ea.mw + l, go = row * ea.mo + l, gf = row * ea.mf + l;
    static_assert(MODE == EPI_STAGE || MODE == EPI_RHS || MODE == EPI_UV || MODE == EPI_UV_RHS || MODE == EPI_IUV,
                  "the updates of ns3d_project_update");
    bool bad = false;
    const ProjCoef c = proj_coef(tab, j, k, l);
    const double AQr[3] = {c.a11 * Qx.x + c.a12 * Qy.x + c.a13 * Qz.x, c.a12 * Qx.x + c.a22 * Qy.x + c.a23 * Qz.x,
                           c.a13 * Qx.x + c.a23 * Qy.x + c.a33 * Qz.x};
    const double AQi[3] = {c.a11 * Qx.y + c.a12 * Qy.y + c.a13 * Qz.y, c.a12 * Qx.y + c.a22 * Qy.y + c.a23 * Qz.y,
                           c.a13 * Qx.y + c.a23 * Qy.y + c.a33 * Qz.y};
    const cplx<double> Q[3] = {Qx, Qy, Qz};
    const double dt = ea.dt;
#pragma unroll
    for (int b = 0; b < 3; b++) {
        cplx<double> r;
        const cplx<double> w = ea.w[b][gw];
        if (MODE == EPI_STAGE) {
            const double G = (1.0 - c.din * ea.dtnu);
            cplx<double> f = mk<double>(0.0, 0.0);
            if (ea.f[b]) f = ea.f[b][gf];
            r.x = dt * AQr[b] + G * w.x + dt * f.x - dt * Q[b].x;
            r.y = dt * AQi[b] + G * w.y + dt * f.y - dt * Q[b].y;
            ea.out[b][go] = r;
            bad |= !finite2(r);
        } else if (MODE == EPI_RHS) {
            const double G = (-c.din * ea.nu);
            cplx<double> f = mk<double>(0.0, 0.0);
            if (ea.f[b]) f = ea.f[b][gf];
            r.x = AQr[b] + G * w.x + f.x - Q[b].x;
            r.y = AQi[b] + G * w.y + f.y - Q[b].y;
            ea.out[b][go] = r;
            bad |= !finite2(r);
        } else if (MODE == EPI_UV) {
            const double G = (1.0 - c.din * ea.dtnu);
            r.x = dt * AQr[b] + G * w.x - dt * Q[b].x;
            r.y = dt * AQi[b] + G * w.y - dt * Q[b].y;
            ea.w[b][gw] = r;
            bad |= !finite2(r);
        } else if (MODE == EPI_UV_RHS) {
            const double G = (-c.din * ea.nu);
            r.x = AQr[b] + G * w.x - Q[b].x;
            r.y = AQi[b] + G * w.y - Q[b].y;
            ea.w[b][gw] = r;
            bad |= !finite2(r);
        } else {  // EPI_IUV
            const double G = (1.0 + c.din * ea.dtnu);
            r.x = (dt * AQr[b] + w.x - dt * Q[b].x) / G;
            r.y = (dt * AQi[b] + w.y - dt * Q[b].y) / G;
            ea.w[b][gw] = r;
            bad |= !finite2(r);
        }
    }
    flag_nonfinite(ea.nf, bad);
}

// set_to_zero_real (Source/advection_2_3.cu:35-70)
__device__ __forceinline__ void ipq_rule(cplx<double>& Qx, cplx<double>& Qy, cplx<double>& Qz, int ipq, bool origin) {
    if (ipq) {
        Qx.x = 0.0;
        Qy.x = 0.0;
        Qz.x = 0.0;
        if (origin) {
            Qx.y = 0.0;
            Qy.y = 0.0;
            Qz.y = 0.0;
        }
    }
}

// ---- P5 kernel: the epilogues of every mode, their operands read ahead.
// Scalar type of the state operands w, u0 and out in memory.
template <int MODE>
using EpiState = typename std::conditional<MODE == EPI_STAGE32 || MODE == EPI_INC || MODE == EPI_INC_FINAL, float,
                                           double>::type;
// The operands of UM consecutive modes of one component (what MODE does not read stays unused).
template <int MODE, int UM> struct EpiUnit {
    cplx<EpiState<MODE>> w[UM], u0[UM];
    cplx<float> lo[UM];
    cplx<double> f[UM];
};
// Wavenumber factor of x-index j, as the host table's 2*pi/Lx*m.
template <int NX> __device__ __forceinline__ double kx_of(const SpecTables& tab, int j) {
    return tab.kb1 * (double)(j >= NX / 2 ? j - NX : j);
}

// P5: x-forward transform and epilogue.  Bound by HBM at 256^3 and above (12 fields
// moved in 8-mode row segments) and by the latency of its gathers below.  The state,
// base and forcing operands are read ahead through buffer resources, UM modes of one
// component at a time (a unit) with RING units in flight, the first ones under the
// transforms, because loads issued mode by mode behind the stores of the mode before
// (which may alias them) left one round trip to each of a thread's modes exposed:
// 32^3 step 110 -> 84 us, 128^3 pass 70 -> 45 us, 256^3 0.402 -> 0.375 ms (FP64).  FP64
// keeps 4 modes a thread (202 VGPRs, 2 waves per SIMD; 8 modes leave no room for the
// operands and spill); from 256 points FP32 takes one unit at a time to stay under
// 128 VGPRs (two 512-thread blocks on a CU: 0.333 -> 0.299 ms).
//
// CHAIN: the P1 of the next stage on the columns just updated: w^ -> M w^ and
// M (i kx w^), both transformed back in x and written to A, so the next stage
// starts at P2 and its P1 never reads the state.  Both precisions repeat the plan of
// the standalone P1, so the results are bitwise its own: FP64 by the mirror image of
// the forward plan, which starts from the values as the epilogue leaves them; FP32 by
// the 8-point plan (EI points per thread) on half of a pencil's threads for each of the
// two transforms, after one exchange through LDS.  256^3 FP64: 0.44 ms on average
// against 0.185 + 0.375 for the two passes; 128^3 57 against 27 + 45 us.
template <typename TB, int NX, int P, int MODE, int E, int CHAIN, int EI = E>
__global__ void __attribute__((amdgpu_waves_per_eu(XFWD_WAVES<TB, NX>, 8))) __launch_bounds__((P * XYPlan<NX, E>::TPP))
k_x_fwd_epi(const cplx<TB>* D, cplx<TB>* A, long nc, int Ny, int Mz, int Ms, int nlt, int nb, SpecTables tab,
            const cplx<TB>* __restrict__ twg, EpiArgs ea, int nt, long bsc, MemberMask mm) {
    using Plan_ = XYPlan<NX, E>;
    constexpr int TPP = Plan_::TPP;
    using F = PencilFFT<TB, NX, TPP, -1, typename Plan_::R, IndexMajor<P>>;
    using TS = EpiState<MODE>;
    constexpr bool F64 = sizeof(TB) == 8;
    constexpr int NO = F::BL * F::RL;    // modes of each component a thread holds after the transform
    __shared__ cplx<TB> lds[2 * NX * P];
    __shared__ cplx<TB> tw[NX];
    const int bid0 = xcd_tile();
    if (bid0 >= nb || member_idle(mm)) return;
    const int bid = tile_order<NS3D_REV_XFWD>(bid0, nb);
    stage_twiddles<TB, NX>(tw, twg);
    const int tid = threadIdx.x, p = tid % P, t = tid / P;
    const int k = bid / nlt, lt = bid % nlt;
    const int l = lt * P + p;
    const bool lv = l < Mz;
    if (ea.dtv) {                        // per-member time step and Reynolds number
        const double dtm = ea.dtv[blockIdx.z], rem = ea.rev[blockIdx.z];
        ea.dt = dtm;
        ea.Re = rem;
        ea.nu = 1.0 / rem;
        ea.dtnu = dtm / rem;
    }
    const long z = blockIdx.z;           // batch member
    D += z * bsc;
    A += z * bsc;
    // D: this thread's elements, plane stride Ny*Ms
    const int strD = Ny * Ms * (int)sizeof(cplx<TB>);
    const int offD = lv ? (k * Ms + l) * (int)sizeof(cplx<TB>) : BUF_OOB;
    const int bytesD = (int)(nc * (long)sizeof(cplx<TB>));
    cplx<TB> qv[3][F::E];
#pragma unroll
    for (int b = 0; b < 3; b++) {
        const auto src = buf_rsrc(D + (long)b * nc, bytesD);
#pragma unroll
        for (int q = 0; q < F::B0; q++) {
            const int o = F::in_active(t, q) ? offD + t * strD : BUF_OOB;
#pragma unroll
            for (int r = 0; r < F::R0; r++)
                qv[b][q * F::R0 + r] = buf_load<TB>(src, lv ? o : BUF_OOB, (F::in_index(0, q, r)) * strD);
        }
    }
    // ---- operands: unit u = modes e0..e0+UM-1 of component b, u = b*UPC + e0/UM
    constexpr int UM = XFWD_UM<TB> < NO ? XFWD_UM<TB> : NO;
    constexpr int UPC = NO / UM, NU = 3 * UPC;
    static_assert(NO % UM == 0, "units cover a component");
    constexpr int RING = XFWD_RING<TB, NX, E> < NU ? XFWD_RING<TB, NX, E> : NU;
    constexpr bool HAS_U0 = MODE == EPI_STAGE || MODE == EPI_STAGE32 || MODE == EPI_INC || MODE == EPI_INC_FINAL;
    constexpr bool HAS_F = HAS_U0 || MODE == EPI_RHS;
    EpiUnit<MODE, UM> un[RING];
    const long nrow = (long)NX * Ny;
    auto rsrc_of = [&](const void* ptr, long shift, int m, int esz) __attribute__((always_inline)) {
        return buf_rsrc((const char*)ptr + shift * esz, (int)(nrow * m * esz));
    };
    auto voff = [&](int m, int esz, int q) __attribute__((always_inline)) {
        return lv && F::out_active(t, q) ? ((t * Ny + k) * m + l) * esz : BUF_OOB;
    };
    // reduced vectors: element i of component b at (vec - 1 + b*(N-1))[i], none for i = 0
    auto rsrc_vec = [&](const double* vec, int b) __attribute__((always_inline)) {
        return buf_rsrc(vec - 1 + (long)b * (nrow * Mz - 1), (int)(nrow * Mz * 8));
    };
    auto voff_vec = [&](int j, int q) __attribute__((always_inline)) { return (j | k | l) == 0 ? BUF_OOB : voff(Mz, 8, q); };
    auto load_unit = [&](auto UC) __attribute__((always_inline)) {
        constexpr int u = decltype(UC)::value, b = u / UPC, e0 = (u % UPC) * UM;
        EpiUnit<MODE, UM>& U = un[u % RING];
        constexpr int es = (int)sizeof(cplx<TS>);
        const auto rw = MODE == EPI_UV_VEC ? rsrc_vec(ea.vin, b) : rsrc_of(ea.w[b], z * ea.bw, ea.mw, es);
#pragma unroll
        for (int i = 0; i < UM; i++) {
            const int e = e0 + i;
            const int q = e / F::RL, so = F::out_index(0, q, e % F::RL) * Ny;
            if constexpr (MODE == EPI_UV_VEC)
                U.w[i] = mk<TS>(0, (TS)buf_load_f64(rw, voff_vec(F::out_index(t, q, e % F::RL), q), so * Mz * 8));
            else if constexpr (MODE != EPI_Q) U.w[i] = buf_load<TS>(rw, voff(ea.mw, es, q), so * ea.mw * es);
        }
        if constexpr (HAS_U0) {
            if (ea.u0[b]) {
                const auto ru = rsrc_of(ea.u0[b], z * ea.bu0, ea.mu0, es);
#pragma unroll
                for (int i = 0; i < UM; i++) {
                    const int e = e0 + i;
                    const int q = e / F::RL, so = F::out_index(0, q, e % F::RL) * Ny;
                    U.u0[i] = buf_load<TS>(ru, voff(ea.mu0, es, q), so * ea.mu0 * es);
                }
            } else {
#pragma unroll
                for (int i = 0; i < UM; i++) U.u0[i] = mk<TS>(0, 0);
            }
        }
        if constexpr (MODE == EPI_INC_FINAL) {
            const auto rl = rsrc_of(ea.out32[b], 0, ea.mw, es);
#pragma unroll
            for (int i = 0; i < UM; i++) {
                const int e = e0 + i;
                const int q = e / F::RL, so = F::out_index(0, q, e % F::RL) * Ny;
                U.lo[i] = buf_load<float>(rl, voff(ea.mw, es, q), so * ea.mw * es);
            }
        }
        if constexpr (HAS_F) {
            if (ea.f[b]) {
                const auto rf = rsrc_of(ea.f[b], 0, ea.mf, 16);
#pragma unroll
                for (int i = 0; i < UM; i++) {
                    const int e = e0 + i;
                    const int q = e / F::RL, so = F::out_index(0, q, e % F::RL) * Ny;
                    U.f[i] = buf_load<double>(rf, voff(ea.mf, 16, q), so * ea.mf * 16);
                }
            } else {
#pragma unroll
                for (int i = 0; i < UM; i++) U.f[i] = mk<double>(0.0, 0.0);
            }
        }
    };
    // chain: the masked modes of this thread's column, and whether any lane has some
    unsigned kept = 0;
    bool chained = false;
    bool col = false;
    if constexpr (CHAIN) {
        col = lv && column_kept(tab, k, l);
        if (col) {
#pragma unroll
            for (int e = 0; e < NO; e++) {
                const int q = e / F::RL, j = F::out_index(t, q, e % F::RL);
                if (F::out_active(t, q) && mask_keep(tab, j, k, l)) kept |= 1u << e;
            }
        }
    }
    const double ky = tab.ky[k], kz = lv ? tab.kz[l] : 0.0;
    // the first RING - 1 units are in flight while the transforms run; the block-wide vote
    // waits for the mask, so it comes after them (before D's loads: 32^3 step 80.9 us, here
    // 79.6; 256^3 3.88 ms, here 3.85)
    if constexpr (MODE != EPI_Q) static_for<0, RING - 1>([&](auto UC) __attribute__((always_inline)) { load_unit(UC); });
    if constexpr (CHAIN) chained = __syncthreads_or(col);
    F::run2(qv[0], qv[1], lds, lds + NX * P, tw, t, p);
    F::run(qv[2], lds, tw, t, p);
    const double kyz2 = ky * ky + kz * kz;
    // projection: AM Q - Q with AM Q = kv (kv.Q)/|k|^2.  FP64: R replaces Q;
    // FP32: Q stays in FP32 and kd = (kv.Q)/|k|^2 is kept in FP64.
    cplx<double> kd[(F64 || MODE == EPI_Q) ? 1 : NO];
    const double qs = MODE == EPI_RHS || MODE == EPI_UV_RHS || MODE == EPI_UV_VEC ? 1.0 : ea.dt;   // weight of (AM Q - Q)
#pragma unroll
    for (int e = 0; e < NO; e++) {
        const int j = F::out_index(t, e / F::RL, e % F::RL);
        cplx<double> Q[3] = {cvt<double>(qv[0][e]), cvt<double>(qv[1][e]), cvt<double>(qv[2][e])};
        ipq_rule(Q[0], Q[1], Q[2], ea.ipq, (j | k | l) == 0);
        if constexpr (MODE == EPI_Q) {
#pragma unroll
            for (int b = 0; b < 3; b++) qv[b][e] = cvt<TB>(Q[b]);
        } else {
            const double kx = kx_of<NX>(tab, j);
            const double k2 = kx * kx + kyz2;
            const double inv = (j | k | l) == 0 ? 0.0 : 1.0 / k2;
            cplx<double> d;
            d.x = (kx * Q[0].x + ky * Q[1].x + kz * Q[2].x) * inv;
            d.y = (kx * Q[0].y + ky * Q[1].y + kz * Q[2].y) * inv;
            const double kv[3] = {kx, ky, kz};
            if constexpr (F64) {
#pragma unroll
                for (int b = 0; b < 3; b++) qv[b][e] = mk<TB>(qs * (kv[b] * d.x - Q[b].x), qs * (kv[b] * d.y - Q[b].y));
            } else {
                kd[e] = d;
#pragma unroll
                for (int b = 0; b < 3; b++) qv[b][e] = cvt<TB>(Q[b]);   // after the IPQ rule
            }
        }
    }
    // chain: inverse transforms of one component's w and dx w, stored to A
    auto chain = [&](int b, cplx<TB>* v, cplx<TB>* d) __attribute__((always_inline)) {
        auto put = [&](auto FC, cplx<TB>* x, int field, int ti) __attribute__((always_inline)) {
            using FX = decltype(FC);
            const auto ra = buf_rsrc(A + (long)field * nc, bytesD);
            by_nt(nt, [&](auto NT) __attribute__((always_inline)) {
#pragma unroll
                for (int q = 0; q < FX::BL; q++) {
                    const int o = col && FX::out_active(ti, q) ? offD + ti * strD : BUF_OOB;
#pragma unroll
                    for (int r = 0; r < FX::RL; r++)
                        buf_store<TB, NT.value>(ra, x[q * FX::RL + r], o, FX::out_index(0, q, r) * strD);
                }
            });
        };
        if constexpr (F64) {
            // the mirror-image plan: its first pass reads what the last forward pass holds
            static_assert(!CHAIN || MIRROR_P1<TB, NX>, "the standalone P1 runs the same plan");
            using FI = PencilFFT<TB, NX, TPP, +1, XInvPlan<TB, NX, E>, IndexMajor<P>, false, true>;
            FI::run2(v, d, lds, lds + NX * P, tw, t, p);
            put(FI{}, v, b, t);
            put(FI{}, d, 3 + b, t);
        } else {
            // the standalone P1's plan on half the threads for each transform
            constexpr int TPI = XYPlan<NX, EI>::TPP;
            static_assert(!CHAIN || PIN_P1<TB, NX>, "the standalone P1 rounds alike");
            static_assert(!CHAIN || TPP == 2 * TPI, "half of a pencil's threads run each of its two inverse transforms");
            using FI = PencilFFT<TB, NX, TPI, +1, typename XYPlan<NX, EI>::R, IndexMajor<P>, false, PIN_P1<TB, NX>>;
#pragma unroll
            for (int e = 0; e < NO; e++) {
                const int q = e / F::RL, j = F::out_index(t, q, e % F::RL);
                if (!F::out_active(t, q)) continue;
                lds[j * P + p] = v[e];
                lds[NX * P + j * P + p] = d[e];
            }
            __syncthreads();
            const int h = t >= TPI ? 1 : 0, ti = t - h * TPI;
            cplx<TB>* half = lds + h * NX * P;
            cplx<TB> x[FI::E];
#pragma unroll
            for (int q = 0; q < FI::B0; q++) {
                if (!FI::in_active(ti, q)) continue;
#pragma unroll
                for (int r = 0; r < FI::R0; r++) x[q * FI::R0 + r] = half[FI::in_index(ti, q, r) * P + p];
            }
            __syncthreads();
            FI::run(x, half, tw, ti, p);
            cplx<TB>* dst = A + (long)(b + 3 * h) * nc + ((long)k * Ms + l);
            const long str = (long)Ny * Ms;
            if (col) by_nt(nt, [&](auto NT) __attribute__((always_inline)) {
#pragma unroll
                for (int q = 0; q < FI::BL; q++) {
                    if (!FI::out_active(ti, q)) continue;
#pragma unroll
                    for (int r = 0; r < FI::RL; r++) st_cplx<NT.value>(dst + FI::out_index(ti, q, r) * str, x[q * FI::RL + r]);
                }
            });
        }
    };
    bool bad = false;
    cplx<TB> cv[CHAIN ? F::E : 1], cd[CHAIN ? F::E : 1];   // (F::E: also the mirror-image plan's registers)
    static_for<0, NU>([&](auto UC) __attribute__((always_inline)) {
        constexpr int u = decltype(UC)::value, b = u / UPC, e0 = (u % UPC) * UM;
        if constexpr (MODE != EPI_Q && u + RING - 1 < NU) load_unit(std::integral_constant<int, u + RING - 1>{});
        const EpiUnit<MODE, UM>& U = un[u % RING];
        constexpr int es = (int)sizeof(cplx<TS>);
        // UV, UV_RHS and IUV update w in place
        constexpr bool INPLACE = MODE == EPI_UV || MODE == EPI_UV_RHS || MODE == EPI_IUV || MODE == EPI_INC_FINAL;
        const int mo = INPLACE ? ea.mw : ea.mo;   // (EPI_UV_VEC stores through its own resource)
        const auto ro = rsrc_of(INPLACE ? ea.w[b] : ea.out[b], INPLACE ? z * ea.bw : z * ea.bo, mo, es);
#pragma unroll
        for (int i = 0; i < UM; i++) {
            const int e = e0 + i;
            const int q = e / F::RL, jo = F::out_index(0, q, e % F::RL), j = t + jo;
            const int vo = voff(mo, es, q), so = jo * Ny * mo * es;
            if constexpr (MODE == EPI_Q) {
                const cplx<double> r = cvt<double>(qv[b][e]);
                buf_store<double>(ro, r, vo, so);
                bad |= vo >= 0 && !finite2(r);
                continue;
            } else {
                const double kx = kx_of<NX>(tab, j);
                const double k2 = kx * kx + kyz2;
                cplx<double> R;
                if constexpr (F64) {
                    R = qv[b][e];
                } else {
                    const double kb = b == 0 ? kx : (b == 1 ? ky : kz);
                    const cplx<double> Q = cvt<double>(qv[b][e]);
                    R = mk<double>(qs * (kb * kd[e].x - Q.x), qs * (kb * kd[e].y - Q.y));
                }
                cplx<double> r, w = cvt<double>(U.w[i]);
                cplx<TS> keepv = mk<TS>(0, 0);   // the stage value as written
                if constexpr (MODE == EPI_STAGE || MODE == EPI_STAGE32) {
                    const double G = 1.0 - k2 * ea.dtnu;
                    r.x = R.x + G * w.x + ea.dt * U.f[i].x;
                    r.y = R.y + G * w.y + ea.dt * U.f[i].y;
                    r.x = ea.a0 * (double)U.u0[i].x + ea.a1 * r.x;
                    r.y = ea.a0 * (double)U.u0[i].y + ea.a1 * r.y;
                    keepv = cvt<TS>(r);
                    buf_store<TS>(ro, keepv, vo, so);
                    bad |= vo >= 0 && !finite2(keepv);
                } else if constexpr (MODE == EPI_INC || MODE == EPI_INC_FINAL) {
                    cplx<double> base = w;
                    if constexpr (MODE == EPI_INC_FINAL) base = base + cvt<double>(U.lo[i]);
                    const cplx<double> d = cvt<double>(U.u0[i]);
                    const double Gd = k2 * ea.dtnu;
                    r.x = ea.a1 * (d.x + (R.x - Gd * (base.x + d.x) + ea.dt * U.f[i].x));
                    r.y = ea.a1 * (d.y + (R.y - Gd * (base.y + d.y) + ea.dt * U.f[i].y));
                    if constexpr (MODE == EPI_INC) {
                        keepv = cvt<TS>(r);
                        buf_store<TS>(ro, keepv, vo, so);
                        bad |= vo >= 0 && !finite2(keepv);
                    } else {
                        r = r + base;
                        keepv = cvt<TS>(r);
                        buf_store<TS>(ro, keepv, vo, so);
                        buf_store<float>(rsrc_of(ea.out32[b], 0, ea.mw, es),
                                         mk<float>((float)(r.x - (double)keepv.x), (float)(r.y - (double)keepv.y)), vo, so);
                        bad |= vo >= 0 && !finite2(r);
                    }
                } else if constexpr (MODE == EPI_RHS || MODE == EPI_UV_RHS) {
                    const double G = -k2 * ea.nu;
                    r.x = R.x + G * w.x;
                    r.y = R.y + G * w.y;
                    if constexpr (MODE == EPI_RHS) r = r + U.f[i];
                    buf_store<double>(ro, r, vo, so);
                    bad |= vo >= 0 && !finite2(r);
                } else if constexpr (MODE == EPI_UV_VEC) {
                    const double G = -k2 * ea.nu;
                    r = mk<double>(R.x + G * w.x, R.y + G * w.y);
                    const int vv = voff_vec(j, q);
                    buf_store_f64(rsrc_vec(ea.vout, b), ea.shift != 0.0 ? r.y - ea.shift * w.y : r.y, vv, jo * Ny * Mz * 8);
                    bad |= vo >= 0 && !finite2(r);
                } else if constexpr (MODE == EPI_UV) {
                    const double G = 1.0 - k2 * ea.dtnu;
                    r = mk<double>(R.x + G * w.x, R.y + G * w.y);
                    buf_store<double>(ro, r, vo, so);
                    bad |= vo >= 0 && !finite2(r);
                } else {  // EPI_IUV
                    const double G = 1.0 + k2 * ea.dtnu;
                    r = mk<double>((w.x + R.x) / G, (w.y + R.y) / G);
                    buf_store<double>(ro, r, vo, so);
                    bad |= vo >= 0 && !finite2(r);
                }
                if constexpr (CHAIN) {
                    cplx<double> s = cvt<double>(keepv);
                    if constexpr (MODE == EPI_INC) s = w + s;   // base + increment
                    if (!(kept >> e & 1u)) s = mk<double>(0.0, 0.0);
                    cv[e] = cvt<TB>(s);
                    cd[e] = ikx<TB>(s, kx);
                }
            }
        }
        if constexpr (CHAIN && u % UPC == UPC - 1) {
            if (chained) chain(b, cv, cd);
        }
    });
    flag_nonfinite(ea.nf, bad);
}

// Pointwise epilogue from stored Q^ (the standalone solve_advection_diffusion_projection*).
template <int MODE>
__global__ void __launch_bounds__(256)
k_update(const cplx<double>* __restrict__ Qx, const cplx<double>* __restrict__ Qy, const cplx<double>* __restrict__ Qz,
         long nc, int Ny, int Mz, SpecTables tab, EpiArgs ea) {
    const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= nc) return;
    const int l = (int)(g % Mz);
    const long t1 = g / Mz;
    const int k = (int)(t1 % Ny), j = (int)(t1 / Ny);
    epilogue<MODE>(ea, tab, j, k, l, Qx[g], Qy[g], Qz[g]);
}

// ---------------------------------------------------------------- z C2R / R2C (single fields)
// Two neighbouring (x,y) pencils share one complex FFT: Y = X_p0 + i X_p1.
template <typename TB, int NZ, int P>
__global__ void __launch_bounds__((P * ZTPP<TB, NZ>))
k_z_c2r(const cplx<TB>* __restrict__ in, TB* __restrict__ out, long npairs, int Mz, int nb, SpecTables tab,
        const cplx<TB>* __restrict__ twg, TB scale) {
    using Z = ZPencil<TB, NZ, P>;
    constexpr int TPP = Z::TPP;
    __shared__ cplx<TB> lds[P * (NZ + Z::PAD)];
    __shared__ cplx<TB> tw[NZ];
    const int bid = xcd_tile();
    if (bid >= nb) return;
    stage_twiddles<TB, NZ>(tw, twg);
    const int tid = threadIdx.x;
    int t, p;
    Z::lanes(tid, t, p);
    const long pair = (long)bid * P + p;
    const bool valid = pair < npairs;
    const long p0 = valid ? 2 * pair : 0, p1 = p0 + 1;
    TB x1[Z::NPT], x2[Z::NPT];
    Z::c2r_pair(x1, x2, in + p0 * Mz, false, in + p1 * Mz, false, valid, tab, lds, tw, t, p, scale);
    if (!valid) return;
#pragma unroll
    for (int q = 0; q < Z::FI::BL; q++) {
        if (!Z::FI::out_active(t, q)) continue;
#pragma unroll
        for (int r = 0; r < Z::FI::RL; r++) {
            const int n = Z::FI::out_index(t, q, r);
            out[p0 * NZ + n] = x1[q * Z::FI::RL + r];
            out[p1 * NZ + n] = x2[q * Z::FI::RL + r];
        }
    }
}

template <typename TB, int NZ, int P>
__global__ void __launch_bounds__((P * ZTPP<TB, NZ>))
k_z_r2c(const TB* __restrict__ in, cplx<TB>* __restrict__ out, long npairs, int Mz, int nb,
        const cplx<TB>* __restrict__ twg) {
    using Z = ZPencil<TB, NZ, P>;
    constexpr int TPP = Z::TPP;
    __shared__ cplx<TB> lds[P * (NZ + Z::PAD)];
    __shared__ cplx<TB> tw[NZ];
    const int bid = xcd_tile();
    if (bid >= nb) return;
    stage_twiddles<TB, NZ>(tw, twg);
    const int tid = threadIdx.x;
    int t, p;
    Z::lanes(tid, t, p);
    const long pair = (long)bid * P + p;
    const bool valid = pair < npairs;
    const long p0 = valid ? 2 * pair : 0, p1 = p0 + 1;
    TB q1[Z::NPT], q2[Z::NPT];
#pragma unroll
    for (int q = 0; q < Z::FF::B0; q++) {
#pragma unroll
        for (int r = 0; r < Z::FF::R0; r++) {
            const int n = Z::FF::in_index(t, q, r);
            const bool on = valid && Z::FF::in_active(t, q);
            q1[q * Z::FF::R0 + r] = on ? in[p0 * NZ + n] : (TB)0;
            q2[q * Z::FF::R0 + r] = on ? in[p1 * NZ + n] : (TB)0;
        }
    }
    Z::r2c_pair(q1, q2, out + p0 * Mz, out + p1 * Mz, valid, lds, tw, t, p);
}

}  // namespace ns3d
