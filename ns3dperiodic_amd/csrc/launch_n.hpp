// launch_n.hpp -- definitions of the launches declared in launch.hpp.  Scratch fields have
// rows padded to mi_of(c) (128-B aligned pencil tiles), nci modes each: region A (6 fields
// per vector field), then region B (9).
#pragma once
#include "launch.hpp"

template <typename TB, typename TS, int NX>
int launch_x_inv(ns3d_ctx* c, const cplx<TS>* const* in, const cplx<TS>* const* in2, int nf, int mw, long bin,
                 const double* vec) {
    const int nz = c->batch, Mi = mi_of(c);
    const long nc = c->nci, bsc = c->bsc;
    cplx<TB>* A = (cplx<TB>*)c->scratch;
    hipStream_t s = c->stream;
    constexpr int E = E_XINV<TB, NX>;
    constexpr int P = PXY_T<TB, NX, E, NS3D_PXINV32, NS3D_BY_RADIX(NX, NS3D_PXINV64, NS3D_R3_PXINV64)>;
    const int nlt = (c->Mz + P - 1) / P;
    const int nb = c->Ny * nlt;
    constexpr int OS = NS3D_OS_XINV;
    dim3 grid = xgrid(nb, 3 * nf * (OS ? 2 : 1), nz), blk(P * XYPlan<NX, E>::TPP);
    if (nf == 1 && in2) {
        if constexpr (std::is_same<TS, float>::value) {
            PtrArr<const cplx<TS>, 3> w{{in[0], in[1], in[2]}};
            PtrArr<const cplx<TS>, 3> w2{{in2[0], in2[1], in2[2]}};
            hipLaunchKernelGGL((k_x_inv_grad<TB, NX, P, 1, E, OS, TS, 1>), grid, blk, 0, s, w, A, nc, c->Ny, c->Mz, mw, Mi, nlt, nb, c->tab,
                               twp<TB>(c, 0), nt_for<TB>(c, P, FIELDS_P1 * nf), bin, bsc, c->mm, w2);
        } else {
            return NS3D_ERR_ARG;
        }
    } else if (nf == 1) {
        PtrArr<const cplx<TS>, 3> w{{in[0], in[1], in[2]}};
        hipLaunchKernelGGL((k_x_inv_grad<TB, NX, P, 1, E, OS, TS>), grid, blk, 0, s, w, A, nc, c->Ny, c->Mz, mw, Mi, nlt, nb, c->tab,
                           twp<TB>(c, 0), nt_for<TB>(c, P, FIELDS_P1 * nf), bin, bsc, c->mm);
    } else if constexpr (std::is_same<TS, double>::value) {
        PtrArr<const zd, 6> w{{in[0], in[1], in[2], in[3], in[4], in[5]}};
        if (vec)
            hipLaunchKernelGGL((k_x_inv_grad<TB, NX, P, 2, E, OS, double, 0, 1>), grid, blk, 0, s, w, A, nc, c->Ny, c->Mz, c->Mz, Mi,
                               nlt, nb, c->tab, twp<TB>(c, 0), nt_for<TB>(c, P, FIELDS_P1 * nf), 0L, bsc, c->mm,
                               PtrArr<const zd, 3>{}, vec);
        else
            hipLaunchKernelGGL((k_x_inv_grad<TB, NX, P, 2, E, OS>), grid, blk, 0, s, w, A, nc, c->Ny, c->Mz, mw, Mi, nlt, nb, c->tab,
                               twp<TB>(c, 0), nt_for<TB>(c, P, FIELDS_P1 * nf), bin, bsc, c->mm);
    } else {
        return NS3D_ERR_ARG;
    }
    return NS3D_OK;
}

template <typename TB, int NY>
int launch_y_inv(ns3d_ctx* c, int nf) {
    const int nz = c->batch, Mi = mi_of(c);
    const long nc = c->nci, bsc = c->bsc;
    cplx<TB>* A = (cplx<TB>*)c->scratch;
    cplx<TB>* B = A + (long)6 * nf * nc;
    hipStream_t s = c->stream;
    constexpr int E = E_YINV<TB>;
    constexpr int P = PXY_T<TB, NY, E, NS3D_BY_RADIX(NY, NS3D_PYINV32, NS3D_R3_PYINV32),
                            NS3D_BY_RADIX(NY, NS3D_PYINV64, NS3D_R3_PYINV64)>;
    const int nlt = (c->Mz + P - 1) / P;
    const int nb = c->Nx * nlt;
    // One output per block (OS) where even three times the blocks leave every wave resident
    // at once, so that a block's latency is the pass's time: FP64 32^3 step 79.6 -> 73.9 us,
    // 48x64x32 111.6 -> 105.9, 96^3 281 -> 267; 128^3 (two rounds) 493 -> 500.  FP32 rounds
    // differently in the two forms and keeps one.
    constexpr int T = P * XYPlan<NY, E>::TPP;
    constexpr long RESIDENT = 5 * 1024;   // waves at 5 to a SIMD
    const long tiles = (long)c->Nx * (c->tab.lmax / P + 1) * c->batch;
    const bool os = sizeof(TB) == 8 && nf == 1 && 9 * tiles * ((T + 63) / 64) <= RESIDENT;
    const dim3 grid = xgrid(nb, 3 * nf, nz), blk(T);
    const int nt = nt_for<TB>(c, P, FIELDS_P2 * nf);
    auto launch = [&](auto kernel, dim3 g) {
        hipLaunchKernelGGL(kernel, g, blk, 0, s, A, B, nc, c->Ny, c->Mz, Mi, nlt, nb, c->tab, twp<TB>(c, 1), nt, bsc, c->mm);
    };
    if (nf == 2) {
        launch(k_y_inv_grad<TB, NY, P, 2, E, 0>, grid);
    } else if constexpr (sizeof(TB) == 8) {
        if (os)
            launch(k_y_inv_grad<TB, NY, P, 1, E, 1>, xgrid(nb, 9, nz));
        else
            launch(k_y_inv_grad<TB, NY, P, 1, E, 0>, grid);
    } else {
        launch(k_y_inv_grad<TB, NY, P, 1, E, 0>, grid);
    }
    return NS3D_OK;
}

// C2R, product, R2C -> C at A
template <typename TB, int NZ>
int launch_z(ns3d_ctx* c, int nf) {
    const int nz = c->batch, Mi = mi_of(c);
    const long nc = c->nci, bsc = c->bsc;
    cplx<TB>* A = (cplx<TB>*)c->scratch;
    cplx<TB>* B = A + (long)6 * nf * nc;
    hipStream_t s = c->stream;
    constexpr int P = PZ<TB, NZ>;
    const int nb = (int)nblk(c->npen, P);
    dim3 grid = xgrid(nb, 1, nz), blk(P * ZTPP<TB, NZ>);
    const TB scale = (TB)(1.0 / (1.0 * c->Nx * c->Ny * c->Nz));
    TB* up = nf == 1 ? (TB*)c->uphys_out : nullptr;
    if (nf == 1)
        hipLaunchKernelGGL((k_z_product<TB, NZ, P, 1>), grid, blk, 0, s, B, A, nc, c->npen, Mi, nb, c->tab, twp<TB>(c, 2), scale,
                           up, c->nr, nt_for<TB>(c, 128, sizeof(TB) == 8 ? FIELDS_P34 : 0.0), bsc, c->mm);
    else
        hipLaunchKernelGGL((k_z_product<TB, NZ, P, 2>), grid, blk, 0, s, B, A, nc, c->npen, Mi, nb, c->tab, twp<TB>(c, 2), scale,
                           (TB*)nullptr, c->nr, nt_for<TB>(c, 128, sizeof(TB) == 8 ? FIELDS_P34 : 0.0), bsc, c->mm);
    return NS3D_OK;
}

template <typename TB, int NY>
int launch_y_fwd(ns3d_ctx* c, int nf, bool chain) {
    const int nz = c->batch, Mi = mi_of(c);
    const long nc = c->nci, bsc = c->bsc;
    cplx<TB>* A = (cplx<TB>*)c->scratch;
    hipStream_t s = c->stream;
    constexpr int E = E_C2C<TB>;
    constexpr int P = PXY_T<TB, NY, E, NS3D_PYFWD32, 8>;
    const int nlt = (c->Mz + P - 1) / P;
    const int nb = c->Nx * nlt;
    dim3 grid = xgrid(nb, 3, nz), blk(P * XYPlan<NY, E>::TPP);
    hipLaunchKernelGGL((k_axis_c2c<TB, NY, P, -1, 1, E>), grid, blk, 0, s, A, d_at<TB>(c, nf, chain), 3, nc, c->Ny, c->Mz, Mi, nlt, nb,
                       twp<TB>(c, 1), nt_for<TB>(c, P, FIELDS_P34), bsc, c->mm);
    return NS3D_OK;
}

template <typename TB, int MODE, int NX>
int launch_x_fwd(ns3d_ctx* c, const EpiArgs& ea, int nf, bool chain) {
    cplx<TB>* A = (cplx<TB>*)c->scratch;
    const cplx<TB>* D = d_at<TB>(c, nf, chain);
    constexpr int E = E_XFWD<TB, NX>;
    constexpr int P0 = sizeof(TB) == 8 ? 8 : NS3D_BY_RADIX(NX, NS3D_PXFWD32, NS3D_R3_PXFWD32);
    constexpr int P = PXY_T<TB, NX, E, P0, P0>;
    const int nlt = (c->Mz + P - 1) / P;
    const int nb = c->Ny * nlt;
    dim3 grid = xgrid(nb, 1, c->batch), blk(P * XYPlan<NX, E>::TPP);
    auto launch = [&](auto CH) {
        hipLaunchKernelGGL((k_x_fwd_epi<TB, NX, P, MODE, E, decltype(CH)::value, E_XINV<TB, NX>>), grid, blk, 0, c->stream, D, A,
                           c->nci, c->Ny, c->Mz, mi_of(c), nlt, nb, c->tab, twp<TB>(c, 0), ea, nt_for<TB>(c, P, FIELDS_P1 * nf), c->bsc, c->mm);
    };
    constexpr bool CAN = CHAINS<TB, NX, MODE> && (MODE == EPI_STAGE || MODE == EPI_STAGE32 || MODE == EPI_INC || MODE == EPI_INC_FINAL);
    if constexpr (CAN) {
        if (chain) launch(std::integral_constant<int, 1>{});
        else launch(std::integral_constant<int, 0>{});
    } else {
        if (chain) return NS3D_ERR_ARG;
        launch(std::integral_constant<int, 0>{});
    }
    return NS3D_OK;
}

template <typename TB, int N, int DIR, int AXIS>
int launch_c2c_as(ns3d_ctx* c, const cplx<TB>* in, cplx<TB>* out) {
    constexpr int E = E_C2C<TB>;
    constexpr int P = PXY<TB, N, E>;
    const int nlt = (c->Mz + P - 1) / P, nb = (AXIS == 0 ? c->Ny : c->Nx) * nlt;
    hipLaunchKernelGGL((k_axis_c2c<TB, N, P, DIR, AXIS, E>), xgrid(nb), dim3(P * XYPlan<N, E>::TPP), 0, c->stream, in, out, 1,
                       c->nc, c->Ny, c->Mz, c->Mz, nlt, nb, twp<TB>(c, AXIS));
    return NS3D_OK;
}
template <typename TB, int N>
int launch_c2c(ns3d_ctx* c, int dir, int axis, const cplx<TB>* in, cplx<TB>* out) {
    if (dir > 0) return axis == 0 ? launch_c2c_as<TB, N, +1, 0>(c, in, out) : launch_c2c_as<TB, N, +1, 1>(c, in, out);
    return axis == 0 ? launch_c2c_as<TB, N, -1, 0>(c, in, out) : launch_c2c_as<TB, N, -1, 1>(c, in, out);
}

template <typename TB, int NZ>
int launch_c2r(ns3d_ctx* c, const cplx<TB>* in, TB* out, bool scale) {
    constexpr int P = PZ<TB, NZ>;
    const long npairs = c->npen / 2;
    const TB sc = scale ? (TB)(1.0 / (1.0 * c->Nx * c->Ny * c->Nz)) : (TB)1;
    const int nb = (int)nblk(npairs, P);
    hipLaunchKernelGGL((k_z_c2r<TB, NZ, P>), xgrid(nb), dim3(P * ZTPP<TB, NZ>), 0, c->stream, in, out, npairs, c->Mz, nb,
                       c->tab, twp<TB>(c, 2), sc);
    return NS3D_OK;
}

template <typename TB, int NZ>
int launch_r2c(ns3d_ctx* c, const TB* in, cplx<TB>* out) {
    constexpr int P = PZ<TB, NZ>;
    const long npairs = c->npen / 2;
    const int nb = (int)nblk(npairs, P);
    hipLaunchKernelGGL((k_z_r2c<TB, NZ, P>), xgrid(nb), dim3(P * ZTPP<TB, NZ>), 0, c->stream, in, out, npairs, c->Mz, nb,
                       twp<TB>(c, 2));
    return NS3D_OK;
}
