// launch.hpp -- the context, the tile shapes of the pencil kernels and the launches of
// each grid length.  The launches are templates on the length, defined in launch_n.hpp
// and instantiated length by length in ns3d_len.hip (one translation unit per group of
// lengths, so they build in parallel); ns3d_api.hip only calls them.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>
#include <vector>

#include "../../include/ns3d.h"
// tile shapes and plans chosen by ns3dperiodic_amd/autotune.py; the #ifndef
// defaults in the kernel headers apply to whatever it does not set
#if !defined(NS3D_NO_TUNED_HEADER) && __has_include("tuned.hpp")
#include "tuned.hpp"
#endif
#include "k_fused.hpp"

using namespace ns3d;

typedef cplx<double> zd;

// pencils per block in the x/y passes: rows of 128 B
#ifndef NS3D_PXY32
#define NS3D_PXY32 16
#endif
template <typename TB> constexpr int PXY0 = sizeof(TB) == 8 ? 8 : NS3D_PXY32;
// Blocks are capped at NS3D_XY_MAXT threads: 1024-thread blocks, which fill
// a CU's 16 waves with one block, lose to 512 (measured at 256^3 and 512^3).
#ifndef NS3D_XY_MAXT
#define NS3D_XY_MAXT 512
#endif
template <typename TB, int N, int E>
constexpr int PXY = PXY0<TB> * XYPlan<N, E>::TPP <= NS3D_XY_MAXT ? PXY0<TB>
                                                                 : (NS3D_XY_MAXT / XYPlan<N, E>::TPP > 0 ? NS3D_XY_MAXT / XYPlan<N, E>::TPP : 1);
// Pencils per block of each fused x/y pass, by precision.
#ifndef NS3D_PXINV32
#define NS3D_PXINV32 8
#endif
#ifndef NS3D_PYINV32
#define NS3D_PYINV32 8
#endif
#ifndef NS3D_PYFWD32
#define NS3D_PYFWD32 16
#endif
#ifndef NS3D_PXFWD32
#define NS3D_PXFWD32 8
#endif
#ifndef NS3D_PXINV64
#define NS3D_PXINV64 8
#endif
#ifndef NS3D_PYINV64
#define NS3D_PYINV64 8
#endif
template <typename TB, int N, int E, int P32, int P64>
constexpr int PXY_T = (sizeof(TB) == 8 ? P64 : P32) * XYPlan<N, E>::TPP <= NS3D_XY_MAXT
                          ? (sizeof(TB) == 8 ? P64 : P32)
                          : (NS3D_XY_MAXT / XYPlan<N, E>::TPP > 0 ? NS3D_XY_MAXT / XYPlan<N, E>::TPP : 1);
// Points per thread of each x/y pass, by precision (measured at 256^3 on MI355X):
// FP64 favours 4 points in the inverse passes, 8 in the forward ones; FP32 the mix below.
#ifndef NS3D_EYINV32
#define NS3D_EYINV32 4
#endif
#ifndef NS3D_EYINV64
#define NS3D_EYINV64 4
#endif
// x-inverse, FP64: 8 points from 384 up, where 4-point blocks of 512 threads hold 5 or 4
// pencils and a row segment no longer fills a 128-B line (384^3 0.973 -> 0.905 ms, 512^3
// 1.86 -> 1.53 ms); not at 320, whose 8-point plan leaves lanes idle in its radix-5 pass
// (0.468 -> 0.712 ms).  The y-inverse pass keeps 4 points (8: 512^3 2.56 -> 2.83-3.10 ms).
template <typename TB, int N>
constexpr int E_XINV = sizeof(TB) == 8 ? (N > 320 ? 8 : 4) : 8;
template <typename TB> constexpr int E_YINV = sizeof(TB) == 8 ? NS3D_EYINV64 : NS3D_EYINV32;
template <typename TB> constexpr int E_C2C = 8;
// 4 points per thread at most up to 256: above, 4-point blocks of 8 pencils would pass
// NS3D_XY_MAXT threads and FP64 tiles would fall below a 128-B line.
template <typename TB, int N> constexpr int E_XFWD = sizeof(TB) == 8 ? (N > 256 ? 8 : 4) : 4;
// one output field per block in the inverse passes (input re-read by 2 or 3 blocks)
#ifndef NS3D_OS_XINV
#define NS3D_OS_XINV 0
#endif
// pencils per block in the z pass: ~128 threads (FP32: NS3D_PZT32)
#ifndef NS3D_PZT32
#define NS3D_PZT32 128
#endif
// (measured: smaller blocks beat whole-wavefront ones, e.g. 96 vs 192 threads at 192^3)
#ifndef NS3D_PZT64
#define NS3D_PZT64 128
#endif
// (FP64 192^3 z pass: 256 threads 0.178 ms, 128 0.187; swizzle groups of 0 / 8 / 16: 0.178 / 0.188 / 0.188)
// Radix-3 lengths from 192 up have their own block shapes (NS3D_R3_*, and
// NS3D_R3_ZSWZ in the z pass), swept at 192^3 (FP64 366 -> 419, FP32 680 ->
// 700, FP32 state 725 -> 768 steps/s); at 48 and 96 these shapes were slower
// than the ones above (swept at 256^3), which those lengths keep.
#ifndef NS3D_R3_PXINV64
#define NS3D_R3_PXINV64 4
#endif
#ifndef NS3D_R3_PYINV64
#define NS3D_R3_PYINV64 4
#endif
#ifndef NS3D_R3_PZT64
#define NS3D_R3_PZT64 256
#endif
#ifndef NS3D_R3_PXFWD32
#define NS3D_R3_PXFWD32 16
#endif
#ifndef NS3D_R3_PYINV32
#define NS3D_R3_PYINV32 4
#endif
#define NS3D_BY_RADIX(N, A, R3) ((N) % 3 == 0 && (N) >= 192 ? (R3) : (A))
template <typename TB, int N>
constexpr int PZT = sizeof(TB) == 8 ? NS3D_BY_RADIX(N, NS3D_PZT64, NS3D_R3_PZT64) : NS3D_PZT32;
template <typename TB, int N>
constexpr int PZ = (PZT<TB, N> / ZTPP<TB, N>) > 0 ? (PZT<TB, N> / ZTPP<TB, N>) : 1;

struct ns3d_ctx {
    int Nx, Ny, Nz, Mz;
    long nc, nr, npen;
    long nci;  // modes per scratch field of the fused passes (rows padded from Mz to mi_of(c))
    int m8, m16;     // Mz rounded up to a multiple of NS3D_ROWPAD64 / NS3D_ROWPAD32 (FP64 / FP32 rows)
    long nc8, nc16;  // Nx*Ny*m8, Nx*Ny*m16
    double Lx, Ly, Lz, Re, dt;
    int precision;
    unsigned flags;
    hipStream_t stream;
    int device;
    int last_error;
    // device tables
    double* dtab = nullptr;
    SpecTables tab;
    void* tw64[3] = {nullptr, nullptr, nullptr};  // x, y, z twiddles (double)
    void* tw32[3] = {nullptr, nullptr, nullptr};  // (float)
    // bulk scratch (A|B regions) in bulk precision; capacity in fields
    void* scratch = nullptr;
    int scratch_fields = 0;
    // incremented whenever a buffer that a captured RK3 step addresses is reallocated
    long long generation = 0;
    // FP64 stage buffers and a Q^ buffer
    zd* stage = nullptr;  // 9 fields: u1[3], u2[3], q[3]
    zd* extra = nullptr;  // 6 fields: tangent map v1[3] + spare
    cplx<float>* s32 = nullptr;  // NS3D_FP32_STATE RK3 loop: state[3], u1[3], u2[3] in FP32
    double* red = nullptr;  // reduction partials (2*RED_BLOCKS + 2)
    double* red_host = nullptr;  // pinned
    void* real_scratch = nullptr;  // physical-space scratch (FP64 or FP32), 4 fields
    // registered base flow for the Krylov callbacks
    zd* base[3] = {nullptr, nullptr, nullptr};
    const zd* bforce[3] = {nullptr, nullptr, nullptr};
    int timesteps_period = 1;
    double tau = 1.0;
    zd* kry = nullptr;  // 3 fields for J.v unpacking
    // Krylov vector kernels: reduction partials, results, pinned host copies, small dense matrix
    double* kv_partial = nullptr;
    double* kv_out = nullptr;
    double* kv_host = nullptr;
    double* kq = nullptr;
    double* kq_host = nullptr;
    // a captured graph of nsteps RK3 steps for fixed state/forcing pointers, dt and Re
    hipGraph_t graph = nullptr;
    hipGraphExec_t graph_exec = nullptr;
    const void* graph_key[6] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    int graph_steps = -1;
    double graph_dt = 0.0, graph_Re = 0.0;
    // passive scalar: physical velocity written by the z pass (bulk precision, 3 real fields)
    void* uphys = nullptr;
    void* uphys_out = nullptr;  // non-null only while a scalar step wants it
    double* theta_stage = nullptr;  // 2 real FP64 fields
    // batches of same-size fields advanced by one set of launches (grid.z = member):
    // members in flight, scratch stride per member (elements), stage buffers per member
    int batch = 1;
    long bsc = 0;
    zd* bstage = nullptr;  // batch members' u1[3], u2[3]: 6 fields of nc8 each per member
    int bstage_members = 0;
    // members sitting out steps, and per-member dt / Re (ns3d_rk3_ssp_batch_members)
    MemberMask mm = {nullptr, 0};
    const double* mdt = nullptr;
    const double* mre = nullptr;
    // graph of ns3d_rk3_ssp_batch_members for fixed pointers, nbatch and nsteps
    hipGraph_t mgraph = nullptr;
    hipGraphExec_t mgraph_exec = nullptr;
    const void* mgraph_key[8] = {};
    int mgraph_nb = -1, mgraph_steps = -1;
    // optional per-pass timing with HIP events on the context stream
    bool prof_on = false;
    std::vector<hipEvent_t> ev_pool;
    std::vector<std::pair<int, int>> ev_used;  // (pass id, index of start event; stop = +1)
    hipEvent_t ev_open = nullptr;
    int ev_open_pass = -1;
    // sticky non-finite flag written by the fused epilogues and the scalar stage
    int* nf = nullptr;
    int* nf_host = nullptr;  // pinned
    // batched probe: partial sums and results (device), results (pinned host)
    double* pb = nullptr;
    double* pb_host = nullptr;
    size_t pb_cap = 0;
};

template <typename TB> const cplx<TB>* twp(const ns3d_ctx* c, int axis) {
    return (const cplx<TB>*)(sizeof(TB) == 8 ? c->tw64[axis] : c->tw32[axis]);
}

inline size_t bulk_bytes(const ns3d_ctx* c) { return c->precision == NS3D_FP64 ? sizeof(zd) : sizeof(cplx<float>); }

// Row stride of the fused passes' scratch fields: Mz rounded up so that every
// P-mode row tile of the x/y passes (128 B) starts on a 128-B line.
#ifndef NS3D_PAD_ROWS
#define NS3D_PAD_ROWS 1
#endif
// Row padding (modes) of the library's own FP64 and FP32 fields: 8 modes, so
// FP64 rows start on 128-B and FP32 rows on 64-B boundaries, which the x and y
// tiles' 8-mode segments need.  256^3, rows of 136 against 144: FP32 steps
// -1.0% (bulk), -1.8% (state), -2.1% (increments), chiefly the x-forward pass
// (-4%: x-planes 136*256 modes apart map onto HBM better than 144*256); FP64
// rows of 144 gained only 0.4% for 6% more memory.
#ifndef NS3D_ROWPAD64
#define NS3D_ROWPAD64 8
#endif
#ifndef NS3D_ROWPAD32
#define NS3D_ROWPAD32 8
#endif
inline int mi_of(const ns3d_ctx* c) {
    const int a = NS3D_PAD_ROWS ? (c->precision == NS3D_FP64 ? NS3D_ROWPAD64 : NS3D_ROWPAD32) : 1;
    return (c->Mz + a - 1) / a * a;
}

inline unsigned nblk(long n, int t) { return (unsigned)((n + t - 1) / t); }
// grid for the XCD-remapped pencil kernels: block count padded to a multiple of 8
inline dim3 xgrid(long nb, int nfy = 1, int nz = 1) {
    return dim3((unsigned)(((nb + 7) / 8) * 8), (unsigned)nfy, (unsigned)nz);
}

// Whether the x-forward pass carries the next stage's P1 (k_x_fwd_epi<..., CHAIN = 1>).
// FP64 up to 256 points in x: above, its operands and the two inverse transforms pass 256
// VGPRs (512^3: 4.10 ms chained against 1.51 + 2.62 ms apart).  FP32: not at radix-5 lengths,
// whose 5-point butterfly is not pinned there; at 512, where a row segment is 32 B, not over the
// FP64 state (five steps chained and apart: FP32 bulk 512x256x256 34.9 and 33.9 ms, 512^3 135.0
// and 131.7; the increments 512x256x256 30.5 and 31.2; the FP32 state 512x64x64 1.58 and 1.66,
// 512^3 106.0 and 106.8, with forcing 119.4 and 118.2).
template <typename TB, int NX, int MODE>
constexpr bool CHAINS = sizeof(TB) == 8 ? MIRROR_P1<TB, NX>
                                          : NX % 5 != 0 && (NX < 512 || MODE != EPI_STAGE);

// D of nf fields.  Where the x-forward pass writes the next stage's P1 output over A
// (chain), D is at the head of region B; else behind C in A, on memory the z pass has not
// just read.  One stage or right-hand side in FP32, D in B against D in A: 96x192x48 80.1
// and 77.8 us, 64x512x64 145.6 and 141.0, 512x64x64 159.1 and 153.0, 128^3 125.1 and 120.6;
// in FP64 and at 192^3 and above within 1%.
template <typename TB> cplx<TB>* d_at(const ns3d_ctx* c, int nf, bool chain) {
    return (cplx<TB>*)c->scratch + (chain ? 6 * nf : 3) * c->nci;
}

// Nontemporal stores of a pass's output, written in full 128-B lines (P modes to a row segment),
// where the next pass does not find it in the 256 MiB Infinity Cache anyway: FP64 from 256 MiB of
// output, FP32 from 128 MiB.  FP64 at 256^3: the pass that reads it next is 4-9% faster (step 4.10
// -> 3.87 ms); smaller outputs are read back from the cache and lose by it (192^3 y-inverse 0.175
// -> 0.195 ms, 128^3 pencil copies 0.022 -> 0.029), and so do partial lines (512^3 y-inverse, 64-B
// segments, 2.56 -> 2.91 ms; 320^3 FP32 y-forward, 96-B segments, 0.155 -> 0.276 ms).  In FP32 only
// the y-forward pass up to 256 points in y fills lines; its reader brings the FP64 state and mostly
// six more fields of A through the cache, so its output is lost to it from half the size on.  Five
// steps without and with, outputs between the two lines: 256^3 15.24 and 15.00 ms (FP32 state 13.27
// and 12.93, increments 13.88 and 13.57), 192x256x256 11.54 and 11.33, 256x192x256 12.02 and 11.81,
// 256x256x320 20.58 and 20.37, 320x256x256 21.66 and 21.42, a step of 16 x 96^3 2.93 and 2.86; above
// both, 384x256x256 26.33 and 26.12, 256x256x512 30.0 and 29.8, 512x256x256 34.31 and 34.23.  (Every
// other segment of FP32 rows of 136 modes starts in the middle of a line; it pays all the same.)
template <typename TB> int nt_for(const ns3d_ctx* c, int P, double fields) {
    return P * sizeof(cplx<TB>) >= 128 &&
           fields * (double)c->nci * c->batch * sizeof(cplx<TB>) > (sizeof(TB) == 8 ? 256.0 : 128.0) * (1 << 20);
}
// fields written: the kept ones of P1's 6 (60% of the columns) and P2's 9 (the planes below the mask's lmax)
constexpr double FIELDS_P1 = 3.6, FIELDS_P2 = 6.0, FIELDS_P34 = 3.0;

// ---------------------------------------------------------------- launches by length
// P1 of nf fields (in2: nf = 1 only, may be null: added to in before the transforms;
// vec: nf = 2 only, may be null: the second vector field as a reduced Krylov vector)
template <typename TB, typename TS, int NX>
int launch_x_inv(ns3d_ctx* c, const cplx<TS>* const* in, const cplx<TS>* const* in2, int nf, int mw, long bin,
                 const double* vec);
template <typename TB, int NY> int launch_y_inv(ns3d_ctx* c, int nf);
template <typename TB, int NZ> int launch_z(ns3d_ctx* c, int nf);
// P4: C (at A) -> D (d_at)
template <typename TB, int NY> int launch_y_fwd(ns3d_ctx* c, int nf, bool chain);
// P5; chain: with the P1 of the next stage (the RK3 loops' modes)
template <typename TB, int MODE, int NX> int launch_x_fwd(ns3d_ctx* c, const EpiArgs& ea, int nf, bool chain);
// standalone transforms of one field in the reference layout
template <typename TB, int N> int launch_c2c(ns3d_ctx* c, int dir, int axis, const cplx<TB>* in, cplx<TB>* out);
template <typename TB, int NZ> int launch_c2r(ns3d_ctx* c, const cplx<TB>* in, TB* out, bool scale);
template <typename TB, int NZ> int launch_r2c(ns3d_ctx* c, const TB* in, cplx<TB>* out);
