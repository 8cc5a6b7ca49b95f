// k_misc.hpp -- precision conversion, pointwise operators, WENO, reductions.
#pragma once
#include "k_fused.hpp"

namespace ns3d {

// ------------------------------------------------------- precision conversion
__global__ void k_d2f_c(const cplx<double>* __restrict__ in, cplx<float>* __restrict__ out, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = cvt<float>(in[i]);
}
__global__ void k_f2d_r(const float* __restrict__ in, double* __restrict__ out, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (double)in[i];
}
__global__ void k_d2f_r(const double* __restrict__ in, float* __restrict__ out, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (float)in[i];
}
__global__ void k_f2d_c(const cplx<float>* __restrict__ in, cplx<double>* __restrict__ out, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = cvt<double>(in[i]);
}
// FP64 field in the reference layout (rows of Mz) <-> FP32 field with rows padded to Mp
__global__ void k_d2f_rows(const cplx<double>* __restrict__ in, cplx<float>* __restrict__ out, long n, int Mz, int Mp) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const long row = i / Mz;
    out[row * Mp + (i - row * Mz)] = cvt<float>(in[i]);
}
__global__ void k_f2d_rows(const cplx<float>* __restrict__ in, cplx<double>* __restrict__ out, long n, int Mz, int Mp) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const long row = i / Mz;
    out[i] = cvt<double>(in[row * Mp + (i - row * Mz)]);
}

// FP64 field in the reference layout <-> the pair (hi, lo) of FP32 fields with
// rows padded to Mp: hi = fp32(u), lo = fp32(u - hi) (u = hi + lo to ~2^-48)
__global__ void k_split_rows(const cplx<double>* __restrict__ in, cplx<float>* __restrict__ hi, cplx<float>* __restrict__ lo,
                             long n, int Mz, int Mp) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const long row = i / Mz, o = row * Mp + (i - row * Mz);
    const cplx<double> u = in[i];
    const cplx<float> h = cvt<float>(u);
    hi[o] = h;
    lo[o] = mk<float>((float)(u.x - (double)h.x), (float)(u.y - (double)h.y));
}
__global__ void k_join_rows(const cplx<float>* __restrict__ hi, const cplx<float>* __restrict__ lo,
                            cplx<double>* __restrict__ out, long n, int Mz, int Mp) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const long row = i / Mz, o = row * Mp + (i - row * Mz);
    const cplx<float> h = hi[o], l = lo[o];
    out[i] = mk<double>((double)h.x + (double)l.x, (double)h.y + (double)l.y);
}

// ------------------------------------------------------- a7: copy / axpby on 3 fields
// single_RK_step_device (Source/RK_time_step.cu:82-115): dst = w0*s0 + w1*s1.
__global__ void __launch_bounds__(256)
k_axpby3(PtrArr<const cplx<double>, 3> s0, double w0, PtrArr<const cplx<double>, 3> s1, double w1,
         PtrArr<cplx<double>, 3> d, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
#pragma unroll
    for (int c = 0; c < 3; c++) {
        const cplx<double> a = s0.p[c][i], b = s1.p[c][i];
        d.p[c][i] = mk<double>(w0 * a.x + w1 * b.x, w0 * a.y + w1 * b.y);
    }
}
// copy_arrays_device (Source/RK_time_step.cu:6-39).
__global__ void __launch_bounds__(256)
k_copy3(PtrArr<const cplx<double>, 3> s, PtrArr<cplx<double>, 3> d, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
#pragma unroll
    for (int c = 0; c < 3; c++) d.p[c][i] = s.p[c][i];
}

// ------------------------------------------------------- a8: divergence
// solve_divergence (Source/divergence.cu:8-30): div^ = i (k . u^) / dt.
__global__ void __launch_bounds__(256)
k_divergence(PtrArr<const cplx<double>, 3> u, cplx<double>* __restrict__ div, long nc, int Ny, int Mz,
             SpecTables tab, double dt) {
    const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= nc) return;
    const int l = (int)(g % Mz);
    const long t1 = g / Mz;
    const int k = (int)(t1 % Ny), j = (int)(t1 / Ny);
    const cplx<double> a = u.p[0][g], b = u.p[1][g], c = u.p[2][g];
    const double kx = tab.kx[j], ky = tab.ky[k], kz = tab.kz[l];
    div[g] = mk<double>((-a.y * kx - b.y * ky - c.y * kz) / dt, (a.x * kx + b.x * ky + c.x * kz) / dt);
}

// ------------------------------------------------------- a10: Krylov packing
// velocities_from_A_vector_reduced_kernel / A_vector_from_velocities_reduced_kernel
// (Source/NS3D_periodic.cu:173-198, 238-250): vec[c*(N-1)+i] <-> Im v^_c[i+1]; v^_c[0] = 0.
__global__ void __launch_bounds__(256)
k_unpack_reduced(const double* __restrict__ vec, PtrArr<cplx<double>, 3> v, long N) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
#pragma unroll
    for (int c = 0; c < 3; c++) v.p[c][i] = mk<double>(0.0, i == 0 ? 0.0 : vec[c * (N - 1) + i - 1]);
}
__global__ void __launch_bounds__(256)
k_pack_reduced(PtrArr<const cplx<double>, 3> v, double* __restrict__ vec, long N) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N - 1) return;
#pragma unroll
    for (int c = 0; c < 3; c++) vec[c * (N - 1) + i] = v.p[c][i + 1].y;
}
// velocities_from_A_vector_kernel / A_vector_from_velocities_kernel (:110-125, :223-236): full length 3N.
__global__ void __launch_bounds__(256)
k_unpack_full(const double* __restrict__ vec, PtrArr<cplx<double>, 3> v, long N) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
#pragma unroll
    for (int c = 0; c < 3; c++) v.p[c][i] = mk<double>(0.0, vec[c * N + i]);
}
__global__ void __launch_bounds__(256)
k_pack_full(PtrArr<const cplx<double>, 3> v, double* __restrict__ vec, long N) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i <= 0 || i >= N) return;  // index 0 is left untouched, as in the reference
#pragma unroll
    for (int c = 0; c < 3; c++) vec[c * N + i] = v.p[c][i].y;
}
// ------------------------------------------------------- a9: WENO advection
// Reference: Source/advection_WENO.cu:47-101 (weno5/weno3), :105-301 (faces), :304-360 (flux).
// A face is one reconstruction, its stencil mirrored to the upwind side, from the
// differences of the scalar along the axis: with f3 the upwind cell's value and e_1..e_4
// the differences outwards, the candidate values are f3 + p_k / 6 and the smoothness
// indicators 13/12 (t_k^2 + 3/13 u_k^2), t and u sums of the e's.  The nonlinear weights
// alpha_k = c_k / (eps + beta_k)^2, here with the common factors taken out, are formed over
// the common denominator prod_k (eps + beta_k)^2, so a face costs one FP64 division
// instead of six; where those products could leave the FP64 range (differences of the
// scalar beyond ~1e33, WENO3 ~1e60) the per-weight form is used.
// Numerators and denominator of one face; FAST: the quotient over the common denominator
// (ok: it and every product of the numerator are in range), else the per-weight form.
// The test of the denominator s covers the numerator: p_k = t_k / 2 +- 3 u_k / 2, so
// |p_k| <= 3.2 sqrt(b_k), and d1 d2 <= s, d0 d2 <= s / 6, d0 d1 <= s / 3 give
// |a_k p_k| <= 4 s^(9/8): under 1e299 for s < 1e265.  WENO3: |a_k e_k| <= s^(5/4), under
// 1e300 for s < 1e240.
template <bool FAST>
__device__ __forceinline__ double weno_increment5(double e1, double e2, double e3, double e4, bool& ok) {
    constexpr double eps = 1.0E-22 * 12.0 / 13.0, g = 3.0 / 13.0;
    const double t0 = e2 - e1, t1 = e3 - e2, t2 = e4 - e3;
    const double u0 = 3.0 * e2 - e1, u1 = e2 + e3, u2 = e4 - 3.0 * e3;
    const double b0 = (t0 * t0 + eps) + g * u0 * u0;
    const double b1 = (t1 * t1 + eps) + g * u1 * u1;
    const double b2 = (t2 * t2 + eps) + g * u2 * u2;
    const double d0 = b0 * b0, d1 = b1 * b1, d2 = b2 * b2;
    const double p0 = 5.0 * e2 - 2.0 * e1, p1 = e2 + 2.0 * e3, p2 = 4.0 * e3 - e4;
    if constexpr (FAST) {
        const double a0 = d1 * d2, a1 = 6.0 * (d0 * d2), a2 = 3.0 * (d0 * d1);
        const double s = a0 + a1 + a2;
        ok = s < 1.0e265 && s > 1.0e-299;
        return (a0 * p0 + a1 * p1 + a2 * p2) / (6.0 * s);
    }
    const double w0 = 1.0 / d0, w1 = 6.0 / d1, w2 = 3.0 / d2, t = 6.0 * (w0 + w1 + w2);
    return w0 / t * p0 + w1 / t * p1 + w2 / t * p2;
}
template <bool FAST>
__device__ __forceinline__ double weno_increment3(double e1, double e2, bool& ok) {
    constexpr double eps = 1.0E-22;
    const double b0 = e1 * e1 + eps, b1 = e2 * e2 + eps;
    const double d0 = b0 * b0, d1 = b1 * b1;
    if constexpr (FAST) {
        const double a0 = d1, a1 = 2.0 * d0, s = a0 + a1;
        ok = s < 1.0e240 && s > 1.0e-299;
        return (a0 * e1 + a1 * e2) / (2.0 * s);
    }
    const double w0 = 1.0 / d0, w1 = 2.0 / d1, t = 2.0 * (w0 + w1);
    return w0 / t * e1 + w1 / t * e2;
}

struct Grid3 {
    int Nx, Ny, Nz;
    __device__ __forceinline__ long at(int j, int k, int l) const {
        j = j >= Nx ? j - Nx : (j < 0 ? j + Nx : j);
        k = k >= Ny ? k - Ny : (k < 0 ? k + Ny : k);
        l = l >= Nz ? l - Nz : (l < 0 ? l + Nz : l);
        return ((long)j * Ny + k) * Nz + l;
    }
};

__device__ __forceinline__ int wrap_add(int i, int o, int n) {
    const int v = i + o;
    return v < 0 ? v + n : (v >= n ? v - n : v);
}

// The face between two cells along one axis, upwinded by the face velocity U:
// flux_{x,y,z}_weno_{L,R} (Source/advection_WENO.cu:105-301).  w[o], o = 1-R..R, is the
// scalar around the lower cell (R = 3 for WENO5, 2 for WENO3, 1 for the first-order
// scheme).  The upper cell's lower face is this same expression, so a face is evaluated
// once.  q9: the z right-biased reconstruction reads offset -1 where -2 belongs
// (Source/advection_WENO.cu:288), i.e. its last difference is zero.
template <int SCHEME, bool FAST>
__device__ __forceinline__ double weno_face(const double* w, double U, bool q9, bool& ok) {
    const bool lo = U >= 0.0;
    const double f = lo ? w[0] : w[1];
    if constexpr (SCHEME == 5) {
        const double m1 = w[0] - w[-1], p1 = w[2] - w[1];
        const double r = weno_increment5<FAST>(lo ? w[-1] - w[-2] : w[3] - w[2], lo ? m1 : p1, w[1] - w[0],
                                               lo ? p1 : (q9 ? 0.0 : m1), ok);
        return lo ? f + r : f - r;
    } else if constexpr (SCHEME == 3) {
        const double r = weno_increment3<FAST>(lo ? w[0] - w[-1] : w[2] - w[1], w[1] - w[0], ok);
        return lo ? f + r : f - r;
    }
    ok = true;
    return f;
}
// N faces, face n of window w + n * stride: the quotients of all of them are independent
// chains, with one branch behind them for those out of range.
template <int SCHEME, int N>
__device__ __forceinline__ void weno_faces(const double* w, int stride, const double* U, bool q9, double* f) {
    bool ok[N], all = true;
#pragma unroll
    for (int n = 0; n < N; n++) {
        f[n] = weno_face<SCHEME, true>(w + n * stride, U[n], q9, ok[n]);
        all = all && ok[n];
    }
    if (SCHEME && !all) {
#pragma unroll
        for (int n = 0; n < N; n++) {
            bool o;
            if (!ok[n]) f[n] = weno_face<SCHEME, false>(w + n * stride, U[n], q9, o);
        }
    }
}

// (u.grad) x with upwind WENO faces chosen by the sign of the face-averaged velocity:
// flux_device + advection (Source/advection_WENO.cu:304-392); out(id, x, adv) per cell.
// VALU bound in WENO5, so each face is evaluated once: a block covers whole z rows and
// marches over `march` x planes; the x face of the step before stays in registers with the
// x window, a thread's YC cells share their y faces, and the z face goes to the upper
// neighbour through LDS (the row is in the block, so no face is left over), as does the
// next plane's row, which is in the x window already.  Six faces a cell, each thread one
// point: WENO5 at 256^3 426 us, 128^3 52.6; this form 225 and 33.5 (y faces evaluated per
// thread, rows read from memory: 246 and 37); first order 235 and 168 us at 256^3.
constexpr int WENO_THREADS = 512;   // a block: whole rows, at most one of the longest
template <int SCHEME, int YC, typename TU, class OUT>
__device__ __forceinline__ void weno_march(const TU* __restrict__ ux, const TU* __restrict__ uy,
                                           const TU* __restrict__ uz, const double* __restrict__ x, const Grid3& G,
                                           int march, double rdx, double rdy, double rdz, bool q9, OUT&& out) {
    constexpr int R = SCHEME == 5 ? 3 : (SCHEME == 3 ? 2 : 1);
    constexpr int W = 2 * R;
    __shared__ double zf[2][YC][WENO_THREADS];
    __shared__ double zx[2][YC][WENO_THREADS];
    const int rows = blockDim.x / G.Nz, nyb = (G.Ny + rows * YC - 1) / (rows * YC);
    const int tile = xcd_tile();
    const int jb = tile / nyb, j0 = jb * march;
    if (j0 >= G.Nx) return;
    const int j1 = min(j0 + march, G.Nx);
    const int t = threadIdx.x, r = t / G.Nz, l = t - r * G.Nz;
    const int k0 = ((tile - jb * nyb) * rows + r) * YC;
    const bool row = r < rows && k0 < G.Ny;
    const int below = l == 0 ? t + G.Nz - 1 : t - 1;
    const long sx = (long)G.Ny * G.Nz;
    // in-plane offsets: the y rows k0-R .. k0+YC-1+R and the z window
    int oy[YC + W], oz[W];
#pragma unroll
    for (int o = 0; o < YC + W; o++) oy[o] = row ? wrap_add(k0, o - R, G.Ny) * G.Nz : 0;
#pragma unroll
    for (int o = 0; o < W; o++) oz[o] = row ? wrap_add(l, o + 1 - R, G.Nz) : 0;
    const int lc = row ? l : 0;
    auto plane = [&](int j) __attribute__((always_inline)) { return x + (long)wrap_add(j, 0, G.Nx) * sx; };
    double wx[YC][W], fx[YC], uc[YC];
#pragma unroll
    for (int c = 0; c < YC; c++) {
        const int oc = oy[c + R] + lc;
#pragma unroll
        for (int o = 0; o < W; o++) wx[c][o] = plane(j0 - R + o)[oc];
        const double ub = (double)ux[(long)wrap_add(j0, -1, G.Nx) * sx + oc];
        uc[c] = (double)ux[(long)j0 * sx + oc];
        const double Ux = 0.5 * (ub + uc[c]);
        weno_faces<SCHEME, 1>(wx[c] + R - 1, 0, &Ux, false, fx + c);
        zx[j0 & 1][c][t] = wx[c][R];
    }
    __syncthreads();
    for (int j = j0; j < j1; j++) {
        const long base = (long)j * sx;
        const double* xj = x + base;
        const double* xr = plane(j + R);
        const TU* un = ux + (long)wrap_add(j, 1, G.Nx) * sx;
        double fe[YC], ue[YC], wc[YC], xc[YC], adv[YC], wy[YC + W], vy[YC + 2];
        // every load of the step first
#pragma unroll
        for (int c = 0; c < YC; c++) {
            const int oc = oy[c + R] + lc;
#pragma unroll
            for (int o = 0; o < W - 1; o++) wx[c][o] = wx[c][o + 1];
            wx[c][W - 1] = xr[oc];
            ue[c] = (double)un[oc];
            xc[c] = wx[c][R - 1];
        }
#pragma unroll
        for (int o = 0; o < YC + W; o++) wy[o] = o >= R && o < R + YC ? xc[o - R] : xj[oy[o] + lc];
#pragma unroll
        for (int o = 0; o < YC + 2; o++) vy[o] = (double)uy[base + oy[o + R - 1] + lc];
        double wz[YC][W], wn[YC];
#pragma unroll
        for (int c = 0; c < YC; c++) {
#pragma unroll
            for (int o = 0; o < W; o++) wz[c][o] = o == R - 1 ? xc[c] : zx[j & 1][c][t - lc + oz[o]];
            wc[c] = (double)uz[base + oy[c + R] + lc];
            wn[c] = (double)uz[base + oy[c + R] + oz[R]];
        }
        double fz[YC], fy[YC + 1], Ux[YC], Uy[YC + 1], Uz[YC];
#pragma unroll
        for (int c = 0; c < YC; c++) {
            Uz[c] = 0.5 * (wc[c] + wn[c]);
            Ux[c] = 0.5 * (uc[c] + ue[c]);
        }
#pragma unroll
        for (int c = 0; c <= YC; c++) Uy[c] = 0.5 * (vy[c] + vy[c + 1]);
        weno_faces<SCHEME, YC>(wz[0] + R - 1, W, Uz, q9, fz);
#pragma unroll
        for (int c = 0; c < YC; c++) {
            zf[j & 1][c][t] = fz[c];
            zx[(j + 1) & 1][c][t] = wx[c][R];
        }
        weno_faces<SCHEME, YC + 1>(wy + R - 1, 1, Uy, false, fy);
        weno_faces<SCHEME, YC>(wx[0] + R - 1, W, Ux, false, fe);
#pragma unroll
        for (int c = 0; c < YC; c++) {
            adv[c] = uc[c] * (fe[c] - fx[c]) * rdx + vy[c + 1] * (fy[c + 1] - fy[c]) * rdy;
            fx[c] = fe[c];
            uc[c] = ue[c];
        }
        __syncthreads();   // two buffers: the next step's writes need no second barrier
#pragma unroll
        for (int c = 0; c < YC; c++) {
            if (row && k0 + c < G.Ny)
                out(base + oy[c + R] + lc, xc[c], adv[c] + wc[c] * (fz[c] - zf[j & 1][c][below]) * rdz);
        }
    }
}

// The same, one cell a thread with its six faces and no barrier: for grids that marching
// blocks do not fill the chip with, where latency is the kernel's time (weno_launch).
template <int SCHEME, typename TU, class OUT>
__device__ __forceinline__ void weno_cells(const TU* __restrict__ ux, const TU* __restrict__ uy,
                                           const TU* __restrict__ uz, const double* __restrict__ x, const Grid3& G,
                                           double rdx, double rdy, double rdz, bool q9, OUT&& out) {
    constexpr int R = SCHEME == 5 ? 3 : (SCHEME == 3 ? 2 : 1);
    const int id = xcd_tile() * blockDim.x + threadIdx.x;
    if (id >= G.Nx * G.Ny * G.Nz) return;
    const int l = id % G.Nz, jk = id / G.Nz, k = jk % G.Ny, j = jk / G.Ny;
    const int n[3] = {G.Nx, G.Ny, G.Nz}, c[3] = {j, k, l}, s[3] = {G.Ny * G.Nz, G.Nz, 1};
    const TU* u[3] = {ux, uy, uz};
    const double rd[3] = {rdx, rdy, rdz}, xc = x[id];
    double w[3][2 * R + 1], uw[3][3], adv = 0.0;
#pragma unroll
    for (int a = 0; a < 3; a++) {
#pragma unroll
        for (int o = -R; o <= R; o++) {
            const int at = id + (wrap_add(c[a], o, n[a]) - c[a]) * s[a];
            w[a][o + R] = o == 0 ? xc : x[at];
            if (o >= -1 && o <= 1) uw[a][o + 1] = (double)u[a][at];
        }
    }
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const double U[2] = {0.5 * (uw[a][0] + uw[a][1]), 0.5 * (uw[a][1] + uw[a][2])};
        double f[2];
        weno_faces<SCHEME, 2>(w[a] + R - 1, 1, U, a == 2 && q9, f);
        adv += uw[a][1] * (f[1] - f[0]) * rd[a];
    }
    out((long)id, xc, adv);
}

// advection kernel + flux_device (Source/advection_WENO.cu:304-392), generalised to any advected scalar x.
// YC = 0: weno_cells.
template <int SCHEME, int YC>
__global__ void __attribute__((amdgpu_waves_per_eu(YC <= 1 ? 4 : 3, 8))) __launch_bounds__(WENO_THREADS)
k_weno(const double* __restrict__ ux, const double* __restrict__ uy, const double* __restrict__ uz,
       const double* __restrict__ x, double* __restrict__ out, Grid3 G, int march, double rdx, double rdy, double rdz,
       int zfix) {
    auto put = [&](long id, double, double adv) __attribute__((always_inline)) { out[id] = adv; };
    if constexpr (YC == 0) weno_cells<SCHEME>(ux, uy, uz, x, G, rdx, rdy, rdz, !zfix, put);
    else weno_march<SCHEME, YC>(ux, uy, uz, x, G, march, rdx, rdy, rdz, !zfix, put);
}

// SSP stage of a passive scalar: out = a0*th_n + a1*(th_s - dt * (u.grad)_WENO th_s),
// u being the masked physical velocity of the same stage (TU = bulk precision).
template <int SCHEME, int YC, typename TU>
__global__ void __attribute__((amdgpu_waves_per_eu(YC <= 1 ? 4 : 3, 8))) __launch_bounds__(WENO_THREADS)
k_weno_stage(const TU* __restrict__ u, long nr, const double* __restrict__ x, const double* xn, double* out, Grid3 G,
             int march, double rdx, double rdy, double rdz, int zfix, double dt, double a0, double a1, int* nf) {
    auto put = [&](long id, double xc, double adv) __attribute__((always_inline)) {
        const double e = xc - dt * adv;
        const double o = xn ? a0 * xn[id] + a1 * e : a1 * e;
        out[id] = o;
        flag_nonfinite(nf, !isfinite(o));
    };
    if constexpr (YC == 0) weno_cells<SCHEME>(u, u + nr, u + 2 * nr, x, G, rdx, rdy, rdz, !zfix, put);
    else weno_march<SCHEME, YC>(u, u + nr, u + 2 * nr, x, G, march, rdx, rdy, rdz, !zfix, put);
}

__global__ void k_set_int(int* __restrict__ p, int v) {
    if (threadIdx.x == 0 && blockIdx.x == 0) p[0] = v;
}

// ------------------------------------------------------- a11: reductions
// Wave64 butterfly reductions via cross-lane shuffles; block partials, then
// a single-block finish.  Sums are deterministic (fixed partition and order).
constexpr int RED_THREADS = 256;
constexpr int RED_BLOCKS = 1024;
// The reference seeds min/max with the integer macro inf = 0x7f800000 (Q8).
constexpr double REF_INF = 2139095040.0;

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ double wave_min(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { const double w = __shfl_xor(v, o, 64); v = w < v ? w : v; }
    return v;
}
__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { const double w = __shfl_xor(v, o, 64); v = w > v ? w : v; }
    return v;
}

template <int OP>  // 0 sum, 1 min+max
__device__ __forceinline__ void block_finish(double a, double b, double* __restrict__ pa, double* __restrict__ pb) {
    __shared__ double sa[RED_THREADS / 64], sb[RED_THREADS / 64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (OP == 0) a = wave_sum(a);
    else { a = wave_min(a); b = wave_max(b); }
    if (lane == 0) { sa[wv] = a; sb[wv] = b; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double x = sa[0], y = sb[0];
        for (int i = 1; i < RED_THREADS / 64; i++) {
            if (OP == 0) x += sa[i];
            else { x = sa[i] < x ? sa[i] : x; y = sb[i] > y ? sb[i] : y; }
        }
        *pa = x;
        if (OP == 1) *pb = y;
    }
}

// Pointwise producers feeding the reductions (value at flat physical index id).
// SRC_SPEC_*: over the nc half-spectrum modes of three spectral fields (a, b,
// c read as interleaved complex), each mode weighted by its Hermitian
// multiplicity (1 on the l = 0 and l = Nz/2 planes, else 2).
// SRC_NONFINITE: 1 for each NaN or Inf among n doubles, else 0 (check_nans_kernel,
// Source/cuda_supp.cu:242-325, which tests isnan only; Inf is counted here too).
enum RedSrc {
    SRC_ARRAY = 0, SRC_ENERGY = 1, SRC_DISSIPATION = 2, SRC_CFL = 3, SRC_SHAPIRO = 4,
    SRC_SPEC_ENERGY = 5, SRC_SPEC_DISSIPATION = 6, SRC_NONFINITE = 7
};
struct RedArgs {
    const double* a;
    const double* b;
    const double* c;
    Grid3 G;
    double dx, dy, dz, p0, p1;  // p0: CFL number or time; p1: Re
    const double* kx;           // wavenumber tables (spectral sources)
    const double* ky;
    const double* kz;
    int Mz;
};

template <int SRC>
__device__ __forceinline__ double red_value(const RedArgs& r, long id) {
    if (SRC == SRC_ARRAY) return r.a[id];
    if (SRC == SRC_NONFINITE) return isfinite(r.a[id]) ? 0.0 : 1.0;
    if (SRC == SRC_SPEC_ENERGY || SRC == SRC_SPEC_DISSIPATION) {
        const int l = (int)(id % r.Mz);
        const long t1 = id / r.Mz;
        const int k = (int)(t1 % r.G.Ny), j = (int)(t1 / r.G.Ny);
        const double w = (l == 0 || 2 * l == r.G.Nz) ? 1.0 : 2.0;
        const double ar = r.a[2 * id], ai = r.a[2 * id + 1];
        const double br = r.b[2 * id], bi = r.b[2 * id + 1];
        const double cr = r.c[2 * id], ci = r.c[2 * id + 1];
        const double e = (ar * ar + ai * ai) + (br * br + bi * bi) + (cr * cr + ci * ci);
        if (SRC == SRC_SPEC_ENERGY) return w * e;
        // |grad u|^2 + (div u)^2 = 2 S:S integrated: |k|^2 |u^|^2 + |k.u^|^2
        const double kx = r.kx[j], ky = r.ky[k], kz = r.kz[l];
        const double dr = kx * ar + ky * br + kz * cr, di = kx * ai + ky * bi + kz * ci;
        return w * (((kx * kx + ky * ky) + kz * kz) * e + (dr * dr + di * di));
    }
    const int l = (int)(id % r.G.Nz);
    const long t1 = id / r.G.Nz;
    const int k = (int)(t1 % r.G.Ny), j = (int)(t1 / r.G.Ny);
    if (SRC == SRC_ENERGY) {  // get_kinetic_energy_device (Source/math_support.cu:744)
        const double uy = r.b[id], uz = r.c[id];
        return 0.5 * (uy * uy + uz * uz) * r.dx * r.dy;
    }
    if (SRC == SRC_DISSIPATION) {  // get_dissipation_device (Source/math_support.cu:777-789)
        const Grid3& G = r.G;
        auto D = [&](const double* f, int ax) {
            if (ax == 0) return (f[G.at(j + 1, k, l)] - f[G.at(j - 1, k, l)]) / r.dx;
            if (ax == 1) return (f[G.at(j, k + 1, l)] - f[G.at(j, k - 1, l)]) / r.dy;
            return (f[G.at(j, k, l + 1)] - f[G.at(j, k, l - 1)]) / r.dz;
        };
        const double ux_x = D(r.a, 0), ux_y = D(r.a, 1), ux_z = D(r.a, 2);
        const double uy_x = D(r.b, 0), uy_y = D(r.b, 1), uy_z = D(r.b, 2);
        const double uz_x = D(r.c, 0), uz_y = D(r.c, 1), uz_z = D(r.c, 2);
        return r.dx * r.dy * r.dz *
               (2.0 * (ux_x * ux_x + uy_y * uy_y + uz_z * uz_z) + (uy_z + uz_y) * (uy_z + uz_y) +
                (ux_z + uz_x) * (ux_z + uz_x) + (ux_y + uy_x) * (ux_y + uy_x));
    }
    if (SRC == SRC_CFL) {  // calculate_CFL_device (Source/cuda_supp.cu:188)
        return r.p0 / ((1.0e-6 + fabs(r.a[id])) / r.dx + (1.0e-6 + fabs(r.b[id])) / r.dy + (1.0e-6 + fabs(r.c[id])) / r.dz);
    }
    // SRC_SHAPIRO: Shapiro_test_case_device (Source/Shapiro_test.cu:26-33)
    const double y = k * r.dy, x = j * r.dx, z = l * r.dz;
    const double f = sqrt(3.0);
    const double dec = exp(-(f * f) * r.p0 / r.p1);
    const double ex = r.a[id] - (-0.5 * (f * cos(x) * sin(y) * sin(z) + sin(x) * cos(y) * cos(z)) * dec);
    const double ey = r.b[id] - (0.5 * (f * sin(x) * cos(y) * sin(z) - cos(x) * sin(y) * cos(z)) * dec);
    const double ez = r.c[id] - (cos(x) * cos(y) * sin(z) * dec);
    return sqrt(ex * ex + ey * ey + ez * ez);
}

template <int OP, int SRC>
__global__ void __launch_bounds__(RED_THREADS)
k_reduce_partial(RedArgs r, long n, double* __restrict__ part) {
    double a = OP == 0 ? 0.0 : REF_INF, b = -REF_INF;
    const long stride = (long)gridDim.x * RED_THREADS;
    for (long id = (long)blockIdx.x * RED_THREADS + threadIdx.x; id < n; id += stride) {
        const double v = red_value<SRC>(r, id);
        if (OP == 0) a += v;
        else { a = v < a ? v : a; b = v > b ? v : b; }
    }
    block_finish<OP>(a, b, part + blockIdx.x, part + gridDim.x + blockIdx.x);
}

template <int OP>
__global__ void __launch_bounds__(RED_THREADS)
k_reduce_final(const double* __restrict__ part, int nb, double* __restrict__ out) {
    double a = OP == 0 ? 0.0 : REF_INF, b = -REF_INF;
    for (int i = threadIdx.x; i < nb; i += RED_THREADS) {
        if (OP == 0) a += part[i];
        else { const double x = part[i], y = part[nb + i]; a = x < a ? x : a; b = y > b ? y : b; }
    }
    block_finish<OP>(a, b, out, out + 1);
}

}  // namespace ns3d
