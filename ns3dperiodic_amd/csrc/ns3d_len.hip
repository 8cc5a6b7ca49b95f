// ns3d_len.hip -- the kernels and launches of a group of grid lengths (launch_n.hpp),
// compiled once for each group with -DNS3D_LENGTHS="L(8) L(512)" or the like.
#include "launch_n.hpp"

#define EPI_BOTH(N, MODE)                                                          \
    template int launch_x_fwd<double, MODE, N>(ns3d_ctx*, const EpiArgs&, int, bool); \
    template int launch_x_fwd<float, MODE, N>(ns3d_ctx*, const EpiArgs&, int, bool);
#define PASSES(T, N)                                                             \
    template int launch_x_inv<T, double, N>(ns3d_ctx*, const zd* const*, const zd* const*, int, int, long, const double*); \
    template int launch_y_inv<T, N>(ns3d_ctx*, int);                             \
    template int launch_z<T, N>(ns3d_ctx*, int);                                 \
    template int launch_y_fwd<T, N>(ns3d_ctx*, int, bool);                       \
    template int launch_c2c<T, N>(ns3d_ctx*, int, int, const cplx<T>*, cplx<T>*); \
    template int launch_c2r<T, N>(ns3d_ctx*, const cplx<T>*, T*, bool);          \
    template int launch_r2c<T, N>(ns3d_ctx*, const T*, cplx<T>*);
#define L(N)                                                                     \
    PASSES(double, N)                                                            \
    PASSES(float, N)                                                             \
    template int launch_x_inv<float, float, N>(ns3d_ctx*, const cplx<float>* const*, const cplx<float>* const*, int, int, long, const double*); \
    EPI_BOTH(N, EPI_Q)                                                           \
    EPI_BOTH(N, EPI_STAGE)                                                       \
    EPI_BOTH(N, EPI_RHS)                                                         \
    EPI_BOTH(N, EPI_UV)                                                          \
    EPI_BOTH(N, EPI_UV_RHS)                                                      \
    EPI_BOTH(N, EPI_UV_VEC)                                                      \
    EPI_BOTH(N, EPI_IUV)                                                         \
    template int launch_x_fwd<float, EPI_STAGE32, N>(ns3d_ctx*, const EpiArgs&, int, bool); \
    template int launch_x_fwd<float, EPI_INC, N>(ns3d_ctx*, const EpiArgs&, int, bool);    \
    template int launch_x_fwd<float, EPI_INC_FINAL, N>(ns3d_ctx*, const EpiArgs&, int, bool);
NS3D_LENGTHS
