// The launchers and kernels of one specialised mesh length, CPW_N: compiled once
// per length of CPW_FAST_SIZES (build.py; CPW_N_FULL: it is in CPW_FULL_SIZES).
#include "mesh_launch.hpp"

namespace cpwgpu {

template int launch_col_fast<float, CPW_N>(cpwgpu_plan_s *, const LocalArgs &, cplx<float> *, int, hipStream_t);
template int launch_col_fast<double, CPW_N>(cpwgpu_plan_s *, const LocalArgs &, cplx<double> *, int, hipStream_t);
template int launch_col_reg<float, CPW_N>(cpwgpu_plan_s *, const LocalArgs &, cplx<float> *, int, hipStream_t);
template int launch_col_reg<double, CPW_N>(cpwgpu_plan_s *, const LocalArgs &, cplx<double> *, int, hipStream_t);
template int launch_plane<float, CPW_N>(cpwgpu_plan_s *, const LocalArgs &, cplx<float> *, const float *, int,
                                        hipStream_t);
template int launch_plane<double, CPW_N>(cpwgpu_plan_s *, const LocalArgs &, cplx<double> *, const double *, int,
                                         hipStream_t);
#if CPW_N_FULL
template int launch_plane_spin<float, CPW_N>(cpwgpu_plan_s *, cplx<float> *, const float *, long, int, int,
                                             hipStream_t);
template int launch_plane_spin<double, CPW_N>(cpwgpu_plan_s *, cplx<double> *, const double *, long, int, int,
                                              hipStream_t);
template int launch_density<CPW_N>(cpwgpu_plan_s *, const cplx<double> *, const double *, int, int, hipStream_t,
                                   double *);
#endif

}  // namespace cpwgpu
