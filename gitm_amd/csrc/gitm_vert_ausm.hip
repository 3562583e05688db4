// gitm_vert_ausm.hip -- the AUSM step of a single grid and of a batch: one
// workgroup per column, NG lanes per level (vert_group.h).
#include "vert_gpu.h"
#include "vert_group.h"

namespace {

// 768 threads hold the tallest column; four wavefronts per SIMD leave a lane
// 128 registers (60 B per lane spilled, 164 with ions).
template <bool IONS>
__global__ void __launch_bounds__(768, 4)
    vert_group_kernel(gv::KParams kp, gitm_vert_columns io) {
  extern __shared__ double lds[];
  GpuCtx cx{kp.err};
  const int col = xcd_column((int)blockIdx.x, (int)gridDim.x);
  gv::run_group_column<IONS>(cx, kp, io, col, lds, kp.dt, col, kp.n_alts);
}

// One workgroup per column of the members mem[0..n-1], whose first_block
// numbers the launch's columns; workgroups are as wide as the widest of them
// needs.
template <bool IONS>
__global__ void __launch_bounds__(768, 4)
    vert_group_batch_kernel(gv::KParams kp, const BatchMember *__restrict__ mem, int n,
                            const double *__restrict__ dt_dev) {
  extern __shared__ double lds[];
  GpuCtx cx{kp.err};
  const int b = xcd_column((int)blockIdx.x, (int)gridDim.x);
  const BatchMember &e = mem[find_member(mem, n, b)];
  if ((int)threadIdx.x >= gv::group_threads(e.io.n_alts)) return;
  const int col = b - e.first_block;
  gv::run_group_column<IONS>(cx, kp, e.io, col, lds, dt_dev ? dt_dev[e.member] : kp.dt,
                             e.col_offset + col, e.io.n_alts);
}

// Columns with ions too tall for vert_group_kernel's LDS: one lane per level
// (vert_column.h), the RK4 carries in device memory (scratch_fields(false, true)
// doubles per level).
__global__ void __launch_bounds__(256) vert_tall_ion_kernel(gv::KParams kp, gitm_vert_columns io) {
  extern __shared__ double lds[];
  GpuCtx cx{kp.err};
  const int col = xcd_column((int)blockIdx.x, (int)gridDim.x);
  gv::run_column<256, GITM_VERT_AUSM, true, false>(cx, kp, io, col, lds, kp.scratch, kp.dt, col,
                                                   io.n_alts, gv::scratch_fields(false, true));
}

// The same for a batch's members mem[0..n-1], as vert_group_batch_kernel: in a
// launch per member those with few columns would leave the chip idle, one after
// the other (16 members of 9 columns: 4.4 ms, 0.30 in one launch).  Columns of
// 227 to 252 levels all have four wavefronts.
__global__ void __launch_bounds__(256)
    vert_tall_ion_batch_kernel(gv::KParams kp, const BatchMember *__restrict__ mem, int n,
                               const double *__restrict__ dt_dev) {
  extern __shared__ double lds[];
  GpuCtx cx{kp.err};
  const int b = xcd_column((int)blockIdx.x, (int)gridDim.x);
  const BatchMember &e = mem[find_member(mem, n, b)];
  if ((int)threadIdx.x >= e.io.n_alts + 4) return;
  const int col = b - e.first_block;
  gv::run_column<256, GITM_VERT_AUSM, true, false>(
      cx, kp, e.io, col, lds, e.scratch, dt_dev ? dt_dev[e.member] : kp.dt, e.col_offset + col,
      e.io.n_alts, gv::scratch_fields(false, true));
}

}  // namespace

// Queues the step of the ncols columns with ions of the n members at mem, all of
// which group_fits refuses and none taller than n_alts.
void launch_ausm_tall_ions(unsigned ncols, int n_alts, hipStream_t stream,
                           const gv::KParams &kp, const BatchMember *mem, int n,
                           const double *dt_dev) {
  hipLaunchKernelGGL(vert_tall_ion_batch_kernel, dim3(ncols), dim3(n_alts + 4),
                     gv::lds_bytes(n_alts, true, false), stream, kp, mem, n, dt_dev);
}

// Queues the step of `ncols` columns of the n members at mem, none taller than
// n_alts.
void launch_ausm_batch(unsigned ncols, int n_alts, hipStream_t stream, const gv::KParams &kp,
                       const BatchMember *mem, int n, const double *dt_dev) {
  const dim3 grid(ncols), block(gv::group_threads(n_alts));
  const size_t lds = gv::group_lds_bytes(n_alts, kp.ions != 0);
  if (kp.ions)
    hipLaunchKernelGGL(vert_group_batch_kernel<true>, grid, block, lds, stream, kp, mem, n,
                       dt_dev);
  else
    hipLaunchKernelGGL(vert_group_batch_kernel<false>, grid, block, lds, stream, kp, mem, n,
                       dt_dev);
}

// One column per workgroup of c's ncols columns.
void launch_ausm(unsigned ncols, hipStream_t stream, const gv::KParams &kp,
                 const gitm_vert_columns &c) {
  const dim3 grid(ncols), block(gv::group_threads(kp.n_alts));
  const size_t lds = gv::group_lds_bytes(kp.n_alts, kp.ions != 0);
  if (!gv::group_fits(kp.n_alts, kp.ions != 0))
    hipLaunchKernelGGL(vert_tall_ion_kernel, grid, dim3(c.n_alts + 4),
                       gv::lds_bytes(c.n_alts, true, false), stream, kp, c);
  else if (kp.ions)
    hipLaunchKernelGGL(vert_group_kernel<true>, grid, block, lds, stream, kp, c);
  else
    hipLaunchKernelGGL(vert_group_kernel<false>, grid, block, lds, stream, kp, c);
}
