// kah_slope_2d.hip -- slope kernels (K1, K3) of the 2D2F form, FP64 storage.
#include "kah_device.h"

namespace kah {

hipError_t launch_slope_2d(const DevArgs& A, bool uni, const int32_t* cells, int n,
                          int maxh, hipStream_t st) {
  return uni ? launch_slope_t<2, 2, true, double>(A, cells, n, maxh, st)
             : launch_slope_t<2, 2, false, double>(A, cells, n, maxh, st);
}

hipError_t launch_slope_chunk_2d(const DevArgs& A, bool uni, const void* recs, const int4* work,
                                int n, int kind, int waves, hipStream_t st) {
  return uni ? launch_slope_chunk_t<2, 2, true, double>(A, recs, work, n, kind, waves, st)
             : launch_slope_chunk_t<2, 2, false, double>(A, recs, work, n, kind, waves, st);
}

hipError_t launch_macro_slope_2d(const DevArgs& A, bool uni, const int32_t* cells, int n,
                                double* sw, hipStream_t st) {
  return uni ? launch_macro_slope_t<2, 2, true, double>(A, cells, n, sw, st)
             : launch_macro_slope_t<2, 2, false, double>(A, cells, n, sw, st);
}

hipError_t launch_overlap_map_2d(const DevArgs& A, const OvJob* jobs, int njobs, uint32_t* map,
                                hipStream_t st) {
  return launch_overlap_map_t<2, 2>(A, jobs, njobs, map, st);
}

hipError_t launch_mirror_2d(const DevArgs& A, bool uni, const int32_t* cells,
                              const int64_t* off, int n, int kind, int unpack, double* buf,
                              const double* mid, const int32_t* benc, double* sw, void* dfw,
                              hipStream_t st) {
  return uni ? launch_mirror_t<2, 2, true, double>(A, cells, off, n, kind, unpack, buf, mid,
                                                     benc, sw, dfw, st)
             : launch_mirror_t<2, 2, false, double>(A, cells, off, n, kind, unpack, buf, mid,
                                                      benc, sw, dfw, st);
}

hipError_t launch_restart_2d(const DevArgs& A, bool uni, const int64_t* row, int64_t N,
                               int64_t Nv, int load, double* ws, int8_t* lev, double* vmid,
                               double* vdf, void* dfw, hipStream_t st) {
  return uni ? launch_restart_t<2, 2, true, double>(A, row, N, Nv, load, ws, lev, vmid, vdf,
                                                      dfw, st)
             : launch_restart_t<2, 2, false, double>(A, row, N, Nv, load, ws, lev, vmid, vdf,
                                                       dfw, st);
}

hipError_t launch_vs_2d(const DevArgs& A, bool uni, int which, const VsArgs& P, int nc,
                          double* out, uint8_t* flags, hipStream_t st) {
  return uni ? launch_vs_t<2, 2, true, double>(A, which, P, nc, out, flags, st)
             : launch_vs_t<2, 2, false, double>(A, which, P, nc, out, flags, st);
}
hipError_t launch_vs_remap_2d(const DevArgs& A, const int64_t* voff_old, const void* df_old,
                                const void* sdf_old, const int32_t* src, const uint8_t* changed,
                                int nc, hipStream_t st) {
  return launch_vs_remap_t<2, 2, double>(A, voff_old, df_old, sdf_old, src, changed, nc, st);
}
hipError_t launch_vs_project_2d(const DevArgs& A, bool uni, const int32_t* cells, int n,
                                  size_t lds, double* scratch, void* dfw, hipStream_t st) {
  return uni ? launch_vs_project_t<2, 2, true, double>(A, cells, n, lds, scratch, dfw, st)
             : launch_vs_project_t<2, 2, false, double>(A, cells, n, lds, scratch, dfw, st);
}

hipError_t launch_ib_2d(const DevArgs& A, bool uni, const IbArgs& B, hipStream_t st) {
  return uni ? launch_ib_t<2, 2, true, double>(A, B, st)
             : launch_ib_t<2, 2, false, double>(A, B, st);
}

}  // namespace kah
