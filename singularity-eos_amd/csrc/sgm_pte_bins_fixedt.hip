// Batched persistent PTE bin kernels (2..6 materials), method PTESolverFixedT.
#include "sgm_pte_kernels.inl"
namespace sgm {
hipError_t launch_pte_bin_fixedt(int nm, const PteArgs &a, const MixParamsDev &P, const int *cells,
                             long n, int *counter, int block, int cpw,
                             int grid, const ParkArgs *park, hipStream_t s) {
  return kern::bin_launch<2>(nm, a, P, cells, n, counter, block, cpw, grid, s, park);
}
hipError_t launch_pte_tail_fixedt(int nm, const PteArgs &a, const MixParamsDev &P,
                              const ParkArgs &park, hipStream_t s) {
  return kern::tail_launch<2>(nm, a, P, park, s);
}
hipError_t launch_pte_batch_fixedt(const PteArgs &a, const MixParamsDev &P, const BatchArgs &b,
                               const int *cells, const long *range, long n, int chunk,
                               hipStream_t s) {
  return kern::batch_launch<2>(a, P, b, cells, range, n, chunk, s);
}
} // namespace sgm
