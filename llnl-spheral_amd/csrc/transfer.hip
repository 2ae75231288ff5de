// The calls that hand fields over: the isotropy test of an uploaded H, and derivative
// fields from slot order to the caller's order.
#include "internal.hh"
#include "dgeom.hh"

namespace sphgpu {

namespace {

// Bound by reading H once (101 MB at 2.1 M rows in 3-D: 0.04 ms; the host loop
// took 8 ms there).  A workgroup that meets a row of another form stores to the
// caller's word; which one does so last makes no difference.
template <int D>
__global__ void __launch_bounds__(256) k_not_isotropic(const double* __restrict__ H, int64_t n, int32_t* flag) {
  constexpr int NS = NSym<D>::value;
  const int64_t i = blockIdx.x * int64_t(256) + threadIdx.x;
  bool iso = true;
  if (i < n) {
    const double* h = H + i * NS;
    int k = 0;
    for (int a = 0; a < D; ++a)
      for (int b = a; b < D; ++b, ++k) iso = iso && (a == b ? h[k] == h[0] : h[k] == 0.0);
  }
  if (!iso) *flag = 1;
}

// One lane per value: the writes and, since slots follow the caller's nodes in
// runs, most reads are whole lines: 0.01 ms for 9 doubles of 125 k nodes, far
// below the copy that follows.
__global__ void __launch_bounds__(256) k_unsort(const double* __restrict__ src, const int32_t* __restrict__ iperm,
                                                int64_t values, int comps, double* __restrict__ dst) {
  const int64_t q = blockIdx.x * int64_t(256) + threadIdx.x;
  if (q >= values) return;
  const int64_t i = q / comps;
  dst[q] = src[int64_t(iperm[i]) * comps + (q - i * comps)];
}

}  // namespace

int32_t* queueIsotropyTest(Sim& s, const double* H, int64_t rows) {
  int32_t* flag = static_cast<int32_t*>(hostStaging(s, 0, sizeof(int32_t)));
  *flag = 0;
  const dim3 grid(unsigned((rows + 255) / 256));
  if (s.dim == 1) hipLaunchKernelGGL(k_not_isotropic<1>, grid, dim3(256), 0, s.stream, H, rows, flag);
  else if (s.dim == 2) hipLaunchKernelGGL(k_not_isotropic<2>, grid, dim3(256), 0, s.stream, H, rows, flag);
  else hipLaunchKernelGGL(k_not_isotropic<3>, grid, dim3(256), 0, s.stream, H, rows, flag);
  SG_CHECK_HIP(hipGetLastError());
  return flag;
}

const double* unsortDerivative(Sim& s, const double* src, int comps) {
  const int64_t values = s.nInt * comps;
  s.unsorted.ensure(sizeof(double) * size_t(values));
  hipLaunchKernelGGL(k_unsort, dim3(unsigned((values + 255) / 256)), dim3(256), 0, s.stream, src,
                     s.iperm.as<int32_t>(), values, comps, s.unsorted.as<double>());
  SG_CHECK_HIP(hipGetLastError());
  return s.unsorted.as<double>();
}

}  // namespace sphgpu
