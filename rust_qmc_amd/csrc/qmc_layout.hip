// qmc_layout.hip -- transposes of the walkers' positions through LDS tiles:
// rows of 64 walkers on the ensemble's side, runs of 32 coordinates on the
// caller's, both contiguous.  On the host, which walks the state with the
// ensemble's stride, reading 65,536 CH4 walkers took 5.96 ms and setting them
// 5.63; now 1.11 and 0.72, nearly all of it the copies (2,048 benzene walkers
// 360 -> 163 us).
#include "qmc_layout.hpp"

namespace qmc {
namespace {

constexpr int TW = 64, TQ = 32;

// columns [0, nz) of pos against the rows of user's W walkers (W <= nz: the
// columns past them are written as zeros; OUT: W = nz)
template <class T, bool OUT>
__global__ void __launch_bounds__(256) positions_kernel(T* __restrict__ pos, int64_t ld, int64_t W, int64_t nz, int n3,
                                                        double* __restrict__ user) {
  __shared__ double tile[TQ][TW + 1];
  const int64_t w0 = (int64_t)blockIdx.x * TW;
  const int q0 = blockIdx.y * TQ;
  auto rows = [&](auto f) {  // (coordinate, walker) pairs, walkers in consecutive lanes
    for (int i = threadIdx.x; i < TQ * TW; i += 256) {
      const int q = i / TW, w = i % TW;
      if (q0 + q < n3 && w0 + w < nz) f(q, w, (int64_t)(q0 + q) * ld + w0 + w);
    }
  };
  auto cols = [&](auto f) {  // coordinates in consecutive lanes
    for (int i = threadIdx.x; i < TQ * TW; i += 256) {
      const int q = i % TQ, w = i / TQ;
      if (q0 + q < n3 && w0 + w < W) f(q, w, (w0 + w) * n3 + q0 + q);
    }
  };
  if constexpr (OUT) {
    rows([&](int q, int w, int64_t at) { tile[q][w] = (double)pos[at]; });
    __syncthreads();
    cols([&](int q, int w, int64_t at) { user[at] = tile[q][w]; });
  } else {
    cols([&](int q, int w, int64_t at) { tile[q][w] = user[at]; });
    __syncthreads();
    rows([&](int q, int w, int64_t at) { pos[at] = w0 + w < W ? (T)tile[q][w] : T(0); });
  }
}

// a launch takes 2^24 walkers, so that its grid stays below 2^32 lanes
template <class T, bool OUT>
hipError_t launch(T* pos, int64_t ld, int64_t n, int64_t nz, int n3, double* user, hipStream_t st) {
  constexpr int64_t step = 1 << 24;
  for (int64_t w = 0; w < nz; w += step) {
    const int64_t m = nz - w < step ? nz - w : step;
    const dim3 grid((unsigned)((m + TW - 1) / TW), (unsigned)((n3 + TQ - 1) / TQ));
    positions_kernel<T, OUT><<<grid, 256, 0, st>>>(pos + w, ld, n - w, m, n3, user + w * n3);
    if (hipError_t e = hipGetLastError()) return e;
  }
  return hipSuccess;
}

}  // namespace

template <class T>
hipError_t positions_out(const T* pos, int64_t ld, int64_t n, int n3, double* out, hipStream_t st) {
  return launch<T, true>(const_cast<T*>(pos), ld, n, n, n3, out, st);
}
template <class T>
hipError_t positions_in(const double* in, int64_t ld, int64_t n, int64_t nz, int n3, T* pos, hipStream_t st) {
  return launch<T, false>(pos, ld, n, nz, n3, const_cast<double*>(in), st);
}
template hipError_t positions_out<double>(const double*, int64_t, int64_t, int, double*, hipStream_t);
template hipError_t positions_out<float>(const float*, int64_t, int64_t, int, double*, hipStream_t);
template hipError_t positions_in<double>(const double*, int64_t, int64_t, int64_t, int, double*, hipStream_t);
template hipError_t positions_in<float>(const double*, int64_t, int64_t, int64_t, int, float*, hipStream_t);

}  // namespace qmc
