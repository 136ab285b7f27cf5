// Receiver CSR of an edge list for the explicit-weight convolution: index checks, int32 senders and the row pointers in
// one launch instead of a chain of elementwise, reduction and histogram launches (the chain took 0.1 ms, more than
// the convolution of a small graph).
#include "common.h"

// Workgroups below n_edge_wg: four edges per thread, send32[e] and the violation counts (adds of the few that occur;
// nothing is added on valid sorted input): bad[0] senders outside [0, n_send), bad[1] receivers outside [0, n),
// bad[2] receivers smaller than their predecessor.  The others: rowptr[k] = first edge with receiver >= k by binary
// search (k = 0 .. n), right when the receivers are sorted and in any case within [0, E].
// Index: int or long long; strides in elements.
template <typename Index>
__global__ void __launch_bounds__(256) mm_edge_csr_kernel(const Index* __restrict__ send, long send_stride,
                                                          const Index* __restrict__ recv, long recv_stride, int E,
                                                          int n, int n_send, int n_edge_wg, int* __restrict__ send32,
                                                          int* __restrict__ rowptr, int* __restrict__ bad) {
  if ((int)blockIdx.x < n_edge_wg) {
    int b0 = 0, b1 = 0, b2 = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const long e = (long)blockIdx.x * 1024 + 256 * k + threadIdx.x;
      if (e >= E) continue;
      if (send32) {
        const Index s = send[e * send_stride];
        send32[e] = (int)s;
        b0 += (s < 0) | (s >= n_send);
      }
      const Index r = recv[e * recv_stride];
      b1 += (r < 0) | (r >= n);
      b2 += e > 0 && r < recv[(e - 1) * recv_stride];
    }
    if (b0) atomicAdd(bad, b0);
    if (b1) atomicAdd(bad + 1, b1);
    if (b2) atomicAdd(bad + 2, b2);
    return;
  }
  const int k = ((int)blockIdx.x - n_edge_wg) * 256 + threadIdx.x;
  if (k > n) return;
  int lo = 0, hi = E;
  while (lo < hi) {
    const int mid = lo + ((hi - lo) >> 1);
    if (recv[mid * recv_stride] < (Index)k) lo = mid + 1;
    else hi = mid;
  }
  rowptr[k] = lo;
}

extern "C" int mm_edge_csr(const void* send, long send_stride, const void* recv, long recv_stride, int index64, int E,
                           int n, int n_send, int* send32, int* rowptr, int* bad, hipStream_t stream) {
  MM_CHECK_ARG(E >= 0 && n >= 0 && n < 2147483647 && n_send >= 0, "bad sizes");
  MM_CHECK_ARG(send_stride >= 0 && recv_stride >= 0, "bad strides");
  MM_CHECK_ARG((send == nullptr) == (send32 == nullptr), "senders and their output come together");
  const int wg = (int)(((long)E + 1023) / 1024);
  const dim3 grid((unsigned)(wg + n / 256 + 1));
  if (index64)
    hipLaunchKernelGGL(mm_edge_csr_kernel<long long>, grid, dim3(256), 0, stream, (const long long*)send, send_stride,
                       (const long long*)recv, recv_stride, E, n, n_send, wg, send32, rowptr, bad);
  else
    hipLaunchKernelGGL(mm_edge_csr_kernel<int>, grid, dim3(256), 0, stream, (const int*)send, send_stride,
                       (const int*)recv, recv_stride, E, n, n_send, wg, send32, rowptr, bad);
  return mm::launch_status("mm_edge_csr");
}
