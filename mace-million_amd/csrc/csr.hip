// Receiver CSR of an edge list for the explicit-weight convolution and of ML-IAP pairs: index checks, int32 senders and the row pointers in
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

// Topology of one receiver chunk [a, b): the node list (the receivers, then the senders outside [a, b) in ascending
// order) and the local sender index of every edge.  A bit per atom marks the outside senders; a prefix sum over the
// bit words gives each its place, so nothing is sorted and the order does not depend on the atomics.  Bound by launches
// for a small chunk and by the edges' senders, read twice, for a large one.  Four launches take the place of 18 tensor
// operations: together with mm_edge_csr for the pairs' receivers and fewer device-to-host reads, a force call on 192 atoms
// goes from 1000 to 736 us, on 12,288 atoms in one chunk from 5.07 to 4.66 ms; 46,080 atoms whose 5 chunks are prepared
// three times a call, from 23.2 to 22.3 ms.
#define MM_TOPO_WORDS 1024   // bit words per workgroup of the prefix sum

__global__ void __launch_bounds__(256) mm_topo_mark_kernel(const int* __restrict__ send, int E, int a, int b, int nt,
                                                           unsigned* mask, int* __restrict__ status) {
  int bad = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const long e = (long)blockIdx.x * 1024 + 256 * k + threadIdx.x;
    if (e >= E) continue;
    const int s = send[e];
    if ((unsigned)s >= (unsigned)nt) {
      ++bad;
      continue;
    }
    if (s >= a && s < b) continue;
    // most senders are marked many times: only a bit that reads as clear is set
    const unsigned bit = 1u << (s & 31);
    if (!(__builtin_nontemporal_load(mask + (s >> 5)) & bit)) atomicOr(mask + (s >> 5), bit);
  }
  if (bad) atomicAdd(status, bad);
}

__device__ __forceinline__ int mm_topo_block_sum(int v, int* s) {
#pragma unroll
  for (int d = 32; d; d >>= 1) v += __shfl_xor(v, d);
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
  __syncthreads();
  v = s[0] + s[1] + s[2] + s[3];
  __syncthreads();
  return v;
}

__global__ void __launch_bounds__(256) mm_topo_count_kernel(const unsigned* __restrict__ mask, int words,
                                                            int* __restrict__ sums) {
  __shared__ int s[4];
  int n = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const long w = (long)blockIdx.x * MM_TOPO_WORDS + 256 * k + threadIdx.x;
    if (w < words) n += __popc(mask[w]);
  }
  n = mm_topo_block_sum(n, s);
  if (threadIdx.x == 0) sums[blockIdx.x] = n;
}

// pre[w] = local index of the first marked atom of word w; nodes; status[1] = marked atoms
__global__ void __launch_bounds__(256) mm_topo_nodes_kernel(const unsigned* __restrict__ mask, int words,
                                                            const int* __restrict__ sums, int a, int nC,
                                                            int* __restrict__ pre, int* __restrict__ nodes,
                                                            int* __restrict__ status) {
  __shared__ int s[4];
  const int tid = threadIdx.x, lane = tid & 63;
  int v = 0;
  for (int j = tid; j < (int)blockIdx.x; j += 256) v += sums[j];
  const int base = mm_topo_block_sum(v, s);
  const long w0 = (long)blockIdx.x * MM_TOPO_WORDS + 4 * tid;
  unsigned m[4];
  int n = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    m[k] = w0 + k < words ? mask[w0 + k] : 0;
    n += __popc(m[k]);
  }
  int inc = n;   // inclusive over the wave
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int u = __shfl_up(inc, d);
    if (lane >= d) inc += u;
  }
  if (lane == 63) s[tid >> 6] = inc;
  __syncthreads();
  int at = nC + base + inc - n;
  for (int w = 0; w < (tid >> 6); ++w) at += s[w];
  if (blockIdx.x == gridDim.x - 1 && tid == 255) status[1] = at + n - nC;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (w0 + k >= words) break;
    pre[w0 + k] = at;
    for (unsigned b = m[k]; b; b &= b - 1) nodes[at++] = (int)(32 * (w0 + k)) + __ffs(b) - 1;
  }
  for (long j = (long)blockIdx.x * 256 + tid; j < nC; j += (long)gridDim.x * 256) nodes[j] = a + (int)j;
}

__global__ void __launch_bounds__(256) mm_topo_local_kernel(const int* __restrict__ send, int E, int a, int b, int nt,
                                                            const unsigned* __restrict__ mask,
                                                            const int* __restrict__ pre, int* __restrict__ ls) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const long e = (long)blockIdx.x * 1024 + 256 * k + threadIdx.x;
    if (e >= E) continue;
    const int s = send[e];
    if ((unsigned)s >= (unsigned)nt) continue;   // counted in status[0]
    ls[e] = s >= a && s < b ? s - a : pre[s >> 5] + __popc(mask[s >> 5] & ((1u << (s & 31)) - 1));
  }
}

extern "C" int mm_chunk_topology(const int* send, int E, int a, int b, int nt, unsigned* scratch, int* nodes, int* ls,
                                 int* status, hipStream_t stream) {
  MM_CHECK_ARG(E >= 0 && nt > 0 && a >= 0 && b >= a && b <= nt, "bad sizes");
  const int words = (nt >> 5) + 1, blocks = (words + MM_TOPO_WORDS - 1) / MM_TOPO_WORDS;
  int* pre = (int*)scratch + words;
  int* sums = pre + words;
  const dim3 edges((unsigned)(((long)E + 1023) / 1024));
  if (E)
    hipLaunchKernelGGL(mm_topo_mark_kernel, edges, dim3(256), 0, stream, send, E, a, b, nt, scratch, status);
  hipLaunchKernelGGL(mm_topo_count_kernel, dim3(blocks), dim3(256), 0, stream, scratch, words, sums);
  hipLaunchKernelGGL(mm_topo_nodes_kernel, dim3(blocks), dim3(256), 0, stream, scratch, words, sums, a, b - a, pre,
                     nodes, status);
  if (E)
    hipLaunchKernelGGL(mm_topo_local_kernel, edges, dim3(256), 0, stream, send, E, a, b, nt, scratch, pre, ls);
  return mm::launch_status("mm_chunk_topology");
}
