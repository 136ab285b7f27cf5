// Receiver CSR of an edge list for the explicit-weight convolution and of ML-IAP pairs: index checks, int32 senders and
// the row pointers in one launch instead of a chain of elementwise, reduction and histogram launches (the chain took
// 0.1 ms, more than the convolution of a small graph).
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
// order) and the local sender index of every edge.  A byte per atom marks the outside senders (plain stores of 1: with
// atomics on bits the marks of 1.5 M edges took 121 us, of 192 atoms 16 us); a prefix sum over words of 32 marks gives
// each its place, so nothing is sorted.  Bound by launches for a small chunk and by the edges' senders, read twice, for
// a large one.  Four launches take the place of 18 tensor operations: together with mm_edge_csr for the pairs'
// receivers and fewer device-to-host reads, a force call on 192 atoms goes from 1000 to 720 us, on 12,288 atoms in one
// chunk from 5.07 to 4.66 ms.
#define MM_TOPO_WORDS 1024   // bit words per workgroup of the prefix sum

__global__ void __launch_bounds__(256) mm_topo_mark_kernel(const int* __restrict__ send, int E, int a, int b, int nt,
                                                           unsigned char* __restrict__ mark,
                                                           int* __restrict__ status) {
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
    if (s < a || s >= b) mark[s] = 1;
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

__global__ void __launch_bounds__(256) mm_topo_count_kernel(const uint4* __restrict__ mark, int words,
                                                            unsigned* __restrict__ mask, int* __restrict__ sums) {
  __shared__ int s[4];
  int n = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const long w = (long)blockIdx.x * MM_TOPO_WORDS + 256 * k + threadIdx.x;
    if (w >= words) continue;
    unsigned m = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint4 v = mark[2 * w + h];
      const unsigned x[4] = {v.x, v.y, v.z, v.w};
      // the low bits of the 4 bytes of x land side by side in bits 24..27 of the product
#pragma unroll
      for (int j = 0; j < 4; ++j) m |= ((x[j] * 0x01020408u) >> 24 & 15u) << (16 * h + 4 * j);
    }
    mask[w] = m;
    n += __popc(m);
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
  MM_CHECK_ARG((size_t)scratch % 16 == 0, "scratch must be 16-byte aligned");
  const int words = (nt >> 5) + 1, blocks = (words + MM_TOPO_WORDS - 1) / MM_TOPO_WORDS;
  unsigned char* mark = (unsigned char*)scratch;   // 32 words bytes
  unsigned* mask = scratch + 8 * (size_t)words;
  int* pre = (int*)mask + words;
  int* sums = pre + words;
  const dim3 edges((unsigned)(((long)E + 1023) / 1024));
  if (E)
    hipLaunchKernelGGL(mm_topo_mark_kernel, edges, dim3(256), 0, stream, send, E, a, b, nt, mark, status);
  hipLaunchKernelGGL(mm_topo_count_kernel, dim3(blocks), dim3(256), 0, stream, (const uint4*)mark, words,
                     mask, sums);
  hipLaunchKernelGGL(mm_topo_nodes_kernel, dim3(blocks), dim3(256), 0, stream, mask, words, sums, a, b - a, pre,
                     nodes, status);
  if (E)
    hipLaunchKernelGGL(mm_topo_local_kernel, edges, dim3(256), 0, stream, send, E, a, b, nt, mask, pre, ls);
  return mm::launch_status("mm_chunk_topology");
}

// Stable sort of E keys in [0, n) with their positions: a least-significant-digit radix sort of 8 bits a pass, as many
// passes as n needs (2 for the 30,000 rows of a chunk).  Per pass: digit counts of tiles of 4,096 keys, a prefix sum
// over each digit's tiles, and the scatter.  In the scatter a wave ranks 64 consecutive keys at a time among equal
// digits with one ballot per bit, on top of counters in LDS, so equal keys stay in order.  Bound by launches (3 a pass)
// and the scattered 8-byte writes.  The merge sort of 64-bit keys, histogram and prefix sum it replaces took 0.3 ms for
// each of a low-memory call's ten sender lists (46,080 atoms, 0.8 M edges each): 22.3 -> 18.6 ms a call.  Unsorted
// pairs of 12,288 atoms: 4.66 -> 4.41 ms a force call.
#define MM_SORT_TILE 4096
#define MM_SORT_ROUNDS (MM_SORT_TILE / 256)

__global__ void __launch_bounds__(256) mm_sort_count_kernel(const int* __restrict__ keys, int E, int shift, int tiles,
                                                            int* __restrict__ counts) {
  __shared__ int h[256];
  h[threadIdx.x] = 0;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < MM_SORT_ROUNDS; ++r) {
    const long e = (long)blockIdx.x * MM_SORT_TILE + 256 * r + threadIdx.x;
    if (e < E) atomicAdd(&h[((unsigned)keys[e] >> shift) & 255], 1);
  }
  __syncthreads();
  counts[(size_t)threadIdx.x * tiles + blockIdx.x] = h[threadIdx.x];
}

// exclusive prefix sum of 256 values, one per thread; the total goes to *total
__device__ __forceinline__ int mm_sort_scan256(int v, int* s, int* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int inc = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int u = __shfl_up(inc, d);
    if (lane >= d) inc += u;
  }
  if (lane == 63) s[wave] = inc;
  __syncthreads();
  int before = 0;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    if (w < wave) before += s[w];
  }
  *total = s[0] + s[1] + s[2] + s[3];
  __syncthreads();
  return before + inc - v;
}

// one workgroup per digit: exclusive prefix sum over its tiles, and its total
__global__ void __launch_bounds__(256) mm_sort_scan_kernel(int* __restrict__ counts, int tiles,
                                                           int* __restrict__ totals) {
  __shared__ int s[4];
  int* __restrict__ row = counts + (size_t)blockIdx.x * tiles;
  int carry = 0;
  for (int t0 = 0; t0 < tiles; t0 += 256) {
    const int t = t0 + threadIdx.x;
    int total;
    const int x = mm_sort_scan256(t < tiles ? row[t] : 0, s, &total);
    if (t < tiles) row[t] = carry + x;
    carry += total;
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// vals null: the positions 0 .. E - 1
__global__ void __launch_bounds__(256) mm_sort_scatter_kernel(const int* __restrict__ keys,
                                                              const int* __restrict__ vals, int E, int shift, int tiles,
                                                              const int* __restrict__ counts,
                                                              const int* __restrict__ totals,
                                                              int* __restrict__ keys_out, int* __restrict__ vals_out) {
  __shared__ int cnt[4][256];
  __shared__ int s[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const long e0 = (long)blockIdx.x * MM_SORT_TILE + wave * (MM_SORT_TILE / 4) + lane;
#pragma unroll
  for (int w = 0; w < 4; ++w) cnt[w][tid] = 0;
  int key[MM_SORT_ROUNDS], rank[MM_SORT_ROUNDS];
#pragma unroll
  for (int r = 0; r < MM_SORT_ROUNDS; ++r) key[r] = e0 + 64 * r < E ? keys[e0 + 64 * r] : 0;
  int unused;
  const int digit0 = mm_sort_scan256(totals[tid], s, &unused);   // its barriers also cover the cleared counters
#pragma unroll
  for (int r = 0; r < MM_SORT_ROUNDS; ++r) {
    const bool ok = e0 + 64 * r < E;
    const int d = ((unsigned)key[r] >> shift) & 255;
    unsigned long long same = __ballot(ok);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const unsigned long long m = __ballot((d >> b) & 1);
      same &= (d >> b) & 1 ? m : ~m;
    }
    const int before = __popcll(same & ((1ull << lane) - 1));
    const int c = cnt[wave][d];
    rank[r] = c + before;
    mm_wave_lds_sync();
    if (ok && before == 0) cnt[wave][d] = c + __popcll(same);
    mm_wave_lds_sync();
  }
  __syncthreads();
  int at = digit0 + counts[(size_t)tid * tiles + blockIdx.x];
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const int c = cnt[w][tid];
    cnt[w][tid] = at;
    at += c;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < MM_SORT_ROUNDS; ++r) {
    const long e = e0 + 64 * r;
    if (e >= E) continue;
    const long o = cnt[wave][((unsigned)key[r] >> shift) & 255] + rank[r];
    keys_out[o] = key[r];
    vals_out[o] = vals ? vals[e] : (int)e;
  }
}

extern "C" int mm_stable_sort(const int* keys, int E, int n, int* keys_out, int* perm, int* scratch,
                              hipStream_t stream) {
  MM_CHECK_ARG(E >= 0 && n >= 0, "bad sizes");
  if (E == 0) return MM_OK;
  const int tiles = (int)(((long)E + MM_SORT_TILE - 1) / MM_SORT_TILE);
  int *tk = scratch, *tv = scratch + E, *counts = scratch + 2 * (size_t)E, *totals = counts + 256 * (size_t)tiles;
  int passes = 1;
  while (passes < 4 && (unsigned)(n > 0 ? n - 1 : 0) >> (8 * passes)) ++passes;
  const int *k = keys, *v = nullptr;
  for (int p = 0; p < passes; ++p) {
    const bool last = (passes - p) & 1;   // the passes alternate and end in the outputs
    int *ko = last ? keys_out : tk, *vo = last ? perm : tv;
    hipLaunchKernelGGL(mm_sort_count_kernel, dim3(tiles), dim3(256), 0, stream, k, E, 8 * p, tiles, counts);
    hipLaunchKernelGGL(mm_sort_scan_kernel, dim3(256), dim3(256), 0, stream, counts, tiles, totals);
    hipLaunchKernelGGL(mm_sort_scatter_kernel, dim3(tiles), dim3(256), 0, stream, k, v, E, 8 * p, tiles, counts, totals,
                       ko, vo);
    k = ko;
    v = vo;
  }
  return mm::launch_status("mm_stable_sort");
}
