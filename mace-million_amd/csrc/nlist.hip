// Cell-list neighbour build, bit-exact with the reference's System / build_neighbors
// (receiver_chunk_mace.py:82-165):
//   wrap      : m = fmod(x, L); m + L where the signs of m and L differ (torch.remainder)
//   cell      : min(floor(m / (L / ncell)), ncell - 1), ncell = max(1, floor(L / r_max)) (host)
//   order     : 10-bit Morton code (x -> bit 3b+2, y -> 3b+1, z -> 3b), stable radix sort -> perm
//   candidates: the 27 cells (c + o) mod ncell for o in (-1, 0, 1)^3, x-offset slowest (meshgrid "ij"), each
//               cell's atoms in sorted order; all atoms 0..N-1 in order if any ncell < 3
//   test      : d = v - L * rint(v / L) (half to even, as torch.round), dd = (dx^2 + dy^2) + dz^2, keep
//               dd < r_max^2 and j != i; candidate order preserved.
// Every fp64 operation is a separately rounded IEEE operation: the file is compiled with -ffp-contract=off and
// the arithmetic scopes carry "#pragma clang fp contract(off)" (HIP's __dmul_rn / __dadd_rn are plain * and +,
// which clang would otherwise fuse into FMAs and so change dd at the last bit).  Output: CSR (rowptr int64 [N+1],
// senders int32 [E]) in the sorted index space.
#include "common.h"
#include "mic.h"

#include <hipcub/hipcub.hpp>

#include <mutex>
#include <string>

__global__ void mm_nl_prepare_kernel(const double* __restrict__ pos_in, long N, double bx, double by, double bz,
                                     double cx, double cy, double cz, int nx, int ny, int nz,
                                     double* __restrict__ pos_w, int* __restrict__ cell,
                                     long long* __restrict__ key, long long* __restrict__ idx) {
#pragma clang fp contract(off)
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i >= N) return;
  const double L[3] = {bx, by, bz};
  const double cs[3] = {cx, cy, cz};
  const int nc[3] = {nx, ny, nz};
  int c[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    double m = fmod(pos_in[3 * i + k], L[k]);
    if (m != 0.0 && ((m < 0.0) != (L[k] < 0.0))) m = __dadd_rn(m, L[k]);
    pos_w[3 * i + k] = m;
    long q = (long)floor(__ddiv_rn(m, cs[k]));
    if (q > nc[k] - 1) q = nc[k] - 1;
    c[k] = (int)q;
    cell[3 * i + k] = c[k];
  }
  long long code = 0;
#pragma unroll
  for (int b = 0; b < 10; ++b) {
    code |= ((long long)((c[0] >> b) & 1)) << (3 * b + 2);
    code |= ((long long)((c[1] >> b) & 1)) << (3 * b + 1);
    code |= ((long long)((c[2] >> b) & 1)) << (3 * b);
  }
  key[i] = code;
  idx[i] = i;
}

__global__ void mm_nl_gather_kernel(const long long* __restrict__ perm, long N, const double* __restrict__ pos_w,
                                    const int* __restrict__ cell, const int* __restrict__ spec_in,
                                    double* __restrict__ pos_s, int* __restrict__ cell_s, int* __restrict__ spec_s) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i >= N) return;
  const long j = perm[i];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    pos_s[3 * i + k] = pos_w[3 * j + k];
    cell_s[3 * i + k] = cell[3 * j + k];
  }
  if (spec_in) spec_s[i] = spec_in[j];
}

// start[cl] = first sorted atom of cell cl (N if empty), count[cl]; atoms of a cell are contiguous after the sort
__global__ void mm_nl_ranges_kernel(const int* __restrict__ cell_s, long N, int ny, int nz, int* __restrict__ start,
                                    int* __restrict__ count) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i >= N) return;
  const int cl = (cell_s[3 * i] * ny + cell_s[3 * i + 1]) * nz + cell_s[3 * i + 2];
  const int prev = i > 0 ? (cell_s[3 * (i - 1)] * ny + cell_s[3 * (i - 1) + 1]) * nz + cell_s[3 * (i - 1) + 2] : -1;
  const int next = i + 1 < N ? (cell_s[3 * (i + 1)] * ny + cell_s[3 * (i + 1) + 1]) * nz + cell_s[3 * (i + 1) + 2]
                             : -1;
  if (cl != prev) start[cl] = (int)i;
  if (cl != next) count[cl] = (int)(i + 1);   // end, turned into a count below
}

__global__ void mm_nl_counts_kernel(int ncells, const int* __restrict__ start, int* __restrict__ count, long N) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncells) return;
  count[c] = start[c] < N ? count[c] - start[c] : 0;
}

__global__ void mm_fill_i32_kernel_nl(int* __restrict__ p, int n, int v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Candidate test of the cell list, one workgroup of 4 waves per cell: all receivers of a cell share their candidates
// (the 27 cells around it), which are staged in LDS MM_NL_CH at a time in candidate order; a wave tests 64 of them
// against four receivers at once and compacts the kept ones with ballots.  blockIdx.y shares a cell's receivers out
// when there are too few cells to fill the GPU.  brute != 0: every atom is a candidate of every receiver, 16 receivers
// per workgroup.
// Bound by the fp64 arithmetic of the tests (27 / 4.2 candidates per kept pair).  196,608 water atoms, 8 A (302 M
// candidates, 42 M pairs): count 945 -> 487 us, fill 1,041 -> 250 us against one thread per receiver with its
// candidates in global memory, three fp64 divisions per test and every test made twice.
//
// FILL = false: NN[i] = kept candidates of receiver i; with masks != nullptr also the ballots, one word per 64
// candidates (masks[i * cap + word], if the cell's candidates fit cap words).
// FILL = true: the kept candidates in order, send[rowptr[i] + k]; from the ballots where the count pass left them,
// otherwise by testing again.
#define MM_NL_CH 1024
#define MM_NL_R 4

template <bool FILL>
__global__ void __launch_bounds__(256) mm_nl_pairs_kernel(const double* __restrict__ pos, long N, double bx, double by,
                                                          double bz, int nx, int ny, int nz,
                                                          const int* __restrict__ start,
                                                          const int* __restrict__ count, double r2, int brute,
                                                          int* __restrict__ NN, const long* __restrict__ rowptr,
                                                          int* __restrict__ send,
                                                          unsigned long long* __restrict__ masks, int cap) {
  __shared__ double sx[MM_NL_CH], sy[MM_NL_CH], sz[MM_NL_CH];
  __shared__ int sj[MM_NL_CH];
  __shared__ int cs[27], cp[28];   // first atom of each candidate cell; candidates before it (cp[27]: all)
  __shared__ int out_of_box;       // a coordinate outside [0, L] (or NaN): the tests take the general minimum image
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  long r0, nr, T;
  if (brute) {
    r0 = (long)blockIdx.x * (4 * MM_NL_R);
    nr = min((long)(4 * MM_NL_R), N - r0);
    T = N;
  } else {
    const int cl = blockIdx.x;
    r0 = start[cl];
    nr = count[cl];
    if (nr == 0) return;
    if (tid < 27) {
      const int cx = cl / (ny * nz), cy = (cl / nz) % ny, cz = cl % nz;
      const int ax = (cx + tid / 9 - 1 + nx) % nx, ay = (cy + (tid / 3) % 3 - 1 + ny) % ny,
                az = (cz + tid % 3 - 1 + nz) % nz;
      const int q = (ax * ny + ay) * nz + az;
      cs[tid] = start[q];
      cp[tid + 1] = count[q];
    }
    __syncthreads();
    if (tid == 0) {
      cp[0] = 0;
      for (int k = 0; k < 27; ++k) cp[k + 1] += cp[k];
    }
    __syncthreads();
    T = cp[27];
  }
  if (tid == 0) out_of_box = 0;
  const bool masked = masks != nullptr && T <= 64L * cap;
  auto inside = [&](double x, double y, double z) {
    return x >= 0 && x <= bx && y >= 0 && y <= by && z >= 0 && z <= bz;
  };
  const double hx = 0.5 * bx, hy = 0.5 * by, hz = 0.5 * bz;
  const int n_ch = (int)((T + MM_NL_CH - 1) / MM_NL_CH);
  for (long rb = (long)blockIdx.y * (4 * MM_NL_R); rb < nr; rb += (long)gridDim.y * (4 * MM_NL_R)) {
    long id[MM_NL_R], base[MM_NL_R];
    double xi[MM_NL_R], yi[MM_NL_R], zi[MM_NL_R];
    int n[MM_NL_R];
    bool on[MM_NL_R];
#pragma unroll
    for (int r = 0; r < MM_NL_R; ++r) {
      const long k = rb + MM_NL_R * wave + r;
      on[r] = k < nr;
      id[r] = r0 + (on[r] ? k : 0);
      n[r] = 0;
      base[r] = FILL ? rowptr[id[r]] : 0;
      if (!(FILL && masked)) {
        xi[r] = pos[3 * id[r]];
        yi[r] = pos[3 * id[r] + 1];
        zi[r] = pos[3 * id[r] + 2];
      }
    }
    for (int ch = 0; ch < n_ch; ++ch) {
      const long c0 = (long)ch * MM_NL_CH;
      const int m = (int)min((long)MM_NL_CH, T - c0);
      if (n_ch > 1 || rb == (long)blockIdx.y * (4 * MM_NL_R)) {   // a single chunk stays staged
        __syncthreads();
        for (int k = tid; k < m; k += 256) {
          long j;
          if (brute) {
            j = c0 + k;
          } else {
            const int g = (int)c0 + k;
            int lo = 0, hi = 26;   // last cell with cp <= g
            while (lo < hi) {
              const int mid = (lo + hi + 1) >> 1;
              if (cp[mid] <= g) lo = mid;
              else hi = mid - 1;
            }
            j = (long)cs[lo] + (g - cp[lo]);
          }
          sj[k] = (int)j;
          if (!(FILL && masked)) {
            const double x = pos[3 * j], y = pos[3 * j + 1], z = pos[3 * j + 2];
            sx[k] = x;
            sy[k] = y;
            sz[k] = z;
            if (!inside(x, y, z)) out_of_box = 1;
          }
        }
        __syncthreads();
      }
      // receivers are candidates of their own cell: every coordinate of the tests has been looked at, the receivers'
      // possibly in another stage of the candidates
      bool general = out_of_box != 0;
      if (!(FILL && masked)) {
#pragma unroll
        for (int r = 0; r < MM_NL_R; ++r) general |= !inside(xi[r], yi[r], zi[r]);
      }
      unsigned long long mine[MM_NL_R];   // lane s: the ballot of step s of this chunk
#pragma unroll
      for (int r = 0; r < MM_NL_R; ++r) {
        mine[r] = 0;
        if (FILL && masked && 64 * lane < m) mine[r] = masks[id[r] * cap + c0 / 64 + lane];
      }
      for (int s = 0; 64 * s < m; ++s) {
        const int k = 64 * s + lane;
        const bool in = k < m;
        const int j = sj[in ? k : 0];
        unsigned long long b[MM_NL_R];
        if (FILL && masked) {
#pragma unroll
          for (int r = 0; r < MM_NL_R; ++r)   // s is uniform: the word goes to scalar registers
            b[r] = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)mine[r], s) |
                   (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(mine[r] >> 32), s) << 32;
        } else {
          const double xj = sx[in ? k : 0], yj = sy[in ? k : 0], zj = sz[in ? k : 0];
          auto test = [&](auto mic) {
#pragma unroll
            for (int r = 0; r < MM_NL_R; ++r) {
#pragma clang fp contract(off)
              const double dx = mic(xi[r] - xj, bx, hx);
              const double dy = mic(yi[r] - yj, by, hy);
              const double dz = mic(zi[r] - zj, bz, hz);
              const double dd = (dx * dx + dy * dy) + dz * dz;
              b[r] = __ballot(in & (dd < r2) & (j != (int)id[r]));
            }
          };
          if (general) test([](double v, double L, double h) { return mm_mic(v, L, h); });
          else test([](double v, double L, double h) { return mm_mic_in_box(v, L, h); });
        }
#pragma unroll
        for (int r = 0; r < MM_NL_R; ++r) {
          if (FILL) {
            if (on[r] & (int)((b[r] >> lane) & 1ull))
              send[base[r] + n[r] + __builtin_amdgcn_mbcnt_hi((unsigned)(b[r] >> 32),
                                                              __builtin_amdgcn_mbcnt_lo((unsigned)b[r], 0))] = j;
          } else {
            mine[r] = lane == s ? b[r] : mine[r];
          }
          n[r] += __popcll(b[r]);
        }
      }
      if (!FILL && masked) {
#pragma unroll
        for (int r = 0; r < MM_NL_R; ++r)
          if (on[r] && 64 * lane < m) masks[id[r] * cap + c0 / 64 + lane] = mine[r];
      }
    }
    if (!FILL && lane == 0) {
#pragma unroll
      for (int r = 0; r < MM_NL_R; ++r)
        if (on[r]) NN[id[r]] = n[r];
    }
  }
}

// The same for boxes of thinly filled cells (gases, slabs and droplets in vacuum), where a workgroup per cell has few
// receivers to share the candidates and many cells to find empty: a wave per receiver.  Lanes 0 .. 26 look up the
// cells, then the wave tests 64 candidates at a time from global memory.  Bound by the latency of that chain.
// Neighbour build, a thread per receiver -> workgroup per cell -> wave per receiver, us: 100,000 atoms of which a cell
// holds 0.1: 161 -> 1,314 -> 163; 1: 192 -> 598 -> 175; 3.7: 265 -> 320 -> 198; 6.4: 343 -> 247 -> 223; 9.4: 395 ->
// 232 -> 258; a droplet of 20,000 atoms in 10^6 cells: 429 -> 753 -> 146.
#define MM_NL_WAVE_WGS (1L << 20)   // workgroups of a launch at most; the waves stride over the receivers

template <bool FILL>
__global__ void __launch_bounds__(256) mm_nl_wave_kernel(const double* __restrict__ pos, const int* __restrict__ cell,
                                                         long N, double bx, double by, double bz, int nx, int ny,
                                                         int nz, const int* __restrict__ start,
                                                         const int* __restrict__ count, double r2,
                                                         int* __restrict__ NN, const long* __restrict__ rowptr,
                                                         int* __restrict__ send,
                                                         unsigned long long* __restrict__ masks, int cap) {
  __shared__ int s_end[4][32], s_off[4][32];   // per cell: candidates up to its end, first atom - candidates before it
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const double hx = 0.5 * bx, hy = 0.5 * by, hz = 0.5 * bz;
  for (long i = (long)blockIdx.x * 4 + wave; i < N; i += (long)gridDim.x * 4) {
    const long base = FILL ? rowptr[i] : 0;
    if (FILL && rowptr[i + 1] == base) continue;
    int st = 0, ct = 0;
    if (lane < 27) {
      const int ax = (cell[3 * i] + lane / 9 - 1 + nx) % nx, ay = (cell[3 * i + 1] + (lane / 3) % 3 - 1 + ny) % ny,
                az = (cell[3 * i + 2] + lane % 3 - 1 + nz) % nz;
      const int q = (ax * ny + ay) * nz + az;
      st = start[q];
      ct = count[q];
    }
    const double xi = pos[3 * i], yi = pos[3 * i + 1], zi = pos[3 * i + 2];
    int inc = ct;
#pragma unroll
    for (int d = 1; d < 32; d <<= 1) {
      const int u = __shfl_up(inc, d);
      if (lane >= d) inc += u;
    }
    const int T = __shfl(inc, 31);   // lanes 27 .. 31 add nothing
    mm_wave_lds_sync();              // the previous receiver's words have been read
    if (lane < 32) {
      s_end[wave][lane] = inc;
      s_off[wave][lane] = st - (inc - ct);
    }
    mm_wave_lds_sync();
    const bool masked = masks != nullptr && T <= 64L * cap;
    int n = 0;
    for (int s = 0; 64 * s < T; ++s) {
      const int g = 64 * s + lane;
      const bool in = g < T;
      int lo = 0, hi = 26;   // first cell that ends beyond g
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (s_end[wave][mid] > g) hi = mid;
        else lo = mid + 1;
      }
      const long j = in ? g + s_off[wave][lo] : i;
      unsigned long long b;
      if (FILL && masked) {
        b = masks[i * cap + s];
      } else {
#pragma clang fp contract(off)
        const double dx = mm_mic(xi - pos[3 * j], bx, hx);
        const double dy = mm_mic(yi - pos[3 * j + 1], by, hy);
        const double dz = mm_mic(zi - pos[3 * j + 2], bz, hz);
        const double dd = (dx * dx + dy * dy) + dz * dz;
        b = __ballot(dd < r2 && j != i);
        if (!FILL && masked && lane == 0) masks[i * cap + s] = b;
      }
      if (FILL && ((b >> lane) & 1ull))
        send[base + n + __builtin_amdgcn_mbcnt_hi((unsigned)(b >> 32),
                                                  __builtin_amdgcn_mbcnt_lo((unsigned)b, 0))] = (int)j;
      n += __popcll(b);
    }
    if (!FILL && lane == 0) NN[i] = n;
  }
}

// Which kernel takes a box.  brute: 16 receivers per workgroup.  A workgroup per cell where a cell holds MM_NL_MEAN
// atoms or more on average (figures above), a cell's receivers shared by up to 8 workgroups while the cells alone give
// the GPU fewer than 4 workgroups per CU; a wave per receiver in thinner boxes, and in boxes of so many cells that a
// launch with a workgroup each would exceed the 2^32 threads of a launch.
#define MM_NL_MEAN 8
template <bool FILL>
static void nl_pairs_launch(const double* pos, const int* cell, long N, const double* box, const int* ncell,
                            const int* start, const int* count, double r2, int brute, int* NN, const long* rowptr,
                            int* send, unsigned long long* masks, int cap, hipStream_t stream) {
  const long cells = (long)ncell[0] * ncell[1] * ncell[2];
  if (!brute && (N < MM_NL_MEAN * cells || cells >= (1L << 23))) {
    hipLaunchKernelGGL(mm_nl_wave_kernel<FILL>, dim3((unsigned)min((N + 3) / 4, MM_NL_WAVE_WGS)), dim3(256), 0, stream,
                       pos, cell, N, box[0], box[1], box[2], ncell[0], ncell[1], ncell[2], start, count, r2, NN,
                       rowptr, send, masks, cap);
    return;
  }
  dim3 grid((unsigned)((N + 4 * MM_NL_R - 1) / (4 * MM_NL_R)));
  if (!brute) {
    unsigned y = 1;
    while (y < 8 && cells * y < 1024) y *= 2;
    grid = dim3((unsigned)cells, y);
  }
  hipLaunchKernelGGL(mm_nl_pairs_kernel<FILL>, grid, dim3(256), 0, stream, pos, N, box[0], box[1], box[2], ncell[0],
                     ncell[1], ncell[2], start, count, r2, brute, NN, rowptr, send, masks, cap);
}

extern "C" int mm_nl_workspace_bytes(long N, size_t* bytes) {
  MM_CHECK_ARG(N >= 0 && N < (1L << 31) && bytes, "bad sizes");
  size_t a = 0, b = 0;
  hipcub::DeviceRadixSort::SortPairs(nullptr, a, (const long long*)nullptr, (long long*)nullptr,
                                     (const long long*)nullptr, (long long*)nullptr, (int)N, 0, 30);
  hipcub::DeviceScan::ExclusiveSum(nullptr, b, (const long*)nullptr, (long*)nullptr, (int)N + 1);
  *bytes = (a > b ? a : b) + 256;
  return MM_OK;
}

extern "C" int mm_nl_prepare(const double* pos_in, long N, const double* box, const int* ncell, const double* cs,
                             double* pos_w, int* cell, long long* key, long long* idx, hipStream_t stream) {
  MM_CHECK_ARG(N >= 0 && box && ncell && cs, "bad arguments");
  for (int k = 0; k < 3; ++k) MM_CHECK_ARG(ncell[k] >= 1 && ncell[k] <= 1024, "ncell out of range (10-bit Morton)");
  if (N == 0) return MM_OK;
  hipLaunchKernelGGL(mm_nl_prepare_kernel, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, stream, pos_in, N, box[0],
                     box[1], box[2], cs[0], cs[1], cs[2], ncell[0], ncell[1], ncell[2], pos_w, cell, key, idx);
  return mm::launch_status("mm_nl_prepare");
}

extern "C" int mm_nl_sort(const long long* key_in, long long* key_out, const long long* idx_in, long long* perm,
                          long N, void* ws, size_t ws_bytes, hipStream_t stream) {
  MM_CHECK_ARG(N >= 0 && N < (1L << 31), "bad sizes");
  if (N == 0) return MM_OK;
  size_t need = 0;
  hipcub::DeviceRadixSort::SortPairs(nullptr, need, key_in, key_out, idx_in, perm, (int)N, 0, 30, stream);
  MM_CHECK_ARG(ws_bytes >= need, "workspace too small");
  if (hipcub::DeviceRadixSort::SortPairs(ws, need, key_in, key_out, idx_in, perm, (int)N, 0, 30, stream) !=
      hipSuccess)
    return mm::launch_status("mm_nl_sort");
  return mm::launch_status("mm_nl_sort");
}

extern "C" int mm_nl_gather(const long long* perm, long N, const double* pos_w, const int* cell, const int* spec_in,
                            double* pos_s, int* cell_s, int* spec_s, hipStream_t stream) {
  MM_CHECK_ARG(N >= 0, "bad sizes");
  if (N == 0) return MM_OK;
  hipLaunchKernelGGL(mm_nl_gather_kernel, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, stream, perm, N, pos_w, cell,
                     spec_in, pos_s, cell_s, spec_s);
  return mm::launch_status("mm_nl_gather");
}

extern "C" int mm_nl_cell_ranges(const int* cell_s, long N, const int* ncell, int* start, int* count,
                                 hipStream_t stream) {
  MM_CHECK_ARG(N >= 0 && ncell, "bad arguments");
  const int ncells = ncell[0] * ncell[1] * ncell[2];
  hipLaunchKernelGGL(mm_fill_i32_kernel_nl, dim3((ncells + 255) / 256), dim3(256), 0, stream, start, ncells, (int)N);
  hipLaunchKernelGGL(mm_fill_i32_kernel_nl, dim3((ncells + 255) / 256), dim3(256), 0, stream, count, ncells, 0);
  if (N > 0)
    hipLaunchKernelGGL(mm_nl_ranges_kernel, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, stream, cell_s, N,
                       ncell[1], ncell[2], start, count);
  hipLaunchKernelGGL(mm_nl_counts_kernel, dim3((ncells + 255) / 256), dim3(256), 0, stream, ncells, start, count, N);
  return mm::launch_status("mm_nl_cell_ranges");
}

extern "C" int mm_nl_count_masked(const double* pos_s, const int* cell_s, long N, const double* box, const int* ncell,
                                  const int* start, const int* count, double r2, int brute, int* NN,
                                  unsigned long long* masks, int cap, hipStream_t stream) {
  MM_CHECK_ARG(N >= 0 && N < (1L << 31) && box && ncell, "bad arguments");
  MM_CHECK_ARG(cap >= 0 && (cap == 0 || masks), "cap words per atom need the mask buffer");
  if (N == 0) return MM_OK;
  nl_pairs_launch<false>(pos_s, cell_s, N, box, ncell, start, count, r2, brute, NN, nullptr, nullptr,
                         cap ? masks : nullptr, cap, stream);
  return mm::launch_status("mm_nl_count");
}

extern "C" int mm_nl_count(const double* pos_s, const int* cell_s, long N, const double* box, const int* ncell,
                           const int* start, const int* count, double r2, int brute, int* NN, hipStream_t stream) {
  return mm_nl_count_masked(pos_s, cell_s, N, box, ncell, start, count, r2, brute, NN, nullptr, 0, stream);
}

extern "C" int mm_nl_scan(const int* NN, long* rowptr, long N, void* ws, size_t ws_bytes, hipStream_t stream) {
  MM_CHECK_ARG(N >= 0 && N < (1L << 31), "bad sizes");
  // rowptr[0] = 0, rowptr[i + 1] = sum_{j <= i} NN[j]: exclusive scan of NN widened to int64, over N + 1 items
  // (the last input item is a zero appended by the widening iterator)
  struct Widen {
    const int* p;
    long n;
    __host__ __device__ long operator()(const long& i) const { return i < n ? (long)p[i] : 0L; }
  };
  hipcub::CountingInputIterator<long> cnt(0);
  hipcub::TransformInputIterator<long, Widen, hipcub::CountingInputIterator<long>> it(cnt, Widen{NN, N});
  size_t need = 0;
  hipcub::DeviceScan::ExclusiveSum(nullptr, need, it, rowptr, (int)N + 1, stream);
  MM_CHECK_ARG(ws_bytes >= need, "workspace too small");
  hipcub::DeviceScan::ExclusiveSum(ws, need, it, rowptr, (int)N + 1, stream);
  return mm::launch_status("mm_nl_scan");
}

// ------------------------------------------------------------------------------------------------------------
// Allocation-free receiver-CSR scan (no counterpart in the reference).  mm_nl_scan_noalloc gives the result of
// mm_nl_scan (rowptr[0] = 0, rowptr[i + 1] = sum_{j <= i} NN[j], int64) without a workspace argument, for callers
// that cannot allocate one (code under HIP-graph capture, serving loops).  Its tile partials live in `scratch`, a
// file-scope device array that every GPU the library runs on holds until the process ends:
//   * N + 1 <= MM_SCAN_MAX_TILES * MM_SCAN_TILE = 134,217,728 counts (larger N is rejected with MM_ERANGE);
//   * the array's device address is looked up once per device (hipGetSymbolAddress, first call on that device);
//   * every partial is written before it is read within one call, so nothing needs clearing between calls;
//   * calls that overlap on one GPU (different streams) share the array and race.
// Three kernels: per-tile sums -> one block scans the tile sums in place -> per-tile scan plus its offset.
#define MM_SCAN_THREADS 256
#define MM_SCAN_ITEMS 16
#define MM_SCAN_TILE (MM_SCAN_THREADS * MM_SCAN_ITEMS)
#define MM_SCAN_MAX_TILES 32768
#define MM_SCAN_OFFSET_THREADS 1024

static __device__ __align__(256) long long scratch[MM_SCAN_MAX_TILES];

// item i of the scan: NN[i] for i < N, 0 for i = N (the appended zero that makes rowptr[N] the total)
__device__ __forceinline__ long long mm_scan_item(const int* __restrict__ NN, long N, long i) {
  return i < N ? (long long)NN[i] : 0LL;
}

// In-place inclusive scan of v[0..n) (n = blockDim.x threads, one value each) in LDS; returns the inclusive value
// of this thread.
__device__ __forceinline__ long long mm_block_inclusive_scan(long long x, long long* lds) {
  const int t = threadIdx.x;
  lds[t] = x;
  __syncthreads();
  for (int d = 1; d < (int)blockDim.x; d <<= 1) {
    const long long y = t >= d ? lds[t - d] : 0LL;
    __syncthreads();
    lds[t] += y;
    __syncthreads();
  }
  return lds[t];
}

__global__ void __launch_bounds__(MM_SCAN_THREADS) mm_scan_tile_sums_kernel(const int* __restrict__ NN, long N,
                                                                             long long* __restrict__ part) {
  __shared__ long long lds[MM_SCAN_THREADS];
  const long base = (long)blockIdx.x * MM_SCAN_TILE + (long)threadIdx.x * MM_SCAN_ITEMS;
  long long s = 0;
#pragma unroll
  for (int k = 0; k < MM_SCAN_ITEMS; ++k) s += mm_scan_item(NN, N, base + k);
  const long long tot = mm_block_inclusive_scan(s, lds);
  if (threadIdx.x == MM_SCAN_THREADS - 1) part[blockIdx.x] = tot;
}

// One block: part[0..tiles) <- exclusive prefix sums of the tile sums.
__global__ void __launch_bounds__(MM_SCAN_OFFSET_THREADS) mm_scan_tile_offsets_kernel(long long* __restrict__ part,
                                                                                        int tiles) {
  __shared__ long long lds[MM_SCAN_OFFSET_THREADS];
  const int per = (tiles + MM_SCAN_OFFSET_THREADS - 1) / MM_SCAN_OFFSET_THREADS;
  const int lo = threadIdx.x * per;
  const int hi = min(lo + per, tiles);
  long long s = 0;
  for (int i = lo; i < hi; ++i) s += part[i];
  long long run = mm_block_inclusive_scan(s, lds) - s;     // exclusive prefix of this thread's run
  for (int i = lo; i < hi; ++i) {
    const long long v = part[i];
    part[i] = run;
    run += v;
  }
}

__global__ void __launch_bounds__(MM_SCAN_THREADS) mm_scan_tile_apply_kernel(const int* __restrict__ NN, long N,
                                                                              const long long* __restrict__ part,
                                                                              long* __restrict__ rowptr) {
  __shared__ long long lds[MM_SCAN_THREADS];
  const long base = (long)blockIdx.x * MM_SCAN_TILE + (long)threadIdx.x * MM_SCAN_ITEMS;
  long long v[MM_SCAN_ITEMS];
  long long s = 0;
#pragma unroll
  for (int k = 0; k < MM_SCAN_ITEMS; ++k) {
    v[k] = mm_scan_item(NN, N, base + k);
    s += v[k];
  }
  long long run = mm_block_inclusive_scan(s, lds) - s + part[blockIdx.x];
#pragma unroll
  for (int k = 0; k < MM_SCAN_ITEMS; ++k) {
    if (base + k <= N) rowptr[base + k] = (long)run;
    run += v[k];
  }
}

namespace {
std::mutex g_scratch_mu;
long long* g_scratch_ptr[64] = {};     // device address of `scratch` per device ordinal

int scan_scratch(long long** out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
    mm::set_error("mm_nl_scan_noalloc: no current HIP device");
    return MM_ELAUNCH;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      mm::set_error(std::string("mm_nl_scan_noalloc: hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
      return MM_ELAUNCH;
    }
    g_scratch_ptr[dev] = (long long*)p;
  }
  *out = g_scratch_ptr[dev];
  return MM_OK;
}
}  // namespace

extern "C" int mm_nl_scan_noalloc(const int* NN, long* rowptr, long N, hipStream_t stream) {
  MM_CHECK_ARG(N >= 0 && rowptr && (N == 0 || NN), "bad arguments");
  const long tiles = (N + 1 + MM_SCAN_TILE - 1) / MM_SCAN_TILE;
  if (tiles > MM_SCAN_MAX_TILES) {
    mm::set_error("mm_nl_scan_noalloc: N = " + std::to_string(N) + " exceeds the scratch limit N + 1 <= " +
                  std::to_string((long)MM_SCAN_MAX_TILES * MM_SCAN_TILE) + " (use mm_nl_scan with a workspace)");
    return MM_ERANGE;
  }
  long long* part = nullptr;
  const int rc = scan_scratch(&part);
  if (rc != MM_OK) return rc;
  hipLaunchKernelGGL(mm_scan_tile_sums_kernel, dim3((unsigned)tiles), dim3(MM_SCAN_THREADS), 0, stream, NN, N,
                     part);
  hipLaunchKernelGGL(mm_scan_tile_offsets_kernel, dim3(1), dim3(MM_SCAN_OFFSET_THREADS), 0, stream, part,
                     (int)tiles);
  hipLaunchKernelGGL(mm_scan_tile_apply_kernel, dim3((unsigned)tiles), dim3(MM_SCAN_THREADS), 0, stream, NN, N,
                     (const long long*)part, rowptr);
  return mm::launch_status("mm_nl_scan_noalloc");
}

extern "C" int mm_nl_fill_masked(const double* pos_s, const int* cell_s, long N, const double* box, const int* ncell,
                                 const int* start, const int* count, double r2, int brute, const long* rowptr,
                                 int* send, const unsigned long long* masks, int cap, hipStream_t stream) {
  MM_CHECK_ARG(N >= 0 && N < (1L << 31) && box && ncell, "bad arguments");
  MM_CHECK_ARG(cap >= 0 && (cap == 0 || masks), "cap words per atom need the mask buffer");
  if (N == 0) return MM_OK;
  nl_pairs_launch<true>(pos_s, cell_s, N, box, ncell, start, count, r2, brute, nullptr, rowptr, send,
                        cap ? (unsigned long long*)masks : nullptr, cap, stream);
  return mm::launch_status("mm_nl_fill");
}

extern "C" int mm_nl_fill(const double* pos_s, const int* cell_s, long N, const double* box, const int* ncell,
                          const int* start, const int* count, double r2, int brute, const long* rowptr, int* send,
                          hipStream_t stream) {
  return mm_nl_fill_masked(pos_s, cell_s, N, box, ncell, start, count, r2, brute, rowptr, send, nullptr, 0, stream);
}

// Per-step pair list of an MD run: the pairs of a skin list (built with r_cut = r_max + skin) whose current
// minimum-image distance is below r_max, in the skin list's order (the same test as mm_nl_pairs_kernel).
// One wave per receiver: 256 candidates per step, kept ones compacted in order with ballots and prefix popcounts.
// FILL = false: NN[i] = number of skin pairs of atom i within r_max; with flags != nullptr also flags[e] = 0 (kept)
// or -1 per skin pair.  FILL = true: the kept pairs in candidate order, send[rowptr[i] + k], and fidx[e] = the
// filtered index of skin pair e or -1; with FROM_FLAGS the keep decisions are read from fidx (the count pass's
// flags, written in place) instead of recomputed from the positions.
template <bool FILL, bool FROM_FLAGS>
__global__ void __launch_bounds__(256) mm_nl_filter_kernel(const double* __restrict__ pos, long N, double bx,
                                                           double by, double bz, const long* __restrict__ rp_s,
                                                           const int* __restrict__ send_s, double r2,
                                                           int* __restrict__ NN, const long* __restrict__ rowptr,
                                                           int* __restrict__ send, int* __restrict__ fidx) {
  const long i = blockIdx.x * 4L + (threadIdx.x >> 6);
  if (i >= N) return;
  const int lane = threadIdx.x & 63;
  double xi = 0, yi = 0, zi = 0;
  if (!FROM_FLAGS) {
    xi = pos[3 * i];
    yi = pos[3 * i + 1];
    zi = pos[3 * i + 2];
  }
  const long end = rp_s[i + 1];
  long n = 0;
  const long base = FILL ? rowptr[i] : 0;
  // 4 x 64 candidates per step: their loads are issued together (a lane past the row reads the row's last
  // candidate and keeps nothing), then the kept ones are compacted in candidate order, 64 at a time
  for (long e0 = rp_s[i]; e0 < end; e0 += 256) {
    int j[4];
    bool keep[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) j[k] = send_s[min(e0 + lane + 64 * k, end - 1)];
    if (FROM_FLAGS) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int flag = fidx[min(e0 + lane + 64 * k, end - 1)];
        keep[k] = (e0 + lane + 64 * k < end) & (flag >= 0);
      }
    } else {
      double px[4], py[4], pz[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        px[k] = pos[3 * (long)j[k]];
        py[k] = pos[3 * (long)j[k] + 1];
        pz[k] = pos[3 * (long)j[k] + 2];
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
#pragma clang fp contract(off)
        const double dx = mm_mic(xi - px[k], bx, 0.5 * bx);
        const double dy = mm_mic(yi - py[k], by, 0.5 * by);
        const double dz = mm_mic(zi - pz[k], bz, 0.5 * bz);
        const double dd = (dx * dx + dy * dy) + dz * dz;
        keep[k] = (e0 + lane + 64 * k < end) & (dd < r2) & (j[k] != i);
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const long e = e0 + lane + 64 * k;
      const unsigned long long m = __ballot(keep[k]);
      if (FILL) {
        const long slot = base + n + __popcll(m & ((1ull << lane) - 1ull));
        if (keep[k]) send[slot] = j[k];
        if (fidx && e < end) fidx[e] = keep[k] ? (int)slot : -1;
      } else if (fidx && e < end) {
        fidx[e] = keep[k] ? 0 : -1;
      }
      n += __popcll(m);
    }
  }
  if (!FILL && lane == 0) NN[i] = (int)n;
}

extern "C" int mm_nl_filter_count(const double* pos, long N, const double* box, const long* rp_s, const int* send_s,
                                  double r2, int* NN, int* flags, hipStream_t stream) {
  MM_CHECK_ARG(N >= 0 && box, "bad arguments");
  if (N == 0) return MM_OK;
  hipLaunchKernelGGL((mm_nl_filter_kernel<false, false>), dim3((unsigned)((N + 3) / 4)), dim3(256), 0, stream, pos,
                     N, box[0], box[1], box[2], rp_s, send_s, r2, NN, (const long*)nullptr, (int*)nullptr, flags);
  return mm::launch_status("mm_nl_filter_count");
}

extern "C" int mm_nl_filter_fill(const double* pos, long N, const double* box, const long* rp_s, const int* send_s,
                                 double r2, const long* rowptr, int* send, int* fidx, int from_flags,
                                 hipStream_t stream) {
  MM_CHECK_ARG(N >= 0 && box, "bad arguments");
  MM_CHECK_ARG(!from_flags || fidx, "from_flags needs the count pass's flags in filtered_index");
  if (N == 0) return MM_OK;
  if (from_flags)
    hipLaunchKernelGGL((mm_nl_filter_kernel<true, true>), dim3((unsigned)((N + 3) / 4)), dim3(256), 0, stream, pos,
                       N, box[0], box[1], box[2], rp_s, send_s, r2, (int*)nullptr, rowptr, send, fidx);
  else
    hipLaunchKernelGGL((mm_nl_filter_kernel<true, false>), dim3((unsigned)((N + 3) / 4)), dim3(256), 0, stream, pos,
                       N, box[0], box[1], box[2], rp_s, send_s, r2, (int*)nullptr, rowptr, send, fidx);
  return mm::launch_status("mm_nl_filter_fill");
}

// rev[e] = index of the pair (j, i) for every pair e = (i, j) of a symmetric CSR pair list (the MD driver's skin
// list), found by scanning row j; no sort and no memory beyond rev.  One wave per receiver i: the senders of 64 of
// its pairs and the bounds of their rows are loaded together, then each 16-lane quarter of the wave searches one
// pair's row, 256 candidates per round (16 loads per lane in flight).  Every sender occurs at most once in a row
// (one minimum image), so at most one lane writes each rev[e]; a pair without a reverse keeps the caller's fill.
__global__ void __launch_bounds__(256) mm_nl_reverse_kernel(long N, const long* __restrict__ rowptr,
                                                            const int* __restrict__ send, int* __restrict__ rev) {
  const long i = blockIdx.x * 4L + (threadIdx.x >> 6);
  if (i >= N) return;
  const int lane = threadIdx.x & 63, q = lane >> 4, lq = lane & 15;
  const long b0 = rowptr[i], b1 = rowptr[i + 1];
  for (long eb = b0; eb < b1; eb += 64) {
    // lanes past the row hold an empty range [0, 0)
    int s0 = 0, len = 0;
    if (eb + lane < b1) {
      const int j = send[eb + lane];
      s0 = (int)rowptr[j];
      len = (int)(rowptr[j + 1] - s0);
    }
    const int n = (int)min(64L, b1 - eb);
    for (int k = 0; k < n; k += 4) {
      const int src = k + q;                       // the pair this quarter searches: eb + src
      const int c0 = __shfl(s0, src), cl = __shfl(len, src);
      for (int c = 0; c < cl; c += 256) {
        int v[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) {
          const int x = c + 16 * t + lq;
          v[t] = x < cl ? send[c0 + x] : -1;
        }
#pragma unroll
        for (int t = 0; t < 16; ++t)
          if (v[t] == (int)i) rev[eb + src] = c0 + c + 16 * t + lq;
      }
    }
  }
}

extern "C" int mm_nl_reverse(const long* rowptr, const int* send, long N, long E, int* rev, hipStream_t stream) {
  MM_CHECK_ARG(N >= 0 && E >= 0 && (N == 0 || (rowptr && send && rev)), "bad arguments");
  if (E > 2147483647L) {
    mm::set_error("mm_nl_reverse: " + std::to_string(E) + " pairs exceed the int32 pair index");
    return MM_ERANGE;
  }
  if (N == 0 || E == 0) return MM_OK;
  hipLaunchKernelGGL(mm_nl_reverse_kernel, dim3((unsigned)((N + 3) / 4)), dim3(256), 0, stream, N, rowptr, send, rev);
  return mm::launch_status("mm_nl_reverse");
}
