// Equivariant linear maps of the node features on the matrix cores, at fp32 accuracy from bf16 products
// (v_mfma_f32_16x16x32_bf16, fp32 accumulation).
//
// Every node-level linear of the two layers is a set of 128x128 channel-mixing blocks applied to 128-channel rows
// of ir_mul features (one row per (node, component)): linear_up, linear (with the density division), skip_tp per
// species (fast_layers.SpeciesSkip, fast_layers.py:41-105 -- here the species rows are gathered by per-species
// row lists instead of computing every species and selecting), the product-block linear, and their transposes in
// the backward passes.  For each output component j of one launch:
//     out[out_row(r), comp_j] (= or +=) scale(r) * sum_q in[in_row(r), src_{j,q}] @ W[w_{j,q}]
//
// Split products.  Every fp32 operand is the sum of three bf16 values, x = x0 + x1 + x2 with x0 = bf16(x),
// x1 = bf16(x - x0), x2 = bf16(x - x0 - x1) (round to nearest even; the differences are exact in fp32), so that
// |x - x0 - x1 - x2| <= 2^-27 |x|.  A product a b is taken as the six bf16 products a_i b_j with i + j <= 2; the
// omitted ones are below 3 * 2^-24 |a b|, the size of an fp32 rounding, and every sum is accumulated in fp32.
// Six 16x16x32 bf16 products take 96 cycles against 256 for the same K = 32 in v_mfma_f32_16x16x4f32.  The
// weights are split once on the host; the input rows are split as they are loaded.
//
// Weights in registers.  A workgroup is 4 waves; each holds 32 of the 128 columns of a weight block (96 registers: 3
// planes x 4 K-steps x 2 tiles) and streams rows past them, 32 rows (a stage) at a time.  The rows of a stage are
// loaded coalesced by the whole workgroup, split once and written to LDS in operand order, one stage ahead of the
// products; a stage is 96 matrix instructions per wave on four independent sums.  The weights are the first operand,
// so that a lane ends with 4 consecutive columns of one row: 16-byte stores.
// Bound: the bf16 products and the rows' traffic, which are near each other (40 x 40 components, 131,072 rows: 0.85 ms
// of products at the 1.21 PFLOP/s of a large matrix product, 0.80 ms of traffic at the 4.67 TB/s of a large copy).
// Before, a workgroup staged the whole weight block (96 KiB) in LDS for 256 rows, and 16 waves read it again for every
// 16 rows: LDS reads cost as much as the products, and nothing of a workgroup's start and end overlapped.  Measured
// (us, before
// -> now; 16 components of 1 source, 16 of 2-3 sources, 40 of 1 source):
//      192 rows:  12.5 -> < 9     27 -> < 10    12.6 -> < 9     (launch calls take 9 us)
//    4,001 rows:   22 -> 20       40 -> 36       56 -> 39
//   16,384 rows:   83 -> 56      174 -> 146     163 -> 149
//  131,072 rows:  474 -> 452    1180 -> 1118   1167 -> 1134
// Several sources: NS stages share each load of a source's weights, with NS stages of sums held.  4 stages from two
// rounds of workgroups on (16 x 2 components, 131,072 rows: 849 us, 1115 us with 1 stage, 920 us with 2, 897 us with
// 3); below that 1 stage, for more workgroups (1,024 rows: 11 us, 19 us with 4).
// Weight blocks: plane p of block b at bf16 offset (3 b + p) 16384; element W[k][n], k = 32 t + 8 g + u, n = 16 nt + i,
// at (((t * 8 + nt) * 4 + g) * 16 + i) * 8 + u, so that lane (i, g) reads its 8 k-values of step t and tile nt as one
// 16-byte load, a wave 1 KiB.  The rows in LDS: 16-byte unit (row tile, plane, k / 8, row), the k / 8 groups 17 units
// apart: the 8-byte writes (32 lanes: one row) and the 16-byte reads (16 lanes: 16 rows) use every bank once.
// Components fastest in the grid: the workgroups of one row block run together, so an output row is written and an
// input row read by neighbouring workgroups.
#include "common.h"

#include <climits>

#define MM_LIN_MAX_COMP 48
#define MM_LIN_MAX_SRC 3
#define MM_LIN_NW 4          // waves per workgroup
#define MM_LIN_ROWS 32       // rows of a stage
#define MM_LIN_WG_ROWS 1024  // rows per workgroup at most
#define MM_LIN_AS 17         // LDS distance (16 B) of the k-groups of a row tile
#define MM_LIN_WG 512        // resident workgroups of the card (2 per CU)
#define MM_LIN_START 2       // cost of a workgroup's start, in stages
#define MM_LIN_NS 4          // stages per load of weights with several sources

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

struct MMLinComp {
  int n_src;
  int in_off[MM_LIN_MAX_SRC];   // float offset of the source chunk inside an input row
  int w_idx[MM_LIN_MAX_SRC];    // weight block index
  int out_off;                  // float offset of the output chunk inside an output row
};

struct MMLinArgs {
  const float* in;        // 16-byte aligned rows
  long in_stride;
  const int* in_rows;     // nullable: in row of logical row id
  float* out;
  long out_stride;
  const int* out_rows;    // nullable
  const uint4* W;         // weight blocks: 3 bf16 planes of 16384 values each (6144 x 16 B per block)
  const float* row_scale; // nullable: per logical row id
  int scale_mode;         // 0: scale = row_scale[id]; 1: scale = 1 / (row_scale[id] + 1)
  const int* list;        // nullable: per group g, list[g * list_stride + r] = logical row id
  const int* list_count;  // per group row count (device): with list, or alone for one group of rows 0 .. n - 1
  long list_stride;
  int n_rows;             // without list
  int w_group_stride;     // weight block offset of group g (species)
  int in_cb;              // 0: input rows component-major; n > 0: 16-channel-block-major rows [8][n][16], a
                          // source chunk at in_off = 128 k being component k of every block
  int accumulate;
  int n_comp;
  MMLinComp comp[MM_LIN_MAX_COMP];
};

// 16 B stores to rows that are only known to be float-aligned
typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));

// x = x0 + x1 + x2 (bf16, round to nearest even; both differences are exact in fp32)
__device__ __forceinline__ void mm_split3_bf16(const floatx4& x, bf16x4& x0, bf16x4& x1, bf16x4& x2) {
  x0 = __builtin_convertvector(x, bf16x4);
  const floatx4 r1 = x - __builtin_convertvector(x0, floatx4);
  x1 = __builtin_convertvector(r1, bf16x4);
  const floatx4 r2 = r1 - __builtin_convertvector(x1, floatx4);
  x2 = __builtin_convertvector(r2, bf16x4);
}

// NS: stages (32 rows) per weight load when a component has several sources.  n_st: stages per workgroup.
template <int NS>
__global__ void __launch_bounds__(64 * MM_LIN_NW, 2) mm_linear_kernel(MMLinArgs args, int n_st) {
  __shared__ uint4 Al[2][2 * 3 * 16 * MM_LIN_AS];   // [buffer][row tile][plane][k / 8][row], k-groups MM_LIN_AS apart
  __shared__ int s_in[MM_LIN_WG_ROWS], s_out[MM_LIN_WG_ROWS];
  __shared__ float s_sc[MM_LIN_WG_ROWS];
  const MMLinComp& cp = args.comp[blockIdx.x];   // kernel-argument memory, read with uniform indices
  const int grp = blockIdx.z;
  const int nrows = args.list_count ? min(args.list_count[grp], args.n_rows) : args.n_rows;
  const int row0 = blockIdx.y * n_st * MM_LIN_ROWS;
  if (row0 >= nrows) return;
  const int n = min(n_st * MM_LIN_ROWS, nrows - row0);   // rows of this workgroup
  const int nst = (n + MM_LIN_ROWS - 1) / MM_LIN_ROWS;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, i = lane & 15, g = lane >> 4;
  const int n_src = cp.n_src;

  // this thread's part of a stage: floats 4 k4 .. + 3 of rows tid >> 5, + 8, + 16, + 24
  const int k4 = tid & 31, rw = tid >> 5;
  const int cb = args.in_cb;
  const int koff = cb ? (k4 >> 2) * 16 * cb + 4 * (k4 & 3) : 4 * k4;
  floatx4 x[4];
  auto load = [&](int st, int q) {
    const float* __restrict__ p = args.in + (cb ? cp.in_off[q] >> 3 : cp.in_off[q]) + koff;   // 16 floats of 128
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = *(const floatx4*)(p + s_in[st * MM_LIN_ROWS + 8 * j + rw] * args.in_stride);
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      bf16x4 h[3];
      mm_split3_bf16(x[j], h[0], h[1], h[2]);
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        uint2* d = (uint2*)&Al[buf][(((j >> 1) * 3 + p) * 16 + (k4 >> 1)) * MM_LIN_AS + 8 * (j & 1) + rw];
        d[k4 & 1] = __builtin_bit_cast(uint2, h[p]);
      }
    }
  };

  bf16x8 B[4][2][3];
  auto load_w = [&](int q) {
    const uint4* __restrict__ Wg = args.W + (size_t)(cp.w_idx[q] + grp * args.w_group_stride) * 6144
                                  + (2 * wave * 4 + g) * 16 + i;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int p = 0; p < 3; ++p) B[t][c][p] = __builtin_bit_cast(bf16x8, Wg[p * 2048 + t * 512 + c * 64]);
  };

  // row indices and scales of the workgroup's rows (rows past the last one repeat it and are not stored); the first
  // weights are loaded behind the indices
  for (int r0 = 0; r0 < nst * MM_LIN_ROWS; r0 += 64 * MM_LIN_NW) {
    const int rr = row0 + min(r0 + tid, n - 1);
    const int id = args.list ? args.list[(size_t)grp * args.list_stride + rr] : rr;
    int ir = id, orow = id;
    float sc = 0.f;
    if (args.in_rows) ir = args.in_rows[id];
    if (args.out_rows) orow = args.out_rows[id];
    if (args.row_scale) sc = args.row_scale[id];
    if (r0 == 0) load_w(0);
    s_in[r0 + tid] = ir;
    s_out[r0 + tid] = orow;
    s_sc[r0 + tid] = !args.row_scale ? 1.f : args.scale_mode == 1 ? 1.f / (sc + 1.f) : sc;
  }
  __syncthreads();
  load(0, 0);
  put(0);
  __syncthreads();
  int buf = 0;
  for (int b = 0; b < nst; b += NS) {
    floatx4 acc[NS][2][2];
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int r = 0; r < 2; ++r) acc[s][r][0] = acc[s][r][1] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int q = 0; q < n_src; ++q) {
      if (n_src > 1 && b + q > 0) load_w(q);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        if (b + s >= nst) break;
        // the next stage of this workgroup: of this source, of the next source, of the next block of stages (after
        // the last one this stage again: a load without a branch leaves the weights' loads countable)
        const bool last_s = s == NS - 1 || b + s + 1 == nst, last_q = q + 1 == n_src;
        const bool more = !(last_s && last_q && b + NS >= nst);
        load(!more || !last_s ? b + s + (more ? 1 : 0) : last_q ? b + NS : b,
             !more || !last_s ? q : last_q ? 0 : q + 1);
        bf16x8 a[2][2][3];
        auto load_a = [&](int t) {
#pragma unroll
          for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int p = 0; p < 3; ++p)
              a[t & 1][r][p] = __builtin_bit_cast(bf16x8, Al[buf][((r * 3 + p) * 16 + 4 * t + g) * MM_LIN_AS + i]);
        };
        load_a(0);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          if (t < 3) load_a(t + 1);
          __builtin_amdgcn_sched_barrier(0);   // the reads of step t + 1 stay ahead of the products of step t
          // four independent sums; per sum the smallest terms first
#pragma unroll
          for (int k = 0; k < 6; ++k) {
            constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
              for (int c = 0; c < 2; ++c)
                acc[s][r][c] =
                    __builtin_amdgcn_mfma_f32_16x16x32_bf16(B[t][c][pb[k]], a[t & 1][r][pa[k]], acc[s][r][c], 0, 0, 0);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (more) {
          put(buf ^ 1);
          __syncthreads();
          buf ^= 1;
        }
      }
    }
    // weights as the first operand: lane (i, g) holds columns 4 g .. + 3 of row i of each tile
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      floatx4u* op[2];
      float sc[2];
      bool ok[2];
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const int rr = (b + s) * MM_LIN_ROWS + 16 * r + i;
        ok[r] = rr < n;
        const int rc = ok[r] ? rr : 0;
        op[r] = (floatx4u*)(args.out + s_out[rc] * args.out_stride + cp.out_off + 32 * wave + 4 * g);
        sc[r] = s_sc[rc];
      }
      if (args.accumulate) {
        floatx4 old[2][2];
#pragma unroll
        for (int r = 0; r < 2; ++r)
          if (ok[r]) {
            old[r][0] = op[r][0];
            old[r][1] = op[r][4];
          }
#pragma unroll
        for (int r = 0; r < 2; ++r)
          if (ok[r]) {
            op[r][0] = old[r][0] + sc[r] * acc[s][r][0];
            op[r][4] = old[r][1] + sc[r] * acc[s][r][1];
          }
      } else {
#pragma unroll
        for (int r = 0; r < 2; ++r)
          if (ok[r]) {
            op[r][0] = sc[r] * acc[s][r][0];
            op[r][4] = sc[r] * acc[s][r][1];
          }
      }
    }
  }
}

// Flat argument form for the C ABI: comp table as int arrays [n_comp][MM_LIN_MAX_SRC] etc.
extern "C" int mm_linear(const float* in, long in_stride, const int* in_rows, float* out, long out_stride,
                         const int* out_rows, const void* W, const float* row_scale, int scale_mode,
                         const int* list, const int* list_count, long list_stride, int n_groups, int w_group_stride,
                         int n_rows_max, int accumulate, int n_comp, const int* comp_nsrc, const int* comp_in_off,
                         const int* comp_w_idx, const int* comp_out_off, int in_cb, hipStream_t stream) {
  MM_CHECK_ARG(n_comp >= 1 && n_comp <= MM_LIN_MAX_COMP, "n_comp out of range");
  MM_CHECK_ARG(n_groups >= 1 && n_rows_max >= 0, "bad sizes");
  MM_CHECK_ARG(list == nullptr || list_count != nullptr, "a row list needs its counts");
  MM_CHECK_ARG(list != nullptr || list_count == nullptr || n_groups == 1, "a device row count without a list is for "
               "one group");
  MM_CHECK_ARG(list != nullptr || n_groups == 1, "groups need row lists");
  MM_CHECK_ARG(in_stride % 4 == 0, "input row stride must be a multiple of 4 floats");
  MM_CHECK_ARG(in_cb >= 0 && (in_cb == 0 || in_stride >= 128L * in_cb), "channel-block-major rows: in_cb >= 0 "
               "components per block, rows of at least 128 in_cb floats");
  MMLinArgs a;
  a.in = in;
  a.in_stride = in_stride;
  a.in_rows = in_rows;
  a.out = out;
  a.out_stride = out_stride;
  a.out_rows = out_rows;
  a.W = (const uint4*)W;
  a.row_scale = row_scale;
  a.scale_mode = scale_mode;
  a.list = list;
  a.list_count = list_count;
  a.list_stride = list_stride;
  a.n_rows = n_rows_max;
  a.w_group_stride = w_group_stride;
  a.in_cb = in_cb;
  a.accumulate = accumulate;
  a.n_comp = n_comp;
  for (int j = 0; j < n_comp; ++j) {
    MM_CHECK_ARG(comp_nsrc[j] >= 1 && comp_nsrc[j] <= MM_LIN_MAX_SRC, "n_src out of range");
    a.comp[j].n_src = comp_nsrc[j];
    for (int q = 0; q < MM_LIN_MAX_SRC; ++q) {
      a.comp[j].in_off[q] = comp_in_off[j * MM_LIN_MAX_SRC + q];
      a.comp[j].w_idx[q] = comp_w_idx[j * MM_LIN_MAX_SRC + q];
      MM_CHECK_ARG(q >= comp_nsrc[j] || a.comp[j].in_off[q] % 4 == 0, "source offsets must be multiples of 4");
      MM_CHECK_ARG(q >= comp_nsrc[j] || in_cb == 0 || (a.comp[j].in_off[q] % 128 == 0 &&
                   a.comp[j].in_off[q] / 128 < in_cb), "channel-block-major sources are whole components < in_cb");
    }
    a.comp[j].out_off = comp_out_off[j];
  }
  if (n_rows_max == 0) return MM_OK;
  bool multi = false;
  for (int j = 0; j < n_comp; ++j) multi |= comp_nsrc[j] > 1;
  // stages per workgroup: the least time in rounds of resident workgroups, a workgroup costing its stages and
  // MM_LIN_START more (first indices, rows and weights).  40 components, 16,384 rows: 149 us; with the fewest
  // workgroups (640 of 32 stages) 182-205 us, with at least 1,024 workgroups 174 us
  const long stages = (n_rows_max + MM_LIN_ROWS - 1) / MM_LIN_ROWS;
  const int ns = multi && stages * n_comp >= 2L * MM_LIN_WG ? MM_LIN_NS : 1;
  long n_st = ns, best = LONG_MAX;
  for (long k = ns; k <= MM_LIN_WG_ROWS / MM_LIN_ROWS; k += ns) {
    const long wgs = (stages + k - 1) / k * n_comp, cost = (wgs + MM_LIN_WG - 1) / MM_LIN_WG * (k + MM_LIN_START);
    if (cost < best) best = cost, n_st = k;
  }
  const dim3 grid(n_comp, (unsigned)((stages + n_st - 1) / n_st), n_groups);
  if (ns == MM_LIN_NS)
    hipLaunchKernelGGL(mm_linear_kernel<MM_LIN_NS>, grid, dim3(64 * MM_LIN_NW), 0, stream, a, (int)n_st);
  else
    hipLaunchKernelGGL(mm_linear_kernel<1>, grid, dim3(64 * MM_LIN_NW), 0, stream, a, (int)n_st);
  return mm::launch_status("mm_linear");
}
