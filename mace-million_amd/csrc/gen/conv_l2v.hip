// generated by mace_onegpu/codegen.py -- layer-2 edge convolution, backward, on the matrix cores
#include "../common.h"
#include "polar.h"

typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));
typedef unsigned uint2v __attribute__((ext_vector_type(2)));
typedef unsigned uint4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned mm_load_u32(const unsigned char* p) {
  unsigned v;
  __builtin_memcpy(&v, p, 4);
  return v;
}

// Slots of the distinct senders of each group of 4 consecutive receivers (spatially close in the Morton order, so
// they share most senders): e_slot[e] = the slot of edge e's sender in its group (255: none, the sender found no slot
// or the edge lies beyond the group's first 1024), g_send[group][slot] = the sender, g_n[group] = slots in use.
// Once per chunk, for the 8 channel blocks of the backward (which hashed the senders 8 times before).
#define MM_SLOT_HASH 2048
extern "C" __global__ void __launch_bounds__(256)
mm_sender_slots_kernel(const int* __restrict__ rowptr, int nC, const int* __restrict__ send,
    unsigned char* __restrict__ e_slot, int* __restrict__ g_send, int* __restrict__ g_n) {
  __shared__ int hkey[MM_SLOT_HASH];
  __shared__ unsigned char hslot[MM_SLOT_HASH];
  __shared__ int nslot;
  const int i0 = blockIdx.x * 4, tid = threadIdx.x;
  const int E0 = rowptr[i0], nE = rowptr[min(i0 + 4, nC)] - E0, nH = min(nE, 1024);
  for (int h = tid; h < MM_SLOT_HASH; h += 256) hkey[h] = -1;
  if (tid == 0) nslot = 0;
  __syncthreads();
  for (int j = tid; j < nH; j += 256) {   // at most 1024 keys: the probing ends at a free entry
    const int s = send[E0 + j];
    unsigned h = ((unsigned)s * 2654435761u) >> 21;
    while (true) {
      const int prev = atomicCAS(&hkey[h], -1, s);
      if (prev == -1) {
        const int sl = atomicAdd(&nslot, 1);
        hslot[h] = sl < 208 ? (unsigned char)sl : 255;
        if (sl < 208) g_send[(size_t)blockIdx.x * 208 + sl] = s;
      }
      if (prev == -1 || prev == s) break;
      h = (h + 1) & (MM_SLOT_HASH - 1);
    }
  }
  __syncthreads();
  for (int j = tid; j < nE; j += 256) {
    unsigned char sl = 255;
    if (j < nH) {
      const int s = send[E0 + j];
      unsigned h = ((unsigned)s * 2654435761u) >> 21;
      while (hkey[h] != s) h = (h + 1) & (MM_SLOT_HASH - 1);
      sl = hslot[h];
    }
    e_slot[E0 + j] = sl;
  }
  if (tid == 0) g_n[blockIdx.x] = min(nslot, 208);
}

extern "C" int mm_sender_slots(const int* rowptr, int nC, const int* send, unsigned char* e_slot, int* g_send, int* g_n,
    hipStream_t stream) {
  MM_CHECK_ARG(nC >= 0, "bad sizes");
  if (nC == 0) return MM_OK;
  hipLaunchKernelGGL(mm_sender_slots_kernel, dim3((nC + 4 - 1) / 4), dim3(256), 0, stream, rowptr, nC, send,
                     e_slot, g_send, g_n);
  return mm::launch_status("mm_sender_slots");
}

extern "C" __global__ void __launch_bounds__(256, 2)
mm_conv2_bwd_vec_kernel(const int* __restrict__ rowptr, int nC, const floatx4* __restrict__ e_pk,
    const floatx4* __restrict__ e_u, const float* __restrict__ X, int x_stride,
    const floatx4* __restrict__ tab, int tab_cb_stride, float inv_h,
    const float* __restrict__ gA, float* __restrict__ part, long part_stride, float* __restrict__ gX,
    const unsigned char* __restrict__ e_slot, const int* __restrict__ g_send,
    const int* __restrict__ g_n) {
  const int cb = mm_xcd_channel_block();
  __shared__ uint4v ya_all[1152];   // per wave: [type][degree][edge][piece] operand rows
  const int grp = blockIdx.x >> 3, i = grp * 4 + (threadIdx.x >> 6);
  __shared__ floatx4 gxs4[3328];   // [slot][component][16 channels]
  __shared__ int ssend[208];
  float* __restrict__ gxs = (float*)gxs4;
  const int ns = g_n[grp];
  const int ir = min(i, nC - 1);   // waves past the last receiver prepare for it and take no edges
  const int lane = threadIdx.x & 63, cl = lane & 15, eg = lane >> 4;
  uint4v* __restrict__ ya = ya_all + (threadIdx.x >> 6) * 288;
  const int c = cb * 16 + cl;
  const int e0 = rowptr[ir], e1 = i < nC ? rowptr[ir + 1] : e0;
  const char* __restrict__ tcb = (const char*)(tab + (size_t)cb * tab_cb_stride);
  const float* __restrict__ gp = gA + (size_t)ir * 5120 + c;
  float g0 = gp[0];
  float g1 = gp[128];
  float g2 = gp[256];
  float g3 = gp[384];
  float g4 = gp[512];
  float g5 = gp[640];
  float g6 = gp[768];
  float g7 = gp[896];
  float g8 = gp[1024];
  float g9 = gp[1152];
  float g10 = gp[1280];
  float g11 = gp[1408];
  float g12 = gp[1536];
  float g13 = gp[1664];
  float g14 = gp[1792];
  float g15 = gp[1920];
  float g16 = gp[2048];
  float g17 = gp[2176];
  float g18 = gp[2304];
  float g19 = gp[2432];
  float g20 = gp[2560];
  float g21 = gp[2688];
  float g22 = gp[2816];
  float g23 = gp[2944];
  float g24 = gp[3072];
  float g25 = gp[3200];
  float g26 = gp[3328];
  float g27 = gp[3456];
  float g28 = gp[3584];
  float g29 = gp[3712];
  float g30 = gp[3840];
  float g31 = gp[3968];
  float g32 = gp[4096];
  float g33 = gp[4224];
  float g34 = gp[4352];
  float g35 = gp[4480];
  float g36 = gp[4608];
  float g37 = gp[4736];
  float g38 = gp[4864];
  float g39 = gp[4992];
  // power-of-two scale of this channel's constants into the fp16 range
  const float mx0 = fmaxf(fmaxf(fabsf(g6), fabsf(g7)), fmaxf(fmaxf(fabsf(g4), fabsf(g5)), fmaxf(fmaxf(fabsf(g2), fabsf(g3)), fmaxf(fmaxf(fabsf(g0), fabsf(g1)), 0.f))));
  const float mx1 = fmaxf(fmaxf(fabsf(g14), fabsf(g15)), fmaxf(fmaxf(fabsf(g12), fabsf(g13)), fmaxf(fmaxf(fabsf(g10), fabsf(g11)), fmaxf(fmaxf(fabsf(g8), fabsf(g9)), mx0))));
  const float mx2 = fmaxf(fmaxf(fabsf(g22), fabsf(g23)), fmaxf(fmaxf(fabsf(g20), fabsf(g21)), fmaxf(fmaxf(fabsf(g18), fabsf(g19)), fmaxf(fmaxf(fabsf(g16), fabsf(g17)), mx1))));
  const float mx3 = fmaxf(fmaxf(fabsf(g30), fabsf(g31)), fmaxf(fmaxf(fabsf(g28), fabsf(g29)), fmaxf(fmaxf(fabsf(g26), fabsf(g27)), fmaxf(fmaxf(fabsf(g24), fabsf(g25)), mx2))));
  const float mx4 = fmaxf(fmaxf(fabsf(g38), fabsf(g39)), fmaxf(fmaxf(fabsf(g36), fabsf(g37)), fmaxf(fmaxf(fabsf(g34), fabsf(g35)), fmaxf(fmaxf(fabsf(g32), fabsf(g33)), mx3))));
  const int gex = max(__float_as_int(mx4) >> 23, 40);
  const float gsc = __int_as_float((265 - gex) << 23);
  const float gun = __int_as_float((gex - 24) << 23);   // 1 / (gsc MM_POLAR_SCALE)
  const float U0_0 = g0 * gsc * MM_POLAR_SCALE;   // l2 = 0: the same u for every edge
  const float U3_1 = g5 * gsc * MM_POLAR_SCALE;   // l2 = 0: the same u for every edge
  const float U3_2 = g6 * gsc * MM_POLAR_SCALE;   // l2 = 0: the same u for every edge
  const float U3_3 = g7 * gsc * MM_POLAR_SCALE;   // l2 = 0: the same u for every edge
  g0 *= gsc;
  g1 *= gsc;
  g2 *= gsc;
  g3 *= gsc;
  g4 *= gsc;
  g5 *= gsc;
  g6 *= gsc;
  g7 *= gsc;
  g8 *= gsc;
  g9 *= gsc;
  g10 *= gsc;
  g11 *= gsc;
  g12 *= gsc;
  g13 *= gsc;
  g14 *= gsc;
  g15 *= gsc;
  g16 *= gsc;
  g17 *= gsc;
  g18 *= gsc;
  g19 *= gsc;
  g20 *= gsc;
  g21 *= gsc;
  g22 *= gsc;
  g23 *= gsc;
  g24 *= gsc;
  g25 *= gsc;
  g26 *= gsc;
  g27 *= gsc;
  g28 *= gsc;
  g29 *= gsc;
  g30 *= gsc;
  g31 *= gsc;
  g32 *= gsc;
  g33 *= gsc;
  g34 *= gsc;
  g35 *= gsc;
  g36 *= gsc;
  g37 *= gsc;
  g38 *= gsc;
  g39 *= gsc;
  // B operands: lane (channel cl, k-group eg) holds fp16 piece 1 - (eg & 1) of its channel's constants
  const bool pb = !(eg & 1);
  uint4v B7_1;
  { unsigned h0, h1; mm_split2_f16(float2v{1.2499999999999998f, 2.4999999999999996f}, float2v{g25, g24}, h0, h1); B7_1[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{fmaf(0.24999999999999997f, g25, 0.8660254037844387f * g23), -0.5f}, float2v{1.f, g22}, h0, h1); B7_1[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-0.25000000000000006f, -2.4999999999999996f}, float2v{g21, g22}, h0, h1); B7_1[2] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-1.25f, 0.f}, float2v{g21, 1.f}, h0, h1); B7_1[3] = pb ? h1 : h0; }
  uint4v B7_2;
  { unsigned h0, h1; mm_split2_f16(float2v{0.f, 2.4999999999999996f}, float2v{1.f, g21}, h0, h1); B7_2[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{1.0f, 0.8660254037844387f}, float2v{g22, g23}, h0, h1); B7_2[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{1.0000000000000004f, 2.4999999999999996f}, float2v{g24, g25}, h0, h1); B7_2[2] = pb ? h1 : h0; }
  B7_2[3] = 0;
  uint4v B7_3;
  { unsigned h0, h1; mm_split2_f16(float2v{1.2499999999999998f, 2.4999999999999996f}, float2v{g21, g22}, h0, h1); B7_3[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-0.24999999999999997f, -0.5f}, float2v{g21, g24}, h0, h1); B7_3[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{fmaf(-0.25000000000000006f, g25, 0.866025403784439f * g23), 2.4999999999999996f}, float2v{1.f, g24}, h0, h1); B7_3[2] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{1.25f, 0.f}, float2v{g25, 1.f}, h0, h1); B7_3[3] = pb ? h1 : h0; }
  uint4v B8_0;
  { unsigned h0, h1; mm_split2_f16(float2v{2.091650066335189f, 5.123475382979799f}, float2v{g26, g27}, h0, h1); B8_0[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{1.620185174601965f, 1.3228756555322956f}, float2v{g28, g29}, h0, h1); B8_0[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{1.6201851746019658f, 5.123475382979799f}, float2v{g30, g31}, h0, h1); B8_0[2] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{2.0916500663351894f, 0.f}, float2v{g32, 1.f}, h0, h1); B8_0[3] = pb ? h1 : h0; }
  uint4v B4_1;
  { unsigned h0, h1; mm_split2_f16(float2v{1.0606601717798207f, 2.121320343559642f}, float2v{g10, g9}, h0, h1); B4_1[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-0.35355339059327384f, 0.f}, float2v{g8, 1.f}, h0, h1); B4_1[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-1.060660171779821f, 0.f}, float2v{g8, 1.f}, h0, h1); B4_1[2] = pb ? h1 : h0; }
  B4_1[3] = 0;
  uint4v B4_2;
  { unsigned h0, h1; mm_split2_f16(float2v{0.f, 2.121320343559642f}, float2v{1.f, g8}, h0, h1); B4_2[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{0.7071067811865478f, 2.121320343559642f}, float2v{g9, g10}, h0, h1); B4_2[1] = pb ? h1 : h0; }
  B4_2[2] = 0;
  B4_2[3] = 0;
  uint4v B4_3;
  { unsigned h0, h1; mm_split2_f16(float2v{1.0606601717798207f, 0.f}, float2v{g8, 1.f}, h0, h1); B4_3[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-0.35355339059327384f, 2.121320343559642f}, float2v{g10, g9}, h0, h1); B4_3[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{1.060660171779821f, 0.f}, float2v{g10, 1.f}, h0, h1); B4_3[2] = pb ? h1 : h0; }
  B4_3[3] = 0;
  uint4v B5_0;
  { unsigned h0, h1; mm_split2_f16(float2v{1.936491673103708f, 3.8729833462074166f}, float2v{g11, g12}, h0, h1); B5_0[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{1.1180339887498953f, 3.872983346207417f}, float2v{g13, g14}, h0, h1); B5_0[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{1.9364916731037083f, 0.f}, float2v{g15, 1.f}, h0, h1); B5_0[2] = pb ? h1 : h0; }
  B5_0[3] = 0;
  uint4v B9_1;
  { unsigned h0, h1; mm_split2_f16(float2v{fmaf(1.369306393762915f, g39, 0.35355339059327373f * g37), fmaf(2.236067977499789f, g38, 1.7320508075688774f * g36)}, float2v{1.f, 1.f}, h0, h1); B9_1[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-0.7071067811865478f, -2.2360679774997894f}, float2v{g35, g34}, h0, h1); B9_1[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{fmaf(-0.3535533905932738f, g35, -1.3693063937629153f * g33), 0.f}, float2v{1.f, 1.f}, h0, h1); B9_1[2] = pb ? h1 : h0; }
  B9_1[3] = 0;
  uint4v B9_2;
  { unsigned h0, h1; mm_split2_f16(float2v{-1.1180339887498947f, -2.8284271247461903f}, float2v{g34, g35}, h0, h1); B9_2[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-0.8660254037844392f, -2.8284271247461903f}, float2v{g36, g37}, h0, h1); B9_2[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-1.118033988749895f, 0.f}, float2v{g38, 1.f}, h0, h1); B9_2[2] = pb ? h1 : h0; }
  B9_2[3] = 0;
  uint4v B9_3;
  { unsigned h0, h1; mm_split2_f16(float2v{fmaf(0.35355339059327373f, g35, -1.369306393762915f * g33), -2.236067977499789f}, float2v{1.f, g34}, h0, h1); B9_3[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-0.7071067811865478f, fmaf(-2.2360679774997894f, g38, 1.7320508075688774f * g36)}, float2v{g37, 1.f}, h0, h1); B9_3[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{fmaf(-1.3693063937629153f, g39, 0.3535533905932738f * g37), 0.f}, float2v{1.f, 1.f}, h0, h1); B9_3[2] = pb ? h1 : h0; }
  B9_3[3] = 0;
  uint2v B1_1;
  { unsigned h0, h1; mm_split2_f16(float2v{0.9999999999999999f, 0.f}, float2v{g1, 1.f}, h0, h1); B1_1[0] = pb ? h1 : h0; }
  B1_1[1] = 0;
  uint2v B1_2;
  { unsigned h0, h1; mm_split2_f16(float2v{0.f, 1.0f}, float2v{1.f, g1}, h0, h1); B1_2[0] = pb ? h1 : h0; }
  B1_2[1] = 0;
  uint2v B1_3;
  B1_3[0] = 0;
  { unsigned h0, h1; mm_split2_f16(float2v{0.9999999999999999f, 0.f}, float2v{g1, 1.f}, h0, h1); B1_3[1] = pb ? h1 : h0; }
  uint2v B2_0;
  { unsigned h0, h1; mm_split2_f16(float2v{1.732050807568877f, 1.7320508075688772f}, float2v{g2, g3}, h0, h1); B2_0[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{1.732050807568877f, 0.f}, float2v{g4, 1.f}, h0, h1); B2_0[1] = pb ? h1 : h0; }
  uint2v B6_1;
  { unsigned h0, h1; mm_split2_f16(float2v{fmaf(1.224744871391589f, g20, 0.7071067811865475f * g18), -1.2247448713915892f}, float2v{1.f, g17}, h0, h1); B6_1[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-1.224744871391589f, 0.f}, float2v{g16, 1.f}, h0, h1); B6_1[1] = pb ? h1 : h0; }
  uint2v B6_2;
  { unsigned h0, h1; mm_split2_f16(float2v{-1.2247448713915892f, -1.4142135623730951f}, float2v{g17, g18}, h0, h1); B6_2[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-1.2247448713915892f, 0.f}, float2v{g19, 1.f}, h0, h1); B6_2[1] = pb ? h1 : h0; }
  uint2v B6_3;
  { unsigned h0, h1; mm_split2_f16(float2v{-1.224744871391589f, -1.2247448713915892f}, float2v{g16, g19}, h0, h1); B6_3[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{fmaf(-1.224744871391589f, g20, 0.7071067811865475f * g18), 0.f}, float2v{1.f, 1.f}, h0, h1); B6_3[1] = pb ? h1 : h0; }
  if ((int)threadIdx.x < ns) ssend[threadIdx.x] = g_send[(size_t)grp * 208 + threadIdx.x];
  for (int j = threadIdx.x; j < ns * 16; j += 256) gxs4[j] = floatx4{0.f, 0.f, 0.f, 0.f};
  __syncthreads();
  if (e0 < e1) {
  floatx4 pkn0, pkn1, pkn2, pkn3, un;   // records and edge vector of the next tile
  unsigned on0, on1, on2, on3;           // its table rows
    pkn0 = e_pk[min(e0 + 4 * eg + 0, e1 - 1)];
    pkn1 = e_pk[min(e0 + 4 * eg + 1, e1 - 1)];
    pkn2 = e_pk[min(e0 + 4 * eg + 2, e1 - 1)];
    pkn3 = e_pk[min(e0 + 4 * eg + 3, e1 - 1)];
    un = e_u[min(e0 + cl, e1 - 1)];
    on0 = (unsigned)__float_as_int(pkn0.y) * 2560u + cl * 16u;
    on1 = (unsigned)__float_as_int(pkn1.y) * 2560u + cl * 16u;
    on2 = (unsigned)__float_as_int(pkn2.y) * 2560u + cl * 16u;
    on3 = (unsigned)__float_as_int(pkn3.y) * 2560u + cl * 16u;
    floatx4 q0_0 = *(const floatx4*)(tcb + on0 + 1792);
    floatx4 q0_1 = *(const floatx4*)(tcb + on1 + 1792);
    floatx4 q0_2 = *(const floatx4*)(tcb + on2 + 1792);
    floatx4 q0_3 = *(const floatx4*)(tcb + on3 + 1792);
    floatx4 q1_0 = *(const floatx4*)(tcb + on0 + 2048);
    floatx4 q1_1 = *(const floatx4*)(tcb + on1 + 2048);
    floatx4 q1_2 = *(const floatx4*)(tcb + on2 + 2048);
    floatx4 q1_3 = *(const floatx4*)(tcb + on3 + 2048);
  for (int eb = e0; eb < e1; eb += 16) {
    const float t0 = pkn0.x;
    const unsigned o0 = on0;
    const float* __restrict__ xp0 = X + (size_t)__float_as_int(pkn0.z) * x_stride + c;
    const float X0_0 = xp0[0];
    const float X1_0 = xp0[128];
    const float X2_0 = xp0[256];
    const float X3_0 = xp0[384];
    const float t1 = pkn1.x;
    const unsigned o1 = on1;
    const float* __restrict__ xp1 = X + (size_t)__float_as_int(pkn1.z) * x_stride + c;
    const float X0_1 = xp1[0];
    const float X1_1 = xp1[128];
    const float X2_1 = xp1[256];
    const float X3_1 = xp1[384];
    const float t2 = pkn2.x;
    const unsigned o2 = on2;
    const float* __restrict__ xp2 = X + (size_t)__float_as_int(pkn2.z) * x_stride + c;
    const float X0_2 = xp2[0];
    const float X1_2 = xp2[128];
    const float X2_2 = xp2[256];
    const float X3_2 = xp2[384];
    const float t3 = pkn3.x;
    const unsigned o3 = on3;
    const float* __restrict__ xp3 = X + (size_t)__float_as_int(pkn3.z) * x_stride + c;
    const float X0_3 = xp3[0];
    const float X1_3 = xp3[128];
    const float X2_3 = xp3[256];
    const float X3_3 = xp3[384];
    const floatx4 ua = un;
    // the next tile's records and edge vector are loaded one tile ahead (the last tile reloads its own end)
    pkn0 = e_pk[min(eb + 16 + 4 * eg + 0, e1 - 1)];
    pkn1 = e_pk[min(eb + 16 + 4 * eg + 1, e1 - 1)];
    pkn2 = e_pk[min(eb + 16 + 4 * eg + 2, e1 - 1)];
    pkn3 = e_pk[min(eb + 16 + 4 * eg + 3, e1 - 1)];
    un = e_u[min(eb + 16 + cl, e1 - 1)];
    const unsigned sl4 = mm_load_u32(e_slot + eb + 4 * eg);   // slots of four edges (the array is padded)
    // A operands of edge eb + cl: lane group 0 the harmonics, 1 and 2 their two derivatives
    {
      float F[16], A[16], s, cp, sp;
      mm_polar(ua.x, ua.y, s, cp, sp);
      mm_polar_operands(ua.x, ua.y, ua.z, s, cp, sp, eg, F, A);
      mm_wave_lds_sync();   // the previous tile's operands have been read
      if (eg < 3) {
        { uint4v a = {}, b = {};
          { unsigned h0, h1; mm_split2_f16(float2v{F[9], F[10]}, float2v{A[9], A[10]}, h0, h1); a[0] = h0; b[0] = h1; }
          { unsigned h0, h1; mm_split2_f16(float2v{F[11], F[12]}, float2v{A[11], A[12]}, h0, h1); a[1] = h0; b[1] = h1; }
          { unsigned h0, h1; mm_split2_f16(float2v{F[13], F[14]}, float2v{A[13], A[14]}, h0, h1); a[2] = h0; b[2] = h1; }
          { unsigned h0, h1; mm_split2_f16(float2v{F[15], 0.f}, float2v{A[15], 0.f}, h0, h1); a[3] = h0; b[3] = h1; }
          uint4v* __restrict__ d = ya + ((eg * 3 + 0) * 16 + cl) * 2;
          d[0] = a; d[1] = b; }
        { uint4v a = {}, b = {};
          { unsigned h0, h1; mm_split2_f16(float2v{F[4], F[5]}, float2v{A[4], A[5]}, h0, h1); a[0] = h0; b[0] = h1; }
          { unsigned h0, h1; mm_split2_f16(float2v{F[6], F[7]}, float2v{A[6], A[7]}, h0, h1); a[1] = h0; b[1] = h1; }
          { unsigned h0, h1; mm_split2_f16(float2v{F[8], 0.f}, float2v{A[8], 0.f}, h0, h1); a[2] = h0; b[2] = h1; }
          uint4v* __restrict__ d = ya + ((eg * 3 + 1) * 16 + cl) * 2;
          d[0] = a; d[1] = b; }
        { uint4v a = {}, b = {};
          { unsigned h0, h1; mm_split2_f16(float2v{F[1], F[2]}, float2v{A[1], A[2]}, h0, h1); a[0] = h0; b[0] = h1; }
          { unsigned h0, h1; mm_split2_f16(float2v{F[3], 0.f}, float2v{A[3], 0.f}, h0, h1); a[1] = h0; b[1] = h1; }
          uint4v* __restrict__ d = ya + ((eg * 3 + 2) * 16 + cl) * 2;
          d[0] = a; d[1] = b; }
      }
      mm_wave_lds_sync();
    }
    float gr0 = 0.f, gt0 = 0.f, gp0 = 0.f;
    float gx0_0 = 0.f;
    float gx1_0 = 0.f;
    float gx2_0 = 0.f;
    float gx3_0 = 0.f;
    float gr1 = 0.f, gt1 = 0.f, gp1 = 0.f;
    float gx0_1 = 0.f;
    float gx1_1 = 0.f;
    float gx2_1 = 0.f;
    float gx3_1 = 0.f;
    float gr2 = 0.f, gt2 = 0.f, gp2 = 0.f;
    float gx0_2 = 0.f;
    float gx1_2 = 0.f;
    float gx2_2 = 0.f;
    float gx3_2 = 0.f;
    float gr3 = 0.f, gt3 = 0.f, gp3 = 0.f;
    float gx0_3 = 0.f;
    float gx1_3 = 0.f;
    float gx2_3 = 0.f;
    float gx3_3 = 0.f;
    const half8v A3_0 = __builtin_bit_cast(half8v, ya[((0) * 16 + cl) * 2 + 1 - (eg >> 1)]);
    const half8v A3_1 = __builtin_bit_cast(half8v, ya[((3) * 16 + cl) * 2 + 1 - (eg >> 1)]);
    const half8v A3_2 = __builtin_bit_cast(half8v, ya[((6) * 16 + cl) * 2 + 1 - (eg >> 1)]);
    const floatx4 D0_7_1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_0, __builtin_bit_cast(half8v, B7_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_7_1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_1, __builtin_bit_cast(half8v, B7_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_7_1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_2, __builtin_bit_cast(half8v, B7_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_7_2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_0, __builtin_bit_cast(half8v, B7_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_7_2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_1, __builtin_bit_cast(half8v, B7_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_7_2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_2, __builtin_bit_cast(half8v, B7_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_7_3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_0, __builtin_bit_cast(half8v, B7_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_7_3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_1, __builtin_bit_cast(half8v, B7_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_7_3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_2, __builtin_bit_cast(half8v, B7_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    {
      const floatx4 q = q0_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx1_0 = fmaf(W, D0_7_1[0], gx1_0);
      gx2_0 = fmaf(W, D0_7_2[0], gx2_0);
      gx3_0 = fmaf(W, D0_7_3[0], gx3_0);
      gr0 = fmaf(fmaf(X3_0, D0_7_3[0], fmaf(X2_0, D0_7_2[0], X1_0 * D0_7_1[0])), D, gr0);
      gt0 = fmaf(fmaf(X3_0, D1_7_3[0], fmaf(X2_0, D1_7_2[0], X1_0 * D1_7_1[0])), W, gt0);
      gp0 = fmaf(fmaf(X3_0, D2_7_3[0], fmaf(X2_0, D2_7_2[0], X1_0 * D2_7_1[0])), W, gp0);
    }
    {
      const floatx4 q = q0_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx1_1 = fmaf(W, D0_7_1[1], gx1_1);
      gx2_1 = fmaf(W, D0_7_2[1], gx2_1);
      gx3_1 = fmaf(W, D0_7_3[1], gx3_1);
      gr1 = fmaf(fmaf(X3_1, D0_7_3[1], fmaf(X2_1, D0_7_2[1], X1_1 * D0_7_1[1])), D, gr1);
      gt1 = fmaf(fmaf(X3_1, D1_7_3[1], fmaf(X2_1, D1_7_2[1], X1_1 * D1_7_1[1])), W, gt1);
      gp1 = fmaf(fmaf(X3_1, D2_7_3[1], fmaf(X2_1, D2_7_2[1], X1_1 * D2_7_1[1])), W, gp1);
    }
    {
      const floatx4 q = q0_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx1_2 = fmaf(W, D0_7_1[2], gx1_2);
      gx2_2 = fmaf(W, D0_7_2[2], gx2_2);
      gx3_2 = fmaf(W, D0_7_3[2], gx3_2);
      gr2 = fmaf(fmaf(X3_2, D0_7_3[2], fmaf(X2_2, D0_7_2[2], X1_2 * D0_7_1[2])), D, gr2);
      gt2 = fmaf(fmaf(X3_2, D1_7_3[2], fmaf(X2_2, D1_7_2[2], X1_2 * D1_7_1[2])), W, gt2);
      gp2 = fmaf(fmaf(X3_2, D2_7_3[2], fmaf(X2_2, D2_7_2[2], X1_2 * D2_7_1[2])), W, gp2);
    }
    {
      const floatx4 q = q0_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx1_3 = fmaf(W, D0_7_1[3], gx1_3);
      gx2_3 = fmaf(W, D0_7_2[3], gx2_3);
      gx3_3 = fmaf(W, D0_7_3[3], gx3_3);
      gr3 = fmaf(fmaf(X3_3, D0_7_3[3], fmaf(X2_3, D0_7_2[3], X1_3 * D0_7_1[3])), D, gr3);
      gt3 = fmaf(fmaf(X3_3, D1_7_3[3], fmaf(X2_3, D1_7_2[3], X1_3 * D1_7_1[3])), W, gt3);
      gp3 = fmaf(fmaf(X3_3, D2_7_3[3], fmaf(X2_3, D2_7_2[3], X1_3 * D2_7_1[3])), W, gp3);
    }
    asm volatile("" : "+v"(gx1_0), "+v"(gx1_1), "+v"(gx1_2), "+v"(gx1_3), "+v"(gx2_0), "+v"(gx2_1), "+v"(gx2_2), "+v"(gx2_3), "+v"(gx3_0), "+v"(gx3_1), "+v"(gx3_2), "+v"(gx3_3));
    floatx4 q2_0 = *(const floatx4*)(tcb + o0 + 1024);
    floatx4 q2_1 = *(const floatx4*)(tcb + o1 + 1024);
    floatx4 q2_2 = *(const floatx4*)(tcb + o2 + 1024);
    floatx4 q2_3 = *(const floatx4*)(tcb + o3 + 1024);
    const floatx4 D0_8_0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_0, __builtin_bit_cast(half8v, B8_0), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_8_0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_1, __builtin_bit_cast(half8v, B8_0), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_8_0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_2, __builtin_bit_cast(half8v, B8_0), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    {
      const floatx4 q = q1_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx0_0 = fmaf(W, D0_8_0[0], gx0_0);
      gr0 = fmaf(X0_0 * D0_8_0[0], D, gr0);
      gt0 = fmaf(X0_0 * D1_8_0[0], W, gt0);
      gp0 = fmaf(X0_0 * D2_8_0[0], W, gp0);
    }
    {
      const floatx4 q = q1_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx0_1 = fmaf(W, D0_8_0[1], gx0_1);
      gr1 = fmaf(X0_1 * D0_8_0[1], D, gr1);
      gt1 = fmaf(X0_1 * D1_8_0[1], W, gt1);
      gp1 = fmaf(X0_1 * D2_8_0[1], W, gp1);
    }
    {
      const floatx4 q = q1_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx0_2 = fmaf(W, D0_8_0[2], gx0_2);
      gr2 = fmaf(X0_2 * D0_8_0[2], D, gr2);
      gt2 = fmaf(X0_2 * D1_8_0[2], W, gt2);
      gp2 = fmaf(X0_2 * D2_8_0[2], W, gp2);
    }
    {
      const floatx4 q = q1_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx0_3 = fmaf(W, D0_8_0[3], gx0_3);
      gr3 = fmaf(X0_3 * D0_8_0[3], D, gr3);
      gt3 = fmaf(X0_3 * D1_8_0[3], W, gt3);
      gp3 = fmaf(X0_3 * D2_8_0[3], W, gp3);
    }
    asm volatile("" : "+v"(gx0_0), "+v"(gx0_1), "+v"(gx0_2), "+v"(gx0_3));
    floatx4 q3_0 = *(const floatx4*)(tcb + o0 + 1280);
    floatx4 q3_1 = *(const floatx4*)(tcb + o1 + 1280);
    floatx4 q3_2 = *(const floatx4*)(tcb + o2 + 1280);
    floatx4 q3_3 = *(const floatx4*)(tcb + o3 + 1280);
    const half8v A2_0 = __builtin_bit_cast(half8v, ya[((1) * 16 + cl) * 2 + 1 - (eg >> 1)]);
    const half8v A2_1 = __builtin_bit_cast(half8v, ya[((4) * 16 + cl) * 2 + 1 - (eg >> 1)]);
    const half8v A2_2 = __builtin_bit_cast(half8v, ya[((7) * 16 + cl) * 2 + 1 - (eg >> 1)]);
    const floatx4 D0_4_1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_0, __builtin_bit_cast(half8v, B4_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_4_1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_1, __builtin_bit_cast(half8v, B4_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_4_1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_2, __builtin_bit_cast(half8v, B4_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_4_2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_0, __builtin_bit_cast(half8v, B4_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_4_2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_1, __builtin_bit_cast(half8v, B4_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_4_2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_2, __builtin_bit_cast(half8v, B4_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_4_3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_0, __builtin_bit_cast(half8v, B4_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_4_3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_1, __builtin_bit_cast(half8v, B4_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_4_3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_2, __builtin_bit_cast(half8v, B4_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    {
      const floatx4 q = q2_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx1_0 = fmaf(W, D0_4_1[0], gx1_0);
      gx2_0 = fmaf(W, D0_4_2[0], gx2_0);
      gx3_0 = fmaf(W, D0_4_3[0], gx3_0);
      gr0 = fmaf(fmaf(X3_0, D0_4_3[0], fmaf(X2_0, D0_4_2[0], X1_0 * D0_4_1[0])), D, gr0);
      gt0 = fmaf(fmaf(X3_0, D1_4_3[0], fmaf(X2_0, D1_4_2[0], X1_0 * D1_4_1[0])), W, gt0);
      gp0 = fmaf(fmaf(X3_0, D2_4_3[0], fmaf(X2_0, D2_4_2[0], X1_0 * D2_4_1[0])), W, gp0);
    }
    {
      const floatx4 q = q2_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx1_1 = fmaf(W, D0_4_1[1], gx1_1);
      gx2_1 = fmaf(W, D0_4_2[1], gx2_1);
      gx3_1 = fmaf(W, D0_4_3[1], gx3_1);
      gr1 = fmaf(fmaf(X3_1, D0_4_3[1], fmaf(X2_1, D0_4_2[1], X1_1 * D0_4_1[1])), D, gr1);
      gt1 = fmaf(fmaf(X3_1, D1_4_3[1], fmaf(X2_1, D1_4_2[1], X1_1 * D1_4_1[1])), W, gt1);
      gp1 = fmaf(fmaf(X3_1, D2_4_3[1], fmaf(X2_1, D2_4_2[1], X1_1 * D2_4_1[1])), W, gp1);
    }
    {
      const floatx4 q = q2_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx1_2 = fmaf(W, D0_4_1[2], gx1_2);
      gx2_2 = fmaf(W, D0_4_2[2], gx2_2);
      gx3_2 = fmaf(W, D0_4_3[2], gx3_2);
      gr2 = fmaf(fmaf(X3_2, D0_4_3[2], fmaf(X2_2, D0_4_2[2], X1_2 * D0_4_1[2])), D, gr2);
      gt2 = fmaf(fmaf(X3_2, D1_4_3[2], fmaf(X2_2, D1_4_2[2], X1_2 * D1_4_1[2])), W, gt2);
      gp2 = fmaf(fmaf(X3_2, D2_4_3[2], fmaf(X2_2, D2_4_2[2], X1_2 * D2_4_1[2])), W, gp2);
    }
    {
      const floatx4 q = q2_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx1_3 = fmaf(W, D0_4_1[3], gx1_3);
      gx2_3 = fmaf(W, D0_4_2[3], gx2_3);
      gx3_3 = fmaf(W, D0_4_3[3], gx3_3);
      gr3 = fmaf(fmaf(X3_3, D0_4_3[3], fmaf(X2_3, D0_4_2[3], X1_3 * D0_4_1[3])), D, gr3);
      gt3 = fmaf(fmaf(X3_3, D1_4_3[3], fmaf(X2_3, D1_4_2[3], X1_3 * D1_4_1[3])), W, gt3);
      gp3 = fmaf(fmaf(X3_3, D2_4_3[3], fmaf(X2_3, D2_4_2[3], X1_3 * D2_4_1[3])), W, gp3);
    }
    asm volatile("" : "+v"(gx1_0), "+v"(gx1_1), "+v"(gx1_2), "+v"(gx1_3), "+v"(gx2_0), "+v"(gx2_1), "+v"(gx2_2), "+v"(gx2_3), "+v"(gx3_0), "+v"(gx3_1), "+v"(gx3_2), "+v"(gx3_3));
    floatx4 q4_0 = *(const floatx4*)(tcb + o0 + 2304);
    floatx4 q4_1 = *(const floatx4*)(tcb + o1 + 2304);
    floatx4 q4_2 = *(const floatx4*)(tcb + o2 + 2304);
    floatx4 q4_3 = *(const floatx4*)(tcb + o3 + 2304);
    const floatx4 D0_5_0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_0, __builtin_bit_cast(half8v, B5_0), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_5_0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_1, __builtin_bit_cast(half8v, B5_0), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_5_0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_2, __builtin_bit_cast(half8v, B5_0), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    {
      const floatx4 q = q3_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx0_0 = fmaf(W, D0_5_0[0], gx0_0);
      gr0 = fmaf(X0_0 * D0_5_0[0], D, gr0);
      gt0 = fmaf(X0_0 * D1_5_0[0], W, gt0);
      gp0 = fmaf(X0_0 * D2_5_0[0], W, gp0);
    }
    {
      const floatx4 q = q3_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx0_1 = fmaf(W, D0_5_0[1], gx0_1);
      gr1 = fmaf(X0_1 * D0_5_0[1], D, gr1);
      gt1 = fmaf(X0_1 * D1_5_0[1], W, gt1);
      gp1 = fmaf(X0_1 * D2_5_0[1], W, gp1);
    }
    {
      const floatx4 q = q3_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx0_2 = fmaf(W, D0_5_0[2], gx0_2);
      gr2 = fmaf(X0_2 * D0_5_0[2], D, gr2);
      gt2 = fmaf(X0_2 * D1_5_0[2], W, gt2);
      gp2 = fmaf(X0_2 * D2_5_0[2], W, gp2);
    }
    {
      const floatx4 q = q3_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx0_3 = fmaf(W, D0_5_0[3], gx0_3);
      gr3 = fmaf(X0_3 * D0_5_0[3], D, gr3);
      gt3 = fmaf(X0_3 * D1_5_0[3], W, gt3);
      gp3 = fmaf(X0_3 * D2_5_0[3], W, gp3);
    }
    asm volatile("" : "+v"(gx0_0), "+v"(gx0_1), "+v"(gx0_2), "+v"(gx0_3));
    floatx4 q5_0 = *(const floatx4*)(tcb + o0 + 256);
    floatx4 q5_1 = *(const floatx4*)(tcb + o1 + 256);
    floatx4 q5_2 = *(const floatx4*)(tcb + o2 + 256);
    floatx4 q5_3 = *(const floatx4*)(tcb + o3 + 256);
    const floatx4 D0_9_1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_0, __builtin_bit_cast(half8v, B9_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_9_1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_1, __builtin_bit_cast(half8v, B9_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_9_1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_2, __builtin_bit_cast(half8v, B9_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_9_2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_0, __builtin_bit_cast(half8v, B9_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_9_2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_1, __builtin_bit_cast(half8v, B9_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_9_2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_2, __builtin_bit_cast(half8v, B9_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_9_3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_0, __builtin_bit_cast(half8v, B9_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_9_3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_1, __builtin_bit_cast(half8v, B9_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_9_3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_2, __builtin_bit_cast(half8v, B9_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    {
      const floatx4 q = q4_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx1_0 = fmaf(W, D0_9_1[0], gx1_0);
      gx2_0 = fmaf(W, D0_9_2[0], gx2_0);
      gx3_0 = fmaf(W, D0_9_3[0], gx3_0);
      gr0 = fmaf(fmaf(X3_0, D0_9_3[0], fmaf(X2_0, D0_9_2[0], X1_0 * D0_9_1[0])), D, gr0);
      gt0 = fmaf(fmaf(X3_0, D1_9_3[0], fmaf(X2_0, D1_9_2[0], X1_0 * D1_9_1[0])), W, gt0);
      gp0 = fmaf(fmaf(X3_0, D2_9_3[0], fmaf(X2_0, D2_9_2[0], X1_0 * D2_9_1[0])), W, gp0);
    }
    {
      const floatx4 q = q4_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx1_1 = fmaf(W, D0_9_1[1], gx1_1);
      gx2_1 = fmaf(W, D0_9_2[1], gx2_1);
      gx3_1 = fmaf(W, D0_9_3[1], gx3_1);
      gr1 = fmaf(fmaf(X3_1, D0_9_3[1], fmaf(X2_1, D0_9_2[1], X1_1 * D0_9_1[1])), D, gr1);
      gt1 = fmaf(fmaf(X3_1, D1_9_3[1], fmaf(X2_1, D1_9_2[1], X1_1 * D1_9_1[1])), W, gt1);
      gp1 = fmaf(fmaf(X3_1, D2_9_3[1], fmaf(X2_1, D2_9_2[1], X1_1 * D2_9_1[1])), W, gp1);
    }
    {
      const floatx4 q = q4_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx1_2 = fmaf(W, D0_9_1[2], gx1_2);
      gx2_2 = fmaf(W, D0_9_2[2], gx2_2);
      gx3_2 = fmaf(W, D0_9_3[2], gx3_2);
      gr2 = fmaf(fmaf(X3_2, D0_9_3[2], fmaf(X2_2, D0_9_2[2], X1_2 * D0_9_1[2])), D, gr2);
      gt2 = fmaf(fmaf(X3_2, D1_9_3[2], fmaf(X2_2, D1_9_2[2], X1_2 * D1_9_1[2])), W, gt2);
      gp2 = fmaf(fmaf(X3_2, D2_9_3[2], fmaf(X2_2, D2_9_2[2], X1_2 * D2_9_1[2])), W, gp2);
    }
    {
      const floatx4 q = q4_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx1_3 = fmaf(W, D0_9_1[3], gx1_3);
      gx2_3 = fmaf(W, D0_9_2[3], gx2_3);
      gx3_3 = fmaf(W, D0_9_3[3], gx3_3);
      gr3 = fmaf(fmaf(X3_3, D0_9_3[3], fmaf(X2_3, D0_9_2[3], X1_3 * D0_9_1[3])), D, gr3);
      gt3 = fmaf(fmaf(X3_3, D1_9_3[3], fmaf(X2_3, D1_9_2[3], X1_3 * D1_9_1[3])), W, gt3);
      gp3 = fmaf(fmaf(X3_3, D2_9_3[3], fmaf(X2_3, D2_9_2[3], X1_3 * D2_9_1[3])), W, gp3);
    }
    asm volatile("" : "+v"(gx1_0), "+v"(gx1_1), "+v"(gx1_2), "+v"(gx1_3), "+v"(gx2_0), "+v"(gx2_1), "+v"(gx2_2), "+v"(gx2_3), "+v"(gx3_0), "+v"(gx3_1), "+v"(gx3_2), "+v"(gx3_3));
    floatx4 q6_0 = *(const floatx4*)(tcb + o0 + 512);
    floatx4 q6_1 = *(const floatx4*)(tcb + o1 + 512);
    floatx4 q6_2 = *(const floatx4*)(tcb + o2 + 512);
    floatx4 q6_3 = *(const floatx4*)(tcb + o3 + 512);
    const half4v A1_0 = __builtin_bit_cast(half4v, *(const uint2v*)&ya[((2) * 16 + cl) * 2 + 1 - (eg >> 1)]);
    const half4v A1_1 = __builtin_bit_cast(half4v, *(const uint2v*)&ya[((5) * 16 + cl) * 2 + 1 - (eg >> 1)]);
    const half4v A1_2 = __builtin_bit_cast(half4v, *(const uint2v*)&ya[((8) * 16 + cl) * 2 + 1 - (eg >> 1)]);
    const floatx4 D0_1_1 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_0, __builtin_bit_cast(half4v, B1_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_1_1 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_1, __builtin_bit_cast(half4v, B1_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_1_1 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_2, __builtin_bit_cast(half4v, B1_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_1_2 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_0, __builtin_bit_cast(half4v, B1_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_1_2 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_1, __builtin_bit_cast(half4v, B1_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_1_2 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_2, __builtin_bit_cast(half4v, B1_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_1_3 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_0, __builtin_bit_cast(half4v, B1_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_1_3 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_1, __builtin_bit_cast(half4v, B1_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_1_3 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_2, __builtin_bit_cast(half4v, B1_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    {
      const floatx4 q = q5_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx1_0 = fmaf(W, D0_1_1[0], gx1_0);
      gx2_0 = fmaf(W, D0_1_2[0], gx2_0);
      gx3_0 = fmaf(W, D0_1_3[0], gx3_0);
      gr0 = fmaf(fmaf(X3_0, D0_1_3[0], fmaf(X2_0, D0_1_2[0], X1_0 * D0_1_1[0])), D, gr0);
      gt0 = fmaf(fmaf(X3_0, D1_1_3[0], fmaf(X2_0, D1_1_2[0], X1_0 * D1_1_1[0])), W, gt0);
      gp0 = fmaf(fmaf(X3_0, D2_1_3[0], fmaf(X2_0, D2_1_2[0], X1_0 * D2_1_1[0])), W, gp0);
    }
    {
      const floatx4 q = q5_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx1_1 = fmaf(W, D0_1_1[1], gx1_1);
      gx2_1 = fmaf(W, D0_1_2[1], gx2_1);
      gx3_1 = fmaf(W, D0_1_3[1], gx3_1);
      gr1 = fmaf(fmaf(X3_1, D0_1_3[1], fmaf(X2_1, D0_1_2[1], X1_1 * D0_1_1[1])), D, gr1);
      gt1 = fmaf(fmaf(X3_1, D1_1_3[1], fmaf(X2_1, D1_1_2[1], X1_1 * D1_1_1[1])), W, gt1);
      gp1 = fmaf(fmaf(X3_1, D2_1_3[1], fmaf(X2_1, D2_1_2[1], X1_1 * D2_1_1[1])), W, gp1);
    }
    {
      const floatx4 q = q5_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx1_2 = fmaf(W, D0_1_1[2], gx1_2);
      gx2_2 = fmaf(W, D0_1_2[2], gx2_2);
      gx3_2 = fmaf(W, D0_1_3[2], gx3_2);
      gr2 = fmaf(fmaf(X3_2, D0_1_3[2], fmaf(X2_2, D0_1_2[2], X1_2 * D0_1_1[2])), D, gr2);
      gt2 = fmaf(fmaf(X3_2, D1_1_3[2], fmaf(X2_2, D1_1_2[2], X1_2 * D1_1_1[2])), W, gt2);
      gp2 = fmaf(fmaf(X3_2, D2_1_3[2], fmaf(X2_2, D2_1_2[2], X1_2 * D2_1_1[2])), W, gp2);
    }
    {
      const floatx4 q = q5_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx1_3 = fmaf(W, D0_1_1[3], gx1_3);
      gx2_3 = fmaf(W, D0_1_2[3], gx2_3);
      gx3_3 = fmaf(W, D0_1_3[3], gx3_3);
      gr3 = fmaf(fmaf(X3_3, D0_1_3[3], fmaf(X2_3, D0_1_2[3], X1_3 * D0_1_1[3])), D, gr3);
      gt3 = fmaf(fmaf(X3_3, D1_1_3[3], fmaf(X2_3, D1_1_2[3], X1_3 * D1_1_1[3])), W, gt3);
      gp3 = fmaf(fmaf(X3_3, D2_1_3[3], fmaf(X2_3, D2_1_2[3], X1_3 * D2_1_1[3])), W, gp3);
    }
    asm volatile("" : "+v"(gx1_0), "+v"(gx1_1), "+v"(gx1_2), "+v"(gx1_3), "+v"(gx2_0), "+v"(gx2_1), "+v"(gx2_2), "+v"(gx2_3), "+v"(gx3_0), "+v"(gx3_1), "+v"(gx3_2), "+v"(gx3_3));
    floatx4 q7_0 = *(const floatx4*)(tcb + o0 + 1536);
    floatx4 q7_1 = *(const floatx4*)(tcb + o1 + 1536);
    floatx4 q7_2 = *(const floatx4*)(tcb + o2 + 1536);
    floatx4 q7_3 = *(const floatx4*)(tcb + o3 + 1536);
    const floatx4 D0_2_0 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_0, __builtin_bit_cast(half4v, B2_0), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_2_0 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_1, __builtin_bit_cast(half4v, B2_0), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_2_0 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_2, __builtin_bit_cast(half4v, B2_0), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    {
      const floatx4 q = q6_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx0_0 = fmaf(W, D0_2_0[0], gx0_0);
      gr0 = fmaf(X0_0 * D0_2_0[0], D, gr0);
      gt0 = fmaf(X0_0 * D1_2_0[0], W, gt0);
      gp0 = fmaf(X0_0 * D2_2_0[0], W, gp0);
    }
    {
      const floatx4 q = q6_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx0_1 = fmaf(W, D0_2_0[1], gx0_1);
      gr1 = fmaf(X0_1 * D0_2_0[1], D, gr1);
      gt1 = fmaf(X0_1 * D1_2_0[1], W, gt1);
      gp1 = fmaf(X0_1 * D2_2_0[1], W, gp1);
    }
    {
      const floatx4 q = q6_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx0_2 = fmaf(W, D0_2_0[2], gx0_2);
      gr2 = fmaf(X0_2 * D0_2_0[2], D, gr2);
      gt2 = fmaf(X0_2 * D1_2_0[2], W, gt2);
      gp2 = fmaf(X0_2 * D2_2_0[2], W, gp2);
    }
    {
      const floatx4 q = q6_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx0_3 = fmaf(W, D0_2_0[3], gx0_3);
      gr3 = fmaf(X0_3 * D0_2_0[3], D, gr3);
      gt3 = fmaf(X0_3 * D1_2_0[3], W, gt3);
      gp3 = fmaf(X0_3 * D2_2_0[3], W, gp3);
    }
    asm volatile("" : "+v"(gx0_0), "+v"(gx0_1), "+v"(gx0_2), "+v"(gx0_3));
    floatx4 q8_0 = *(const floatx4*)(tcb + o0 + 0);
    floatx4 q8_1 = *(const floatx4*)(tcb + o1 + 0);
    floatx4 q8_2 = *(const floatx4*)(tcb + o2 + 0);
    floatx4 q8_3 = *(const floatx4*)(tcb + o3 + 0);
    const floatx4 D0_6_1 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_0, __builtin_bit_cast(half4v, B6_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_6_1 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_1, __builtin_bit_cast(half4v, B6_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_6_1 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_2, __builtin_bit_cast(half4v, B6_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_6_2 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_0, __builtin_bit_cast(half4v, B6_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_6_2 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_1, __builtin_bit_cast(half4v, B6_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_6_2 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_2, __builtin_bit_cast(half4v, B6_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_6_3 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_0, __builtin_bit_cast(half4v, B6_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_6_3 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_1, __builtin_bit_cast(half4v, B6_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_6_3 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_2, __builtin_bit_cast(half4v, B6_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    {
      const floatx4 q = q7_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx1_0 = fmaf(W, D0_6_1[0], gx1_0);
      gx2_0 = fmaf(W, D0_6_2[0], gx2_0);
      gx3_0 = fmaf(W, D0_6_3[0], gx3_0);
      gr0 = fmaf(fmaf(X3_0, D0_6_3[0], fmaf(X2_0, D0_6_2[0], X1_0 * D0_6_1[0])), D, gr0);
      gt0 = fmaf(fmaf(X3_0, D1_6_3[0], fmaf(X2_0, D1_6_2[0], X1_0 * D1_6_1[0])), W, gt0);
      gp0 = fmaf(fmaf(X3_0, D2_6_3[0], fmaf(X2_0, D2_6_2[0], X1_0 * D2_6_1[0])), W, gp0);
    }
    {
      const floatx4 q = q7_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx1_1 = fmaf(W, D0_6_1[1], gx1_1);
      gx2_1 = fmaf(W, D0_6_2[1], gx2_1);
      gx3_1 = fmaf(W, D0_6_3[1], gx3_1);
      gr1 = fmaf(fmaf(X3_1, D0_6_3[1], fmaf(X2_1, D0_6_2[1], X1_1 * D0_6_1[1])), D, gr1);
      gt1 = fmaf(fmaf(X3_1, D1_6_3[1], fmaf(X2_1, D1_6_2[1], X1_1 * D1_6_1[1])), W, gt1);
      gp1 = fmaf(fmaf(X3_1, D2_6_3[1], fmaf(X2_1, D2_6_2[1], X1_1 * D2_6_1[1])), W, gp1);
    }
    {
      const floatx4 q = q7_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx1_2 = fmaf(W, D0_6_1[2], gx1_2);
      gx2_2 = fmaf(W, D0_6_2[2], gx2_2);
      gx3_2 = fmaf(W, D0_6_3[2], gx3_2);
      gr2 = fmaf(fmaf(X3_2, D0_6_3[2], fmaf(X2_2, D0_6_2[2], X1_2 * D0_6_1[2])), D, gr2);
      gt2 = fmaf(fmaf(X3_2, D1_6_3[2], fmaf(X2_2, D1_6_2[2], X1_2 * D1_6_1[2])), W, gt2);
      gp2 = fmaf(fmaf(X3_2, D2_6_3[2], fmaf(X2_2, D2_6_2[2], X1_2 * D2_6_1[2])), W, gp2);
    }
    {
      const floatx4 q = q7_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx1_3 = fmaf(W, D0_6_1[3], gx1_3);
      gx2_3 = fmaf(W, D0_6_2[3], gx2_3);
      gx3_3 = fmaf(W, D0_6_3[3], gx3_3);
      gr3 = fmaf(fmaf(X3_3, D0_6_3[3], fmaf(X2_3, D0_6_2[3], X1_3 * D0_6_1[3])), D, gr3);
      gt3 = fmaf(fmaf(X3_3, D1_6_3[3], fmaf(X2_3, D1_6_2[3], X1_3 * D1_6_1[3])), W, gt3);
      gp3 = fmaf(fmaf(X3_3, D2_6_3[3], fmaf(X2_3, D2_6_2[3], X1_3 * D2_6_1[3])), W, gp3);
    }
    asm volatile("" : "+v"(gx1_0), "+v"(gx1_1), "+v"(gx1_2), "+v"(gx1_3), "+v"(gx2_0), "+v"(gx2_1), "+v"(gx2_2), "+v"(gx2_3), "+v"(gx3_0), "+v"(gx3_1), "+v"(gx3_2), "+v"(gx3_3));
    floatx4 q9_0 = *(const floatx4*)(tcb + o0 + 768);
    floatx4 q9_1 = *(const floatx4*)(tcb + o1 + 768);
    floatx4 q9_2 = *(const floatx4*)(tcb + o2 + 768);
    floatx4 q9_3 = *(const floatx4*)(tcb + o3 + 768);
    {
      const floatx4 q = q8_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx0_0 = fmaf(W, U0_0, gx0_0);
      gr0 = fmaf(X0_0 * U0_0, D, gr0);
    }
    {
      const floatx4 q = q8_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx0_1 = fmaf(W, U0_0, gx0_1);
      gr1 = fmaf(X0_1 * U0_0, D, gr1);
    }
    {
      const floatx4 q = q8_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx0_2 = fmaf(W, U0_0, gx0_2);
      gr2 = fmaf(X0_2 * U0_0, D, gr2);
    }
    {
      const floatx4 q = q8_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx0_3 = fmaf(W, U0_0, gx0_3);
      gr3 = fmaf(X0_3 * U0_0, D, gr3);
    }
    asm volatile("" : "+v"(gx0_0), "+v"(gx0_1), "+v"(gx0_2), "+v"(gx0_3));
    on0 = (unsigned)__float_as_int(pkn0.y) * 2560u + cl * 16u;
    on1 = (unsigned)__float_as_int(pkn1.y) * 2560u + cl * 16u;
    on2 = (unsigned)__float_as_int(pkn2.y) * 2560u + cl * 16u;
    on3 = (unsigned)__float_as_int(pkn3.y) * 2560u + cl * 16u;
    q0_0 = *(const floatx4*)(tcb + on0 + 1792);
    q0_1 = *(const floatx4*)(tcb + on1 + 1792);
    q0_2 = *(const floatx4*)(tcb + on2 + 1792);
    q0_3 = *(const floatx4*)(tcb + on3 + 1792);
    {
      const floatx4 q = q9_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx1_0 = fmaf(W, U3_1, gx1_0);
      gx2_0 = fmaf(W, U3_2, gx2_0);
      gx3_0 = fmaf(W, U3_3, gx3_0);
      gr0 = fmaf(fmaf(X3_0, U3_3, fmaf(X2_0, U3_2, X1_0 * U3_1)), D, gr0);
    }
    {
      const floatx4 q = q9_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx1_1 = fmaf(W, U3_1, gx1_1);
      gx2_1 = fmaf(W, U3_2, gx2_1);
      gx3_1 = fmaf(W, U3_3, gx3_1);
      gr1 = fmaf(fmaf(X3_1, U3_3, fmaf(X2_1, U3_2, X1_1 * U3_1)), D, gr1);
    }
    {
      const floatx4 q = q9_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx1_2 = fmaf(W, U3_1, gx1_2);
      gx2_2 = fmaf(W, U3_2, gx2_2);
      gx3_2 = fmaf(W, U3_3, gx3_2);
      gr2 = fmaf(fmaf(X3_2, U3_3, fmaf(X2_2, U3_2, X1_2 * U3_1)), D, gr2);
    }
    {
      const floatx4 q = q9_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx1_3 = fmaf(W, U3_1, gx1_3);
      gx2_3 = fmaf(W, U3_2, gx2_3);
      gx3_3 = fmaf(W, U3_3, gx3_3);
      gr3 = fmaf(fmaf(X3_3, U3_3, fmaf(X2_3, U3_2, X1_3 * U3_1)), D, gr3);
    }
    asm volatile("" : "+v"(gx1_0), "+v"(gx1_1), "+v"(gx1_2), "+v"(gx1_3), "+v"(gx2_0), "+v"(gx2_1), "+v"(gx2_2), "+v"(gx2_3), "+v"(gx3_0), "+v"(gx3_1), "+v"(gx3_2), "+v"(gx3_3));
    q1_0 = *(const floatx4*)(tcb + on0 + 2048);
    q1_1 = *(const floatx4*)(tcb + on1 + 2048);
    q1_2 = *(const floatx4*)(tcb + on2 + 2048);
    q1_3 = *(const floatx4*)(tcb + on3 + 2048);
    const int n_own = min(e1 - (eb + 4 * eg), 4);   // this lane's edges inside the receiver's range (may be <= 0)
    // sums over the 16 channels of the row: transpose-reduction, lane cl = 3 v + j ends with value j of edge v
    gr0 *= gun;
    gt0 *= gun;
    gp0 *= gun;
    gr1 *= gun;
    gt1 *= gun;
    gp1 *= gun;
    gr2 *= gun;
    gt2 *= gun;
    gp2 *= gun;
    gr3 *= gun;
    gt3 *= gun;
    gp3 *= gun;
    const bool b3 = cl & 8, b2 = cl & 4, b1 = cl & 2, b0 = cl & 1;
    const float s8_0 = (b3 ? gp2 : gr0) + mm_dpp<0x140>(b3 ? gr0 : gp2);
    const float s8_1 = (b3 ? gr3 : gt0) + mm_dpp<0x140>(b3 ? gt0 : gr3);
    const float s8_2 = (b3 ? gt3 : gp0) + mm_dpp<0x140>(b3 ? gp0 : gt3);
    const float s8_3 = (b3 ? gp3 : gr1) + mm_dpp<0x140>(b3 ? gr1 : gp3);
    const float s8_4 = (b3 ? 0.f : gt1) + mm_dpp<0x140>(b3 ? gt1 : 0.f);
    const float s8_5 = (b3 ? 0.f : gp1) + mm_dpp<0x140>(b3 ? gp1 : 0.f);
    const float s8_6 = (b3 ? 0.f : gr2) + mm_dpp<0x140>(b3 ? gr2 : 0.f);
    const float s8_7 = (b3 ? 0.f : gt2) + mm_dpp<0x140>(b3 ? gt2 : 0.f);
    const float s4_0 = (b2 ? s8_4 : s8_0) + mm_dpp<0x141>(b2 ? s8_0 : s8_4);
    const float s4_1 = (b2 ? s8_5 : s8_1) + mm_dpp<0x141>(b2 ? s8_1 : s8_5);
    const float s4_2 = (b2 ? s8_6 : s8_2) + mm_dpp<0x141>(b2 ? s8_2 : s8_6);
    const float s4_3 = (b2 ? s8_7 : s8_3) + mm_dpp<0x141>(b2 ? s8_3 : s8_7);
    const float s2_0 = (b1 ? s4_2 : s4_0) + mm_dpp<0x1B>(b1 ? s4_0 : s4_2);
    const float s2_1 = (b1 ? s4_3 : s4_1) + mm_dpp<0x1B>(b1 ? s4_1 : s4_3);
    float sum = (b0 ? s2_1 : s2_0) + mm_dpp<0xB1>(b0 ? s2_0 : s2_1);
    const float tc = cl < 3 ? t0 : cl < 6 ? t1 : cl < 9 ? t2 : t3;
    if (cl == 0 || cl == 3 || cl == 6 || cl == 9) sum *= mm_spline_dxdr(tc, inv_h);   // zero below the table start
    if (cl < 12 && cl < 3 * n_own)
      part[(size_t)cb * part_stride + (size_t)(eb + 4 * eg) * 3 + cl] = sum;
    const unsigned sl0 = (sl4 >> 0) & 255u;
    const unsigned sl1 = (sl4 >> 8) & 255u;
    const unsigned sl2 = (sl4 >> 16) & 255u;
    const unsigned sl3 = (sl4 >> 24) & 255u;
    // the group's LDS accumulators of the senders by 32-bit compare-and-swap, all issued together and repeated only
    // where another wave came between; edges without a slot add to gX directly
    if (__all(n_own == 4 && !(sl0 == 255 || sl1 == 255 || sl2 == 255 || sl3 == 255))) {
      unsigned* __restrict__ l0 = (unsigned*)gxs + sl0 * 64 + cl;
      unsigned* __restrict__ l1 = (unsigned*)gxs + sl1 * 64 + cl;
      unsigned* __restrict__ l2 = (unsigned*)gxs + sl2 * 64 + cl;
      unsigned* __restrict__ l3 = (unsigned*)gxs + sl3 * 64 + cl;
      unsigned a0_0 = l0[0];
      unsigned a1_0 = l0[16];
      unsigned a2_0 = l0[32];
      unsigned a3_0 = l0[48];
      unsigned a0_1 = l1[0];
      unsigned a1_1 = l1[16];
      unsigned a2_1 = l1[32];
      unsigned a3_1 = l1[48];
      unsigned a0_2 = l2[0];
      unsigned a1_2 = l2[16];
      unsigned a2_2 = l2[32];
      unsigned a3_2 = l2[48];
      unsigned a0_3 = l3[0];
      unsigned a1_3 = l3[16];
      unsigned a2_3 = l3[32];
      unsigned a3_3 = l3[48];
      unsigned r0_0 = atomicCAS(l0 + 0, a0_0, __float_as_uint(fmaf(gx0_0, gun, __uint_as_float(a0_0))));
      unsigned r1_0 = atomicCAS(l0 + 16, a1_0, __float_as_uint(fmaf(gx1_0, gun, __uint_as_float(a1_0))));
      unsigned r2_0 = atomicCAS(l0 + 32, a2_0, __float_as_uint(fmaf(gx2_0, gun, __uint_as_float(a2_0))));
      unsigned r3_0 = atomicCAS(l0 + 48, a3_0, __float_as_uint(fmaf(gx3_0, gun, __uint_as_float(a3_0))));
      unsigned r0_1 = atomicCAS(l1 + 0, a0_1, __float_as_uint(fmaf(gx0_1, gun, __uint_as_float(a0_1))));
      unsigned r1_1 = atomicCAS(l1 + 16, a1_1, __float_as_uint(fmaf(gx1_1, gun, __uint_as_float(a1_1))));
      unsigned r2_1 = atomicCAS(l1 + 32, a2_1, __float_as_uint(fmaf(gx2_1, gun, __uint_as_float(a2_1))));
      unsigned r3_1 = atomicCAS(l1 + 48, a3_1, __float_as_uint(fmaf(gx3_1, gun, __uint_as_float(a3_1))));
      unsigned r0_2 = atomicCAS(l2 + 0, a0_2, __float_as_uint(fmaf(gx0_2, gun, __uint_as_float(a0_2))));
      unsigned r1_2 = atomicCAS(l2 + 16, a1_2, __float_as_uint(fmaf(gx1_2, gun, __uint_as_float(a1_2))));
      unsigned r2_2 = atomicCAS(l2 + 32, a2_2, __float_as_uint(fmaf(gx2_2, gun, __uint_as_float(a2_2))));
      unsigned r3_2 = atomicCAS(l2 + 48, a3_2, __float_as_uint(fmaf(gx3_2, gun, __uint_as_float(a3_2))));
      unsigned r0_3 = atomicCAS(l3 + 0, a0_3, __float_as_uint(fmaf(gx0_3, gun, __uint_as_float(a0_3))));
      unsigned r1_3 = atomicCAS(l3 + 16, a1_3, __float_as_uint(fmaf(gx1_3, gun, __uint_as_float(a1_3))));
      unsigned r2_3 = atomicCAS(l3 + 32, a2_3, __float_as_uint(fmaf(gx2_3, gun, __uint_as_float(a2_3))));
      unsigned r3_3 = atomicCAS(l3 + 48, a3_3, __float_as_uint(fmaf(gx3_3, gun, __uint_as_float(a3_3))));
      if ((r0_0 != a0_0) | (r1_0 != a1_0) | (r2_0 != a2_0) | (r3_0 != a3_0) | (r0_1 != a0_1) | (r1_1 != a1_1) | (r2_1 != a2_1) | (r3_1 != a3_1) | (r0_2 != a0_2) | (r1_2 != a1_2) | (r2_2 != a2_2) | (r3_2 != a3_2) | (r0_3 != a0_3) | (r1_3 != a1_3) | (r2_3 != a2_3) | (r3_3 != a3_3)) {
        while (r0_0 != a0_0) { a0_0 = r0_0; r0_0 = atomicCAS(l0 + 0, a0_0, __float_as_uint(fmaf(gx0_0, gun, __uint_as_float(a0_0)))); }
        while (r1_0 != a1_0) { a1_0 = r1_0; r1_0 = atomicCAS(l0 + 16, a1_0, __float_as_uint(fmaf(gx1_0, gun, __uint_as_float(a1_0)))); }
        while (r2_0 != a2_0) { a2_0 = r2_0; r2_0 = atomicCAS(l0 + 32, a2_0, __float_as_uint(fmaf(gx2_0, gun, __uint_as_float(a2_0)))); }
        while (r3_0 != a3_0) { a3_0 = r3_0; r3_0 = atomicCAS(l0 + 48, a3_0, __float_as_uint(fmaf(gx3_0, gun, __uint_as_float(a3_0)))); }
        while (r0_1 != a0_1) { a0_1 = r0_1; r0_1 = atomicCAS(l1 + 0, a0_1, __float_as_uint(fmaf(gx0_1, gun, __uint_as_float(a0_1)))); }
        while (r1_1 != a1_1) { a1_1 = r1_1; r1_1 = atomicCAS(l1 + 16, a1_1, __float_as_uint(fmaf(gx1_1, gun, __uint_as_float(a1_1)))); }
        while (r2_1 != a2_1) { a2_1 = r2_1; r2_1 = atomicCAS(l1 + 32, a2_1, __float_as_uint(fmaf(gx2_1, gun, __uint_as_float(a2_1)))); }
        while (r3_1 != a3_1) { a3_1 = r3_1; r3_1 = atomicCAS(l1 + 48, a3_1, __float_as_uint(fmaf(gx3_1, gun, __uint_as_float(a3_1)))); }
        while (r0_2 != a0_2) { a0_2 = r0_2; r0_2 = atomicCAS(l2 + 0, a0_2, __float_as_uint(fmaf(gx0_2, gun, __uint_as_float(a0_2)))); }
        while (r1_2 != a1_2) { a1_2 = r1_2; r1_2 = atomicCAS(l2 + 16, a1_2, __float_as_uint(fmaf(gx1_2, gun, __uint_as_float(a1_2)))); }
        while (r2_2 != a2_2) { a2_2 = r2_2; r2_2 = atomicCAS(l2 + 32, a2_2, __float_as_uint(fmaf(gx2_2, gun, __uint_as_float(a2_2)))); }
        while (r3_2 != a3_2) { a3_2 = r3_2; r3_2 = atomicCAS(l2 + 48, a3_2, __float_as_uint(fmaf(gx3_2, gun, __uint_as_float(a3_2)))); }
        while (r0_3 != a0_3) { a0_3 = r0_3; r0_3 = atomicCAS(l3 + 0, a0_3, __float_as_uint(fmaf(gx0_3, gun, __uint_as_float(a0_3)))); }
        while (r1_3 != a1_3) { a1_3 = r1_3; r1_3 = atomicCAS(l3 + 16, a1_3, __float_as_uint(fmaf(gx1_3, gun, __uint_as_float(a1_3)))); }
        while (r2_3 != a2_3) { a2_3 = r2_3; r2_3 = atomicCAS(l3 + 32, a2_3, __float_as_uint(fmaf(gx2_3, gun, __uint_as_float(a2_3)))); }
        while (r3_3 != a3_3) { a3_3 = r3_3; r3_3 = atomicCAS(l3 + 48, a3_3, __float_as_uint(fmaf(gx3_3, gun, __uint_as_float(a3_3)))); }
      }
    } else {
      if (0 < n_own) {
        if (sl0 != 255) {
          mm_lds_add4_f32(gxs + sl0 * 64 + cl, gx0_0 * gun, gx1_0 * gun, gx2_0 * gun, gx3_0 * gun);
        } else {
          float* __restrict__ gxp = gX + (size_t)__float_as_int(e_pk[eb + 4 * eg + 0].z) * 512 + cb * 64 + cl;
          atomicAdd(gxp + 0, gx0_0 * gun);
          atomicAdd(gxp + 16, gx1_0 * gun);
          atomicAdd(gxp + 32, gx2_0 * gun);
          atomicAdd(gxp + 48, gx3_0 * gun);
        }
      }
      if (1 < n_own) {
        if (sl1 != 255) {
          mm_lds_add4_f32(gxs + sl1 * 64 + cl, gx0_1 * gun, gx1_1 * gun, gx2_1 * gun, gx3_1 * gun);
        } else {
          float* __restrict__ gxp = gX + (size_t)__float_as_int(e_pk[eb + 4 * eg + 1].z) * 512 + cb * 64 + cl;
          atomicAdd(gxp + 0, gx0_1 * gun);
          atomicAdd(gxp + 16, gx1_1 * gun);
          atomicAdd(gxp + 32, gx2_1 * gun);
          atomicAdd(gxp + 48, gx3_1 * gun);
        }
      }
      if (2 < n_own) {
        if (sl2 != 255) {
          mm_lds_add4_f32(gxs + sl2 * 64 + cl, gx0_2 * gun, gx1_2 * gun, gx2_2 * gun, gx3_2 * gun);
        } else {
          float* __restrict__ gxp = gX + (size_t)__float_as_int(e_pk[eb + 4 * eg + 2].z) * 512 + cb * 64 + cl;
          atomicAdd(gxp + 0, gx0_2 * gun);
          atomicAdd(gxp + 16, gx1_2 * gun);
          atomicAdd(gxp + 32, gx2_2 * gun);
          atomicAdd(gxp + 48, gx3_2 * gun);
        }
      }
      if (3 < n_own) {
        if (sl3 != 255) {
          mm_lds_add4_f32(gxs + sl3 * 64 + cl, gx0_3 * gun, gx1_3 * gun, gx2_3 * gun, gx3_3 * gun);
        } else {
          float* __restrict__ gxp = gX + (size_t)__float_as_int(e_pk[eb + 4 * eg + 3].z) * 512 + cb * 64 + cl;
          atomicAdd(gxp + 0, gx0_3 * gun);
          atomicAdd(gxp + 16, gx1_3 * gun);
          atomicAdd(gxp + 32, gx2_3 * gun);
          atomicAdd(gxp + 48, gx3_3 * gun);
        }
      }
    }
  }
  }   // edges
  __syncthreads();
  for (int j = threadIdx.x; j < ns * 64; j += 256) {
    const int sl = j >> 6, r = j & 63;   // a slot: 256 contiguous bytes [component][channel] of its sender's row
    atomicAdd(gX + (size_t)ssend[sl] * 512 + cb * 64 + r, gxs[j]);
  }
}

extern "C" int mm_conv2_bwd_vec(const int* rowptr, int nC, const float* e_pk, const float* e_u,
    const float* X, int x_stride, const float* tab, int n_tab, int M, float inv_h, const float* gA,
    float* part, long part_stride, float* gX, const unsigned char* e_slot, const int* g_send, const int* g_n, hipStream_t stream) {
  MM_CHECK_ARG(nC >= 0 && M >= 2 && n_tab >= 1, "bad sizes");
  MM_CHECK_ARG(e_slot && g_send && g_n, "the groups' sender slots (mm_sender_slots) are required");
  MM_CHECK_ARG(gX != nullptr, "the sender-feature gradient buffer is required");
  MM_CHECK_ARG((long)n_tab * (M - 1) * 2560 < (1L << 32), "a channel block's tables exceed 4 GiB");
  if (nC == 0) return MM_OK;
  hipLaunchKernelGGL(mm_conv2_bwd_vec_kernel, dim3(8 * ((nC + 3) / 4)), dim3(256), 0, stream, rowptr, nC,
                     (const floatx4*)e_pk, (const floatx4*)e_u, X, x_stride, (const floatx4*)tab,
                     n_tab * (M - 1) * 160, inv_h, gA, part, part_stride, gX, e_slot, g_send, g_n);
  return mm::launch_status("mm_conv2_bwd_vec");
}

extern "C" __global__ void __launch_bounds__(256, 2)
mm_conv2_bwd_vec_det_kernel(const int* __restrict__ rowptr, int nC, const floatx4* __restrict__ e_pk,
    const floatx4* __restrict__ e_u, const float* __restrict__ X, int x_stride,
    const floatx4* __restrict__ tab, int tab_cb_stride, float inv_h,
    const float* __restrict__ gA, float* __restrict__ part, long part_stride, float* __restrict__ gX) {
  const int cb = mm_xcd_channel_block();
  __shared__ uint4v ya_all[1152];   // per wave: [type][degree][edge][piece] operand rows
  const int grp = blockIdx.x >> 3, i = grp * 4 + (threadIdx.x >> 6);
  if (i >= nC) return;
  const int ir = i;
  const int lane = threadIdx.x & 63, cl = lane & 15, eg = lane >> 4;
  uint4v* __restrict__ ya = ya_all + (threadIdx.x >> 6) * 288;
  const int c = cb * 16 + cl;
  const int e0 = rowptr[ir], e1 = i < nC ? rowptr[ir + 1] : e0;
  const char* __restrict__ tcb = (const char*)(tab + (size_t)cb * tab_cb_stride);
  const float* __restrict__ gp = gA + (size_t)ir * 5120 + c;
  float g0 = gp[0];
  float g1 = gp[128];
  float g2 = gp[256];
  float g3 = gp[384];
  float g4 = gp[512];
  float g5 = gp[640];
  float g6 = gp[768];
  float g7 = gp[896];
  float g8 = gp[1024];
  float g9 = gp[1152];
  float g10 = gp[1280];
  float g11 = gp[1408];
  float g12 = gp[1536];
  float g13 = gp[1664];
  float g14 = gp[1792];
  float g15 = gp[1920];
  float g16 = gp[2048];
  float g17 = gp[2176];
  float g18 = gp[2304];
  float g19 = gp[2432];
  float g20 = gp[2560];
  float g21 = gp[2688];
  float g22 = gp[2816];
  float g23 = gp[2944];
  float g24 = gp[3072];
  float g25 = gp[3200];
  float g26 = gp[3328];
  float g27 = gp[3456];
  float g28 = gp[3584];
  float g29 = gp[3712];
  float g30 = gp[3840];
  float g31 = gp[3968];
  float g32 = gp[4096];
  float g33 = gp[4224];
  float g34 = gp[4352];
  float g35 = gp[4480];
  float g36 = gp[4608];
  float g37 = gp[4736];
  float g38 = gp[4864];
  float g39 = gp[4992];
  // power-of-two scale of this channel's constants into the fp16 range
  const float mx0 = fmaxf(fmaxf(fabsf(g6), fabsf(g7)), fmaxf(fmaxf(fabsf(g4), fabsf(g5)), fmaxf(fmaxf(fabsf(g2), fabsf(g3)), fmaxf(fmaxf(fabsf(g0), fabsf(g1)), 0.f))));
  const float mx1 = fmaxf(fmaxf(fabsf(g14), fabsf(g15)), fmaxf(fmaxf(fabsf(g12), fabsf(g13)), fmaxf(fmaxf(fabsf(g10), fabsf(g11)), fmaxf(fmaxf(fabsf(g8), fabsf(g9)), mx0))));
  const float mx2 = fmaxf(fmaxf(fabsf(g22), fabsf(g23)), fmaxf(fmaxf(fabsf(g20), fabsf(g21)), fmaxf(fmaxf(fabsf(g18), fabsf(g19)), fmaxf(fmaxf(fabsf(g16), fabsf(g17)), mx1))));
  const float mx3 = fmaxf(fmaxf(fabsf(g30), fabsf(g31)), fmaxf(fmaxf(fabsf(g28), fabsf(g29)), fmaxf(fmaxf(fabsf(g26), fabsf(g27)), fmaxf(fmaxf(fabsf(g24), fabsf(g25)), mx2))));
  const float mx4 = fmaxf(fmaxf(fabsf(g38), fabsf(g39)), fmaxf(fmaxf(fabsf(g36), fabsf(g37)), fmaxf(fmaxf(fabsf(g34), fabsf(g35)), fmaxf(fmaxf(fabsf(g32), fabsf(g33)), mx3))));
  const int gex = max(__float_as_int(mx4) >> 23, 40);
  const float gsc = __int_as_float((265 - gex) << 23);
  const float gun = __int_as_float((gex - 24) << 23);   // 1 / (gsc MM_POLAR_SCALE)
  const float U0_0 = g0 * gsc * MM_POLAR_SCALE;   // l2 = 0: the same u for every edge
  const float U3_1 = g5 * gsc * MM_POLAR_SCALE;   // l2 = 0: the same u for every edge
  const float U3_2 = g6 * gsc * MM_POLAR_SCALE;   // l2 = 0: the same u for every edge
  const float U3_3 = g7 * gsc * MM_POLAR_SCALE;   // l2 = 0: the same u for every edge
  g0 *= gsc;
  g1 *= gsc;
  g2 *= gsc;
  g3 *= gsc;
  g4 *= gsc;
  g5 *= gsc;
  g6 *= gsc;
  g7 *= gsc;
  g8 *= gsc;
  g9 *= gsc;
  g10 *= gsc;
  g11 *= gsc;
  g12 *= gsc;
  g13 *= gsc;
  g14 *= gsc;
  g15 *= gsc;
  g16 *= gsc;
  g17 *= gsc;
  g18 *= gsc;
  g19 *= gsc;
  g20 *= gsc;
  g21 *= gsc;
  g22 *= gsc;
  g23 *= gsc;
  g24 *= gsc;
  g25 *= gsc;
  g26 *= gsc;
  g27 *= gsc;
  g28 *= gsc;
  g29 *= gsc;
  g30 *= gsc;
  g31 *= gsc;
  g32 *= gsc;
  g33 *= gsc;
  g34 *= gsc;
  g35 *= gsc;
  g36 *= gsc;
  g37 *= gsc;
  g38 *= gsc;
  g39 *= gsc;
  // B operands: lane (channel cl, k-group eg) holds fp16 piece 1 - (eg & 1) of its channel's constants
  const bool pb = !(eg & 1);
  uint4v B7_1;
  { unsigned h0, h1; mm_split2_f16(float2v{1.2499999999999998f, 2.4999999999999996f}, float2v{g25, g24}, h0, h1); B7_1[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{fmaf(0.24999999999999997f, g25, 0.8660254037844387f * g23), -0.5f}, float2v{1.f, g22}, h0, h1); B7_1[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-0.25000000000000006f, -2.4999999999999996f}, float2v{g21, g22}, h0, h1); B7_1[2] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-1.25f, 0.f}, float2v{g21, 1.f}, h0, h1); B7_1[3] = pb ? h1 : h0; }
  uint4v B7_2;
  { unsigned h0, h1; mm_split2_f16(float2v{0.f, 2.4999999999999996f}, float2v{1.f, g21}, h0, h1); B7_2[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{1.0f, 0.8660254037844387f}, float2v{g22, g23}, h0, h1); B7_2[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{1.0000000000000004f, 2.4999999999999996f}, float2v{g24, g25}, h0, h1); B7_2[2] = pb ? h1 : h0; }
  B7_2[3] = 0;
  uint4v B7_3;
  { unsigned h0, h1; mm_split2_f16(float2v{1.2499999999999998f, 2.4999999999999996f}, float2v{g21, g22}, h0, h1); B7_3[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-0.24999999999999997f, -0.5f}, float2v{g21, g24}, h0, h1); B7_3[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{fmaf(-0.25000000000000006f, g25, 0.866025403784439f * g23), 2.4999999999999996f}, float2v{1.f, g24}, h0, h1); B7_3[2] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{1.25f, 0.f}, float2v{g25, 1.f}, h0, h1); B7_3[3] = pb ? h1 : h0; }
  uint4v B8_0;
  { unsigned h0, h1; mm_split2_f16(float2v{2.091650066335189f, 5.123475382979799f}, float2v{g26, g27}, h0, h1); B8_0[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{1.620185174601965f, 1.3228756555322956f}, float2v{g28, g29}, h0, h1); B8_0[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{1.6201851746019658f, 5.123475382979799f}, float2v{g30, g31}, h0, h1); B8_0[2] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{2.0916500663351894f, 0.f}, float2v{g32, 1.f}, h0, h1); B8_0[3] = pb ? h1 : h0; }
  uint4v B4_1;
  { unsigned h0, h1; mm_split2_f16(float2v{1.0606601717798207f, 2.121320343559642f}, float2v{g10, g9}, h0, h1); B4_1[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-0.35355339059327384f, 0.f}, float2v{g8, 1.f}, h0, h1); B4_1[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-1.060660171779821f, 0.f}, float2v{g8, 1.f}, h0, h1); B4_1[2] = pb ? h1 : h0; }
  B4_1[3] = 0;
  uint4v B4_2;
  { unsigned h0, h1; mm_split2_f16(float2v{0.f, 2.121320343559642f}, float2v{1.f, g8}, h0, h1); B4_2[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{0.7071067811865478f, 2.121320343559642f}, float2v{g9, g10}, h0, h1); B4_2[1] = pb ? h1 : h0; }
  B4_2[2] = 0;
  B4_2[3] = 0;
  uint4v B4_3;
  { unsigned h0, h1; mm_split2_f16(float2v{1.0606601717798207f, 0.f}, float2v{g8, 1.f}, h0, h1); B4_3[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-0.35355339059327384f, 2.121320343559642f}, float2v{g10, g9}, h0, h1); B4_3[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{1.060660171779821f, 0.f}, float2v{g10, 1.f}, h0, h1); B4_3[2] = pb ? h1 : h0; }
  B4_3[3] = 0;
  uint4v B5_0;
  { unsigned h0, h1; mm_split2_f16(float2v{1.936491673103708f, 3.8729833462074166f}, float2v{g11, g12}, h0, h1); B5_0[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{1.1180339887498953f, 3.872983346207417f}, float2v{g13, g14}, h0, h1); B5_0[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{1.9364916731037083f, 0.f}, float2v{g15, 1.f}, h0, h1); B5_0[2] = pb ? h1 : h0; }
  B5_0[3] = 0;
  uint4v B9_1;
  { unsigned h0, h1; mm_split2_f16(float2v{fmaf(1.369306393762915f, g39, 0.35355339059327373f * g37), fmaf(2.236067977499789f, g38, 1.7320508075688774f * g36)}, float2v{1.f, 1.f}, h0, h1); B9_1[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-0.7071067811865478f, -2.2360679774997894f}, float2v{g35, g34}, h0, h1); B9_1[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{fmaf(-0.3535533905932738f, g35, -1.3693063937629153f * g33), 0.f}, float2v{1.f, 1.f}, h0, h1); B9_1[2] = pb ? h1 : h0; }
  B9_1[3] = 0;
  uint4v B9_2;
  { unsigned h0, h1; mm_split2_f16(float2v{-1.1180339887498947f, -2.8284271247461903f}, float2v{g34, g35}, h0, h1); B9_2[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-0.8660254037844392f, -2.8284271247461903f}, float2v{g36, g37}, h0, h1); B9_2[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-1.118033988749895f, 0.f}, float2v{g38, 1.f}, h0, h1); B9_2[2] = pb ? h1 : h0; }
  B9_2[3] = 0;
  uint4v B9_3;
  { unsigned h0, h1; mm_split2_f16(float2v{fmaf(0.35355339059327373f, g35, -1.369306393762915f * g33), -2.236067977499789f}, float2v{1.f, g34}, h0, h1); B9_3[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-0.7071067811865478f, fmaf(-2.2360679774997894f, g38, 1.7320508075688774f * g36)}, float2v{g37, 1.f}, h0, h1); B9_3[1] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{fmaf(-1.3693063937629153f, g39, 0.3535533905932738f * g37), 0.f}, float2v{1.f, 1.f}, h0, h1); B9_3[2] = pb ? h1 : h0; }
  B9_3[3] = 0;
  uint2v B1_1;
  { unsigned h0, h1; mm_split2_f16(float2v{0.9999999999999999f, 0.f}, float2v{g1, 1.f}, h0, h1); B1_1[0] = pb ? h1 : h0; }
  B1_1[1] = 0;
  uint2v B1_2;
  { unsigned h0, h1; mm_split2_f16(float2v{0.f, 1.0f}, float2v{1.f, g1}, h0, h1); B1_2[0] = pb ? h1 : h0; }
  B1_2[1] = 0;
  uint2v B1_3;
  B1_3[0] = 0;
  { unsigned h0, h1; mm_split2_f16(float2v{0.9999999999999999f, 0.f}, float2v{g1, 1.f}, h0, h1); B1_3[1] = pb ? h1 : h0; }
  uint2v B2_0;
  { unsigned h0, h1; mm_split2_f16(float2v{1.732050807568877f, 1.7320508075688772f}, float2v{g2, g3}, h0, h1); B2_0[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{1.732050807568877f, 0.f}, float2v{g4, 1.f}, h0, h1); B2_0[1] = pb ? h1 : h0; }
  uint2v B6_1;
  { unsigned h0, h1; mm_split2_f16(float2v{fmaf(1.224744871391589f, g20, 0.7071067811865475f * g18), -1.2247448713915892f}, float2v{1.f, g17}, h0, h1); B6_1[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-1.224744871391589f, 0.f}, float2v{g16, 1.f}, h0, h1); B6_1[1] = pb ? h1 : h0; }
  uint2v B6_2;
  { unsigned h0, h1; mm_split2_f16(float2v{-1.2247448713915892f, -1.4142135623730951f}, float2v{g17, g18}, h0, h1); B6_2[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{-1.2247448713915892f, 0.f}, float2v{g19, 1.f}, h0, h1); B6_2[1] = pb ? h1 : h0; }
  uint2v B6_3;
  { unsigned h0, h1; mm_split2_f16(float2v{-1.224744871391589f, -1.2247448713915892f}, float2v{g16, g19}, h0, h1); B6_3[0] = pb ? h1 : h0; }
  { unsigned h0, h1; mm_split2_f16(float2v{fmaf(-1.224744871391589f, g20, 0.7071067811865475f * g18), 0.f}, float2v{1.f, 1.f}, h0, h1); B6_3[1] = pb ? h1 : h0; }
  if (e0 < e1) {
  floatx4 pkn0, pkn1, pkn2, pkn3, un;   // records and edge vector of the next tile
  unsigned on0, on1, on2, on3;           // its table rows
    pkn0 = e_pk[min(e0 + 4 * eg + 0, e1 - 1)];
    pkn1 = e_pk[min(e0 + 4 * eg + 1, e1 - 1)];
    pkn2 = e_pk[min(e0 + 4 * eg + 2, e1 - 1)];
    pkn3 = e_pk[min(e0 + 4 * eg + 3, e1 - 1)];
    un = e_u[min(e0 + cl, e1 - 1)];
    on0 = (unsigned)__float_as_int(pkn0.y) * 2560u + cl * 16u;
    on1 = (unsigned)__float_as_int(pkn1.y) * 2560u + cl * 16u;
    on2 = (unsigned)__float_as_int(pkn2.y) * 2560u + cl * 16u;
    on3 = (unsigned)__float_as_int(pkn3.y) * 2560u + cl * 16u;
    floatx4 q0_0 = *(const floatx4*)(tcb + on0 + 1792);
    floatx4 q0_1 = *(const floatx4*)(tcb + on1 + 1792);
    floatx4 q0_2 = *(const floatx4*)(tcb + on2 + 1792);
    floatx4 q0_3 = *(const floatx4*)(tcb + on3 + 1792);
    floatx4 q1_0 = *(const floatx4*)(tcb + on0 + 2048);
    floatx4 q1_1 = *(const floatx4*)(tcb + on1 + 2048);
    floatx4 q1_2 = *(const floatx4*)(tcb + on2 + 2048);
    floatx4 q1_3 = *(const floatx4*)(tcb + on3 + 2048);
  for (int eb = e0; eb < e1; eb += 16) {
    const float t0 = pkn0.x;
    const unsigned o0 = on0;
    const float* __restrict__ xp0 = X + (size_t)__float_as_int(pkn0.z) * x_stride + c;
    const float X0_0 = xp0[0];
    const float X1_0 = xp0[128];
    const float X2_0 = xp0[256];
    const float X3_0 = xp0[384];
    const float t1 = pkn1.x;
    const unsigned o1 = on1;
    const float* __restrict__ xp1 = X + (size_t)__float_as_int(pkn1.z) * x_stride + c;
    const float X0_1 = xp1[0];
    const float X1_1 = xp1[128];
    const float X2_1 = xp1[256];
    const float X3_1 = xp1[384];
    const float t2 = pkn2.x;
    const unsigned o2 = on2;
    const float* __restrict__ xp2 = X + (size_t)__float_as_int(pkn2.z) * x_stride + c;
    const float X0_2 = xp2[0];
    const float X1_2 = xp2[128];
    const float X2_2 = xp2[256];
    const float X3_2 = xp2[384];
    const float t3 = pkn3.x;
    const unsigned o3 = on3;
    const float* __restrict__ xp3 = X + (size_t)__float_as_int(pkn3.z) * x_stride + c;
    const float X0_3 = xp3[0];
    const float X1_3 = xp3[128];
    const float X2_3 = xp3[256];
    const float X3_3 = xp3[384];
    const floatx4 ua = un;
    // the next tile's records and edge vector are loaded one tile ahead (the last tile reloads its own end)
    pkn0 = e_pk[min(eb + 16 + 4 * eg + 0, e1 - 1)];
    pkn1 = e_pk[min(eb + 16 + 4 * eg + 1, e1 - 1)];
    pkn2 = e_pk[min(eb + 16 + 4 * eg + 2, e1 - 1)];
    pkn3 = e_pk[min(eb + 16 + 4 * eg + 3, e1 - 1)];
    un = e_u[min(eb + 16 + cl, e1 - 1)];
    // A operands of edge eb + cl: lane group 0 the harmonics, 1 and 2 their two derivatives
    {
      float F[16], A[16], s, cp, sp;
      mm_polar(ua.x, ua.y, s, cp, sp);
      mm_polar_operands(ua.x, ua.y, ua.z, s, cp, sp, eg, F, A);
      mm_wave_lds_sync();   // the previous tile's operands have been read
      if (eg < 3) {
        { uint4v a = {}, b = {};
          { unsigned h0, h1; mm_split2_f16(float2v{F[9], F[10]}, float2v{A[9], A[10]}, h0, h1); a[0] = h0; b[0] = h1; }
          { unsigned h0, h1; mm_split2_f16(float2v{F[11], F[12]}, float2v{A[11], A[12]}, h0, h1); a[1] = h0; b[1] = h1; }
          { unsigned h0, h1; mm_split2_f16(float2v{F[13], F[14]}, float2v{A[13], A[14]}, h0, h1); a[2] = h0; b[2] = h1; }
          { unsigned h0, h1; mm_split2_f16(float2v{F[15], 0.f}, float2v{A[15], 0.f}, h0, h1); a[3] = h0; b[3] = h1; }
          uint4v* __restrict__ d = ya + ((eg * 3 + 0) * 16 + cl) * 2;
          d[0] = a; d[1] = b; }
        { uint4v a = {}, b = {};
          { unsigned h0, h1; mm_split2_f16(float2v{F[4], F[5]}, float2v{A[4], A[5]}, h0, h1); a[0] = h0; b[0] = h1; }
          { unsigned h0, h1; mm_split2_f16(float2v{F[6], F[7]}, float2v{A[6], A[7]}, h0, h1); a[1] = h0; b[1] = h1; }
          { unsigned h0, h1; mm_split2_f16(float2v{F[8], 0.f}, float2v{A[8], 0.f}, h0, h1); a[2] = h0; b[2] = h1; }
          uint4v* __restrict__ d = ya + ((eg * 3 + 1) * 16 + cl) * 2;
          d[0] = a; d[1] = b; }
        { uint4v a = {}, b = {};
          { unsigned h0, h1; mm_split2_f16(float2v{F[1], F[2]}, float2v{A[1], A[2]}, h0, h1); a[0] = h0; b[0] = h1; }
          { unsigned h0, h1; mm_split2_f16(float2v{F[3], 0.f}, float2v{A[3], 0.f}, h0, h1); a[1] = h0; b[1] = h1; }
          uint4v* __restrict__ d = ya + ((eg * 3 + 2) * 16 + cl) * 2;
          d[0] = a; d[1] = b; }
      }
      mm_wave_lds_sync();
    }
    float gr0 = 0.f, gt0 = 0.f, gp0 = 0.f;
    float gx0_0 = 0.f;
    float gx1_0 = 0.f;
    float gx2_0 = 0.f;
    float gx3_0 = 0.f;
    float gr1 = 0.f, gt1 = 0.f, gp1 = 0.f;
    float gx0_1 = 0.f;
    float gx1_1 = 0.f;
    float gx2_1 = 0.f;
    float gx3_1 = 0.f;
    float gr2 = 0.f, gt2 = 0.f, gp2 = 0.f;
    float gx0_2 = 0.f;
    float gx1_2 = 0.f;
    float gx2_2 = 0.f;
    float gx3_2 = 0.f;
    float gr3 = 0.f, gt3 = 0.f, gp3 = 0.f;
    float gx0_3 = 0.f;
    float gx1_3 = 0.f;
    float gx2_3 = 0.f;
    float gx3_3 = 0.f;
    const half8v A3_0 = __builtin_bit_cast(half8v, ya[((0) * 16 + cl) * 2 + 1 - (eg >> 1)]);
    const half8v A3_1 = __builtin_bit_cast(half8v, ya[((3) * 16 + cl) * 2 + 1 - (eg >> 1)]);
    const half8v A3_2 = __builtin_bit_cast(half8v, ya[((6) * 16 + cl) * 2 + 1 - (eg >> 1)]);
    const floatx4 D0_7_1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_0, __builtin_bit_cast(half8v, B7_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_7_1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_1, __builtin_bit_cast(half8v, B7_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_7_1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_2, __builtin_bit_cast(half8v, B7_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_7_2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_0, __builtin_bit_cast(half8v, B7_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_7_2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_1, __builtin_bit_cast(half8v, B7_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_7_2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_2, __builtin_bit_cast(half8v, B7_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_7_3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_0, __builtin_bit_cast(half8v, B7_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_7_3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_1, __builtin_bit_cast(half8v, B7_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_7_3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_2, __builtin_bit_cast(half8v, B7_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    {
      const floatx4 q = q0_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx1_0 = fmaf(W, D0_7_1[0], gx1_0);
      gx2_0 = fmaf(W, D0_7_2[0], gx2_0);
      gx3_0 = fmaf(W, D0_7_3[0], gx3_0);
      gr0 = fmaf(fmaf(X3_0, D0_7_3[0], fmaf(X2_0, D0_7_2[0], X1_0 * D0_7_1[0])), D, gr0);
      gt0 = fmaf(fmaf(X3_0, D1_7_3[0], fmaf(X2_0, D1_7_2[0], X1_0 * D1_7_1[0])), W, gt0);
      gp0 = fmaf(fmaf(X3_0, D2_7_3[0], fmaf(X2_0, D2_7_2[0], X1_0 * D2_7_1[0])), W, gp0);
    }
    {
      const floatx4 q = q0_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx1_1 = fmaf(W, D0_7_1[1], gx1_1);
      gx2_1 = fmaf(W, D0_7_2[1], gx2_1);
      gx3_1 = fmaf(W, D0_7_3[1], gx3_1);
      gr1 = fmaf(fmaf(X3_1, D0_7_3[1], fmaf(X2_1, D0_7_2[1], X1_1 * D0_7_1[1])), D, gr1);
      gt1 = fmaf(fmaf(X3_1, D1_7_3[1], fmaf(X2_1, D1_7_2[1], X1_1 * D1_7_1[1])), W, gt1);
      gp1 = fmaf(fmaf(X3_1, D2_7_3[1], fmaf(X2_1, D2_7_2[1], X1_1 * D2_7_1[1])), W, gp1);
    }
    {
      const floatx4 q = q0_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx1_2 = fmaf(W, D0_7_1[2], gx1_2);
      gx2_2 = fmaf(W, D0_7_2[2], gx2_2);
      gx3_2 = fmaf(W, D0_7_3[2], gx3_2);
      gr2 = fmaf(fmaf(X3_2, D0_7_3[2], fmaf(X2_2, D0_7_2[2], X1_2 * D0_7_1[2])), D, gr2);
      gt2 = fmaf(fmaf(X3_2, D1_7_3[2], fmaf(X2_2, D1_7_2[2], X1_2 * D1_7_1[2])), W, gt2);
      gp2 = fmaf(fmaf(X3_2, D2_7_3[2], fmaf(X2_2, D2_7_2[2], X1_2 * D2_7_1[2])), W, gp2);
    }
    {
      const floatx4 q = q0_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx1_3 = fmaf(W, D0_7_1[3], gx1_3);
      gx2_3 = fmaf(W, D0_7_2[3], gx2_3);
      gx3_3 = fmaf(W, D0_7_3[3], gx3_3);
      gr3 = fmaf(fmaf(X3_3, D0_7_3[3], fmaf(X2_3, D0_7_2[3], X1_3 * D0_7_1[3])), D, gr3);
      gt3 = fmaf(fmaf(X3_3, D1_7_3[3], fmaf(X2_3, D1_7_2[3], X1_3 * D1_7_1[3])), W, gt3);
      gp3 = fmaf(fmaf(X3_3, D2_7_3[3], fmaf(X2_3, D2_7_2[3], X1_3 * D2_7_1[3])), W, gp3);
    }
    asm volatile("" : "+v"(gx1_0), "+v"(gx1_1), "+v"(gx1_2), "+v"(gx1_3), "+v"(gx2_0), "+v"(gx2_1), "+v"(gx2_2), "+v"(gx2_3), "+v"(gx3_0), "+v"(gx3_1), "+v"(gx3_2), "+v"(gx3_3));
    floatx4 q2_0 = *(const floatx4*)(tcb + o0 + 1024);
    floatx4 q2_1 = *(const floatx4*)(tcb + o1 + 1024);
    floatx4 q2_2 = *(const floatx4*)(tcb + o2 + 1024);
    floatx4 q2_3 = *(const floatx4*)(tcb + o3 + 1024);
    const floatx4 D0_8_0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_0, __builtin_bit_cast(half8v, B8_0), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_8_0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_1, __builtin_bit_cast(half8v, B8_0), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_8_0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A3_2, __builtin_bit_cast(half8v, B8_0), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    {
      const floatx4 q = q1_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx0_0 = fmaf(W, D0_8_0[0], gx0_0);
      gr0 = fmaf(X0_0 * D0_8_0[0], D, gr0);
      gt0 = fmaf(X0_0 * D1_8_0[0], W, gt0);
      gp0 = fmaf(X0_0 * D2_8_0[0], W, gp0);
    }
    {
      const floatx4 q = q1_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx0_1 = fmaf(W, D0_8_0[1], gx0_1);
      gr1 = fmaf(X0_1 * D0_8_0[1], D, gr1);
      gt1 = fmaf(X0_1 * D1_8_0[1], W, gt1);
      gp1 = fmaf(X0_1 * D2_8_0[1], W, gp1);
    }
    {
      const floatx4 q = q1_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx0_2 = fmaf(W, D0_8_0[2], gx0_2);
      gr2 = fmaf(X0_2 * D0_8_0[2], D, gr2);
      gt2 = fmaf(X0_2 * D1_8_0[2], W, gt2);
      gp2 = fmaf(X0_2 * D2_8_0[2], W, gp2);
    }
    {
      const floatx4 q = q1_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx0_3 = fmaf(W, D0_8_0[3], gx0_3);
      gr3 = fmaf(X0_3 * D0_8_0[3], D, gr3);
      gt3 = fmaf(X0_3 * D1_8_0[3], W, gt3);
      gp3 = fmaf(X0_3 * D2_8_0[3], W, gp3);
    }
    asm volatile("" : "+v"(gx0_0), "+v"(gx0_1), "+v"(gx0_2), "+v"(gx0_3));
    floatx4 q3_0 = *(const floatx4*)(tcb + o0 + 1280);
    floatx4 q3_1 = *(const floatx4*)(tcb + o1 + 1280);
    floatx4 q3_2 = *(const floatx4*)(tcb + o2 + 1280);
    floatx4 q3_3 = *(const floatx4*)(tcb + o3 + 1280);
    const half8v A2_0 = __builtin_bit_cast(half8v, ya[((1) * 16 + cl) * 2 + 1 - (eg >> 1)]);
    const half8v A2_1 = __builtin_bit_cast(half8v, ya[((4) * 16 + cl) * 2 + 1 - (eg >> 1)]);
    const half8v A2_2 = __builtin_bit_cast(half8v, ya[((7) * 16 + cl) * 2 + 1 - (eg >> 1)]);
    const floatx4 D0_4_1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_0, __builtin_bit_cast(half8v, B4_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_4_1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_1, __builtin_bit_cast(half8v, B4_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_4_1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_2, __builtin_bit_cast(half8v, B4_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_4_2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_0, __builtin_bit_cast(half8v, B4_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_4_2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_1, __builtin_bit_cast(half8v, B4_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_4_2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_2, __builtin_bit_cast(half8v, B4_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_4_3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_0, __builtin_bit_cast(half8v, B4_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_4_3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_1, __builtin_bit_cast(half8v, B4_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_4_3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_2, __builtin_bit_cast(half8v, B4_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    {
      const floatx4 q = q2_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx1_0 = fmaf(W, D0_4_1[0], gx1_0);
      gx2_0 = fmaf(W, D0_4_2[0], gx2_0);
      gx3_0 = fmaf(W, D0_4_3[0], gx3_0);
      gr0 = fmaf(fmaf(X3_0, D0_4_3[0], fmaf(X2_0, D0_4_2[0], X1_0 * D0_4_1[0])), D, gr0);
      gt0 = fmaf(fmaf(X3_0, D1_4_3[0], fmaf(X2_0, D1_4_2[0], X1_0 * D1_4_1[0])), W, gt0);
      gp0 = fmaf(fmaf(X3_0, D2_4_3[0], fmaf(X2_0, D2_4_2[0], X1_0 * D2_4_1[0])), W, gp0);
    }
    {
      const floatx4 q = q2_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx1_1 = fmaf(W, D0_4_1[1], gx1_1);
      gx2_1 = fmaf(W, D0_4_2[1], gx2_1);
      gx3_1 = fmaf(W, D0_4_3[1], gx3_1);
      gr1 = fmaf(fmaf(X3_1, D0_4_3[1], fmaf(X2_1, D0_4_2[1], X1_1 * D0_4_1[1])), D, gr1);
      gt1 = fmaf(fmaf(X3_1, D1_4_3[1], fmaf(X2_1, D1_4_2[1], X1_1 * D1_4_1[1])), W, gt1);
      gp1 = fmaf(fmaf(X3_1, D2_4_3[1], fmaf(X2_1, D2_4_2[1], X1_1 * D2_4_1[1])), W, gp1);
    }
    {
      const floatx4 q = q2_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx1_2 = fmaf(W, D0_4_1[2], gx1_2);
      gx2_2 = fmaf(W, D0_4_2[2], gx2_2);
      gx3_2 = fmaf(W, D0_4_3[2], gx3_2);
      gr2 = fmaf(fmaf(X3_2, D0_4_3[2], fmaf(X2_2, D0_4_2[2], X1_2 * D0_4_1[2])), D, gr2);
      gt2 = fmaf(fmaf(X3_2, D1_4_3[2], fmaf(X2_2, D1_4_2[2], X1_2 * D1_4_1[2])), W, gt2);
      gp2 = fmaf(fmaf(X3_2, D2_4_3[2], fmaf(X2_2, D2_4_2[2], X1_2 * D2_4_1[2])), W, gp2);
    }
    {
      const floatx4 q = q2_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx1_3 = fmaf(W, D0_4_1[3], gx1_3);
      gx2_3 = fmaf(W, D0_4_2[3], gx2_3);
      gx3_3 = fmaf(W, D0_4_3[3], gx3_3);
      gr3 = fmaf(fmaf(X3_3, D0_4_3[3], fmaf(X2_3, D0_4_2[3], X1_3 * D0_4_1[3])), D, gr3);
      gt3 = fmaf(fmaf(X3_3, D1_4_3[3], fmaf(X2_3, D1_4_2[3], X1_3 * D1_4_1[3])), W, gt3);
      gp3 = fmaf(fmaf(X3_3, D2_4_3[3], fmaf(X2_3, D2_4_2[3], X1_3 * D2_4_1[3])), W, gp3);
    }
    asm volatile("" : "+v"(gx1_0), "+v"(gx1_1), "+v"(gx1_2), "+v"(gx1_3), "+v"(gx2_0), "+v"(gx2_1), "+v"(gx2_2), "+v"(gx2_3), "+v"(gx3_0), "+v"(gx3_1), "+v"(gx3_2), "+v"(gx3_3));
    floatx4 q4_0 = *(const floatx4*)(tcb + o0 + 2304);
    floatx4 q4_1 = *(const floatx4*)(tcb + o1 + 2304);
    floatx4 q4_2 = *(const floatx4*)(tcb + o2 + 2304);
    floatx4 q4_3 = *(const floatx4*)(tcb + o3 + 2304);
    const floatx4 D0_5_0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_0, __builtin_bit_cast(half8v, B5_0), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_5_0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_1, __builtin_bit_cast(half8v, B5_0), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_5_0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_2, __builtin_bit_cast(half8v, B5_0), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    {
      const floatx4 q = q3_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx0_0 = fmaf(W, D0_5_0[0], gx0_0);
      gr0 = fmaf(X0_0 * D0_5_0[0], D, gr0);
      gt0 = fmaf(X0_0 * D1_5_0[0], W, gt0);
      gp0 = fmaf(X0_0 * D2_5_0[0], W, gp0);
    }
    {
      const floatx4 q = q3_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx0_1 = fmaf(W, D0_5_0[1], gx0_1);
      gr1 = fmaf(X0_1 * D0_5_0[1], D, gr1);
      gt1 = fmaf(X0_1 * D1_5_0[1], W, gt1);
      gp1 = fmaf(X0_1 * D2_5_0[1], W, gp1);
    }
    {
      const floatx4 q = q3_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx0_2 = fmaf(W, D0_5_0[2], gx0_2);
      gr2 = fmaf(X0_2 * D0_5_0[2], D, gr2);
      gt2 = fmaf(X0_2 * D1_5_0[2], W, gt2);
      gp2 = fmaf(X0_2 * D2_5_0[2], W, gp2);
    }
    {
      const floatx4 q = q3_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx0_3 = fmaf(W, D0_5_0[3], gx0_3);
      gr3 = fmaf(X0_3 * D0_5_0[3], D, gr3);
      gt3 = fmaf(X0_3 * D1_5_0[3], W, gt3);
      gp3 = fmaf(X0_3 * D2_5_0[3], W, gp3);
    }
    asm volatile("" : "+v"(gx0_0), "+v"(gx0_1), "+v"(gx0_2), "+v"(gx0_3));
    floatx4 q5_0 = *(const floatx4*)(tcb + o0 + 256);
    floatx4 q5_1 = *(const floatx4*)(tcb + o1 + 256);
    floatx4 q5_2 = *(const floatx4*)(tcb + o2 + 256);
    floatx4 q5_3 = *(const floatx4*)(tcb + o3 + 256);
    const floatx4 D0_9_1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_0, __builtin_bit_cast(half8v, B9_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_9_1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_1, __builtin_bit_cast(half8v, B9_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_9_1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_2, __builtin_bit_cast(half8v, B9_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_9_2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_0, __builtin_bit_cast(half8v, B9_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_9_2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_1, __builtin_bit_cast(half8v, B9_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_9_2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_2, __builtin_bit_cast(half8v, B9_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_9_3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_0, __builtin_bit_cast(half8v, B9_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_9_3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_1, __builtin_bit_cast(half8v, B9_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_9_3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(A2_2, __builtin_bit_cast(half8v, B9_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    {
      const floatx4 q = q4_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx1_0 = fmaf(W, D0_9_1[0], gx1_0);
      gx2_0 = fmaf(W, D0_9_2[0], gx2_0);
      gx3_0 = fmaf(W, D0_9_3[0], gx3_0);
      gr0 = fmaf(fmaf(X3_0, D0_9_3[0], fmaf(X2_0, D0_9_2[0], X1_0 * D0_9_1[0])), D, gr0);
      gt0 = fmaf(fmaf(X3_0, D1_9_3[0], fmaf(X2_0, D1_9_2[0], X1_0 * D1_9_1[0])), W, gt0);
      gp0 = fmaf(fmaf(X3_0, D2_9_3[0], fmaf(X2_0, D2_9_2[0], X1_0 * D2_9_1[0])), W, gp0);
    }
    {
      const floatx4 q = q4_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx1_1 = fmaf(W, D0_9_1[1], gx1_1);
      gx2_1 = fmaf(W, D0_9_2[1], gx2_1);
      gx3_1 = fmaf(W, D0_9_3[1], gx3_1);
      gr1 = fmaf(fmaf(X3_1, D0_9_3[1], fmaf(X2_1, D0_9_2[1], X1_1 * D0_9_1[1])), D, gr1);
      gt1 = fmaf(fmaf(X3_1, D1_9_3[1], fmaf(X2_1, D1_9_2[1], X1_1 * D1_9_1[1])), W, gt1);
      gp1 = fmaf(fmaf(X3_1, D2_9_3[1], fmaf(X2_1, D2_9_2[1], X1_1 * D2_9_1[1])), W, gp1);
    }
    {
      const floatx4 q = q4_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx1_2 = fmaf(W, D0_9_1[2], gx1_2);
      gx2_2 = fmaf(W, D0_9_2[2], gx2_2);
      gx3_2 = fmaf(W, D0_9_3[2], gx3_2);
      gr2 = fmaf(fmaf(X3_2, D0_9_3[2], fmaf(X2_2, D0_9_2[2], X1_2 * D0_9_1[2])), D, gr2);
      gt2 = fmaf(fmaf(X3_2, D1_9_3[2], fmaf(X2_2, D1_9_2[2], X1_2 * D1_9_1[2])), W, gt2);
      gp2 = fmaf(fmaf(X3_2, D2_9_3[2], fmaf(X2_2, D2_9_2[2], X1_2 * D2_9_1[2])), W, gp2);
    }
    {
      const floatx4 q = q4_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx1_3 = fmaf(W, D0_9_1[3], gx1_3);
      gx2_3 = fmaf(W, D0_9_2[3], gx2_3);
      gx3_3 = fmaf(W, D0_9_3[3], gx3_3);
      gr3 = fmaf(fmaf(X3_3, D0_9_3[3], fmaf(X2_3, D0_9_2[3], X1_3 * D0_9_1[3])), D, gr3);
      gt3 = fmaf(fmaf(X3_3, D1_9_3[3], fmaf(X2_3, D1_9_2[3], X1_3 * D1_9_1[3])), W, gt3);
      gp3 = fmaf(fmaf(X3_3, D2_9_3[3], fmaf(X2_3, D2_9_2[3], X1_3 * D2_9_1[3])), W, gp3);
    }
    asm volatile("" : "+v"(gx1_0), "+v"(gx1_1), "+v"(gx1_2), "+v"(gx1_3), "+v"(gx2_0), "+v"(gx2_1), "+v"(gx2_2), "+v"(gx2_3), "+v"(gx3_0), "+v"(gx3_1), "+v"(gx3_2), "+v"(gx3_3));
    floatx4 q6_0 = *(const floatx4*)(tcb + o0 + 512);
    floatx4 q6_1 = *(const floatx4*)(tcb + o1 + 512);
    floatx4 q6_2 = *(const floatx4*)(tcb + o2 + 512);
    floatx4 q6_3 = *(const floatx4*)(tcb + o3 + 512);
    const half4v A1_0 = __builtin_bit_cast(half4v, *(const uint2v*)&ya[((2) * 16 + cl) * 2 + 1 - (eg >> 1)]);
    const half4v A1_1 = __builtin_bit_cast(half4v, *(const uint2v*)&ya[((5) * 16 + cl) * 2 + 1 - (eg >> 1)]);
    const half4v A1_2 = __builtin_bit_cast(half4v, *(const uint2v*)&ya[((8) * 16 + cl) * 2 + 1 - (eg >> 1)]);
    const floatx4 D0_1_1 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_0, __builtin_bit_cast(half4v, B1_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_1_1 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_1, __builtin_bit_cast(half4v, B1_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_1_1 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_2, __builtin_bit_cast(half4v, B1_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_1_2 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_0, __builtin_bit_cast(half4v, B1_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_1_2 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_1, __builtin_bit_cast(half4v, B1_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_1_2 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_2, __builtin_bit_cast(half4v, B1_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_1_3 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_0, __builtin_bit_cast(half4v, B1_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_1_3 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_1, __builtin_bit_cast(half4v, B1_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_1_3 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_2, __builtin_bit_cast(half4v, B1_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    {
      const floatx4 q = q5_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx1_0 = fmaf(W, D0_1_1[0], gx1_0);
      gx2_0 = fmaf(W, D0_1_2[0], gx2_0);
      gx3_0 = fmaf(W, D0_1_3[0], gx3_0);
      gr0 = fmaf(fmaf(X3_0, D0_1_3[0], fmaf(X2_0, D0_1_2[0], X1_0 * D0_1_1[0])), D, gr0);
      gt0 = fmaf(fmaf(X3_0, D1_1_3[0], fmaf(X2_0, D1_1_2[0], X1_0 * D1_1_1[0])), W, gt0);
      gp0 = fmaf(fmaf(X3_0, D2_1_3[0], fmaf(X2_0, D2_1_2[0], X1_0 * D2_1_1[0])), W, gp0);
    }
    {
      const floatx4 q = q5_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx1_1 = fmaf(W, D0_1_1[1], gx1_1);
      gx2_1 = fmaf(W, D0_1_2[1], gx2_1);
      gx3_1 = fmaf(W, D0_1_3[1], gx3_1);
      gr1 = fmaf(fmaf(X3_1, D0_1_3[1], fmaf(X2_1, D0_1_2[1], X1_1 * D0_1_1[1])), D, gr1);
      gt1 = fmaf(fmaf(X3_1, D1_1_3[1], fmaf(X2_1, D1_1_2[1], X1_1 * D1_1_1[1])), W, gt1);
      gp1 = fmaf(fmaf(X3_1, D2_1_3[1], fmaf(X2_1, D2_1_2[1], X1_1 * D2_1_1[1])), W, gp1);
    }
    {
      const floatx4 q = q5_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx1_2 = fmaf(W, D0_1_1[2], gx1_2);
      gx2_2 = fmaf(W, D0_1_2[2], gx2_2);
      gx3_2 = fmaf(W, D0_1_3[2], gx3_2);
      gr2 = fmaf(fmaf(X3_2, D0_1_3[2], fmaf(X2_2, D0_1_2[2], X1_2 * D0_1_1[2])), D, gr2);
      gt2 = fmaf(fmaf(X3_2, D1_1_3[2], fmaf(X2_2, D1_1_2[2], X1_2 * D1_1_1[2])), W, gt2);
      gp2 = fmaf(fmaf(X3_2, D2_1_3[2], fmaf(X2_2, D2_1_2[2], X1_2 * D2_1_1[2])), W, gp2);
    }
    {
      const floatx4 q = q5_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx1_3 = fmaf(W, D0_1_1[3], gx1_3);
      gx2_3 = fmaf(W, D0_1_2[3], gx2_3);
      gx3_3 = fmaf(W, D0_1_3[3], gx3_3);
      gr3 = fmaf(fmaf(X3_3, D0_1_3[3], fmaf(X2_3, D0_1_2[3], X1_3 * D0_1_1[3])), D, gr3);
      gt3 = fmaf(fmaf(X3_3, D1_1_3[3], fmaf(X2_3, D1_1_2[3], X1_3 * D1_1_1[3])), W, gt3);
      gp3 = fmaf(fmaf(X3_3, D2_1_3[3], fmaf(X2_3, D2_1_2[3], X1_3 * D2_1_1[3])), W, gp3);
    }
    asm volatile("" : "+v"(gx1_0), "+v"(gx1_1), "+v"(gx1_2), "+v"(gx1_3), "+v"(gx2_0), "+v"(gx2_1), "+v"(gx2_2), "+v"(gx2_3), "+v"(gx3_0), "+v"(gx3_1), "+v"(gx3_2), "+v"(gx3_3));
    floatx4 q7_0 = *(const floatx4*)(tcb + o0 + 1536);
    floatx4 q7_1 = *(const floatx4*)(tcb + o1 + 1536);
    floatx4 q7_2 = *(const floatx4*)(tcb + o2 + 1536);
    floatx4 q7_3 = *(const floatx4*)(tcb + o3 + 1536);
    const floatx4 D0_2_0 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_0, __builtin_bit_cast(half4v, B2_0), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_2_0 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_1, __builtin_bit_cast(half4v, B2_0), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_2_0 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_2, __builtin_bit_cast(half4v, B2_0), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    {
      const floatx4 q = q6_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx0_0 = fmaf(W, D0_2_0[0], gx0_0);
      gr0 = fmaf(X0_0 * D0_2_0[0], D, gr0);
      gt0 = fmaf(X0_0 * D1_2_0[0], W, gt0);
      gp0 = fmaf(X0_0 * D2_2_0[0], W, gp0);
    }
    {
      const floatx4 q = q6_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx0_1 = fmaf(W, D0_2_0[1], gx0_1);
      gr1 = fmaf(X0_1 * D0_2_0[1], D, gr1);
      gt1 = fmaf(X0_1 * D1_2_0[1], W, gt1);
      gp1 = fmaf(X0_1 * D2_2_0[1], W, gp1);
    }
    {
      const floatx4 q = q6_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx0_2 = fmaf(W, D0_2_0[2], gx0_2);
      gr2 = fmaf(X0_2 * D0_2_0[2], D, gr2);
      gt2 = fmaf(X0_2 * D1_2_0[2], W, gt2);
      gp2 = fmaf(X0_2 * D2_2_0[2], W, gp2);
    }
    {
      const floatx4 q = q6_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx0_3 = fmaf(W, D0_2_0[3], gx0_3);
      gr3 = fmaf(X0_3 * D0_2_0[3], D, gr3);
      gt3 = fmaf(X0_3 * D1_2_0[3], W, gt3);
      gp3 = fmaf(X0_3 * D2_2_0[3], W, gp3);
    }
    asm volatile("" : "+v"(gx0_0), "+v"(gx0_1), "+v"(gx0_2), "+v"(gx0_3));
    floatx4 q8_0 = *(const floatx4*)(tcb + o0 + 0);
    floatx4 q8_1 = *(const floatx4*)(tcb + o1 + 0);
    floatx4 q8_2 = *(const floatx4*)(tcb + o2 + 0);
    floatx4 q8_3 = *(const floatx4*)(tcb + o3 + 0);
    const floatx4 D0_6_1 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_0, __builtin_bit_cast(half4v, B6_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_6_1 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_1, __builtin_bit_cast(half4v, B6_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_6_1 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_2, __builtin_bit_cast(half4v, B6_1), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_6_2 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_0, __builtin_bit_cast(half4v, B6_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_6_2 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_1, __builtin_bit_cast(half4v, B6_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_6_2 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_2, __builtin_bit_cast(half4v, B6_2), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D0_6_3 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_0, __builtin_bit_cast(half4v, B6_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D1_6_3 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_1, __builtin_bit_cast(half4v, B6_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const floatx4 D2_6_3 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1_2, __builtin_bit_cast(half4v, B6_3), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    {
      const floatx4 q = q7_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx1_0 = fmaf(W, D0_6_1[0], gx1_0);
      gx2_0 = fmaf(W, D0_6_2[0], gx2_0);
      gx3_0 = fmaf(W, D0_6_3[0], gx3_0);
      gr0 = fmaf(fmaf(X3_0, D0_6_3[0], fmaf(X2_0, D0_6_2[0], X1_0 * D0_6_1[0])), D, gr0);
      gt0 = fmaf(fmaf(X3_0, D1_6_3[0], fmaf(X2_0, D1_6_2[0], X1_0 * D1_6_1[0])), W, gt0);
      gp0 = fmaf(fmaf(X3_0, D2_6_3[0], fmaf(X2_0, D2_6_2[0], X1_0 * D2_6_1[0])), W, gp0);
    }
    {
      const floatx4 q = q7_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx1_1 = fmaf(W, D0_6_1[1], gx1_1);
      gx2_1 = fmaf(W, D0_6_2[1], gx2_1);
      gx3_1 = fmaf(W, D0_6_3[1], gx3_1);
      gr1 = fmaf(fmaf(X3_1, D0_6_3[1], fmaf(X2_1, D0_6_2[1], X1_1 * D0_6_1[1])), D, gr1);
      gt1 = fmaf(fmaf(X3_1, D1_6_3[1], fmaf(X2_1, D1_6_2[1], X1_1 * D1_6_1[1])), W, gt1);
      gp1 = fmaf(fmaf(X3_1, D2_6_3[1], fmaf(X2_1, D2_6_2[1], X1_1 * D2_6_1[1])), W, gp1);
    }
    {
      const floatx4 q = q7_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx1_2 = fmaf(W, D0_6_1[2], gx1_2);
      gx2_2 = fmaf(W, D0_6_2[2], gx2_2);
      gx3_2 = fmaf(W, D0_6_3[2], gx3_2);
      gr2 = fmaf(fmaf(X3_2, D0_6_3[2], fmaf(X2_2, D0_6_2[2], X1_2 * D0_6_1[2])), D, gr2);
      gt2 = fmaf(fmaf(X3_2, D1_6_3[2], fmaf(X2_2, D1_6_2[2], X1_2 * D1_6_1[2])), W, gt2);
      gp2 = fmaf(fmaf(X3_2, D2_6_3[2], fmaf(X2_2, D2_6_2[2], X1_2 * D2_6_1[2])), W, gp2);
    }
    {
      const floatx4 q = q7_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx1_3 = fmaf(W, D0_6_1[3], gx1_3);
      gx2_3 = fmaf(W, D0_6_2[3], gx2_3);
      gx3_3 = fmaf(W, D0_6_3[3], gx3_3);
      gr3 = fmaf(fmaf(X3_3, D0_6_3[3], fmaf(X2_3, D0_6_2[3], X1_3 * D0_6_1[3])), D, gr3);
      gt3 = fmaf(fmaf(X3_3, D1_6_3[3], fmaf(X2_3, D1_6_2[3], X1_3 * D1_6_1[3])), W, gt3);
      gp3 = fmaf(fmaf(X3_3, D2_6_3[3], fmaf(X2_3, D2_6_2[3], X1_3 * D2_6_1[3])), W, gp3);
    }
    asm volatile("" : "+v"(gx1_0), "+v"(gx1_1), "+v"(gx1_2), "+v"(gx1_3), "+v"(gx2_0), "+v"(gx2_1), "+v"(gx2_2), "+v"(gx2_3), "+v"(gx3_0), "+v"(gx3_1), "+v"(gx3_2), "+v"(gx3_3));
    floatx4 q9_0 = *(const floatx4*)(tcb + o0 + 768);
    floatx4 q9_1 = *(const floatx4*)(tcb + o1 + 768);
    floatx4 q9_2 = *(const floatx4*)(tcb + o2 + 768);
    floatx4 q9_3 = *(const floatx4*)(tcb + o3 + 768);
    {
      const floatx4 q = q8_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx0_0 = fmaf(W, U0_0, gx0_0);
      gr0 = fmaf(X0_0 * U0_0, D, gr0);
    }
    {
      const floatx4 q = q8_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx0_1 = fmaf(W, U0_0, gx0_1);
      gr1 = fmaf(X0_1 * U0_0, D, gr1);
    }
    {
      const floatx4 q = q8_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx0_2 = fmaf(W, U0_0, gx0_2);
      gr2 = fmaf(X0_2 * U0_0, D, gr2);
    }
    {
      const floatx4 q = q8_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx0_3 = fmaf(W, U0_0, gx0_3);
      gr3 = fmaf(X0_3 * U0_0, D, gr3);
    }
    asm volatile("" : "+v"(gx0_0), "+v"(gx0_1), "+v"(gx0_2), "+v"(gx0_3));
    on0 = (unsigned)__float_as_int(pkn0.y) * 2560u + cl * 16u;
    on1 = (unsigned)__float_as_int(pkn1.y) * 2560u + cl * 16u;
    on2 = (unsigned)__float_as_int(pkn2.y) * 2560u + cl * 16u;
    on3 = (unsigned)__float_as_int(pkn3.y) * 2560u + cl * 16u;
    q0_0 = *(const floatx4*)(tcb + on0 + 1792);
    q0_1 = *(const floatx4*)(tcb + on1 + 1792);
    q0_2 = *(const floatx4*)(tcb + on2 + 1792);
    q0_3 = *(const floatx4*)(tcb + on3 + 1792);
    {
      const floatx4 q = q9_0;
      const float a = fmaf(q.w, t0, q.z);
      const float b = fmaf(a, t0, q.y);
      const float W = fmaf(b, t0, q.x);
      const float D = fmaf(fmaf(q.w, t0, a), t0, b);
      gx1_0 = fmaf(W, U3_1, gx1_0);
      gx2_0 = fmaf(W, U3_2, gx2_0);
      gx3_0 = fmaf(W, U3_3, gx3_0);
      gr0 = fmaf(fmaf(X3_0, U3_3, fmaf(X2_0, U3_2, X1_0 * U3_1)), D, gr0);
    }
    {
      const floatx4 q = q9_1;
      const float a = fmaf(q.w, t1, q.z);
      const float b = fmaf(a, t1, q.y);
      const float W = fmaf(b, t1, q.x);
      const float D = fmaf(fmaf(q.w, t1, a), t1, b);
      gx1_1 = fmaf(W, U3_1, gx1_1);
      gx2_1 = fmaf(W, U3_2, gx2_1);
      gx3_1 = fmaf(W, U3_3, gx3_1);
      gr1 = fmaf(fmaf(X3_1, U3_3, fmaf(X2_1, U3_2, X1_1 * U3_1)), D, gr1);
    }
    {
      const floatx4 q = q9_2;
      const float a = fmaf(q.w, t2, q.z);
      const float b = fmaf(a, t2, q.y);
      const float W = fmaf(b, t2, q.x);
      const float D = fmaf(fmaf(q.w, t2, a), t2, b);
      gx1_2 = fmaf(W, U3_1, gx1_2);
      gx2_2 = fmaf(W, U3_2, gx2_2);
      gx3_2 = fmaf(W, U3_3, gx3_2);
      gr2 = fmaf(fmaf(X3_2, U3_3, fmaf(X2_2, U3_2, X1_2 * U3_1)), D, gr2);
    }
    {
      const floatx4 q = q9_3;
      const float a = fmaf(q.w, t3, q.z);
      const float b = fmaf(a, t3, q.y);
      const float W = fmaf(b, t3, q.x);
      const float D = fmaf(fmaf(q.w, t3, a), t3, b);
      gx1_3 = fmaf(W, U3_1, gx1_3);
      gx2_3 = fmaf(W, U3_2, gx2_3);
      gx3_3 = fmaf(W, U3_3, gx3_3);
      gr3 = fmaf(fmaf(X3_3, U3_3, fmaf(X2_3, U3_2, X1_3 * U3_1)), D, gr3);
    }
    asm volatile("" : "+v"(gx1_0), "+v"(gx1_1), "+v"(gx1_2), "+v"(gx1_3), "+v"(gx2_0), "+v"(gx2_1), "+v"(gx2_2), "+v"(gx2_3), "+v"(gx3_0), "+v"(gx3_1), "+v"(gx3_2), "+v"(gx3_3));
    q1_0 = *(const floatx4*)(tcb + on0 + 2048);
    q1_1 = *(const floatx4*)(tcb + on1 + 2048);
    q1_2 = *(const floatx4*)(tcb + on2 + 2048);
    q1_3 = *(const floatx4*)(tcb + on3 + 2048);
    const int n_own = min(e1 - (eb + 4 * eg), 4);   // this lane's edges inside the receiver's range (may be <= 0)
    // sums over the 16 channels of the row: transpose-reduction, lane cl = 3 v + j ends with value j of edge v
    gr0 *= gun;
    gt0 *= gun;
    gp0 *= gun;
    gr1 *= gun;
    gt1 *= gun;
    gp1 *= gun;
    gr2 *= gun;
    gt2 *= gun;
    gp2 *= gun;
    gr3 *= gun;
    gt3 *= gun;
    gp3 *= gun;
    const bool b3 = cl & 8, b2 = cl & 4, b1 = cl & 2, b0 = cl & 1;
    const float s8_0 = (b3 ? gp2 : gr0) + mm_dpp<0x140>(b3 ? gr0 : gp2);
    const float s8_1 = (b3 ? gr3 : gt0) + mm_dpp<0x140>(b3 ? gt0 : gr3);
    const float s8_2 = (b3 ? gt3 : gp0) + mm_dpp<0x140>(b3 ? gp0 : gt3);
    const float s8_3 = (b3 ? gp3 : gr1) + mm_dpp<0x140>(b3 ? gr1 : gp3);
    const float s8_4 = (b3 ? 0.f : gt1) + mm_dpp<0x140>(b3 ? gt1 : 0.f);
    const float s8_5 = (b3 ? 0.f : gp1) + mm_dpp<0x140>(b3 ? gp1 : 0.f);
    const float s8_6 = (b3 ? 0.f : gr2) + mm_dpp<0x140>(b3 ? gr2 : 0.f);
    const float s8_7 = (b3 ? 0.f : gt2) + mm_dpp<0x140>(b3 ? gt2 : 0.f);
    const float s4_0 = (b2 ? s8_4 : s8_0) + mm_dpp<0x141>(b2 ? s8_0 : s8_4);
    const float s4_1 = (b2 ? s8_5 : s8_1) + mm_dpp<0x141>(b2 ? s8_1 : s8_5);
    const float s4_2 = (b2 ? s8_6 : s8_2) + mm_dpp<0x141>(b2 ? s8_2 : s8_6);
    const float s4_3 = (b2 ? s8_7 : s8_3) + mm_dpp<0x141>(b2 ? s8_3 : s8_7);
    const float s2_0 = (b1 ? s4_2 : s4_0) + mm_dpp<0x1B>(b1 ? s4_0 : s4_2);
    const float s2_1 = (b1 ? s4_3 : s4_1) + mm_dpp<0x1B>(b1 ? s4_1 : s4_3);
    float sum = (b0 ? s2_1 : s2_0) + mm_dpp<0xB1>(b0 ? s2_0 : s2_1);
    const float tc = cl < 3 ? t0 : cl < 6 ? t1 : cl < 9 ? t2 : t3;
    if (cl == 0 || cl == 3 || cl == 6 || cl == 9) sum *= mm_spline_dxdr(tc, inv_h);   // zero below the table start
    if (cl < 12 && cl < 3 * n_own)
      part[(size_t)cb * part_stride + (size_t)(eb + 4 * eg) * 3 + cl] = sum;
    if (0 < n_own) {
      float* __restrict__ gxp = gX + (size_t)(eb + 4 * eg + 0) * 512 + cb * 64 + cl;
      gxp[0] = gx0_0 * gun;
      gxp[16] = gx1_0 * gun;
      gxp[32] = gx2_0 * gun;
      gxp[48] = gx3_0 * gun;
    }
    if (1 < n_own) {
      float* __restrict__ gxp = gX + (size_t)(eb + 4 * eg + 1) * 512 + cb * 64 + cl;
      gxp[0] = gx0_1 * gun;
      gxp[16] = gx1_1 * gun;
      gxp[32] = gx2_1 * gun;
      gxp[48] = gx3_1 * gun;
    }
    if (2 < n_own) {
      float* __restrict__ gxp = gX + (size_t)(eb + 4 * eg + 2) * 512 + cb * 64 + cl;
      gxp[0] = gx0_2 * gun;
      gxp[16] = gx1_2 * gun;
      gxp[32] = gx2_2 * gun;
      gxp[48] = gx3_2 * gun;
    }
    if (3 < n_own) {
      float* __restrict__ gxp = gX + (size_t)(eb + 4 * eg + 3) * 512 + cb * 64 + cl;
      gxp[0] = gx0_3 * gun;
      gxp[16] = gx1_3 * gun;
      gxp[32] = gx2_3 * gun;
      gxp[48] = gx3_3 * gun;
    }
  }
  }   // edges
}

extern "C" int mm_conv2_bwd_vec_det(const int* rowptr, int nC, const float* e_pk, const float* e_u,
    const float* X, int x_stride, const float* tab, int n_tab, int M, float inv_h, const float* gA,
    float* part, long part_stride, float* gX, hipStream_t stream) {
  MM_CHECK_ARG(nC >= 0 && M >= 2 && n_tab >= 1, "bad sizes");
  MM_CHECK_ARG(gX != nullptr, "the sender-feature gradient buffer is required");
  MM_CHECK_ARG((long)n_tab * (M - 1) * 2560 < (1L << 32), "a channel block's tables exceed 4 GiB");
  if (nC == 0) return MM_OK;
  hipLaunchKernelGGL(mm_conv2_bwd_vec_det_kernel, dim3(8 * ((nC + 3) / 4)), dim3(256), 0, stream, rowptr, nC,
                     (const floatx4*)e_pk, (const floatx4*)e_u, X, x_stride, (const floatx4*)tab,
                     n_tab * (M - 1) * 160, inv_h, gA, part, part_stride, gX);
  return mm::launch_status("mm_conv2_bwd_vec_det");
}

