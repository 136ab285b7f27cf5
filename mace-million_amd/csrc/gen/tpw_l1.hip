// generated by mace_onegpu/codegen.py -- explicit-weight channelwise TP 'l1'
// nX=1, nW=4, nO=16, terms=16
//
// out[i, o, c] = sum_{p in [rowptr[i], rowptr[i+1])} sum_terms coef * W[e, w, c] * X[send[e], k, c] * Y[e, m],
// e = eid[p] (or p when eid is null): receiver-CSR over a permutation, so edges need not be stored sorted.
// Forward: one wave per receiver and channel half, 2 channel(s) per lane (c = 64 h + lane + 64 j),
// 1 wave(s) per receiver, 2 edge(s) loaded together.  Backward: 2 channel(s) per lane, 1 wave(s)
// per receiver, 2 edge(s) loaded together; dL/dY partials: 1 per edge (one per channel half).
#include "../common.h"

extern "C" __global__ void __launch_bounds__(256)
mm_tpw_l1_fwd_kernel(const int* __restrict__ rowptr, int nR, const int* __restrict__ eid,
    const int* __restrict__ send, const float* __restrict__ Y, long y_stride, const float* __restrict__ W,
    long w_stride, const float* __restrict__ X, long x_stride, float* __restrict__ out, long out_stride) {
  const int gw = blockIdx.x * 4 + (threadIdx.x >> 6);   // global wave: receiver i, sub-wave h
  const int i = gw, h = 0;
  if (i >= nR) return;
  const int lane = threadIdx.x & 63;
  const int c = h * 64 + lane;
  const int p0 = rowptr[i], p1 = rowptr[i + 1];
  float acc0_0 = 0.f;
  float acc0_1 = 0.f;
  float acc1_0 = 0.f;
  float acc1_1 = 0.f;
  float acc2_0 = 0.f;
  float acc2_1 = 0.f;
  float acc3_0 = 0.f;
  float acc3_1 = 0.f;
  float acc4_0 = 0.f;
  float acc4_1 = 0.f;
  float acc5_0 = 0.f;
  float acc5_1 = 0.f;
  float acc6_0 = 0.f;
  float acc6_1 = 0.f;
  float acc7_0 = 0.f;
  float acc7_1 = 0.f;
  float acc8_0 = 0.f;
  float acc8_1 = 0.f;
  float acc9_0 = 0.f;
  float acc9_1 = 0.f;
  float acc10_0 = 0.f;
  float acc10_1 = 0.f;
  float acc11_0 = 0.f;
  float acc11_1 = 0.f;
  float acc12_0 = 0.f;
  float acc12_1 = 0.f;
  float acc13_0 = 0.f;
  float acc13_1 = 0.f;
  float acc14_0 = 0.f;
  float acc14_1 = 0.f;
  float acc15_0 = 0.f;
  float acc15_1 = 0.f;
  for (int p = p0; p < p1; p += 2) {
    const bool two = p + 1 < p1;   // wave-uniform
    const int ea = __builtin_amdgcn_readfirstlane(eid ? eid[p] : p);
    const int sa = __builtin_amdgcn_readfirstlane(send[ea]);
    const float* __restrict__ wpa = W + (size_t)ea * w_stride + c;
    const float W0_0_a = wpa[0];
    const float W0_1_a = wpa[64];
    const float W1_0_a = wpa[128];
    const float W1_1_a = wpa[192];
    const float W2_0_a = wpa[256];
    const float W2_1_a = wpa[320];
    const float W3_0_a = wpa[384];
    const float W3_1_a = wpa[448];
    const float* __restrict__ xpa = X + (size_t)sa * x_stride + c;
    const float X0_0_a = xpa[0];
    const float X0_1_a = xpa[64];
    const float* __restrict__ ypa = Y + (size_t)ea * y_stride;
    const float Y0_a = ypa[0];
    const float Y1_a = ypa[1];
    const float Y2_a = ypa[2];
    const float Y3_a = ypa[3];
    const float Y4_a = ypa[4];
    const float Y5_a = ypa[5];
    const float Y6_a = ypa[6];
    const float Y7_a = ypa[7];
    const float Y8_a = ypa[8];
    const float Y9_a = ypa[9];
    const float Y10_a = ypa[10];
    const float Y11_a = ypa[11];
    const float Y12_a = ypa[12];
    const float Y13_a = ypa[13];
    const float Y14_a = ypa[14];
    const float Y15_a = ypa[15];
    const int eb = two ? __builtin_amdgcn_readfirstlane(eid ? eid[p + 1] : p + 1) : ea;
    const int sb = __builtin_amdgcn_readfirstlane(send[eb]);
    const float* __restrict__ wpb = W + (size_t)eb * w_stride + c;
    const float W0_0_b = wpb[0];
    const float W0_1_b = wpb[64];
    const float W1_0_b = wpb[128];
    const float W1_1_b = wpb[192];
    const float W2_0_b = wpb[256];
    const float W2_1_b = wpb[320];
    const float W3_0_b = wpb[384];
    const float W3_1_b = wpb[448];
    const float* __restrict__ xpb = X + (size_t)sb * x_stride + c;
    const float X0_0_b = xpb[0];
    const float X0_1_b = xpb[64];
    const float* __restrict__ ypb = Y + (size_t)eb * y_stride;
    const float Y0_b = ypb[0];
    const float Y1_b = ypb[1];
    const float Y2_b = ypb[2];
    const float Y3_b = ypb[3];
    const float Y4_b = ypb[4];
    const float Y5_b = ypb[5];
    const float Y6_b = ypb[6];
    const float Y7_b = ypb[7];
    const float Y8_b = ypb[8];
    const float Y9_b = ypb[9];
    const float Y10_b = ypb[10];
    const float Y11_b = ypb[11];
    const float Y12_b = ypb[12];
    const float Y13_b = ypb[13];
    const float Y14_b = ypb[14];
    const float Y15_b = ypb[15];
    { const float q = W0_0_a * X0_0_a;
      acc0_0 = fmaf(q, Y0_a, acc0_0);
    }
    { const float q = W0_1_a * X0_1_a;
      acc0_1 = fmaf(q, Y0_a, acc0_1);
    }
    { const float q = W1_0_a * X0_0_a;
      acc1_0 = fmaf(q, Y1_a, acc1_0);
      acc2_0 = fmaf(q, Y2_a, acc2_0);
      acc3_0 = fmaf(q, Y3_a, acc3_0);
    }
    { const float q = W1_1_a * X0_1_a;
      acc1_1 = fmaf(q, Y1_a, acc1_1);
      acc2_1 = fmaf(q, Y2_a, acc2_1);
      acc3_1 = fmaf(q, Y3_a, acc3_1);
    }
    { const float q = W2_0_a * X0_0_a;
      acc4_0 = fmaf(q, Y4_a, acc4_0);
      acc5_0 = fmaf(q, Y5_a, acc5_0);
      acc6_0 = fmaf(q, Y6_a, acc6_0);
      acc7_0 = fmaf(q, Y7_a, acc7_0);
      acc8_0 = fmaf(q, Y8_a, acc8_0);
    }
    { const float q = W2_1_a * X0_1_a;
      acc4_1 = fmaf(q, Y4_a, acc4_1);
      acc5_1 = fmaf(q, Y5_a, acc5_1);
      acc6_1 = fmaf(q, Y6_a, acc6_1);
      acc7_1 = fmaf(q, Y7_a, acc7_1);
      acc8_1 = fmaf(q, Y8_a, acc8_1);
    }
    { const float q = W3_0_a * X0_0_a;
      acc9_0 = fmaf(q, Y9_a, acc9_0);
      acc10_0 = fmaf(q, Y10_a, acc10_0);
      acc11_0 = fmaf(q, Y11_a, acc11_0);
      acc12_0 = fmaf(q, Y12_a, acc12_0);
      acc13_0 = fmaf(q, Y13_a, acc13_0);
      acc14_0 = fmaf(q, Y14_a, acc14_0);
      acc15_0 = fmaf(q, Y15_a, acc15_0);
    }
    { const float q = W3_1_a * X0_1_a;
      acc9_1 = fmaf(q, Y9_a, acc9_1);
      acc10_1 = fmaf(q, Y10_a, acc10_1);
      acc11_1 = fmaf(q, Y11_a, acc11_1);
      acc12_1 = fmaf(q, Y12_a, acc12_1);
      acc13_1 = fmaf(q, Y13_a, acc13_1);
      acc14_1 = fmaf(q, Y14_a, acc14_1);
      acc15_1 = fmaf(q, Y15_a, acc15_1);
    }
    if (two) {
    { const float q = W0_0_b * X0_0_b;
      acc0_0 = fmaf(q, Y0_b, acc0_0);
    }
    { const float q = W0_1_b * X0_1_b;
      acc0_1 = fmaf(q, Y0_b, acc0_1);
    }
    { const float q = W1_0_b * X0_0_b;
      acc1_0 = fmaf(q, Y1_b, acc1_0);
      acc2_0 = fmaf(q, Y2_b, acc2_0);
      acc3_0 = fmaf(q, Y3_b, acc3_0);
    }
    { const float q = W1_1_b * X0_1_b;
      acc1_1 = fmaf(q, Y1_b, acc1_1);
      acc2_1 = fmaf(q, Y2_b, acc2_1);
      acc3_1 = fmaf(q, Y3_b, acc3_1);
    }
    { const float q = W2_0_b * X0_0_b;
      acc4_0 = fmaf(q, Y4_b, acc4_0);
      acc5_0 = fmaf(q, Y5_b, acc5_0);
      acc6_0 = fmaf(q, Y6_b, acc6_0);
      acc7_0 = fmaf(q, Y7_b, acc7_0);
      acc8_0 = fmaf(q, Y8_b, acc8_0);
    }
    { const float q = W2_1_b * X0_1_b;
      acc4_1 = fmaf(q, Y4_b, acc4_1);
      acc5_1 = fmaf(q, Y5_b, acc5_1);
      acc6_1 = fmaf(q, Y6_b, acc6_1);
      acc7_1 = fmaf(q, Y7_b, acc7_1);
      acc8_1 = fmaf(q, Y8_b, acc8_1);
    }
    { const float q = W3_0_b * X0_0_b;
      acc9_0 = fmaf(q, Y9_b, acc9_0);
      acc10_0 = fmaf(q, Y10_b, acc10_0);
      acc11_0 = fmaf(q, Y11_b, acc11_0);
      acc12_0 = fmaf(q, Y12_b, acc12_0);
      acc13_0 = fmaf(q, Y13_b, acc13_0);
      acc14_0 = fmaf(q, Y14_b, acc14_0);
      acc15_0 = fmaf(q, Y15_b, acc15_0);
    }
    { const float q = W3_1_b * X0_1_b;
      acc9_1 = fmaf(q, Y9_b, acc9_1);
      acc10_1 = fmaf(q, Y10_b, acc10_1);
      acc11_1 = fmaf(q, Y11_b, acc11_1);
      acc12_1 = fmaf(q, Y12_b, acc12_1);
      acc13_1 = fmaf(q, Y13_b, acc13_1);
      acc14_1 = fmaf(q, Y14_b, acc14_1);
      acc15_1 = fmaf(q, Y15_b, acc15_1);
    }
    }
  }
  float* __restrict__ op = out + (size_t)i * out_stride + c;
  op[0] = acc0_0;
  op[64] = acc0_1;
  op[128] = acc1_0;
  op[192] = acc1_1;
  op[256] = acc2_0;
  op[320] = acc2_1;
  op[384] = acc3_0;
  op[448] = acc3_1;
  op[512] = acc4_0;
  op[576] = acc4_1;
  op[640] = acc5_0;
  op[704] = acc5_1;
  op[768] = acc6_0;
  op[832] = acc6_1;
  op[896] = acc7_0;
  op[960] = acc7_1;
  op[1024] = acc8_0;
  op[1088] = acc8_1;
  op[1152] = acc9_0;
  op[1216] = acc9_1;
  op[1280] = acc10_0;
  op[1344] = acc10_1;
  op[1408] = acc11_0;
  op[1472] = acc11_1;
  op[1536] = acc12_0;
  op[1600] = acc12_1;
  op[1664] = acc13_0;
  op[1728] = acc13_1;
  op[1792] = acc14_0;
  op[1856] = acc14_1;
  op[1920] = acc15_0;
  op[1984] = acc15_1;
}

extern "C" __global__ void __launch_bounds__(256)
mm_tpw_l1_fwd_shared_kernel(const int* __restrict__ rowptr, int nR, const int* __restrict__ eid,
    const int* __restrict__ send, const float* __restrict__ Y, long y_stride, const float* __restrict__ W,
    long w_stride, const float* __restrict__ X, long x_stride, float* __restrict__ out, long out_stride) {
  __shared__ float red[32 * 64];   // one wave's sums [accumulator][lane]
  const int wave = threadIdx.x >> 6;
  const int gw = blockIdx.x;   // receiver i, sub-wave h
  const int i = gw, h = 0;
  if (i >= nR) return;
  const int lane = threadIdx.x & 63;
  const int c = h * 64 + lane;
  const int r0 = rowptr[i], nr = rowptr[i + 1] - r0;
  const int p0 = r0 + (int)((long)nr * wave / 4), p1 = r0 + (int)((long)nr * (wave + 1) / 4);
  float acc0_0 = 0.f;
  float acc0_1 = 0.f;
  float acc1_0 = 0.f;
  float acc1_1 = 0.f;
  float acc2_0 = 0.f;
  float acc2_1 = 0.f;
  float acc3_0 = 0.f;
  float acc3_1 = 0.f;
  float acc4_0 = 0.f;
  float acc4_1 = 0.f;
  float acc5_0 = 0.f;
  float acc5_1 = 0.f;
  float acc6_0 = 0.f;
  float acc6_1 = 0.f;
  float acc7_0 = 0.f;
  float acc7_1 = 0.f;
  float acc8_0 = 0.f;
  float acc8_1 = 0.f;
  float acc9_0 = 0.f;
  float acc9_1 = 0.f;
  float acc10_0 = 0.f;
  float acc10_1 = 0.f;
  float acc11_0 = 0.f;
  float acc11_1 = 0.f;
  float acc12_0 = 0.f;
  float acc12_1 = 0.f;
  float acc13_0 = 0.f;
  float acc13_1 = 0.f;
  float acc14_0 = 0.f;
  float acc14_1 = 0.f;
  float acc15_0 = 0.f;
  float acc15_1 = 0.f;
  for (int p = p0; p < p1; p += 2) {
    const bool two = p + 1 < p1;   // wave-uniform
    const int ea = __builtin_amdgcn_readfirstlane(eid ? eid[p] : p);
    const int sa = __builtin_amdgcn_readfirstlane(send[ea]);
    const float* __restrict__ wpa = W + (size_t)ea * w_stride + c;
    const float W0_0_a = wpa[0];
    const float W0_1_a = wpa[64];
    const float W1_0_a = wpa[128];
    const float W1_1_a = wpa[192];
    const float W2_0_a = wpa[256];
    const float W2_1_a = wpa[320];
    const float W3_0_a = wpa[384];
    const float W3_1_a = wpa[448];
    const float* __restrict__ xpa = X + (size_t)sa * x_stride + c;
    const float X0_0_a = xpa[0];
    const float X0_1_a = xpa[64];
    const float* __restrict__ ypa = Y + (size_t)ea * y_stride;
    const float Y0_a = ypa[0];
    const float Y1_a = ypa[1];
    const float Y2_a = ypa[2];
    const float Y3_a = ypa[3];
    const float Y4_a = ypa[4];
    const float Y5_a = ypa[5];
    const float Y6_a = ypa[6];
    const float Y7_a = ypa[7];
    const float Y8_a = ypa[8];
    const float Y9_a = ypa[9];
    const float Y10_a = ypa[10];
    const float Y11_a = ypa[11];
    const float Y12_a = ypa[12];
    const float Y13_a = ypa[13];
    const float Y14_a = ypa[14];
    const float Y15_a = ypa[15];
    const int eb = two ? __builtin_amdgcn_readfirstlane(eid ? eid[p + 1] : p + 1) : ea;
    const int sb = __builtin_amdgcn_readfirstlane(send[eb]);
    const float* __restrict__ wpb = W + (size_t)eb * w_stride + c;
    const float W0_0_b = wpb[0];
    const float W0_1_b = wpb[64];
    const float W1_0_b = wpb[128];
    const float W1_1_b = wpb[192];
    const float W2_0_b = wpb[256];
    const float W2_1_b = wpb[320];
    const float W3_0_b = wpb[384];
    const float W3_1_b = wpb[448];
    const float* __restrict__ xpb = X + (size_t)sb * x_stride + c;
    const float X0_0_b = xpb[0];
    const float X0_1_b = xpb[64];
    const float* __restrict__ ypb = Y + (size_t)eb * y_stride;
    const float Y0_b = ypb[0];
    const float Y1_b = ypb[1];
    const float Y2_b = ypb[2];
    const float Y3_b = ypb[3];
    const float Y4_b = ypb[4];
    const float Y5_b = ypb[5];
    const float Y6_b = ypb[6];
    const float Y7_b = ypb[7];
    const float Y8_b = ypb[8];
    const float Y9_b = ypb[9];
    const float Y10_b = ypb[10];
    const float Y11_b = ypb[11];
    const float Y12_b = ypb[12];
    const float Y13_b = ypb[13];
    const float Y14_b = ypb[14];
    const float Y15_b = ypb[15];
    { const float q = W0_0_a * X0_0_a;
      acc0_0 = fmaf(q, Y0_a, acc0_0);
    }
    { const float q = W0_1_a * X0_1_a;
      acc0_1 = fmaf(q, Y0_a, acc0_1);
    }
    { const float q = W1_0_a * X0_0_a;
      acc1_0 = fmaf(q, Y1_a, acc1_0);
      acc2_0 = fmaf(q, Y2_a, acc2_0);
      acc3_0 = fmaf(q, Y3_a, acc3_0);
    }
    { const float q = W1_1_a * X0_1_a;
      acc1_1 = fmaf(q, Y1_a, acc1_1);
      acc2_1 = fmaf(q, Y2_a, acc2_1);
      acc3_1 = fmaf(q, Y3_a, acc3_1);
    }
    { const float q = W2_0_a * X0_0_a;
      acc4_0 = fmaf(q, Y4_a, acc4_0);
      acc5_0 = fmaf(q, Y5_a, acc5_0);
      acc6_0 = fmaf(q, Y6_a, acc6_0);
      acc7_0 = fmaf(q, Y7_a, acc7_0);
      acc8_0 = fmaf(q, Y8_a, acc8_0);
    }
    { const float q = W2_1_a * X0_1_a;
      acc4_1 = fmaf(q, Y4_a, acc4_1);
      acc5_1 = fmaf(q, Y5_a, acc5_1);
      acc6_1 = fmaf(q, Y6_a, acc6_1);
      acc7_1 = fmaf(q, Y7_a, acc7_1);
      acc8_1 = fmaf(q, Y8_a, acc8_1);
    }
    { const float q = W3_0_a * X0_0_a;
      acc9_0 = fmaf(q, Y9_a, acc9_0);
      acc10_0 = fmaf(q, Y10_a, acc10_0);
      acc11_0 = fmaf(q, Y11_a, acc11_0);
      acc12_0 = fmaf(q, Y12_a, acc12_0);
      acc13_0 = fmaf(q, Y13_a, acc13_0);
      acc14_0 = fmaf(q, Y14_a, acc14_0);
      acc15_0 = fmaf(q, Y15_a, acc15_0);
    }
    { const float q = W3_1_a * X0_1_a;
      acc9_1 = fmaf(q, Y9_a, acc9_1);
      acc10_1 = fmaf(q, Y10_a, acc10_1);
      acc11_1 = fmaf(q, Y11_a, acc11_1);
      acc12_1 = fmaf(q, Y12_a, acc12_1);
      acc13_1 = fmaf(q, Y13_a, acc13_1);
      acc14_1 = fmaf(q, Y14_a, acc14_1);
      acc15_1 = fmaf(q, Y15_a, acc15_1);
    }
    if (two) {
    { const float q = W0_0_b * X0_0_b;
      acc0_0 = fmaf(q, Y0_b, acc0_0);
    }
    { const float q = W0_1_b * X0_1_b;
      acc0_1 = fmaf(q, Y0_b, acc0_1);
    }
    { const float q = W1_0_b * X0_0_b;
      acc1_0 = fmaf(q, Y1_b, acc1_0);
      acc2_0 = fmaf(q, Y2_b, acc2_0);
      acc3_0 = fmaf(q, Y3_b, acc3_0);
    }
    { const float q = W1_1_b * X0_1_b;
      acc1_1 = fmaf(q, Y1_b, acc1_1);
      acc2_1 = fmaf(q, Y2_b, acc2_1);
      acc3_1 = fmaf(q, Y3_b, acc3_1);
    }
    { const float q = W2_0_b * X0_0_b;
      acc4_0 = fmaf(q, Y4_b, acc4_0);
      acc5_0 = fmaf(q, Y5_b, acc5_0);
      acc6_0 = fmaf(q, Y6_b, acc6_0);
      acc7_0 = fmaf(q, Y7_b, acc7_0);
      acc8_0 = fmaf(q, Y8_b, acc8_0);
    }
    { const float q = W2_1_b * X0_1_b;
      acc4_1 = fmaf(q, Y4_b, acc4_1);
      acc5_1 = fmaf(q, Y5_b, acc5_1);
      acc6_1 = fmaf(q, Y6_b, acc6_1);
      acc7_1 = fmaf(q, Y7_b, acc7_1);
      acc8_1 = fmaf(q, Y8_b, acc8_1);
    }
    { const float q = W3_0_b * X0_0_b;
      acc9_0 = fmaf(q, Y9_b, acc9_0);
      acc10_0 = fmaf(q, Y10_b, acc10_0);
      acc11_0 = fmaf(q, Y11_b, acc11_0);
      acc12_0 = fmaf(q, Y12_b, acc12_0);
      acc13_0 = fmaf(q, Y13_b, acc13_0);
      acc14_0 = fmaf(q, Y14_b, acc14_0);
      acc15_0 = fmaf(q, Y15_b, acc15_0);
    }
    { const float q = W3_1_b * X0_1_b;
      acc9_1 = fmaf(q, Y9_b, acc9_1);
      acc10_1 = fmaf(q, Y10_b, acc10_1);
      acc11_1 = fmaf(q, Y11_b, acc11_1);
      acc12_1 = fmaf(q, Y12_b, acc12_1);
      acc13_1 = fmaf(q, Y13_b, acc13_1);
      acc14_1 = fmaf(q, Y14_b, acc14_1);
      acc15_1 = fmaf(q, Y15_b, acc15_1);
    }
    }
  }
  for (int s = 1; s < 4; ++s) {   // the waves' sums in wave order
    if (wave == s) {
      red[0 + lane] = acc0_0;
      red[64 + lane] = acc0_1;
      red[128 + lane] = acc1_0;
      red[192 + lane] = acc1_1;
      red[256 + lane] = acc2_0;
      red[320 + lane] = acc2_1;
      red[384 + lane] = acc3_0;
      red[448 + lane] = acc3_1;
      red[512 + lane] = acc4_0;
      red[576 + lane] = acc4_1;
      red[640 + lane] = acc5_0;
      red[704 + lane] = acc5_1;
      red[768 + lane] = acc6_0;
      red[832 + lane] = acc6_1;
      red[896 + lane] = acc7_0;
      red[960 + lane] = acc7_1;
      red[1024 + lane] = acc8_0;
      red[1088 + lane] = acc8_1;
      red[1152 + lane] = acc9_0;
      red[1216 + lane] = acc9_1;
      red[1280 + lane] = acc10_0;
      red[1344 + lane] = acc10_1;
      red[1408 + lane] = acc11_0;
      red[1472 + lane] = acc11_1;
      red[1536 + lane] = acc12_0;
      red[1600 + lane] = acc12_1;
      red[1664 + lane] = acc13_0;
      red[1728 + lane] = acc13_1;
      red[1792 + lane] = acc14_0;
      red[1856 + lane] = acc14_1;
      red[1920 + lane] = acc15_0;
      red[1984 + lane] = acc15_1;
    }
    __syncthreads();
    if (wave == 0) {
      acc0_0 += red[0 + lane];
      acc0_1 += red[64 + lane];
      acc1_0 += red[128 + lane];
      acc1_1 += red[192 + lane];
      acc2_0 += red[256 + lane];
      acc2_1 += red[320 + lane];
      acc3_0 += red[384 + lane];
      acc3_1 += red[448 + lane];
      acc4_0 += red[512 + lane];
      acc4_1 += red[576 + lane];
      acc5_0 += red[640 + lane];
      acc5_1 += red[704 + lane];
      acc6_0 += red[768 + lane];
      acc6_1 += red[832 + lane];
      acc7_0 += red[896 + lane];
      acc7_1 += red[960 + lane];
      acc8_0 += red[1024 + lane];
      acc8_1 += red[1088 + lane];
      acc9_0 += red[1152 + lane];
      acc9_1 += red[1216 + lane];
      acc10_0 += red[1280 + lane];
      acc10_1 += red[1344 + lane];
      acc11_0 += red[1408 + lane];
      acc11_1 += red[1472 + lane];
      acc12_0 += red[1536 + lane];
      acc12_1 += red[1600 + lane];
      acc13_0 += red[1664 + lane];
      acc13_1 += red[1728 + lane];
      acc14_0 += red[1792 + lane];
      acc14_1 += red[1856 + lane];
      acc15_0 += red[1920 + lane];
      acc15_1 += red[1984 + lane];
    }
    __syncthreads();
  }
  if (wave) return;
  float* __restrict__ op = out + (size_t)i * out_stride + c;
  op[0] = acc0_0;
  op[64] = acc0_1;
  op[128] = acc1_0;
  op[192] = acc1_1;
  op[256] = acc2_0;
  op[320] = acc2_1;
  op[384] = acc3_0;
  op[448] = acc3_1;
  op[512] = acc4_0;
  op[576] = acc4_1;
  op[640] = acc5_0;
  op[704] = acc5_1;
  op[768] = acc6_0;
  op[832] = acc6_1;
  op[896] = acc7_0;
  op[960] = acc7_1;
  op[1024] = acc8_0;
  op[1088] = acc8_1;
  op[1152] = acc9_0;
  op[1216] = acc9_1;
  op[1280] = acc10_0;
  op[1344] = acc10_1;
  op[1408] = acc11_0;
  op[1472] = acc11_1;
  op[1536] = acc12_0;
  op[1600] = acc12_1;
  op[1664] = acc13_0;
  op[1728] = acc13_1;
  op[1792] = acc14_0;
  op[1856] = acc14_1;
  op[1920] = acc15_0;
  op[1984] = acc15_1;
}

// Backward from gO = dL/dout: gW[e, w, c] (written), gYp[part][e][m] = partial sums of dL/dY[e, m] over
// the channels and paths of one wave (1 partial(s): channel half h x path group g, part
// h * 1 + g; summed by the caller), gX[send, k, c] (atomic adds).  Null outputs are skipped.
extern "C" __global__ void __launch_bounds__(256)
mm_tpw_l1_bwd_kernel(const int* __restrict__ rowptr, int nR, const int* __restrict__ eid,
    const int* __restrict__ send, const float* __restrict__ Y, long y_stride, const float* __restrict__ W,
    long w_stride, const float* __restrict__ X, long x_stride, const float* __restrict__ gO, long g_stride,
    float* __restrict__ gW, long gw_stride, float* __restrict__ gYp, long gy_cb_stride,
    float* __restrict__ gX, long gx_stride) {
  const int gw = blockIdx.x * 4 + (threadIdx.x >> 6);   // global wave: receiver i, sub-wave h
  const int i = gw, h = 0;
  if (i >= nR) return;
  const int lane = threadIdx.x & 63;
  const int c = h * 64 + lane;
  const int p0 = rowptr[i], p1 = rowptr[i + 1];
  const int part = h;
  const int cl = lane & 15;
  const bool b3 = cl & 8, b2 = cl & 4, b1 = cl & 2, b0 = cl & 1;
  const float* __restrict__ gp = gO + (size_t)i * g_stride + c;
  const float g0_0 = gp[0];
  const float g0_1 = gp[64];
  const float g1_0 = gp[128];
  const float g1_1 = gp[192];
  const float g2_0 = gp[256];
  const float g2_1 = gp[320];
  const float g3_0 = gp[384];
  const float g3_1 = gp[448];
  const float g4_0 = gp[512];
  const float g4_1 = gp[576];
  const float g5_0 = gp[640];
  const float g5_1 = gp[704];
  const float g6_0 = gp[768];
  const float g6_1 = gp[832];
  const float g7_0 = gp[896];
  const float g7_1 = gp[960];
  const float g8_0 = gp[1024];
  const float g8_1 = gp[1088];
  const float g9_0 = gp[1152];
  const float g9_1 = gp[1216];
  const float g10_0 = gp[1280];
  const float g10_1 = gp[1344];
  const float g11_0 = gp[1408];
  const float g11_1 = gp[1472];
  const float g12_0 = gp[1536];
  const float g12_1 = gp[1600];
  const float g13_0 = gp[1664];
  const float g13_1 = gp[1728];
  const float g14_0 = gp[1792];
  const float g14_1 = gp[1856];
  const float g15_0 = gp[1920];
  const float g15_1 = gp[1984];
  const float G0_0 = g0_0;
  const float G0_1 = g0_1;
  const float G1_0 = g1_0;
  const float G1_1 = g1_1;
  const float G2_0 = g2_0;
  const float G2_1 = g2_1;
  const float G3_0 = g3_0;
  const float G3_1 = g3_1;
  const float G4_0 = g4_0;
  const float G4_1 = g4_1;
  const float G5_0 = g5_0;
  const float G5_1 = g5_1;
  const float G6_0 = g6_0;
  const float G6_1 = g6_1;
  const float G7_0 = g7_0;
  const float G7_1 = g7_1;
  const float G8_0 = g8_0;
  const float G8_1 = g8_1;
  const float G9_0 = g9_0;
  const float G9_1 = g9_1;
  const float G10_0 = g10_0;
  const float G10_1 = g10_1;
  const float G11_0 = g11_0;
  const float G11_1 = g11_1;
  const float G12_0 = g12_0;
  const float G12_1 = g12_1;
  const float G13_0 = g13_0;
  const float G13_1 = g13_1;
  const float G14_0 = g14_0;
  const float G14_1 = g14_1;
  const float G15_0 = g15_0;
  const float G15_1 = g15_1;
  for (int p = p0; p < p1; p += 2) {
    const bool two = p + 1 < p1;   // wave-uniform
    const int ea = __builtin_amdgcn_readfirstlane(eid ? eid[p] : p);
    const int sa = __builtin_amdgcn_readfirstlane(send[ea]);
    const float* __restrict__ wpa = W + (size_t)ea * w_stride + c;
    const float W0_0_a = wpa[0];
    const float W0_1_a = wpa[64];
    const float W1_0_a = wpa[128];
    const float W1_1_a = wpa[192];
    const float W2_0_a = wpa[256];
    const float W2_1_a = wpa[320];
    const float W3_0_a = wpa[384];
    const float W3_1_a = wpa[448];
    const float* __restrict__ xpa = X + (size_t)sa * x_stride + c;
    const float X0_0_a = xpa[0];
    const float X0_1_a = xpa[64];
    const float* __restrict__ ypa = Y + (size_t)ea * y_stride;
    const float Y0_a = ypa[0];
    const float Y1_a = ypa[1];
    const float Y2_a = ypa[2];
    const float Y3_a = ypa[3];
    const float Y4_a = ypa[4];
    const float Y5_a = ypa[5];
    const float Y6_a = ypa[6];
    const float Y7_a = ypa[7];
    const float Y8_a = ypa[8];
    const float Y9_a = ypa[9];
    const float Y10_a = ypa[10];
    const float Y11_a = ypa[11];
    const float Y12_a = ypa[12];
    const float Y13_a = ypa[13];
    const float Y14_a = ypa[14];
    const float Y15_a = ypa[15];
    const int eb = two ? __builtin_amdgcn_readfirstlane(eid ? eid[p + 1] : p + 1) : ea;
    const int sb = __builtin_amdgcn_readfirstlane(send[eb]);
    const float* __restrict__ wpb = W + (size_t)eb * w_stride + c;
    const float W0_0_b = wpb[0];
    const float W0_1_b = wpb[64];
    const float W1_0_b = wpb[128];
    const float W1_1_b = wpb[192];
    const float W2_0_b = wpb[256];
    const float W2_1_b = wpb[320];
    const float W3_0_b = wpb[384];
    const float W3_1_b = wpb[448];
    const float* __restrict__ xpb = X + (size_t)sb * x_stride + c;
    const float X0_0_b = xpb[0];
    const float X0_1_b = xpb[64];
    const float* __restrict__ ypb = Y + (size_t)eb * y_stride;
    const float Y0_b = ypb[0];
    const float Y1_b = ypb[1];
    const float Y2_b = ypb[2];
    const float Y3_b = ypb[3];
    const float Y4_b = ypb[4];
    const float Y5_b = ypb[5];
    const float Y6_b = ypb[6];
    const float Y7_b = ypb[7];
    const float Y8_b = ypb[8];
    const float Y9_b = ypb[9];
    const float Y10_b = ypb[10];
    const float Y11_b = ypb[11];
    const float Y12_b = ypb[12];
    const float Y13_b = ypb[13];
    const float Y14_b = ypb[14];
    const float Y15_b = ypb[15];
    float gy0 = 0.f;
    float gy1 = 0.f;
    float gy2 = 0.f;
    float gy3 = 0.f;
    float gy4 = 0.f;
    float gy5 = 0.f;
    float gy6 = 0.f;
    float gy7 = 0.f;
    float gy8 = 0.f;
    float gy9 = 0.f;
    float gy10 = 0.f;
    float gy11 = 0.f;
    float gy12 = 0.f;
    float gy13 = 0.f;
    float gy14 = 0.f;
    float gy15 = 0.f;
    float gx0_0 = 0.f;
    float gx0_1 = 0.f;
    float* __restrict__ gwp = gW ? gW + (size_t)ea * gw_stride + c : nullptr;
    {
      float gw0 = 0.f;
      float gw1 = 0.f;
      { const float q = W0_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y0_a, G0_0, u); gy0 = fmaf(q, G0_0, gy0);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W0_0_a, u, gx0_0);
      }
      { const float q = W0_1_a * X0_1_a; float u = 0.f;
        u = fmaf(Y0_a, G0_1, u); gy0 = fmaf(q, G0_1, gy0);
        gw1 = fmaf(X0_1_a, u, gw1); gx0_1 = fmaf(W0_1_a, u, gx0_1);
      }
      if (gwp) gwp[0] = gw0;
      if (gwp) gwp[64] = gw1;
    }
    {
      float gw0 = 0.f;
      float gw1 = 0.f;
      { const float q = W1_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y1_a, G1_0, u); gy1 = fmaf(q, G1_0, gy1);
        u = fmaf(Y2_a, G2_0, u); gy2 = fmaf(q, G2_0, gy2);
        u = fmaf(Y3_a, G3_0, u); gy3 = fmaf(q, G3_0, gy3);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W1_0_a, u, gx0_0);
      }
      { const float q = W1_1_a * X0_1_a; float u = 0.f;
        u = fmaf(Y1_a, G1_1, u); gy1 = fmaf(q, G1_1, gy1);
        u = fmaf(Y2_a, G2_1, u); gy2 = fmaf(q, G2_1, gy2);
        u = fmaf(Y3_a, G3_1, u); gy3 = fmaf(q, G3_1, gy3);
        gw1 = fmaf(X0_1_a, u, gw1); gx0_1 = fmaf(W1_1_a, u, gx0_1);
      }
      if (gwp) gwp[128] = gw0;
      if (gwp) gwp[192] = gw1;
    }
    {
      float gw0 = 0.f;
      float gw1 = 0.f;
      { const float q = W2_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y4_a, G4_0, u); gy4 = fmaf(q, G4_0, gy4);
        u = fmaf(Y5_a, G5_0, u); gy5 = fmaf(q, G5_0, gy5);
        u = fmaf(Y6_a, G6_0, u); gy6 = fmaf(q, G6_0, gy6);
        u = fmaf(Y7_a, G7_0, u); gy7 = fmaf(q, G7_0, gy7);
        u = fmaf(Y8_a, G8_0, u); gy8 = fmaf(q, G8_0, gy8);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W2_0_a, u, gx0_0);
      }
      { const float q = W2_1_a * X0_1_a; float u = 0.f;
        u = fmaf(Y4_a, G4_1, u); gy4 = fmaf(q, G4_1, gy4);
        u = fmaf(Y5_a, G5_1, u); gy5 = fmaf(q, G5_1, gy5);
        u = fmaf(Y6_a, G6_1, u); gy6 = fmaf(q, G6_1, gy6);
        u = fmaf(Y7_a, G7_1, u); gy7 = fmaf(q, G7_1, gy7);
        u = fmaf(Y8_a, G8_1, u); gy8 = fmaf(q, G8_1, gy8);
        gw1 = fmaf(X0_1_a, u, gw1); gx0_1 = fmaf(W2_1_a, u, gx0_1);
      }
      if (gwp) gwp[256] = gw0;
      if (gwp) gwp[320] = gw1;
    }
    {
      float gw0 = 0.f;
      float gw1 = 0.f;
      { const float q = W3_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y9_a, G9_0, u); gy9 = fmaf(q, G9_0, gy9);
        u = fmaf(Y10_a, G10_0, u); gy10 = fmaf(q, G10_0, gy10);
        u = fmaf(Y11_a, G11_0, u); gy11 = fmaf(q, G11_0, gy11);
        u = fmaf(Y12_a, G12_0, u); gy12 = fmaf(q, G12_0, gy12);
        u = fmaf(Y13_a, G13_0, u); gy13 = fmaf(q, G13_0, gy13);
        u = fmaf(Y14_a, G14_0, u); gy14 = fmaf(q, G14_0, gy14);
        u = fmaf(Y15_a, G15_0, u); gy15 = fmaf(q, G15_0, gy15);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W3_0_a, u, gx0_0);
      }
      { const float q = W3_1_a * X0_1_a; float u = 0.f;
        u = fmaf(Y9_a, G9_1, u); gy9 = fmaf(q, G9_1, gy9);
        u = fmaf(Y10_a, G10_1, u); gy10 = fmaf(q, G10_1, gy10);
        u = fmaf(Y11_a, G11_1, u); gy11 = fmaf(q, G11_1, gy11);
        u = fmaf(Y12_a, G12_1, u); gy12 = fmaf(q, G12_1, gy12);
        u = fmaf(Y13_a, G13_1, u); gy13 = fmaf(q, G13_1, gy13);
        u = fmaf(Y14_a, G14_1, u); gy14 = fmaf(q, G14_1, gy14);
        u = fmaf(Y15_a, G15_1, u); gy15 = fmaf(q, G15_1, gy15);
        gw1 = fmaf(X0_1_a, u, gw1); gx0_1 = fmaf(W3_1_a, u, gx0_1);
      }
      if (gwp) gwp[384] = gw0;
      if (gwp) gwp[448] = gw1;
    }
    if (gYp) {
      // transpose-reduction over each 16-lane row (lane cl ends with the row's sum of gy_cl), then the 4 rows
      const float s8_0 = (b3 ? gy8 : gy0) + mm_dpp<0x140>(b3 ? gy0 : gy8);
      const float s8_1 = (b3 ? gy9 : gy1) + mm_dpp<0x140>(b3 ? gy1 : gy9);
      const float s8_2 = (b3 ? gy10 : gy2) + mm_dpp<0x140>(b3 ? gy2 : gy10);
      const float s8_3 = (b3 ? gy11 : gy3) + mm_dpp<0x140>(b3 ? gy3 : gy11);
      const float s8_4 = (b3 ? gy12 : gy4) + mm_dpp<0x140>(b3 ? gy4 : gy12);
      const float s8_5 = (b3 ? gy13 : gy5) + mm_dpp<0x140>(b3 ? gy5 : gy13);
      const float s8_6 = (b3 ? gy14 : gy6) + mm_dpp<0x140>(b3 ? gy6 : gy14);
      const float s8_7 = (b3 ? gy15 : gy7) + mm_dpp<0x140>(b3 ? gy7 : gy15);
      const float s4_0 = (b2 ? s8_4 : s8_0) + mm_dpp<0x141>(b2 ? s8_0 : s8_4);
      const float s4_1 = (b2 ? s8_5 : s8_1) + mm_dpp<0x141>(b2 ? s8_1 : s8_5);
      const float s4_2 = (b2 ? s8_6 : s8_2) + mm_dpp<0x141>(b2 ? s8_2 : s8_6);
      const float s4_3 = (b2 ? s8_7 : s8_3) + mm_dpp<0x141>(b2 ? s8_3 : s8_7);
      const float s2_0 = (b1 ? s4_2 : s4_0) + mm_dpp<0x1B>(b1 ? s4_0 : s4_2);
      const float s2_1 = (b1 ? s4_3 : s4_1) + mm_dpp<0x1B>(b1 ? s4_1 : s4_3);
      float gyl = (b0 ? s2_1 : s2_0) + mm_dpp<0xB1>(b0 ? s2_0 : s2_1);
      gyl += __shfl_xor(gyl, 16);
      gyl += __shfl_xor(gyl, 32);
      if (lane < 16) gYp[(size_t)part * gy_cb_stride + (size_t)ea * 16 + lane] = gyl;
    }
    if (gX) {
      float* __restrict__ gxp = gX + (size_t)sa * gx_stride + c;
      atomicAdd(gxp + 0, gx0_0);
      atomicAdd(gxp + 64, gx0_1);
    }
    if (two) {
    float gy0 = 0.f;
    float gy1 = 0.f;
    float gy2 = 0.f;
    float gy3 = 0.f;
    float gy4 = 0.f;
    float gy5 = 0.f;
    float gy6 = 0.f;
    float gy7 = 0.f;
    float gy8 = 0.f;
    float gy9 = 0.f;
    float gy10 = 0.f;
    float gy11 = 0.f;
    float gy12 = 0.f;
    float gy13 = 0.f;
    float gy14 = 0.f;
    float gy15 = 0.f;
    float gx0_0 = 0.f;
    float gx0_1 = 0.f;
    float* __restrict__ gwp = gW ? gW + (size_t)eb * gw_stride + c : nullptr;
    {
      float gw0 = 0.f;
      float gw1 = 0.f;
      { const float q = W0_0_b * X0_0_b; float u = 0.f;
        u = fmaf(Y0_b, G0_0, u); gy0 = fmaf(q, G0_0, gy0);
        gw0 = fmaf(X0_0_b, u, gw0); gx0_0 = fmaf(W0_0_b, u, gx0_0);
      }
      { const float q = W0_1_b * X0_1_b; float u = 0.f;
        u = fmaf(Y0_b, G0_1, u); gy0 = fmaf(q, G0_1, gy0);
        gw1 = fmaf(X0_1_b, u, gw1); gx0_1 = fmaf(W0_1_b, u, gx0_1);
      }
      if (gwp) gwp[0] = gw0;
      if (gwp) gwp[64] = gw1;
    }
    {
      float gw0 = 0.f;
      float gw1 = 0.f;
      { const float q = W1_0_b * X0_0_b; float u = 0.f;
        u = fmaf(Y1_b, G1_0, u); gy1 = fmaf(q, G1_0, gy1);
        u = fmaf(Y2_b, G2_0, u); gy2 = fmaf(q, G2_0, gy2);
        u = fmaf(Y3_b, G3_0, u); gy3 = fmaf(q, G3_0, gy3);
        gw0 = fmaf(X0_0_b, u, gw0); gx0_0 = fmaf(W1_0_b, u, gx0_0);
      }
      { const float q = W1_1_b * X0_1_b; float u = 0.f;
        u = fmaf(Y1_b, G1_1, u); gy1 = fmaf(q, G1_1, gy1);
        u = fmaf(Y2_b, G2_1, u); gy2 = fmaf(q, G2_1, gy2);
        u = fmaf(Y3_b, G3_1, u); gy3 = fmaf(q, G3_1, gy3);
        gw1 = fmaf(X0_1_b, u, gw1); gx0_1 = fmaf(W1_1_b, u, gx0_1);
      }
      if (gwp) gwp[128] = gw0;
      if (gwp) gwp[192] = gw1;
    }
    {
      float gw0 = 0.f;
      float gw1 = 0.f;
      { const float q = W2_0_b * X0_0_b; float u = 0.f;
        u = fmaf(Y4_b, G4_0, u); gy4 = fmaf(q, G4_0, gy4);
        u = fmaf(Y5_b, G5_0, u); gy5 = fmaf(q, G5_0, gy5);
        u = fmaf(Y6_b, G6_0, u); gy6 = fmaf(q, G6_0, gy6);
        u = fmaf(Y7_b, G7_0, u); gy7 = fmaf(q, G7_0, gy7);
        u = fmaf(Y8_b, G8_0, u); gy8 = fmaf(q, G8_0, gy8);
        gw0 = fmaf(X0_0_b, u, gw0); gx0_0 = fmaf(W2_0_b, u, gx0_0);
      }
      { const float q = W2_1_b * X0_1_b; float u = 0.f;
        u = fmaf(Y4_b, G4_1, u); gy4 = fmaf(q, G4_1, gy4);
        u = fmaf(Y5_b, G5_1, u); gy5 = fmaf(q, G5_1, gy5);
        u = fmaf(Y6_b, G6_1, u); gy6 = fmaf(q, G6_1, gy6);
        u = fmaf(Y7_b, G7_1, u); gy7 = fmaf(q, G7_1, gy7);
        u = fmaf(Y8_b, G8_1, u); gy8 = fmaf(q, G8_1, gy8);
        gw1 = fmaf(X0_1_b, u, gw1); gx0_1 = fmaf(W2_1_b, u, gx0_1);
      }
      if (gwp) gwp[256] = gw0;
      if (gwp) gwp[320] = gw1;
    }
    {
      float gw0 = 0.f;
      float gw1 = 0.f;
      { const float q = W3_0_b * X0_0_b; float u = 0.f;
        u = fmaf(Y9_b, G9_0, u); gy9 = fmaf(q, G9_0, gy9);
        u = fmaf(Y10_b, G10_0, u); gy10 = fmaf(q, G10_0, gy10);
        u = fmaf(Y11_b, G11_0, u); gy11 = fmaf(q, G11_0, gy11);
        u = fmaf(Y12_b, G12_0, u); gy12 = fmaf(q, G12_0, gy12);
        u = fmaf(Y13_b, G13_0, u); gy13 = fmaf(q, G13_0, gy13);
        u = fmaf(Y14_b, G14_0, u); gy14 = fmaf(q, G14_0, gy14);
        u = fmaf(Y15_b, G15_0, u); gy15 = fmaf(q, G15_0, gy15);
        gw0 = fmaf(X0_0_b, u, gw0); gx0_0 = fmaf(W3_0_b, u, gx0_0);
      }
      { const float q = W3_1_b * X0_1_b; float u = 0.f;
        u = fmaf(Y9_b, G9_1, u); gy9 = fmaf(q, G9_1, gy9);
        u = fmaf(Y10_b, G10_1, u); gy10 = fmaf(q, G10_1, gy10);
        u = fmaf(Y11_b, G11_1, u); gy11 = fmaf(q, G11_1, gy11);
        u = fmaf(Y12_b, G12_1, u); gy12 = fmaf(q, G12_1, gy12);
        u = fmaf(Y13_b, G13_1, u); gy13 = fmaf(q, G13_1, gy13);
        u = fmaf(Y14_b, G14_1, u); gy14 = fmaf(q, G14_1, gy14);
        u = fmaf(Y15_b, G15_1, u); gy15 = fmaf(q, G15_1, gy15);
        gw1 = fmaf(X0_1_b, u, gw1); gx0_1 = fmaf(W3_1_b, u, gx0_1);
      }
      if (gwp) gwp[384] = gw0;
      if (gwp) gwp[448] = gw1;
    }
    if (gYp) {
      // transpose-reduction over each 16-lane row (lane cl ends with the row's sum of gy_cl), then the 4 rows
      const float s8_0 = (b3 ? gy8 : gy0) + mm_dpp<0x140>(b3 ? gy0 : gy8);
      const float s8_1 = (b3 ? gy9 : gy1) + mm_dpp<0x140>(b3 ? gy1 : gy9);
      const float s8_2 = (b3 ? gy10 : gy2) + mm_dpp<0x140>(b3 ? gy2 : gy10);
      const float s8_3 = (b3 ? gy11 : gy3) + mm_dpp<0x140>(b3 ? gy3 : gy11);
      const float s8_4 = (b3 ? gy12 : gy4) + mm_dpp<0x140>(b3 ? gy4 : gy12);
      const float s8_5 = (b3 ? gy13 : gy5) + mm_dpp<0x140>(b3 ? gy5 : gy13);
      const float s8_6 = (b3 ? gy14 : gy6) + mm_dpp<0x140>(b3 ? gy6 : gy14);
      const float s8_7 = (b3 ? gy15 : gy7) + mm_dpp<0x140>(b3 ? gy7 : gy15);
      const float s4_0 = (b2 ? s8_4 : s8_0) + mm_dpp<0x141>(b2 ? s8_0 : s8_4);
      const float s4_1 = (b2 ? s8_5 : s8_1) + mm_dpp<0x141>(b2 ? s8_1 : s8_5);
      const float s4_2 = (b2 ? s8_6 : s8_2) + mm_dpp<0x141>(b2 ? s8_2 : s8_6);
      const float s4_3 = (b2 ? s8_7 : s8_3) + mm_dpp<0x141>(b2 ? s8_3 : s8_7);
      const float s2_0 = (b1 ? s4_2 : s4_0) + mm_dpp<0x1B>(b1 ? s4_0 : s4_2);
      const float s2_1 = (b1 ? s4_3 : s4_1) + mm_dpp<0x1B>(b1 ? s4_1 : s4_3);
      float gyl = (b0 ? s2_1 : s2_0) + mm_dpp<0xB1>(b0 ? s2_0 : s2_1);
      gyl += __shfl_xor(gyl, 16);
      gyl += __shfl_xor(gyl, 32);
      if (lane < 16) gYp[(size_t)part * gy_cb_stride + (size_t)eb * 16 + lane] = gyl;
    }
    if (gX) {
      float* __restrict__ gxp = gX + (size_t)sb * gx_stride + c;
      atomicAdd(gxp + 0, gx0_0);
      atomicAdd(gxp + 64, gx0_1);
    }
    }
  }
}

// Backward from gO = dL/dout: gW[e, w, c] (written), gYp[part][e][m] = partial sums of dL/dY[e, m] over
// the channels and paths of one wave (1 partial(s): channel half h x path group g, part
// h * 1 + g; summed by the caller), gX[send, k, c] (atomic adds).  Null outputs are skipped.
extern "C" __global__ void __launch_bounds__(256)
mm_tpw_l1_bwd_shared_kernel(const int* __restrict__ rowptr, int nR, const int* __restrict__ eid,
    const int* __restrict__ send, const float* __restrict__ Y, long y_stride, const float* __restrict__ W,
    long w_stride, const float* __restrict__ X, long x_stride, const float* __restrict__ gO, long g_stride,
    float* __restrict__ gW, long gw_stride, float* __restrict__ gYp, long gy_cb_stride,
    float* __restrict__ gX, long gx_stride) {
  const int wave = threadIdx.x >> 6;
  const int gw = blockIdx.x;   // receiver i, sub-wave h
  const int i = gw, h = 0;
  if (i >= nR) return;
  const int lane = threadIdx.x & 63;
  const int c = h * 64 + lane;
  const int r0 = rowptr[i], nr = rowptr[i + 1] - r0;
  const int p0 = r0 + (int)((long)nr * wave / 4), p1 = r0 + (int)((long)nr * (wave + 1) / 4);
  const int part = h;
  const int cl = lane & 15;
  const bool b3 = cl & 8, b2 = cl & 4, b1 = cl & 2, b0 = cl & 1;
  const float* __restrict__ gp = gO + (size_t)i * g_stride + c;
  const float g0_0 = gp[0];
  const float g0_1 = gp[64];
  const float g1_0 = gp[128];
  const float g1_1 = gp[192];
  const float g2_0 = gp[256];
  const float g2_1 = gp[320];
  const float g3_0 = gp[384];
  const float g3_1 = gp[448];
  const float g4_0 = gp[512];
  const float g4_1 = gp[576];
  const float g5_0 = gp[640];
  const float g5_1 = gp[704];
  const float g6_0 = gp[768];
  const float g6_1 = gp[832];
  const float g7_0 = gp[896];
  const float g7_1 = gp[960];
  const float g8_0 = gp[1024];
  const float g8_1 = gp[1088];
  const float g9_0 = gp[1152];
  const float g9_1 = gp[1216];
  const float g10_0 = gp[1280];
  const float g10_1 = gp[1344];
  const float g11_0 = gp[1408];
  const float g11_1 = gp[1472];
  const float g12_0 = gp[1536];
  const float g12_1 = gp[1600];
  const float g13_0 = gp[1664];
  const float g13_1 = gp[1728];
  const float g14_0 = gp[1792];
  const float g14_1 = gp[1856];
  const float g15_0 = gp[1920];
  const float g15_1 = gp[1984];
  const float G0_0 = g0_0;
  const float G0_1 = g0_1;
  const float G1_0 = g1_0;
  const float G1_1 = g1_1;
  const float G2_0 = g2_0;
  const float G2_1 = g2_1;
  const float G3_0 = g3_0;
  const float G3_1 = g3_1;
  const float G4_0 = g4_0;
  const float G4_1 = g4_1;
  const float G5_0 = g5_0;
  const float G5_1 = g5_1;
  const float G6_0 = g6_0;
  const float G6_1 = g6_1;
  const float G7_0 = g7_0;
  const float G7_1 = g7_1;
  const float G8_0 = g8_0;
  const float G8_1 = g8_1;
  const float G9_0 = g9_0;
  const float G9_1 = g9_1;
  const float G10_0 = g10_0;
  const float G10_1 = g10_1;
  const float G11_0 = g11_0;
  const float G11_1 = g11_1;
  const float G12_0 = g12_0;
  const float G12_1 = g12_1;
  const float G13_0 = g13_0;
  const float G13_1 = g13_1;
  const float G14_0 = g14_0;
  const float G14_1 = g14_1;
  const float G15_0 = g15_0;
  const float G15_1 = g15_1;
  for (int p = p0; p < p1; p += 2) {
    const bool two = p + 1 < p1;   // wave-uniform
    const int ea = __builtin_amdgcn_readfirstlane(eid ? eid[p] : p);
    const int sa = __builtin_amdgcn_readfirstlane(send[ea]);
    const float* __restrict__ wpa = W + (size_t)ea * w_stride + c;
    const float W0_0_a = wpa[0];
    const float W0_1_a = wpa[64];
    const float W1_0_a = wpa[128];
    const float W1_1_a = wpa[192];
    const float W2_0_a = wpa[256];
    const float W2_1_a = wpa[320];
    const float W3_0_a = wpa[384];
    const float W3_1_a = wpa[448];
    const float* __restrict__ xpa = X + (size_t)sa * x_stride + c;
    const float X0_0_a = xpa[0];
    const float X0_1_a = xpa[64];
    const float* __restrict__ ypa = Y + (size_t)ea * y_stride;
    const float Y0_a = ypa[0];
    const float Y1_a = ypa[1];
    const float Y2_a = ypa[2];
    const float Y3_a = ypa[3];
    const float Y4_a = ypa[4];
    const float Y5_a = ypa[5];
    const float Y6_a = ypa[6];
    const float Y7_a = ypa[7];
    const float Y8_a = ypa[8];
    const float Y9_a = ypa[9];
    const float Y10_a = ypa[10];
    const float Y11_a = ypa[11];
    const float Y12_a = ypa[12];
    const float Y13_a = ypa[13];
    const float Y14_a = ypa[14];
    const float Y15_a = ypa[15];
    const int eb = two ? __builtin_amdgcn_readfirstlane(eid ? eid[p + 1] : p + 1) : ea;
    const int sb = __builtin_amdgcn_readfirstlane(send[eb]);
    const float* __restrict__ wpb = W + (size_t)eb * w_stride + c;
    const float W0_0_b = wpb[0];
    const float W0_1_b = wpb[64];
    const float W1_0_b = wpb[128];
    const float W1_1_b = wpb[192];
    const float W2_0_b = wpb[256];
    const float W2_1_b = wpb[320];
    const float W3_0_b = wpb[384];
    const float W3_1_b = wpb[448];
    const float* __restrict__ xpb = X + (size_t)sb * x_stride + c;
    const float X0_0_b = xpb[0];
    const float X0_1_b = xpb[64];
    const float* __restrict__ ypb = Y + (size_t)eb * y_stride;
    const float Y0_b = ypb[0];
    const float Y1_b = ypb[1];
    const float Y2_b = ypb[2];
    const float Y3_b = ypb[3];
    const float Y4_b = ypb[4];
    const float Y5_b = ypb[5];
    const float Y6_b = ypb[6];
    const float Y7_b = ypb[7];
    const float Y8_b = ypb[8];
    const float Y9_b = ypb[9];
    const float Y10_b = ypb[10];
    const float Y11_b = ypb[11];
    const float Y12_b = ypb[12];
    const float Y13_b = ypb[13];
    const float Y14_b = ypb[14];
    const float Y15_b = ypb[15];
    float gy0 = 0.f;
    float gy1 = 0.f;
    float gy2 = 0.f;
    float gy3 = 0.f;
    float gy4 = 0.f;
    float gy5 = 0.f;
    float gy6 = 0.f;
    float gy7 = 0.f;
    float gy8 = 0.f;
    float gy9 = 0.f;
    float gy10 = 0.f;
    float gy11 = 0.f;
    float gy12 = 0.f;
    float gy13 = 0.f;
    float gy14 = 0.f;
    float gy15 = 0.f;
    float gx0_0 = 0.f;
    float gx0_1 = 0.f;
    float* __restrict__ gwp = gW ? gW + (size_t)ea * gw_stride + c : nullptr;
    {
      float gw0 = 0.f;
      float gw1 = 0.f;
      { const float q = W0_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y0_a, G0_0, u); gy0 = fmaf(q, G0_0, gy0);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W0_0_a, u, gx0_0);
      }
      { const float q = W0_1_a * X0_1_a; float u = 0.f;
        u = fmaf(Y0_a, G0_1, u); gy0 = fmaf(q, G0_1, gy0);
        gw1 = fmaf(X0_1_a, u, gw1); gx0_1 = fmaf(W0_1_a, u, gx0_1);
      }
      if (gwp) gwp[0] = gw0;
      if (gwp) gwp[64] = gw1;
    }
    {
      float gw0 = 0.f;
      float gw1 = 0.f;
      { const float q = W1_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y1_a, G1_0, u); gy1 = fmaf(q, G1_0, gy1);
        u = fmaf(Y2_a, G2_0, u); gy2 = fmaf(q, G2_0, gy2);
        u = fmaf(Y3_a, G3_0, u); gy3 = fmaf(q, G3_0, gy3);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W1_0_a, u, gx0_0);
      }
      { const float q = W1_1_a * X0_1_a; float u = 0.f;
        u = fmaf(Y1_a, G1_1, u); gy1 = fmaf(q, G1_1, gy1);
        u = fmaf(Y2_a, G2_1, u); gy2 = fmaf(q, G2_1, gy2);
        u = fmaf(Y3_a, G3_1, u); gy3 = fmaf(q, G3_1, gy3);
        gw1 = fmaf(X0_1_a, u, gw1); gx0_1 = fmaf(W1_1_a, u, gx0_1);
      }
      if (gwp) gwp[128] = gw0;
      if (gwp) gwp[192] = gw1;
    }
    {
      float gw0 = 0.f;
      float gw1 = 0.f;
      { const float q = W2_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y4_a, G4_0, u); gy4 = fmaf(q, G4_0, gy4);
        u = fmaf(Y5_a, G5_0, u); gy5 = fmaf(q, G5_0, gy5);
        u = fmaf(Y6_a, G6_0, u); gy6 = fmaf(q, G6_0, gy6);
        u = fmaf(Y7_a, G7_0, u); gy7 = fmaf(q, G7_0, gy7);
        u = fmaf(Y8_a, G8_0, u); gy8 = fmaf(q, G8_0, gy8);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W2_0_a, u, gx0_0);
      }
      { const float q = W2_1_a * X0_1_a; float u = 0.f;
        u = fmaf(Y4_a, G4_1, u); gy4 = fmaf(q, G4_1, gy4);
        u = fmaf(Y5_a, G5_1, u); gy5 = fmaf(q, G5_1, gy5);
        u = fmaf(Y6_a, G6_1, u); gy6 = fmaf(q, G6_1, gy6);
        u = fmaf(Y7_a, G7_1, u); gy7 = fmaf(q, G7_1, gy7);
        u = fmaf(Y8_a, G8_1, u); gy8 = fmaf(q, G8_1, gy8);
        gw1 = fmaf(X0_1_a, u, gw1); gx0_1 = fmaf(W2_1_a, u, gx0_1);
      }
      if (gwp) gwp[256] = gw0;
      if (gwp) gwp[320] = gw1;
    }
    {
      float gw0 = 0.f;
      float gw1 = 0.f;
      { const float q = W3_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y9_a, G9_0, u); gy9 = fmaf(q, G9_0, gy9);
        u = fmaf(Y10_a, G10_0, u); gy10 = fmaf(q, G10_0, gy10);
        u = fmaf(Y11_a, G11_0, u); gy11 = fmaf(q, G11_0, gy11);
        u = fmaf(Y12_a, G12_0, u); gy12 = fmaf(q, G12_0, gy12);
        u = fmaf(Y13_a, G13_0, u); gy13 = fmaf(q, G13_0, gy13);
        u = fmaf(Y14_a, G14_0, u); gy14 = fmaf(q, G14_0, gy14);
        u = fmaf(Y15_a, G15_0, u); gy15 = fmaf(q, G15_0, gy15);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W3_0_a, u, gx0_0);
      }
      { const float q = W3_1_a * X0_1_a; float u = 0.f;
        u = fmaf(Y9_a, G9_1, u); gy9 = fmaf(q, G9_1, gy9);
        u = fmaf(Y10_a, G10_1, u); gy10 = fmaf(q, G10_1, gy10);
        u = fmaf(Y11_a, G11_1, u); gy11 = fmaf(q, G11_1, gy11);
        u = fmaf(Y12_a, G12_1, u); gy12 = fmaf(q, G12_1, gy12);
        u = fmaf(Y13_a, G13_1, u); gy13 = fmaf(q, G13_1, gy13);
        u = fmaf(Y14_a, G14_1, u); gy14 = fmaf(q, G14_1, gy14);
        u = fmaf(Y15_a, G15_1, u); gy15 = fmaf(q, G15_1, gy15);
        gw1 = fmaf(X0_1_a, u, gw1); gx0_1 = fmaf(W3_1_a, u, gx0_1);
      }
      if (gwp) gwp[384] = gw0;
      if (gwp) gwp[448] = gw1;
    }
    if (gYp) {
      // transpose-reduction over each 16-lane row (lane cl ends with the row's sum of gy_cl), then the 4 rows
      const float s8_0 = (b3 ? gy8 : gy0) + mm_dpp<0x140>(b3 ? gy0 : gy8);
      const float s8_1 = (b3 ? gy9 : gy1) + mm_dpp<0x140>(b3 ? gy1 : gy9);
      const float s8_2 = (b3 ? gy10 : gy2) + mm_dpp<0x140>(b3 ? gy2 : gy10);
      const float s8_3 = (b3 ? gy11 : gy3) + mm_dpp<0x140>(b3 ? gy3 : gy11);
      const float s8_4 = (b3 ? gy12 : gy4) + mm_dpp<0x140>(b3 ? gy4 : gy12);
      const float s8_5 = (b3 ? gy13 : gy5) + mm_dpp<0x140>(b3 ? gy5 : gy13);
      const float s8_6 = (b3 ? gy14 : gy6) + mm_dpp<0x140>(b3 ? gy6 : gy14);
      const float s8_7 = (b3 ? gy15 : gy7) + mm_dpp<0x140>(b3 ? gy7 : gy15);
      const float s4_0 = (b2 ? s8_4 : s8_0) + mm_dpp<0x141>(b2 ? s8_0 : s8_4);
      const float s4_1 = (b2 ? s8_5 : s8_1) + mm_dpp<0x141>(b2 ? s8_1 : s8_5);
      const float s4_2 = (b2 ? s8_6 : s8_2) + mm_dpp<0x141>(b2 ? s8_2 : s8_6);
      const float s4_3 = (b2 ? s8_7 : s8_3) + mm_dpp<0x141>(b2 ? s8_3 : s8_7);
      const float s2_0 = (b1 ? s4_2 : s4_0) + mm_dpp<0x1B>(b1 ? s4_0 : s4_2);
      const float s2_1 = (b1 ? s4_3 : s4_1) + mm_dpp<0x1B>(b1 ? s4_1 : s4_3);
      float gyl = (b0 ? s2_1 : s2_0) + mm_dpp<0xB1>(b0 ? s2_0 : s2_1);
      gyl += __shfl_xor(gyl, 16);
      gyl += __shfl_xor(gyl, 32);
      if (lane < 16) gYp[(size_t)part * gy_cb_stride + (size_t)ea * 16 + lane] = gyl;
    }
    if (gX) {
      float* __restrict__ gxp = gX + (size_t)sa * gx_stride + c;
      atomicAdd(gxp + 0, gx0_0);
      atomicAdd(gxp + 64, gx0_1);
    }
    if (two) {
    float gy0 = 0.f;
    float gy1 = 0.f;
    float gy2 = 0.f;
    float gy3 = 0.f;
    float gy4 = 0.f;
    float gy5 = 0.f;
    float gy6 = 0.f;
    float gy7 = 0.f;
    float gy8 = 0.f;
    float gy9 = 0.f;
    float gy10 = 0.f;
    float gy11 = 0.f;
    float gy12 = 0.f;
    float gy13 = 0.f;
    float gy14 = 0.f;
    float gy15 = 0.f;
    float gx0_0 = 0.f;
    float gx0_1 = 0.f;
    float* __restrict__ gwp = gW ? gW + (size_t)eb * gw_stride + c : nullptr;
    {
      float gw0 = 0.f;
      float gw1 = 0.f;
      { const float q = W0_0_b * X0_0_b; float u = 0.f;
        u = fmaf(Y0_b, G0_0, u); gy0 = fmaf(q, G0_0, gy0);
        gw0 = fmaf(X0_0_b, u, gw0); gx0_0 = fmaf(W0_0_b, u, gx0_0);
      }
      { const float q = W0_1_b * X0_1_b; float u = 0.f;
        u = fmaf(Y0_b, G0_1, u); gy0 = fmaf(q, G0_1, gy0);
        gw1 = fmaf(X0_1_b, u, gw1); gx0_1 = fmaf(W0_1_b, u, gx0_1);
      }
      if (gwp) gwp[0] = gw0;
      if (gwp) gwp[64] = gw1;
    }
    {
      float gw0 = 0.f;
      float gw1 = 0.f;
      { const float q = W1_0_b * X0_0_b; float u = 0.f;
        u = fmaf(Y1_b, G1_0, u); gy1 = fmaf(q, G1_0, gy1);
        u = fmaf(Y2_b, G2_0, u); gy2 = fmaf(q, G2_0, gy2);
        u = fmaf(Y3_b, G3_0, u); gy3 = fmaf(q, G3_0, gy3);
        gw0 = fmaf(X0_0_b, u, gw0); gx0_0 = fmaf(W1_0_b, u, gx0_0);
      }
      { const float q = W1_1_b * X0_1_b; float u = 0.f;
        u = fmaf(Y1_b, G1_1, u); gy1 = fmaf(q, G1_1, gy1);
        u = fmaf(Y2_b, G2_1, u); gy2 = fmaf(q, G2_1, gy2);
        u = fmaf(Y3_b, G3_1, u); gy3 = fmaf(q, G3_1, gy3);
        gw1 = fmaf(X0_1_b, u, gw1); gx0_1 = fmaf(W1_1_b, u, gx0_1);
      }
      if (gwp) gwp[128] = gw0;
      if (gwp) gwp[192] = gw1;
    }
    {
      float gw0 = 0.f;
      float gw1 = 0.f;
      { const float q = W2_0_b * X0_0_b; float u = 0.f;
        u = fmaf(Y4_b, G4_0, u); gy4 = fmaf(q, G4_0, gy4);
        u = fmaf(Y5_b, G5_0, u); gy5 = fmaf(q, G5_0, gy5);
        u = fmaf(Y6_b, G6_0, u); gy6 = fmaf(q, G6_0, gy6);
        u = fmaf(Y7_b, G7_0, u); gy7 = fmaf(q, G7_0, gy7);
        u = fmaf(Y8_b, G8_0, u); gy8 = fmaf(q, G8_0, gy8);
        gw0 = fmaf(X0_0_b, u, gw0); gx0_0 = fmaf(W2_0_b, u, gx0_0);
      }
      { const float q = W2_1_b * X0_1_b; float u = 0.f;
        u = fmaf(Y4_b, G4_1, u); gy4 = fmaf(q, G4_1, gy4);
        u = fmaf(Y5_b, G5_1, u); gy5 = fmaf(q, G5_1, gy5);
        u = fmaf(Y6_b, G6_1, u); gy6 = fmaf(q, G6_1, gy6);
        u = fmaf(Y7_b, G7_1, u); gy7 = fmaf(q, G7_1, gy7);
        u = fmaf(Y8_b, G8_1, u); gy8 = fmaf(q, G8_1, gy8);
        gw1 = fmaf(X0_1_b, u, gw1); gx0_1 = fmaf(W2_1_b, u, gx0_1);
      }
      if (gwp) gwp[256] = gw0;
      if (gwp) gwp[320] = gw1;
    }
    {
      float gw0 = 0.f;
      float gw1 = 0.f;
      { const float q = W3_0_b * X0_0_b; float u = 0.f;
        u = fmaf(Y9_b, G9_0, u); gy9 = fmaf(q, G9_0, gy9);
        u = fmaf(Y10_b, G10_0, u); gy10 = fmaf(q, G10_0, gy10);
        u = fmaf(Y11_b, G11_0, u); gy11 = fmaf(q, G11_0, gy11);
        u = fmaf(Y12_b, G12_0, u); gy12 = fmaf(q, G12_0, gy12);
        u = fmaf(Y13_b, G13_0, u); gy13 = fmaf(q, G13_0, gy13);
        u = fmaf(Y14_b, G14_0, u); gy14 = fmaf(q, G14_0, gy14);
        u = fmaf(Y15_b, G15_0, u); gy15 = fmaf(q, G15_0, gy15);
        gw0 = fmaf(X0_0_b, u, gw0); gx0_0 = fmaf(W3_0_b, u, gx0_0);
      }
      { const float q = W3_1_b * X0_1_b; float u = 0.f;
        u = fmaf(Y9_b, G9_1, u); gy9 = fmaf(q, G9_1, gy9);
        u = fmaf(Y10_b, G10_1, u); gy10 = fmaf(q, G10_1, gy10);
        u = fmaf(Y11_b, G11_1, u); gy11 = fmaf(q, G11_1, gy11);
        u = fmaf(Y12_b, G12_1, u); gy12 = fmaf(q, G12_1, gy12);
        u = fmaf(Y13_b, G13_1, u); gy13 = fmaf(q, G13_1, gy13);
        u = fmaf(Y14_b, G14_1, u); gy14 = fmaf(q, G14_1, gy14);
        u = fmaf(Y15_b, G15_1, u); gy15 = fmaf(q, G15_1, gy15);
        gw1 = fmaf(X0_1_b, u, gw1); gx0_1 = fmaf(W3_1_b, u, gx0_1);
      }
      if (gwp) gwp[384] = gw0;
      if (gwp) gwp[448] = gw1;
    }
    if (gYp) {
      // transpose-reduction over each 16-lane row (lane cl ends with the row's sum of gy_cl), then the 4 rows
      const float s8_0 = (b3 ? gy8 : gy0) + mm_dpp<0x140>(b3 ? gy0 : gy8);
      const float s8_1 = (b3 ? gy9 : gy1) + mm_dpp<0x140>(b3 ? gy1 : gy9);
      const float s8_2 = (b3 ? gy10 : gy2) + mm_dpp<0x140>(b3 ? gy2 : gy10);
      const float s8_3 = (b3 ? gy11 : gy3) + mm_dpp<0x140>(b3 ? gy3 : gy11);
      const float s8_4 = (b3 ? gy12 : gy4) + mm_dpp<0x140>(b3 ? gy4 : gy12);
      const float s8_5 = (b3 ? gy13 : gy5) + mm_dpp<0x140>(b3 ? gy5 : gy13);
      const float s8_6 = (b3 ? gy14 : gy6) + mm_dpp<0x140>(b3 ? gy6 : gy14);
      const float s8_7 = (b3 ? gy15 : gy7) + mm_dpp<0x140>(b3 ? gy7 : gy15);
      const float s4_0 = (b2 ? s8_4 : s8_0) + mm_dpp<0x141>(b2 ? s8_0 : s8_4);
      const float s4_1 = (b2 ? s8_5 : s8_1) + mm_dpp<0x141>(b2 ? s8_1 : s8_5);
      const float s4_2 = (b2 ? s8_6 : s8_2) + mm_dpp<0x141>(b2 ? s8_2 : s8_6);
      const float s4_3 = (b2 ? s8_7 : s8_3) + mm_dpp<0x141>(b2 ? s8_3 : s8_7);
      const float s2_0 = (b1 ? s4_2 : s4_0) + mm_dpp<0x1B>(b1 ? s4_0 : s4_2);
      const float s2_1 = (b1 ? s4_3 : s4_1) + mm_dpp<0x1B>(b1 ? s4_1 : s4_3);
      float gyl = (b0 ? s2_1 : s2_0) + mm_dpp<0xB1>(b0 ? s2_0 : s2_1);
      gyl += __shfl_xor(gyl, 16);
      gyl += __shfl_xor(gyl, 32);
      if (lane < 16) gYp[(size_t)part * gy_cb_stride + (size_t)eb * 16 + lane] = gyl;
    }
    if (gX) {
      float* __restrict__ gxp = gX + (size_t)sb * gx_stride + c;
      atomicAdd(gxp + 0, gx0_0);
      atomicAdd(gxp + 64, gx0_1);
    }
    }
  }
}

extern "C" int mm_tpw_l1_fwd_n(long E, const int* rowptr, int nR, const int* eid, const int* send, const float* Y,
    long y_stride, const float* W, long w_stride, const float* X, long x_stride, float* out, long out_stride,
    hipStream_t stream) {
  MM_CHECK_ARG(nR >= 0, "bad sizes");
  MM_CHECK_ARG(y_stride >= 16 && w_stride >= 512 && x_stride >= 128 && out_stride >= 2048,
               "row strides smaller than the path table's widths");
  if (nR == 0) return MM_OK;
  const long waves = (long)nR * 1;
  // E < 0: unknown, shared where the receivers alone leave most of the chip idle
  // (a launch takes fewer than 2^32 threads)
  const bool shared = E < 0 ? waves <= 2048 : true && waves < (1L << 24) && E >= 4L * nR;
  dim3 grid((unsigned)(shared ? waves : (waves + 3) / 4)), block(256);
  hipLaunchKernelGGL(shared ? mm_tpw_l1_fwd_shared_kernel : mm_tpw_l1_fwd_kernel, grid, block, 0, stream, rowptr, nR, eid, send, Y, y_stride, W,
                     w_stride, X, x_stride, out, out_stride);
  return mm::launch_status("mm_tpw_l1_fwd");
}

extern "C" int mm_tpw_l1_fwd(const int* rowptr, int nR, const int* eid, const int* send, const float* Y,
    long y_stride, const float* W, long w_stride, const float* X, long x_stride,
    float* out, long out_stride, hipStream_t stream) {
  return mm_tpw_l1_fwd_n(-1, rowptr, nR, eid, send, Y, y_stride, W, w_stride, X, x_stride, out, out_stride, stream);
}

extern "C" int mm_tpw_l1_bwd_n(long E, const int* rowptr, int nR, const int* eid, const int* send, const float* Y,
    long y_stride, const float* W, long w_stride, const float* X, long x_stride, const float* gO, long g_stride,
    float* gW, long gw_stride, float* gYp, long gy_cb_stride, float* gX, long gx_stride, hipStream_t stream) {
  MM_CHECK_ARG(nR >= 0, "bad sizes");
  MM_CHECK_ARG(y_stride >= 16 && w_stride >= 512 && x_stride >= 128 && g_stride >= 2048,
               "row strides smaller than the path table's widths");
  MM_CHECK_ARG(!gW || gw_stride >= 512, "gW row stride");
  MM_CHECK_ARG(!gX || gx_stride >= 128, "gX row stride");
  if (nR == 0) return MM_OK;
  const long waves = (long)nR * 1;
  // E < 0: unknown, shared where the receivers alone leave most of the chip idle
  // (a launch takes fewer than 2^32 threads)
  const bool shared = E < 0 ? waves <= 2048 : true && waves < (1L << 24) && E >= 4L * nR;
  dim3 grid((unsigned)(shared ? waves : (waves + 3) / 4)), block(256);
  hipLaunchKernelGGL(shared ? mm_tpw_l1_bwd_shared_kernel : mm_tpw_l1_bwd_kernel, grid, block, 0, stream, rowptr, nR, eid, send, Y, y_stride, W,
                     w_stride, X, x_stride, gO, g_stride, gW, gw_stride, gYp, gy_cb_stride, gX, gx_stride);
  return mm::launch_status("mm_tpw_l1_bwd");
}

extern "C" int mm_tpw_l1_bwd(const int* rowptr, int nR, const int* eid, const int* send, const float* Y,
    long y_stride, const float* W, long w_stride, const float* X, long x_stride,
    const float* gO, long g_stride, float* gW, long gw_stride, float* gYp, long gy_cb_stride, float* gX,
    long gx_stride, hipStream_t stream) {
  return mm_tpw_l1_bwd_n(-1, rowptr, nR, eid, send, Y, y_stride, W, w_stride, X, x_stride, gO, g_stride, gW, gw_stride, gYp, gy_cb_stride, gX, gx_stride, stream);
}
