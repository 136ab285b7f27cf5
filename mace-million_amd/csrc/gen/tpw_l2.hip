// generated by mace_onegpu/codegen.py -- explicit-weight channelwise TP 'l2'
// nX=4, nW=10, nO=40, terms=86
//
// out[i, o, c] = sum_{p in [rowptr[i], rowptr[i+1])} sum_terms coef * W[e, w, c] * X[send[e], k, c] * Y[e, m],
// e = eid[p] (or p when eid is null): receiver-CSR over a permutation, so edges need not be stored sorted.
// Forward: one wave per receiver and channel half, 2 channel(s) per lane (c = 64 h + lane + 64 j),
// 1 wave(s) per receiver, 2 edge(s) loaded together.  Backward: 1 channel(s) per lane, 2 wave(s)
// per receiver, 2 edge(s) loaded together; dL/dY partials: 2 per edge (one per channel half).
#include "../common.h"

extern "C" __global__ void __launch_bounds__(256)
mm_tpw_l2_fwd_kernel(const int* __restrict__ rowptr, int nR, const int* __restrict__ eid,
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
  float acc16_0 = 0.f;
  float acc16_1 = 0.f;
  float acc17_0 = 0.f;
  float acc17_1 = 0.f;
  float acc18_0 = 0.f;
  float acc18_1 = 0.f;
  float acc19_0 = 0.f;
  float acc19_1 = 0.f;
  float acc20_0 = 0.f;
  float acc20_1 = 0.f;
  float acc21_0 = 0.f;
  float acc21_1 = 0.f;
  float acc22_0 = 0.f;
  float acc22_1 = 0.f;
  float acc23_0 = 0.f;
  float acc23_1 = 0.f;
  float acc24_0 = 0.f;
  float acc24_1 = 0.f;
  float acc25_0 = 0.f;
  float acc25_1 = 0.f;
  float acc26_0 = 0.f;
  float acc26_1 = 0.f;
  float acc27_0 = 0.f;
  float acc27_1 = 0.f;
  float acc28_0 = 0.f;
  float acc28_1 = 0.f;
  float acc29_0 = 0.f;
  float acc29_1 = 0.f;
  float acc30_0 = 0.f;
  float acc30_1 = 0.f;
  float acc31_0 = 0.f;
  float acc31_1 = 0.f;
  float acc32_0 = 0.f;
  float acc32_1 = 0.f;
  float acc33_0 = 0.f;
  float acc33_1 = 0.f;
  float acc34_0 = 0.f;
  float acc34_1 = 0.f;
  float acc35_0 = 0.f;
  float acc35_1 = 0.f;
  float acc36_0 = 0.f;
  float acc36_1 = 0.f;
  float acc37_0 = 0.f;
  float acc37_1 = 0.f;
  float acc38_0 = 0.f;
  float acc38_1 = 0.f;
  float acc39_0 = 0.f;
  float acc39_1 = 0.f;
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
    const float W4_0_a = wpa[512];
    const float W4_1_a = wpa[576];
    const float W5_0_a = wpa[640];
    const float W5_1_a = wpa[704];
    const float W6_0_a = wpa[768];
    const float W6_1_a = wpa[832];
    const float W7_0_a = wpa[896];
    const float W7_1_a = wpa[960];
    const float W8_0_a = wpa[1024];
    const float W8_1_a = wpa[1088];
    const float W9_0_a = wpa[1152];
    const float W9_1_a = wpa[1216];
    const float* __restrict__ xpa = X + (size_t)sa * x_stride + c;
    const float X0_0_a = xpa[0];
    const float X0_1_a = xpa[64];
    const float X1_0_a = xpa[128];
    const float X1_1_a = xpa[192];
    const float X2_0_a = xpa[256];
    const float X2_1_a = xpa[320];
    const float X3_0_a = xpa[384];
    const float X3_1_a = xpa[448];
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
    const float W4_0_b = wpb[512];
    const float W4_1_b = wpb[576];
    const float W5_0_b = wpb[640];
    const float W5_1_b = wpb[704];
    const float W6_0_b = wpb[768];
    const float W6_1_b = wpb[832];
    const float W7_0_b = wpb[896];
    const float W7_1_b = wpb[960];
    const float W8_0_b = wpb[1024];
    const float W8_1_b = wpb[1088];
    const float W9_0_b = wpb[1152];
    const float W9_1_b = wpb[1216];
    const float* __restrict__ xpb = X + (size_t)sb * x_stride + c;
    const float X0_0_b = xpb[0];
    const float X0_1_b = xpb[64];
    const float X1_0_b = xpb[128];
    const float X1_1_b = xpb[192];
    const float X2_0_b = xpb[256];
    const float X2_1_b = xpb[320];
    const float X3_0_b = xpb[384];
    const float X3_1_b = xpb[448];
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
    { const float q = W1_0_a * X1_0_a;
      const float q0 = 0.5773502691896257f * q;
      acc1_0 = fmaf(q0, Y1_a, acc1_0);
    }
    { const float q = W1_1_a * X1_1_a;
      const float q0 = 0.5773502691896257f * q;
      acc1_1 = fmaf(q0, Y1_a, acc1_1);
    }
    { const float q = W1_0_a * X2_0_a;
      const float q0 = 0.5773502691896258f * q;
      acc1_0 = fmaf(q0, Y2_a, acc1_0);
    }
    { const float q = W1_1_a * X2_1_a;
      const float q0 = 0.5773502691896258f * q;
      acc1_1 = fmaf(q0, Y2_a, acc1_1);
    }
    { const float q = W1_0_a * X3_0_a;
      const float q0 = 0.5773502691896257f * q;
      acc1_0 = fmaf(q0, Y3_a, acc1_0);
    }
    { const float q = W1_1_a * X3_1_a;
      const float q0 = 0.5773502691896257f * q;
      acc1_1 = fmaf(q0, Y3_a, acc1_1);
    }
    { const float q = W2_0_a * X0_0_a;
      acc2_0 = fmaf(q, Y1_a, acc2_0);
      acc3_0 = fmaf(q, Y2_a, acc3_0);
      acc4_0 = fmaf(q, Y3_a, acc4_0);
    }
    { const float q = W2_1_a * X0_1_a;
      acc2_1 = fmaf(q, Y1_a, acc2_1);
      acc3_1 = fmaf(q, Y2_a, acc3_1);
      acc4_1 = fmaf(q, Y3_a, acc4_1);
    }
    { const float q = W3_0_a * X1_0_a;
      acc5_0 = fmaf(q, Y0_a, acc5_0);
    }
    { const float q = W3_1_a * X1_1_a;
      acc5_1 = fmaf(q, Y0_a, acc5_1);
    }
    { const float q = W3_0_a * X2_0_a;
      acc6_0 = fmaf(q, Y0_a, acc6_0);
    }
    { const float q = W3_1_a * X2_1_a;
      acc6_1 = fmaf(q, Y0_a, acc6_1);
    }
    { const float q = W3_0_a * X3_0_a;
      acc7_0 = fmaf(q, Y0_a, acc7_0);
    }
    { const float q = W3_1_a * X3_1_a;
      acc7_1 = fmaf(q, Y0_a, acc7_1);
    }
    { const float q = W4_0_a * X1_0_a;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc10_0 = fmaf(q0, Y4_a, acc10_0);
      acc9_0 = fmaf(q0, Y5_a, acc9_0);
      acc8_0 = fmaf(-q1, Y6_a, acc8_0);
      acc8_0 = fmaf(-q0, Y8_a, acc8_0);
    }
    { const float q = W4_1_a * X1_1_a;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc10_1 = fmaf(q0, Y4_a, acc10_1);
      acc9_1 = fmaf(q0, Y5_a, acc9_1);
      acc8_1 = fmaf(-q1, Y6_a, acc8_1);
      acc8_1 = fmaf(-q0, Y8_a, acc8_1);
    }
    { const float q = W4_0_a * X2_0_a;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.632455532033676f * q;
      acc8_0 = fmaf(q0, Y5_a, acc8_0);
      acc9_0 = fmaf(q1, Y6_a, acc9_0);
      acc10_0 = fmaf(q0, Y7_a, acc10_0);
    }
    { const float q = W4_1_a * X2_1_a;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.632455532033676f * q;
      acc8_1 = fmaf(q0, Y5_a, acc8_1);
      acc9_1 = fmaf(q1, Y6_a, acc9_1);
      acc10_1 = fmaf(q0, Y7_a, acc10_1);
    }
    { const float q = W4_0_a * X3_0_a;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc8_0 = fmaf(q0, Y4_a, acc8_0);
      acc10_0 = fmaf(-q1, Y6_a, acc10_0);
      acc9_0 = fmaf(q0, Y7_a, acc9_0);
      acc10_0 = fmaf(q0, Y8_a, acc10_0);
    }
    { const float q = W4_1_a * X3_1_a;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc8_1 = fmaf(q0, Y4_a, acc8_1);
      acc10_1 = fmaf(-q1, Y6_a, acc10_1);
      acc9_1 = fmaf(q0, Y7_a, acc9_1);
      acc10_1 = fmaf(q0, Y8_a, acc10_1);
    }
    { const float q = W5_0_a * X0_0_a;
      acc11_0 = fmaf(q, Y4_a, acc11_0);
      acc12_0 = fmaf(q, Y5_a, acc12_0);
      acc13_0 = fmaf(q, Y6_a, acc13_0);
      acc14_0 = fmaf(q, Y7_a, acc14_0);
      acc15_0 = fmaf(q, Y8_a, acc15_0);
    }
    { const float q = W5_1_a * X0_1_a;
      acc11_1 = fmaf(q, Y4_a, acc11_1);
      acc12_1 = fmaf(q, Y5_a, acc12_1);
      acc13_1 = fmaf(q, Y6_a, acc13_1);
      acc14_1 = fmaf(q, Y7_a, acc14_1);
      acc15_1 = fmaf(q, Y8_a, acc15_1);
    }
    { const float q = W6_0_a * X1_0_a;
      const float q0 = 0.408248290463863f * q;
      const float q1 = 0.7071067811865475f * q;
      acc18_0 = fmaf(q0, Y1_a, acc18_0);
      acc20_0 = fmaf(q1, Y1_a, acc20_0);
      acc17_0 = fmaf(-q1, Y2_a, acc17_0);
      acc16_0 = fmaf(-q1, Y3_a, acc16_0);
    }
    { const float q = W6_1_a * X1_1_a;
      const float q0 = 0.408248290463863f * q;
      const float q1 = 0.7071067811865475f * q;
      acc18_1 = fmaf(q0, Y1_a, acc18_1);
      acc20_1 = fmaf(q1, Y1_a, acc20_1);
      acc17_1 = fmaf(-q1, Y2_a, acc17_1);
      acc16_1 = fmaf(-q1, Y3_a, acc16_1);
    }
    { const float q = W6_0_a * X2_0_a;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.8164965809277261f * q;
      acc17_0 = fmaf(-q0, Y1_a, acc17_0);
      acc18_0 = fmaf(-q1, Y2_a, acc18_0);
      acc19_0 = fmaf(-q0, Y3_a, acc19_0);
    }
    { const float q = W6_1_a * X2_1_a;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.8164965809277261f * q;
      acc17_1 = fmaf(-q0, Y1_a, acc17_1);
      acc18_1 = fmaf(-q1, Y2_a, acc18_1);
      acc19_1 = fmaf(-q0, Y3_a, acc19_1);
    }
    { const float q = W6_0_a * X3_0_a;
      const float q0 = 0.7071067811865475f * q;
      const float q1 = 0.408248290463863f * q;
      acc16_0 = fmaf(-q0, Y1_a, acc16_0);
      acc19_0 = fmaf(-q0, Y2_a, acc19_0);
      acc18_0 = fmaf(q1, Y3_a, acc18_0);
      acc20_0 = fmaf(-q0, Y3_a, acc20_0);
    }
    { const float q = W6_1_a * X3_1_a;
      const float q0 = 0.7071067811865475f * q;
      const float q1 = 0.408248290463863f * q;
      acc16_1 = fmaf(-q0, Y1_a, acc16_1);
      acc19_1 = fmaf(-q0, Y2_a, acc19_1);
      acc18_1 = fmaf(q1, Y3_a, acc18_1);
      acc20_1 = fmaf(-q0, Y3_a, acc20_1);
    }
    { const float q = W7_0_a * X1_0_a;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.5345224838248488f * q;
      const float q3 = 0.15430334996209188f * q;
      const float q4 = 0.3779644730092272f * q;
      acc25_0 = fmaf(q0, Y9_a, acc25_0);
      acc24_0 = fmaf(q1, Y10_a, acc24_0);
      acc23_0 = fmaf(q2, Y11_a, acc23_0);
      acc25_0 = fmaf(q3, Y11_a, acc25_0);
      acc22_0 = fmaf(-q4, Y12_a, acc22_0);
      acc21_0 = fmaf(-q3, Y13_a, acc21_0);
      acc22_0 = fmaf(-q1, Y14_a, acc22_0);
      acc21_0 = fmaf(-q0, Y15_a, acc21_0);
    }
    { const float q = W7_1_a * X1_1_a;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.5345224838248488f * q;
      const float q3 = 0.15430334996209188f * q;
      const float q4 = 0.3779644730092272f * q;
      acc25_1 = fmaf(q0, Y9_a, acc25_1);
      acc24_1 = fmaf(q1, Y10_a, acc24_1);
      acc23_1 = fmaf(q2, Y11_a, acc23_1);
      acc25_1 = fmaf(q3, Y11_a, acc25_1);
      acc22_1 = fmaf(-q4, Y12_a, acc22_1);
      acc21_1 = fmaf(-q3, Y13_a, acc21_1);
      acc22_1 = fmaf(-q1, Y14_a, acc22_1);
      acc21_1 = fmaf(-q0, Y15_a, acc21_1);
    }
    { const float q = W7_0_a * X2_0_a;
      const float q0 = 0.48795003647426655f * q;
      const float q1 = 0.6172133998483676f * q;
      const float q2 = 0.6546536707079772f * q;
      acc21_0 = fmaf(q0, Y10_a, acc21_0);
      acc22_0 = fmaf(q1, Y11_a, acc22_0);
      acc23_0 = fmaf(q2, Y12_a, acc23_0);
      acc24_0 = fmaf(q1, Y13_a, acc24_0);
      acc25_0 = fmaf(q0, Y14_a, acc25_0);
    }
    { const float q = W7_1_a * X2_1_a;
      const float q0 = 0.48795003647426655f * q;
      const float q1 = 0.6172133998483676f * q;
      const float q2 = 0.6546536707079772f * q;
      acc21_1 = fmaf(q0, Y10_a, acc21_1);
      acc22_1 = fmaf(q1, Y11_a, acc22_1);
      acc23_1 = fmaf(q2, Y12_a, acc23_1);
      acc24_1 = fmaf(q1, Y13_a, acc24_1);
      acc25_1 = fmaf(q0, Y14_a, acc25_1);
    }
    { const float q = W7_0_a * X3_0_a;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.15430334996209188f * q;
      const float q3 = 0.3779644730092272f * q;
      const float q4 = 0.5345224838248488f * q;
      acc21_0 = fmaf(q0, Y9_a, acc21_0);
      acc22_0 = fmaf(q1, Y10_a, acc22_0);
      acc21_0 = fmaf(-q2, Y11_a, acc21_0);
      acc24_0 = fmaf(-q3, Y12_a, acc24_0);
      acc23_0 = fmaf(q4, Y13_a, acc23_0);
      acc25_0 = fmaf(-q2, Y13_a, acc25_0);
      acc24_0 = fmaf(q1, Y14_a, acc24_0);
      acc25_0 = fmaf(q0, Y15_a, acc25_0);
    }
    { const float q = W7_1_a * X3_1_a;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.15430334996209188f * q;
      const float q3 = 0.3779644730092272f * q;
      const float q4 = 0.5345224838248488f * q;
      acc21_1 = fmaf(q0, Y9_a, acc21_1);
      acc22_1 = fmaf(q1, Y10_a, acc22_1);
      acc21_1 = fmaf(-q2, Y11_a, acc21_1);
      acc24_1 = fmaf(-q3, Y12_a, acc24_1);
      acc23_1 = fmaf(q4, Y13_a, acc23_1);
      acc25_1 = fmaf(-q2, Y13_a, acc25_1);
      acc24_1 = fmaf(q1, Y14_a, acc24_1);
      acc25_1 = fmaf(q0, Y15_a, acc25_1);
    }
    { const float q = W8_0_a * X0_0_a;
      acc26_0 = fmaf(q, Y9_a, acc26_0);
      acc27_0 = fmaf(q, Y10_a, acc27_0);
      acc28_0 = fmaf(q, Y11_a, acc28_0);
      acc29_0 = fmaf(q, Y12_a, acc29_0);
      acc30_0 = fmaf(q, Y13_a, acc30_0);
      acc31_0 = fmaf(q, Y14_a, acc31_0);
      acc32_0 = fmaf(q, Y15_a, acc32_0);
    }
    { const float q = W8_1_a * X0_1_a;
      acc26_1 = fmaf(q, Y9_a, acc26_1);
      acc27_1 = fmaf(q, Y10_a, acc27_1);
      acc28_1 = fmaf(q, Y11_a, acc28_1);
      acc29_1 = fmaf(q, Y12_a, acc29_1);
      acc30_1 = fmaf(q, Y13_a, acc30_1);
      acc31_1 = fmaf(q, Y14_a, acc31_1);
      acc32_1 = fmaf(q, Y15_a, acc32_1);
    }
    { const float q = W9_0_a * X1_0_a;
      const float q0 = 0.18257418583505539f * q;
      const float q1 = 0.7071067811865476f * q;
      const float q2 = 0.447213595499958f * q;
      const float q3 = 0.5773502691896256f * q;
      const float q4 = 0.632455532033676f * q;
      acc37_0 = fmaf(q0, Y4_a, acc37_0);
      acc39_0 = fmaf(q1, Y4_a, acc39_0);
      acc36_0 = fmaf(q2, Y5_a, acc36_0);
      acc38_0 = fmaf(q3, Y5_a, acc38_0);
      acc35_0 = fmaf(-q4, Y6_a, acc35_0);
      acc34_0 = fmaf(-q3, Y7_a, acc34_0);
      acc33_0 = fmaf(-q1, Y8_a, acc33_0);
      acc35_0 = fmaf(-q0, Y8_a, acc35_0);
    }
    { const float q = W9_1_a * X1_1_a;
      const float q0 = 0.18257418583505539f * q;
      const float q1 = 0.7071067811865476f * q;
      const float q2 = 0.447213595499958f * q;
      const float q3 = 0.5773502691896256f * q;
      const float q4 = 0.632455532033676f * q;
      acc37_1 = fmaf(q0, Y4_a, acc37_1);
      acc39_1 = fmaf(q1, Y4_a, acc39_1);
      acc36_1 = fmaf(q2, Y5_a, acc36_1);
      acc38_1 = fmaf(q3, Y5_a, acc38_1);
      acc35_1 = fmaf(-q4, Y6_a, acc35_1);
      acc34_1 = fmaf(-q3, Y7_a, acc34_1);
      acc33_1 = fmaf(-q1, Y8_a, acc33_1);
      acc35_1 = fmaf(-q0, Y8_a, acc35_1);
    }
    { const float q = W9_0_a * X2_0_a;
      const float q0 = 0.5773502691896258f * q;
      const float q1 = 0.7302967433402215f * q;
      const float q2 = 0.7745966692414836f * q;
      acc34_0 = fmaf(-q0, Y4_a, acc34_0);
      acc35_0 = fmaf(-q1, Y5_a, acc35_0);
      acc36_0 = fmaf(-q2, Y6_a, acc36_0);
      acc37_0 = fmaf(-q1, Y7_a, acc37_0);
      acc38_0 = fmaf(-q0, Y8_a, acc38_0);
    }
    { const float q = W9_1_a * X2_1_a;
      const float q0 = 0.5773502691896258f * q;
      const float q1 = 0.7302967433402215f * q;
      const float q2 = 0.7745966692414836f * q;
      acc34_1 = fmaf(-q0, Y4_a, acc34_1);
      acc35_1 = fmaf(-q1, Y5_a, acc35_1);
      acc36_1 = fmaf(-q2, Y6_a, acc36_1);
      acc37_1 = fmaf(-q1, Y7_a, acc37_1);
      acc38_1 = fmaf(-q0, Y8_a, acc38_1);
    }
    { const float q = W9_0_a * X3_0_a;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.18257418583505539f * q;
      const float q2 = 0.5773502691896256f * q;
      const float q3 = 0.632455532033676f * q;
      const float q4 = 0.447213595499958f * q;
      acc33_0 = fmaf(-q0, Y4_a, acc33_0);
      acc35_0 = fmaf(q1, Y4_a, acc35_0);
      acc34_0 = fmaf(-q2, Y5_a, acc34_0);
      acc37_0 = fmaf(-q3, Y6_a, acc37_0);
      acc36_0 = fmaf(q4, Y7_a, acc36_0);
      acc38_0 = fmaf(-q2, Y7_a, acc38_0);
      acc37_0 = fmaf(q1, Y8_a, acc37_0);
      acc39_0 = fmaf(-q0, Y8_a, acc39_0);
    }
    { const float q = W9_1_a * X3_1_a;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.18257418583505539f * q;
      const float q2 = 0.5773502691896256f * q;
      const float q3 = 0.632455532033676f * q;
      const float q4 = 0.447213595499958f * q;
      acc33_1 = fmaf(-q0, Y4_a, acc33_1);
      acc35_1 = fmaf(q1, Y4_a, acc35_1);
      acc34_1 = fmaf(-q2, Y5_a, acc34_1);
      acc37_1 = fmaf(-q3, Y6_a, acc37_1);
      acc36_1 = fmaf(q4, Y7_a, acc36_1);
      acc38_1 = fmaf(-q2, Y7_a, acc38_1);
      acc37_1 = fmaf(q1, Y8_a, acc37_1);
      acc39_1 = fmaf(-q0, Y8_a, acc39_1);
    }
    if (two) {
    { const float q = W0_0_b * X0_0_b;
      acc0_0 = fmaf(q, Y0_b, acc0_0);
    }
    { const float q = W0_1_b * X0_1_b;
      acc0_1 = fmaf(q, Y0_b, acc0_1);
    }
    { const float q = W1_0_b * X1_0_b;
      const float q0 = 0.5773502691896257f * q;
      acc1_0 = fmaf(q0, Y1_b, acc1_0);
    }
    { const float q = W1_1_b * X1_1_b;
      const float q0 = 0.5773502691896257f * q;
      acc1_1 = fmaf(q0, Y1_b, acc1_1);
    }
    { const float q = W1_0_b * X2_0_b;
      const float q0 = 0.5773502691896258f * q;
      acc1_0 = fmaf(q0, Y2_b, acc1_0);
    }
    { const float q = W1_1_b * X2_1_b;
      const float q0 = 0.5773502691896258f * q;
      acc1_1 = fmaf(q0, Y2_b, acc1_1);
    }
    { const float q = W1_0_b * X3_0_b;
      const float q0 = 0.5773502691896257f * q;
      acc1_0 = fmaf(q0, Y3_b, acc1_0);
    }
    { const float q = W1_1_b * X3_1_b;
      const float q0 = 0.5773502691896257f * q;
      acc1_1 = fmaf(q0, Y3_b, acc1_1);
    }
    { const float q = W2_0_b * X0_0_b;
      acc2_0 = fmaf(q, Y1_b, acc2_0);
      acc3_0 = fmaf(q, Y2_b, acc3_0);
      acc4_0 = fmaf(q, Y3_b, acc4_0);
    }
    { const float q = W2_1_b * X0_1_b;
      acc2_1 = fmaf(q, Y1_b, acc2_1);
      acc3_1 = fmaf(q, Y2_b, acc3_1);
      acc4_1 = fmaf(q, Y3_b, acc4_1);
    }
    { const float q = W3_0_b * X1_0_b;
      acc5_0 = fmaf(q, Y0_b, acc5_0);
    }
    { const float q = W3_1_b * X1_1_b;
      acc5_1 = fmaf(q, Y0_b, acc5_1);
    }
    { const float q = W3_0_b * X2_0_b;
      acc6_0 = fmaf(q, Y0_b, acc6_0);
    }
    { const float q = W3_1_b * X2_1_b;
      acc6_1 = fmaf(q, Y0_b, acc6_1);
    }
    { const float q = W3_0_b * X3_0_b;
      acc7_0 = fmaf(q, Y0_b, acc7_0);
    }
    { const float q = W3_1_b * X3_1_b;
      acc7_1 = fmaf(q, Y0_b, acc7_1);
    }
    { const float q = W4_0_b * X1_0_b;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc10_0 = fmaf(q0, Y4_b, acc10_0);
      acc9_0 = fmaf(q0, Y5_b, acc9_0);
      acc8_0 = fmaf(-q1, Y6_b, acc8_0);
      acc8_0 = fmaf(-q0, Y8_b, acc8_0);
    }
    { const float q = W4_1_b * X1_1_b;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc10_1 = fmaf(q0, Y4_b, acc10_1);
      acc9_1 = fmaf(q0, Y5_b, acc9_1);
      acc8_1 = fmaf(-q1, Y6_b, acc8_1);
      acc8_1 = fmaf(-q0, Y8_b, acc8_1);
    }
    { const float q = W4_0_b * X2_0_b;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.632455532033676f * q;
      acc8_0 = fmaf(q0, Y5_b, acc8_0);
      acc9_0 = fmaf(q1, Y6_b, acc9_0);
      acc10_0 = fmaf(q0, Y7_b, acc10_0);
    }
    { const float q = W4_1_b * X2_1_b;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.632455532033676f * q;
      acc8_1 = fmaf(q0, Y5_b, acc8_1);
      acc9_1 = fmaf(q1, Y6_b, acc9_1);
      acc10_1 = fmaf(q0, Y7_b, acc10_1);
    }
    { const float q = W4_0_b * X3_0_b;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc8_0 = fmaf(q0, Y4_b, acc8_0);
      acc10_0 = fmaf(-q1, Y6_b, acc10_0);
      acc9_0 = fmaf(q0, Y7_b, acc9_0);
      acc10_0 = fmaf(q0, Y8_b, acc10_0);
    }
    { const float q = W4_1_b * X3_1_b;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc8_1 = fmaf(q0, Y4_b, acc8_1);
      acc10_1 = fmaf(-q1, Y6_b, acc10_1);
      acc9_1 = fmaf(q0, Y7_b, acc9_1);
      acc10_1 = fmaf(q0, Y8_b, acc10_1);
    }
    { const float q = W5_0_b * X0_0_b;
      acc11_0 = fmaf(q, Y4_b, acc11_0);
      acc12_0 = fmaf(q, Y5_b, acc12_0);
      acc13_0 = fmaf(q, Y6_b, acc13_0);
      acc14_0 = fmaf(q, Y7_b, acc14_0);
      acc15_0 = fmaf(q, Y8_b, acc15_0);
    }
    { const float q = W5_1_b * X0_1_b;
      acc11_1 = fmaf(q, Y4_b, acc11_1);
      acc12_1 = fmaf(q, Y5_b, acc12_1);
      acc13_1 = fmaf(q, Y6_b, acc13_1);
      acc14_1 = fmaf(q, Y7_b, acc14_1);
      acc15_1 = fmaf(q, Y8_b, acc15_1);
    }
    { const float q = W6_0_b * X1_0_b;
      const float q0 = 0.408248290463863f * q;
      const float q1 = 0.7071067811865475f * q;
      acc18_0 = fmaf(q0, Y1_b, acc18_0);
      acc20_0 = fmaf(q1, Y1_b, acc20_0);
      acc17_0 = fmaf(-q1, Y2_b, acc17_0);
      acc16_0 = fmaf(-q1, Y3_b, acc16_0);
    }
    { const float q = W6_1_b * X1_1_b;
      const float q0 = 0.408248290463863f * q;
      const float q1 = 0.7071067811865475f * q;
      acc18_1 = fmaf(q0, Y1_b, acc18_1);
      acc20_1 = fmaf(q1, Y1_b, acc20_1);
      acc17_1 = fmaf(-q1, Y2_b, acc17_1);
      acc16_1 = fmaf(-q1, Y3_b, acc16_1);
    }
    { const float q = W6_0_b * X2_0_b;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.8164965809277261f * q;
      acc17_0 = fmaf(-q0, Y1_b, acc17_0);
      acc18_0 = fmaf(-q1, Y2_b, acc18_0);
      acc19_0 = fmaf(-q0, Y3_b, acc19_0);
    }
    { const float q = W6_1_b * X2_1_b;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.8164965809277261f * q;
      acc17_1 = fmaf(-q0, Y1_b, acc17_1);
      acc18_1 = fmaf(-q1, Y2_b, acc18_1);
      acc19_1 = fmaf(-q0, Y3_b, acc19_1);
    }
    { const float q = W6_0_b * X3_0_b;
      const float q0 = 0.7071067811865475f * q;
      const float q1 = 0.408248290463863f * q;
      acc16_0 = fmaf(-q0, Y1_b, acc16_0);
      acc19_0 = fmaf(-q0, Y2_b, acc19_0);
      acc18_0 = fmaf(q1, Y3_b, acc18_0);
      acc20_0 = fmaf(-q0, Y3_b, acc20_0);
    }
    { const float q = W6_1_b * X3_1_b;
      const float q0 = 0.7071067811865475f * q;
      const float q1 = 0.408248290463863f * q;
      acc16_1 = fmaf(-q0, Y1_b, acc16_1);
      acc19_1 = fmaf(-q0, Y2_b, acc19_1);
      acc18_1 = fmaf(q1, Y3_b, acc18_1);
      acc20_1 = fmaf(-q0, Y3_b, acc20_1);
    }
    { const float q = W7_0_b * X1_0_b;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.5345224838248488f * q;
      const float q3 = 0.15430334996209188f * q;
      const float q4 = 0.3779644730092272f * q;
      acc25_0 = fmaf(q0, Y9_b, acc25_0);
      acc24_0 = fmaf(q1, Y10_b, acc24_0);
      acc23_0 = fmaf(q2, Y11_b, acc23_0);
      acc25_0 = fmaf(q3, Y11_b, acc25_0);
      acc22_0 = fmaf(-q4, Y12_b, acc22_0);
      acc21_0 = fmaf(-q3, Y13_b, acc21_0);
      acc22_0 = fmaf(-q1, Y14_b, acc22_0);
      acc21_0 = fmaf(-q0, Y15_b, acc21_0);
    }
    { const float q = W7_1_b * X1_1_b;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.5345224838248488f * q;
      const float q3 = 0.15430334996209188f * q;
      const float q4 = 0.3779644730092272f * q;
      acc25_1 = fmaf(q0, Y9_b, acc25_1);
      acc24_1 = fmaf(q1, Y10_b, acc24_1);
      acc23_1 = fmaf(q2, Y11_b, acc23_1);
      acc25_1 = fmaf(q3, Y11_b, acc25_1);
      acc22_1 = fmaf(-q4, Y12_b, acc22_1);
      acc21_1 = fmaf(-q3, Y13_b, acc21_1);
      acc22_1 = fmaf(-q1, Y14_b, acc22_1);
      acc21_1 = fmaf(-q0, Y15_b, acc21_1);
    }
    { const float q = W7_0_b * X2_0_b;
      const float q0 = 0.48795003647426655f * q;
      const float q1 = 0.6172133998483676f * q;
      const float q2 = 0.6546536707079772f * q;
      acc21_0 = fmaf(q0, Y10_b, acc21_0);
      acc22_0 = fmaf(q1, Y11_b, acc22_0);
      acc23_0 = fmaf(q2, Y12_b, acc23_0);
      acc24_0 = fmaf(q1, Y13_b, acc24_0);
      acc25_0 = fmaf(q0, Y14_b, acc25_0);
    }
    { const float q = W7_1_b * X2_1_b;
      const float q0 = 0.48795003647426655f * q;
      const float q1 = 0.6172133998483676f * q;
      const float q2 = 0.6546536707079772f * q;
      acc21_1 = fmaf(q0, Y10_b, acc21_1);
      acc22_1 = fmaf(q1, Y11_b, acc22_1);
      acc23_1 = fmaf(q2, Y12_b, acc23_1);
      acc24_1 = fmaf(q1, Y13_b, acc24_1);
      acc25_1 = fmaf(q0, Y14_b, acc25_1);
    }
    { const float q = W7_0_b * X3_0_b;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.15430334996209188f * q;
      const float q3 = 0.3779644730092272f * q;
      const float q4 = 0.5345224838248488f * q;
      acc21_0 = fmaf(q0, Y9_b, acc21_0);
      acc22_0 = fmaf(q1, Y10_b, acc22_0);
      acc21_0 = fmaf(-q2, Y11_b, acc21_0);
      acc24_0 = fmaf(-q3, Y12_b, acc24_0);
      acc23_0 = fmaf(q4, Y13_b, acc23_0);
      acc25_0 = fmaf(-q2, Y13_b, acc25_0);
      acc24_0 = fmaf(q1, Y14_b, acc24_0);
      acc25_0 = fmaf(q0, Y15_b, acc25_0);
    }
    { const float q = W7_1_b * X3_1_b;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.15430334996209188f * q;
      const float q3 = 0.3779644730092272f * q;
      const float q4 = 0.5345224838248488f * q;
      acc21_1 = fmaf(q0, Y9_b, acc21_1);
      acc22_1 = fmaf(q1, Y10_b, acc22_1);
      acc21_1 = fmaf(-q2, Y11_b, acc21_1);
      acc24_1 = fmaf(-q3, Y12_b, acc24_1);
      acc23_1 = fmaf(q4, Y13_b, acc23_1);
      acc25_1 = fmaf(-q2, Y13_b, acc25_1);
      acc24_1 = fmaf(q1, Y14_b, acc24_1);
      acc25_1 = fmaf(q0, Y15_b, acc25_1);
    }
    { const float q = W8_0_b * X0_0_b;
      acc26_0 = fmaf(q, Y9_b, acc26_0);
      acc27_0 = fmaf(q, Y10_b, acc27_0);
      acc28_0 = fmaf(q, Y11_b, acc28_0);
      acc29_0 = fmaf(q, Y12_b, acc29_0);
      acc30_0 = fmaf(q, Y13_b, acc30_0);
      acc31_0 = fmaf(q, Y14_b, acc31_0);
      acc32_0 = fmaf(q, Y15_b, acc32_0);
    }
    { const float q = W8_1_b * X0_1_b;
      acc26_1 = fmaf(q, Y9_b, acc26_1);
      acc27_1 = fmaf(q, Y10_b, acc27_1);
      acc28_1 = fmaf(q, Y11_b, acc28_1);
      acc29_1 = fmaf(q, Y12_b, acc29_1);
      acc30_1 = fmaf(q, Y13_b, acc30_1);
      acc31_1 = fmaf(q, Y14_b, acc31_1);
      acc32_1 = fmaf(q, Y15_b, acc32_1);
    }
    { const float q = W9_0_b * X1_0_b;
      const float q0 = 0.18257418583505539f * q;
      const float q1 = 0.7071067811865476f * q;
      const float q2 = 0.447213595499958f * q;
      const float q3 = 0.5773502691896256f * q;
      const float q4 = 0.632455532033676f * q;
      acc37_0 = fmaf(q0, Y4_b, acc37_0);
      acc39_0 = fmaf(q1, Y4_b, acc39_0);
      acc36_0 = fmaf(q2, Y5_b, acc36_0);
      acc38_0 = fmaf(q3, Y5_b, acc38_0);
      acc35_0 = fmaf(-q4, Y6_b, acc35_0);
      acc34_0 = fmaf(-q3, Y7_b, acc34_0);
      acc33_0 = fmaf(-q1, Y8_b, acc33_0);
      acc35_0 = fmaf(-q0, Y8_b, acc35_0);
    }
    { const float q = W9_1_b * X1_1_b;
      const float q0 = 0.18257418583505539f * q;
      const float q1 = 0.7071067811865476f * q;
      const float q2 = 0.447213595499958f * q;
      const float q3 = 0.5773502691896256f * q;
      const float q4 = 0.632455532033676f * q;
      acc37_1 = fmaf(q0, Y4_b, acc37_1);
      acc39_1 = fmaf(q1, Y4_b, acc39_1);
      acc36_1 = fmaf(q2, Y5_b, acc36_1);
      acc38_1 = fmaf(q3, Y5_b, acc38_1);
      acc35_1 = fmaf(-q4, Y6_b, acc35_1);
      acc34_1 = fmaf(-q3, Y7_b, acc34_1);
      acc33_1 = fmaf(-q1, Y8_b, acc33_1);
      acc35_1 = fmaf(-q0, Y8_b, acc35_1);
    }
    { const float q = W9_0_b * X2_0_b;
      const float q0 = 0.5773502691896258f * q;
      const float q1 = 0.7302967433402215f * q;
      const float q2 = 0.7745966692414836f * q;
      acc34_0 = fmaf(-q0, Y4_b, acc34_0);
      acc35_0 = fmaf(-q1, Y5_b, acc35_0);
      acc36_0 = fmaf(-q2, Y6_b, acc36_0);
      acc37_0 = fmaf(-q1, Y7_b, acc37_0);
      acc38_0 = fmaf(-q0, Y8_b, acc38_0);
    }
    { const float q = W9_1_b * X2_1_b;
      const float q0 = 0.5773502691896258f * q;
      const float q1 = 0.7302967433402215f * q;
      const float q2 = 0.7745966692414836f * q;
      acc34_1 = fmaf(-q0, Y4_b, acc34_1);
      acc35_1 = fmaf(-q1, Y5_b, acc35_1);
      acc36_1 = fmaf(-q2, Y6_b, acc36_1);
      acc37_1 = fmaf(-q1, Y7_b, acc37_1);
      acc38_1 = fmaf(-q0, Y8_b, acc38_1);
    }
    { const float q = W9_0_b * X3_0_b;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.18257418583505539f * q;
      const float q2 = 0.5773502691896256f * q;
      const float q3 = 0.632455532033676f * q;
      const float q4 = 0.447213595499958f * q;
      acc33_0 = fmaf(-q0, Y4_b, acc33_0);
      acc35_0 = fmaf(q1, Y4_b, acc35_0);
      acc34_0 = fmaf(-q2, Y5_b, acc34_0);
      acc37_0 = fmaf(-q3, Y6_b, acc37_0);
      acc36_0 = fmaf(q4, Y7_b, acc36_0);
      acc38_0 = fmaf(-q2, Y7_b, acc38_0);
      acc37_0 = fmaf(q1, Y8_b, acc37_0);
      acc39_0 = fmaf(-q0, Y8_b, acc39_0);
    }
    { const float q = W9_1_b * X3_1_b;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.18257418583505539f * q;
      const float q2 = 0.5773502691896256f * q;
      const float q3 = 0.632455532033676f * q;
      const float q4 = 0.447213595499958f * q;
      acc33_1 = fmaf(-q0, Y4_b, acc33_1);
      acc35_1 = fmaf(q1, Y4_b, acc35_1);
      acc34_1 = fmaf(-q2, Y5_b, acc34_1);
      acc37_1 = fmaf(-q3, Y6_b, acc37_1);
      acc36_1 = fmaf(q4, Y7_b, acc36_1);
      acc38_1 = fmaf(-q2, Y7_b, acc38_1);
      acc37_1 = fmaf(q1, Y8_b, acc37_1);
      acc39_1 = fmaf(-q0, Y8_b, acc39_1);
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
  op[2048] = acc16_0;
  op[2112] = acc16_1;
  op[2176] = acc17_0;
  op[2240] = acc17_1;
  op[2304] = acc18_0;
  op[2368] = acc18_1;
  op[2432] = acc19_0;
  op[2496] = acc19_1;
  op[2560] = acc20_0;
  op[2624] = acc20_1;
  op[2688] = acc21_0;
  op[2752] = acc21_1;
  op[2816] = acc22_0;
  op[2880] = acc22_1;
  op[2944] = acc23_0;
  op[3008] = acc23_1;
  op[3072] = acc24_0;
  op[3136] = acc24_1;
  op[3200] = acc25_0;
  op[3264] = acc25_1;
  op[3328] = acc26_0;
  op[3392] = acc26_1;
  op[3456] = acc27_0;
  op[3520] = acc27_1;
  op[3584] = acc28_0;
  op[3648] = acc28_1;
  op[3712] = acc29_0;
  op[3776] = acc29_1;
  op[3840] = acc30_0;
  op[3904] = acc30_1;
  op[3968] = acc31_0;
  op[4032] = acc31_1;
  op[4096] = acc32_0;
  op[4160] = acc32_1;
  op[4224] = acc33_0;
  op[4288] = acc33_1;
  op[4352] = acc34_0;
  op[4416] = acc34_1;
  op[4480] = acc35_0;
  op[4544] = acc35_1;
  op[4608] = acc36_0;
  op[4672] = acc36_1;
  op[4736] = acc37_0;
  op[4800] = acc37_1;
  op[4864] = acc38_0;
  op[4928] = acc38_1;
  op[4992] = acc39_0;
  op[5056] = acc39_1;
}

extern "C" __global__ void __launch_bounds__(256)
mm_tpw_l2_fwd_shared_kernel(const int* __restrict__ rowptr, int nR, const int* __restrict__ eid,
    const int* __restrict__ send, const float* __restrict__ Y, long y_stride, const float* __restrict__ W,
    long w_stride, const float* __restrict__ X, long x_stride, float* __restrict__ out, long out_stride) {
  __shared__ float red[80 * 64];   // one wave's sums [accumulator][lane]
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
  float acc16_0 = 0.f;
  float acc16_1 = 0.f;
  float acc17_0 = 0.f;
  float acc17_1 = 0.f;
  float acc18_0 = 0.f;
  float acc18_1 = 0.f;
  float acc19_0 = 0.f;
  float acc19_1 = 0.f;
  float acc20_0 = 0.f;
  float acc20_1 = 0.f;
  float acc21_0 = 0.f;
  float acc21_1 = 0.f;
  float acc22_0 = 0.f;
  float acc22_1 = 0.f;
  float acc23_0 = 0.f;
  float acc23_1 = 0.f;
  float acc24_0 = 0.f;
  float acc24_1 = 0.f;
  float acc25_0 = 0.f;
  float acc25_1 = 0.f;
  float acc26_0 = 0.f;
  float acc26_1 = 0.f;
  float acc27_0 = 0.f;
  float acc27_1 = 0.f;
  float acc28_0 = 0.f;
  float acc28_1 = 0.f;
  float acc29_0 = 0.f;
  float acc29_1 = 0.f;
  float acc30_0 = 0.f;
  float acc30_1 = 0.f;
  float acc31_0 = 0.f;
  float acc31_1 = 0.f;
  float acc32_0 = 0.f;
  float acc32_1 = 0.f;
  float acc33_0 = 0.f;
  float acc33_1 = 0.f;
  float acc34_0 = 0.f;
  float acc34_1 = 0.f;
  float acc35_0 = 0.f;
  float acc35_1 = 0.f;
  float acc36_0 = 0.f;
  float acc36_1 = 0.f;
  float acc37_0 = 0.f;
  float acc37_1 = 0.f;
  float acc38_0 = 0.f;
  float acc38_1 = 0.f;
  float acc39_0 = 0.f;
  float acc39_1 = 0.f;
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
    const float W4_0_a = wpa[512];
    const float W4_1_a = wpa[576];
    const float W5_0_a = wpa[640];
    const float W5_1_a = wpa[704];
    const float W6_0_a = wpa[768];
    const float W6_1_a = wpa[832];
    const float W7_0_a = wpa[896];
    const float W7_1_a = wpa[960];
    const float W8_0_a = wpa[1024];
    const float W8_1_a = wpa[1088];
    const float W9_0_a = wpa[1152];
    const float W9_1_a = wpa[1216];
    const float* __restrict__ xpa = X + (size_t)sa * x_stride + c;
    const float X0_0_a = xpa[0];
    const float X0_1_a = xpa[64];
    const float X1_0_a = xpa[128];
    const float X1_1_a = xpa[192];
    const float X2_0_a = xpa[256];
    const float X2_1_a = xpa[320];
    const float X3_0_a = xpa[384];
    const float X3_1_a = xpa[448];
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
    const float W4_0_b = wpb[512];
    const float W4_1_b = wpb[576];
    const float W5_0_b = wpb[640];
    const float W5_1_b = wpb[704];
    const float W6_0_b = wpb[768];
    const float W6_1_b = wpb[832];
    const float W7_0_b = wpb[896];
    const float W7_1_b = wpb[960];
    const float W8_0_b = wpb[1024];
    const float W8_1_b = wpb[1088];
    const float W9_0_b = wpb[1152];
    const float W9_1_b = wpb[1216];
    const float* __restrict__ xpb = X + (size_t)sb * x_stride + c;
    const float X0_0_b = xpb[0];
    const float X0_1_b = xpb[64];
    const float X1_0_b = xpb[128];
    const float X1_1_b = xpb[192];
    const float X2_0_b = xpb[256];
    const float X2_1_b = xpb[320];
    const float X3_0_b = xpb[384];
    const float X3_1_b = xpb[448];
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
    { const float q = W1_0_a * X1_0_a;
      const float q0 = 0.5773502691896257f * q;
      acc1_0 = fmaf(q0, Y1_a, acc1_0);
    }
    { const float q = W1_1_a * X1_1_a;
      const float q0 = 0.5773502691896257f * q;
      acc1_1 = fmaf(q0, Y1_a, acc1_1);
    }
    { const float q = W1_0_a * X2_0_a;
      const float q0 = 0.5773502691896258f * q;
      acc1_0 = fmaf(q0, Y2_a, acc1_0);
    }
    { const float q = W1_1_a * X2_1_a;
      const float q0 = 0.5773502691896258f * q;
      acc1_1 = fmaf(q0, Y2_a, acc1_1);
    }
    { const float q = W1_0_a * X3_0_a;
      const float q0 = 0.5773502691896257f * q;
      acc1_0 = fmaf(q0, Y3_a, acc1_0);
    }
    { const float q = W1_1_a * X3_1_a;
      const float q0 = 0.5773502691896257f * q;
      acc1_1 = fmaf(q0, Y3_a, acc1_1);
    }
    { const float q = W2_0_a * X0_0_a;
      acc2_0 = fmaf(q, Y1_a, acc2_0);
      acc3_0 = fmaf(q, Y2_a, acc3_0);
      acc4_0 = fmaf(q, Y3_a, acc4_0);
    }
    { const float q = W2_1_a * X0_1_a;
      acc2_1 = fmaf(q, Y1_a, acc2_1);
      acc3_1 = fmaf(q, Y2_a, acc3_1);
      acc4_1 = fmaf(q, Y3_a, acc4_1);
    }
    { const float q = W3_0_a * X1_0_a;
      acc5_0 = fmaf(q, Y0_a, acc5_0);
    }
    { const float q = W3_1_a * X1_1_a;
      acc5_1 = fmaf(q, Y0_a, acc5_1);
    }
    { const float q = W3_0_a * X2_0_a;
      acc6_0 = fmaf(q, Y0_a, acc6_0);
    }
    { const float q = W3_1_a * X2_1_a;
      acc6_1 = fmaf(q, Y0_a, acc6_1);
    }
    { const float q = W3_0_a * X3_0_a;
      acc7_0 = fmaf(q, Y0_a, acc7_0);
    }
    { const float q = W3_1_a * X3_1_a;
      acc7_1 = fmaf(q, Y0_a, acc7_1);
    }
    { const float q = W4_0_a * X1_0_a;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc10_0 = fmaf(q0, Y4_a, acc10_0);
      acc9_0 = fmaf(q0, Y5_a, acc9_0);
      acc8_0 = fmaf(-q1, Y6_a, acc8_0);
      acc8_0 = fmaf(-q0, Y8_a, acc8_0);
    }
    { const float q = W4_1_a * X1_1_a;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc10_1 = fmaf(q0, Y4_a, acc10_1);
      acc9_1 = fmaf(q0, Y5_a, acc9_1);
      acc8_1 = fmaf(-q1, Y6_a, acc8_1);
      acc8_1 = fmaf(-q0, Y8_a, acc8_1);
    }
    { const float q = W4_0_a * X2_0_a;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.632455532033676f * q;
      acc8_0 = fmaf(q0, Y5_a, acc8_0);
      acc9_0 = fmaf(q1, Y6_a, acc9_0);
      acc10_0 = fmaf(q0, Y7_a, acc10_0);
    }
    { const float q = W4_1_a * X2_1_a;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.632455532033676f * q;
      acc8_1 = fmaf(q0, Y5_a, acc8_1);
      acc9_1 = fmaf(q1, Y6_a, acc9_1);
      acc10_1 = fmaf(q0, Y7_a, acc10_1);
    }
    { const float q = W4_0_a * X3_0_a;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc8_0 = fmaf(q0, Y4_a, acc8_0);
      acc10_0 = fmaf(-q1, Y6_a, acc10_0);
      acc9_0 = fmaf(q0, Y7_a, acc9_0);
      acc10_0 = fmaf(q0, Y8_a, acc10_0);
    }
    { const float q = W4_1_a * X3_1_a;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc8_1 = fmaf(q0, Y4_a, acc8_1);
      acc10_1 = fmaf(-q1, Y6_a, acc10_1);
      acc9_1 = fmaf(q0, Y7_a, acc9_1);
      acc10_1 = fmaf(q0, Y8_a, acc10_1);
    }
    { const float q = W5_0_a * X0_0_a;
      acc11_0 = fmaf(q, Y4_a, acc11_0);
      acc12_0 = fmaf(q, Y5_a, acc12_0);
      acc13_0 = fmaf(q, Y6_a, acc13_0);
      acc14_0 = fmaf(q, Y7_a, acc14_0);
      acc15_0 = fmaf(q, Y8_a, acc15_0);
    }
    { const float q = W5_1_a * X0_1_a;
      acc11_1 = fmaf(q, Y4_a, acc11_1);
      acc12_1 = fmaf(q, Y5_a, acc12_1);
      acc13_1 = fmaf(q, Y6_a, acc13_1);
      acc14_1 = fmaf(q, Y7_a, acc14_1);
      acc15_1 = fmaf(q, Y8_a, acc15_1);
    }
    { const float q = W6_0_a * X1_0_a;
      const float q0 = 0.408248290463863f * q;
      const float q1 = 0.7071067811865475f * q;
      acc18_0 = fmaf(q0, Y1_a, acc18_0);
      acc20_0 = fmaf(q1, Y1_a, acc20_0);
      acc17_0 = fmaf(-q1, Y2_a, acc17_0);
      acc16_0 = fmaf(-q1, Y3_a, acc16_0);
    }
    { const float q = W6_1_a * X1_1_a;
      const float q0 = 0.408248290463863f * q;
      const float q1 = 0.7071067811865475f * q;
      acc18_1 = fmaf(q0, Y1_a, acc18_1);
      acc20_1 = fmaf(q1, Y1_a, acc20_1);
      acc17_1 = fmaf(-q1, Y2_a, acc17_1);
      acc16_1 = fmaf(-q1, Y3_a, acc16_1);
    }
    { const float q = W6_0_a * X2_0_a;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.8164965809277261f * q;
      acc17_0 = fmaf(-q0, Y1_a, acc17_0);
      acc18_0 = fmaf(-q1, Y2_a, acc18_0);
      acc19_0 = fmaf(-q0, Y3_a, acc19_0);
    }
    { const float q = W6_1_a * X2_1_a;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.8164965809277261f * q;
      acc17_1 = fmaf(-q0, Y1_a, acc17_1);
      acc18_1 = fmaf(-q1, Y2_a, acc18_1);
      acc19_1 = fmaf(-q0, Y3_a, acc19_1);
    }
    { const float q = W6_0_a * X3_0_a;
      const float q0 = 0.7071067811865475f * q;
      const float q1 = 0.408248290463863f * q;
      acc16_0 = fmaf(-q0, Y1_a, acc16_0);
      acc19_0 = fmaf(-q0, Y2_a, acc19_0);
      acc18_0 = fmaf(q1, Y3_a, acc18_0);
      acc20_0 = fmaf(-q0, Y3_a, acc20_0);
    }
    { const float q = W6_1_a * X3_1_a;
      const float q0 = 0.7071067811865475f * q;
      const float q1 = 0.408248290463863f * q;
      acc16_1 = fmaf(-q0, Y1_a, acc16_1);
      acc19_1 = fmaf(-q0, Y2_a, acc19_1);
      acc18_1 = fmaf(q1, Y3_a, acc18_1);
      acc20_1 = fmaf(-q0, Y3_a, acc20_1);
    }
    { const float q = W7_0_a * X1_0_a;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.5345224838248488f * q;
      const float q3 = 0.15430334996209188f * q;
      const float q4 = 0.3779644730092272f * q;
      acc25_0 = fmaf(q0, Y9_a, acc25_0);
      acc24_0 = fmaf(q1, Y10_a, acc24_0);
      acc23_0 = fmaf(q2, Y11_a, acc23_0);
      acc25_0 = fmaf(q3, Y11_a, acc25_0);
      acc22_0 = fmaf(-q4, Y12_a, acc22_0);
      acc21_0 = fmaf(-q3, Y13_a, acc21_0);
      acc22_0 = fmaf(-q1, Y14_a, acc22_0);
      acc21_0 = fmaf(-q0, Y15_a, acc21_0);
    }
    { const float q = W7_1_a * X1_1_a;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.5345224838248488f * q;
      const float q3 = 0.15430334996209188f * q;
      const float q4 = 0.3779644730092272f * q;
      acc25_1 = fmaf(q0, Y9_a, acc25_1);
      acc24_1 = fmaf(q1, Y10_a, acc24_1);
      acc23_1 = fmaf(q2, Y11_a, acc23_1);
      acc25_1 = fmaf(q3, Y11_a, acc25_1);
      acc22_1 = fmaf(-q4, Y12_a, acc22_1);
      acc21_1 = fmaf(-q3, Y13_a, acc21_1);
      acc22_1 = fmaf(-q1, Y14_a, acc22_1);
      acc21_1 = fmaf(-q0, Y15_a, acc21_1);
    }
    { const float q = W7_0_a * X2_0_a;
      const float q0 = 0.48795003647426655f * q;
      const float q1 = 0.6172133998483676f * q;
      const float q2 = 0.6546536707079772f * q;
      acc21_0 = fmaf(q0, Y10_a, acc21_0);
      acc22_0 = fmaf(q1, Y11_a, acc22_0);
      acc23_0 = fmaf(q2, Y12_a, acc23_0);
      acc24_0 = fmaf(q1, Y13_a, acc24_0);
      acc25_0 = fmaf(q0, Y14_a, acc25_0);
    }
    { const float q = W7_1_a * X2_1_a;
      const float q0 = 0.48795003647426655f * q;
      const float q1 = 0.6172133998483676f * q;
      const float q2 = 0.6546536707079772f * q;
      acc21_1 = fmaf(q0, Y10_a, acc21_1);
      acc22_1 = fmaf(q1, Y11_a, acc22_1);
      acc23_1 = fmaf(q2, Y12_a, acc23_1);
      acc24_1 = fmaf(q1, Y13_a, acc24_1);
      acc25_1 = fmaf(q0, Y14_a, acc25_1);
    }
    { const float q = W7_0_a * X3_0_a;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.15430334996209188f * q;
      const float q3 = 0.3779644730092272f * q;
      const float q4 = 0.5345224838248488f * q;
      acc21_0 = fmaf(q0, Y9_a, acc21_0);
      acc22_0 = fmaf(q1, Y10_a, acc22_0);
      acc21_0 = fmaf(-q2, Y11_a, acc21_0);
      acc24_0 = fmaf(-q3, Y12_a, acc24_0);
      acc23_0 = fmaf(q4, Y13_a, acc23_0);
      acc25_0 = fmaf(-q2, Y13_a, acc25_0);
      acc24_0 = fmaf(q1, Y14_a, acc24_0);
      acc25_0 = fmaf(q0, Y15_a, acc25_0);
    }
    { const float q = W7_1_a * X3_1_a;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.15430334996209188f * q;
      const float q3 = 0.3779644730092272f * q;
      const float q4 = 0.5345224838248488f * q;
      acc21_1 = fmaf(q0, Y9_a, acc21_1);
      acc22_1 = fmaf(q1, Y10_a, acc22_1);
      acc21_1 = fmaf(-q2, Y11_a, acc21_1);
      acc24_1 = fmaf(-q3, Y12_a, acc24_1);
      acc23_1 = fmaf(q4, Y13_a, acc23_1);
      acc25_1 = fmaf(-q2, Y13_a, acc25_1);
      acc24_1 = fmaf(q1, Y14_a, acc24_1);
      acc25_1 = fmaf(q0, Y15_a, acc25_1);
    }
    { const float q = W8_0_a * X0_0_a;
      acc26_0 = fmaf(q, Y9_a, acc26_0);
      acc27_0 = fmaf(q, Y10_a, acc27_0);
      acc28_0 = fmaf(q, Y11_a, acc28_0);
      acc29_0 = fmaf(q, Y12_a, acc29_0);
      acc30_0 = fmaf(q, Y13_a, acc30_0);
      acc31_0 = fmaf(q, Y14_a, acc31_0);
      acc32_0 = fmaf(q, Y15_a, acc32_0);
    }
    { const float q = W8_1_a * X0_1_a;
      acc26_1 = fmaf(q, Y9_a, acc26_1);
      acc27_1 = fmaf(q, Y10_a, acc27_1);
      acc28_1 = fmaf(q, Y11_a, acc28_1);
      acc29_1 = fmaf(q, Y12_a, acc29_1);
      acc30_1 = fmaf(q, Y13_a, acc30_1);
      acc31_1 = fmaf(q, Y14_a, acc31_1);
      acc32_1 = fmaf(q, Y15_a, acc32_1);
    }
    { const float q = W9_0_a * X1_0_a;
      const float q0 = 0.18257418583505539f * q;
      const float q1 = 0.7071067811865476f * q;
      const float q2 = 0.447213595499958f * q;
      const float q3 = 0.5773502691896256f * q;
      const float q4 = 0.632455532033676f * q;
      acc37_0 = fmaf(q0, Y4_a, acc37_0);
      acc39_0 = fmaf(q1, Y4_a, acc39_0);
      acc36_0 = fmaf(q2, Y5_a, acc36_0);
      acc38_0 = fmaf(q3, Y5_a, acc38_0);
      acc35_0 = fmaf(-q4, Y6_a, acc35_0);
      acc34_0 = fmaf(-q3, Y7_a, acc34_0);
      acc33_0 = fmaf(-q1, Y8_a, acc33_0);
      acc35_0 = fmaf(-q0, Y8_a, acc35_0);
    }
    { const float q = W9_1_a * X1_1_a;
      const float q0 = 0.18257418583505539f * q;
      const float q1 = 0.7071067811865476f * q;
      const float q2 = 0.447213595499958f * q;
      const float q3 = 0.5773502691896256f * q;
      const float q4 = 0.632455532033676f * q;
      acc37_1 = fmaf(q0, Y4_a, acc37_1);
      acc39_1 = fmaf(q1, Y4_a, acc39_1);
      acc36_1 = fmaf(q2, Y5_a, acc36_1);
      acc38_1 = fmaf(q3, Y5_a, acc38_1);
      acc35_1 = fmaf(-q4, Y6_a, acc35_1);
      acc34_1 = fmaf(-q3, Y7_a, acc34_1);
      acc33_1 = fmaf(-q1, Y8_a, acc33_1);
      acc35_1 = fmaf(-q0, Y8_a, acc35_1);
    }
    { const float q = W9_0_a * X2_0_a;
      const float q0 = 0.5773502691896258f * q;
      const float q1 = 0.7302967433402215f * q;
      const float q2 = 0.7745966692414836f * q;
      acc34_0 = fmaf(-q0, Y4_a, acc34_0);
      acc35_0 = fmaf(-q1, Y5_a, acc35_0);
      acc36_0 = fmaf(-q2, Y6_a, acc36_0);
      acc37_0 = fmaf(-q1, Y7_a, acc37_0);
      acc38_0 = fmaf(-q0, Y8_a, acc38_0);
    }
    { const float q = W9_1_a * X2_1_a;
      const float q0 = 0.5773502691896258f * q;
      const float q1 = 0.7302967433402215f * q;
      const float q2 = 0.7745966692414836f * q;
      acc34_1 = fmaf(-q0, Y4_a, acc34_1);
      acc35_1 = fmaf(-q1, Y5_a, acc35_1);
      acc36_1 = fmaf(-q2, Y6_a, acc36_1);
      acc37_1 = fmaf(-q1, Y7_a, acc37_1);
      acc38_1 = fmaf(-q0, Y8_a, acc38_1);
    }
    { const float q = W9_0_a * X3_0_a;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.18257418583505539f * q;
      const float q2 = 0.5773502691896256f * q;
      const float q3 = 0.632455532033676f * q;
      const float q4 = 0.447213595499958f * q;
      acc33_0 = fmaf(-q0, Y4_a, acc33_0);
      acc35_0 = fmaf(q1, Y4_a, acc35_0);
      acc34_0 = fmaf(-q2, Y5_a, acc34_0);
      acc37_0 = fmaf(-q3, Y6_a, acc37_0);
      acc36_0 = fmaf(q4, Y7_a, acc36_0);
      acc38_0 = fmaf(-q2, Y7_a, acc38_0);
      acc37_0 = fmaf(q1, Y8_a, acc37_0);
      acc39_0 = fmaf(-q0, Y8_a, acc39_0);
    }
    { const float q = W9_1_a * X3_1_a;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.18257418583505539f * q;
      const float q2 = 0.5773502691896256f * q;
      const float q3 = 0.632455532033676f * q;
      const float q4 = 0.447213595499958f * q;
      acc33_1 = fmaf(-q0, Y4_a, acc33_1);
      acc35_1 = fmaf(q1, Y4_a, acc35_1);
      acc34_1 = fmaf(-q2, Y5_a, acc34_1);
      acc37_1 = fmaf(-q3, Y6_a, acc37_1);
      acc36_1 = fmaf(q4, Y7_a, acc36_1);
      acc38_1 = fmaf(-q2, Y7_a, acc38_1);
      acc37_1 = fmaf(q1, Y8_a, acc37_1);
      acc39_1 = fmaf(-q0, Y8_a, acc39_1);
    }
    if (two) {
    { const float q = W0_0_b * X0_0_b;
      acc0_0 = fmaf(q, Y0_b, acc0_0);
    }
    { const float q = W0_1_b * X0_1_b;
      acc0_1 = fmaf(q, Y0_b, acc0_1);
    }
    { const float q = W1_0_b * X1_0_b;
      const float q0 = 0.5773502691896257f * q;
      acc1_0 = fmaf(q0, Y1_b, acc1_0);
    }
    { const float q = W1_1_b * X1_1_b;
      const float q0 = 0.5773502691896257f * q;
      acc1_1 = fmaf(q0, Y1_b, acc1_1);
    }
    { const float q = W1_0_b * X2_0_b;
      const float q0 = 0.5773502691896258f * q;
      acc1_0 = fmaf(q0, Y2_b, acc1_0);
    }
    { const float q = W1_1_b * X2_1_b;
      const float q0 = 0.5773502691896258f * q;
      acc1_1 = fmaf(q0, Y2_b, acc1_1);
    }
    { const float q = W1_0_b * X3_0_b;
      const float q0 = 0.5773502691896257f * q;
      acc1_0 = fmaf(q0, Y3_b, acc1_0);
    }
    { const float q = W1_1_b * X3_1_b;
      const float q0 = 0.5773502691896257f * q;
      acc1_1 = fmaf(q0, Y3_b, acc1_1);
    }
    { const float q = W2_0_b * X0_0_b;
      acc2_0 = fmaf(q, Y1_b, acc2_0);
      acc3_0 = fmaf(q, Y2_b, acc3_0);
      acc4_0 = fmaf(q, Y3_b, acc4_0);
    }
    { const float q = W2_1_b * X0_1_b;
      acc2_1 = fmaf(q, Y1_b, acc2_1);
      acc3_1 = fmaf(q, Y2_b, acc3_1);
      acc4_1 = fmaf(q, Y3_b, acc4_1);
    }
    { const float q = W3_0_b * X1_0_b;
      acc5_0 = fmaf(q, Y0_b, acc5_0);
    }
    { const float q = W3_1_b * X1_1_b;
      acc5_1 = fmaf(q, Y0_b, acc5_1);
    }
    { const float q = W3_0_b * X2_0_b;
      acc6_0 = fmaf(q, Y0_b, acc6_0);
    }
    { const float q = W3_1_b * X2_1_b;
      acc6_1 = fmaf(q, Y0_b, acc6_1);
    }
    { const float q = W3_0_b * X3_0_b;
      acc7_0 = fmaf(q, Y0_b, acc7_0);
    }
    { const float q = W3_1_b * X3_1_b;
      acc7_1 = fmaf(q, Y0_b, acc7_1);
    }
    { const float q = W4_0_b * X1_0_b;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc10_0 = fmaf(q0, Y4_b, acc10_0);
      acc9_0 = fmaf(q0, Y5_b, acc9_0);
      acc8_0 = fmaf(-q1, Y6_b, acc8_0);
      acc8_0 = fmaf(-q0, Y8_b, acc8_0);
    }
    { const float q = W4_1_b * X1_1_b;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc10_1 = fmaf(q0, Y4_b, acc10_1);
      acc9_1 = fmaf(q0, Y5_b, acc9_1);
      acc8_1 = fmaf(-q1, Y6_b, acc8_1);
      acc8_1 = fmaf(-q0, Y8_b, acc8_1);
    }
    { const float q = W4_0_b * X2_0_b;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.632455532033676f * q;
      acc8_0 = fmaf(q0, Y5_b, acc8_0);
      acc9_0 = fmaf(q1, Y6_b, acc9_0);
      acc10_0 = fmaf(q0, Y7_b, acc10_0);
    }
    { const float q = W4_1_b * X2_1_b;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.632455532033676f * q;
      acc8_1 = fmaf(q0, Y5_b, acc8_1);
      acc9_1 = fmaf(q1, Y6_b, acc9_1);
      acc10_1 = fmaf(q0, Y7_b, acc10_1);
    }
    { const float q = W4_0_b * X3_0_b;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc8_0 = fmaf(q0, Y4_b, acc8_0);
      acc10_0 = fmaf(-q1, Y6_b, acc10_0);
      acc9_0 = fmaf(q0, Y7_b, acc9_0);
      acc10_0 = fmaf(q0, Y8_b, acc10_0);
    }
    { const float q = W4_1_b * X3_1_b;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc8_1 = fmaf(q0, Y4_b, acc8_1);
      acc10_1 = fmaf(-q1, Y6_b, acc10_1);
      acc9_1 = fmaf(q0, Y7_b, acc9_1);
      acc10_1 = fmaf(q0, Y8_b, acc10_1);
    }
    { const float q = W5_0_b * X0_0_b;
      acc11_0 = fmaf(q, Y4_b, acc11_0);
      acc12_0 = fmaf(q, Y5_b, acc12_0);
      acc13_0 = fmaf(q, Y6_b, acc13_0);
      acc14_0 = fmaf(q, Y7_b, acc14_0);
      acc15_0 = fmaf(q, Y8_b, acc15_0);
    }
    { const float q = W5_1_b * X0_1_b;
      acc11_1 = fmaf(q, Y4_b, acc11_1);
      acc12_1 = fmaf(q, Y5_b, acc12_1);
      acc13_1 = fmaf(q, Y6_b, acc13_1);
      acc14_1 = fmaf(q, Y7_b, acc14_1);
      acc15_1 = fmaf(q, Y8_b, acc15_1);
    }
    { const float q = W6_0_b * X1_0_b;
      const float q0 = 0.408248290463863f * q;
      const float q1 = 0.7071067811865475f * q;
      acc18_0 = fmaf(q0, Y1_b, acc18_0);
      acc20_0 = fmaf(q1, Y1_b, acc20_0);
      acc17_0 = fmaf(-q1, Y2_b, acc17_0);
      acc16_0 = fmaf(-q1, Y3_b, acc16_0);
    }
    { const float q = W6_1_b * X1_1_b;
      const float q0 = 0.408248290463863f * q;
      const float q1 = 0.7071067811865475f * q;
      acc18_1 = fmaf(q0, Y1_b, acc18_1);
      acc20_1 = fmaf(q1, Y1_b, acc20_1);
      acc17_1 = fmaf(-q1, Y2_b, acc17_1);
      acc16_1 = fmaf(-q1, Y3_b, acc16_1);
    }
    { const float q = W6_0_b * X2_0_b;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.8164965809277261f * q;
      acc17_0 = fmaf(-q0, Y1_b, acc17_0);
      acc18_0 = fmaf(-q1, Y2_b, acc18_0);
      acc19_0 = fmaf(-q0, Y3_b, acc19_0);
    }
    { const float q = W6_1_b * X2_1_b;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.8164965809277261f * q;
      acc17_1 = fmaf(-q0, Y1_b, acc17_1);
      acc18_1 = fmaf(-q1, Y2_b, acc18_1);
      acc19_1 = fmaf(-q0, Y3_b, acc19_1);
    }
    { const float q = W6_0_b * X3_0_b;
      const float q0 = 0.7071067811865475f * q;
      const float q1 = 0.408248290463863f * q;
      acc16_0 = fmaf(-q0, Y1_b, acc16_0);
      acc19_0 = fmaf(-q0, Y2_b, acc19_0);
      acc18_0 = fmaf(q1, Y3_b, acc18_0);
      acc20_0 = fmaf(-q0, Y3_b, acc20_0);
    }
    { const float q = W6_1_b * X3_1_b;
      const float q0 = 0.7071067811865475f * q;
      const float q1 = 0.408248290463863f * q;
      acc16_1 = fmaf(-q0, Y1_b, acc16_1);
      acc19_1 = fmaf(-q0, Y2_b, acc19_1);
      acc18_1 = fmaf(q1, Y3_b, acc18_1);
      acc20_1 = fmaf(-q0, Y3_b, acc20_1);
    }
    { const float q = W7_0_b * X1_0_b;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.5345224838248488f * q;
      const float q3 = 0.15430334996209188f * q;
      const float q4 = 0.3779644730092272f * q;
      acc25_0 = fmaf(q0, Y9_b, acc25_0);
      acc24_0 = fmaf(q1, Y10_b, acc24_0);
      acc23_0 = fmaf(q2, Y11_b, acc23_0);
      acc25_0 = fmaf(q3, Y11_b, acc25_0);
      acc22_0 = fmaf(-q4, Y12_b, acc22_0);
      acc21_0 = fmaf(-q3, Y13_b, acc21_0);
      acc22_0 = fmaf(-q1, Y14_b, acc22_0);
      acc21_0 = fmaf(-q0, Y15_b, acc21_0);
    }
    { const float q = W7_1_b * X1_1_b;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.5345224838248488f * q;
      const float q3 = 0.15430334996209188f * q;
      const float q4 = 0.3779644730092272f * q;
      acc25_1 = fmaf(q0, Y9_b, acc25_1);
      acc24_1 = fmaf(q1, Y10_b, acc24_1);
      acc23_1 = fmaf(q2, Y11_b, acc23_1);
      acc25_1 = fmaf(q3, Y11_b, acc25_1);
      acc22_1 = fmaf(-q4, Y12_b, acc22_1);
      acc21_1 = fmaf(-q3, Y13_b, acc21_1);
      acc22_1 = fmaf(-q1, Y14_b, acc22_1);
      acc21_1 = fmaf(-q0, Y15_b, acc21_1);
    }
    { const float q = W7_0_b * X2_0_b;
      const float q0 = 0.48795003647426655f * q;
      const float q1 = 0.6172133998483676f * q;
      const float q2 = 0.6546536707079772f * q;
      acc21_0 = fmaf(q0, Y10_b, acc21_0);
      acc22_0 = fmaf(q1, Y11_b, acc22_0);
      acc23_0 = fmaf(q2, Y12_b, acc23_0);
      acc24_0 = fmaf(q1, Y13_b, acc24_0);
      acc25_0 = fmaf(q0, Y14_b, acc25_0);
    }
    { const float q = W7_1_b * X2_1_b;
      const float q0 = 0.48795003647426655f * q;
      const float q1 = 0.6172133998483676f * q;
      const float q2 = 0.6546536707079772f * q;
      acc21_1 = fmaf(q0, Y10_b, acc21_1);
      acc22_1 = fmaf(q1, Y11_b, acc22_1);
      acc23_1 = fmaf(q2, Y12_b, acc23_1);
      acc24_1 = fmaf(q1, Y13_b, acc24_1);
      acc25_1 = fmaf(q0, Y14_b, acc25_1);
    }
    { const float q = W7_0_b * X3_0_b;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.15430334996209188f * q;
      const float q3 = 0.3779644730092272f * q;
      const float q4 = 0.5345224838248488f * q;
      acc21_0 = fmaf(q0, Y9_b, acc21_0);
      acc22_0 = fmaf(q1, Y10_b, acc22_0);
      acc21_0 = fmaf(-q2, Y11_b, acc21_0);
      acc24_0 = fmaf(-q3, Y12_b, acc24_0);
      acc23_0 = fmaf(q4, Y13_b, acc23_0);
      acc25_0 = fmaf(-q2, Y13_b, acc25_0);
      acc24_0 = fmaf(q1, Y14_b, acc24_0);
      acc25_0 = fmaf(q0, Y15_b, acc25_0);
    }
    { const float q = W7_1_b * X3_1_b;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.15430334996209188f * q;
      const float q3 = 0.3779644730092272f * q;
      const float q4 = 0.5345224838248488f * q;
      acc21_1 = fmaf(q0, Y9_b, acc21_1);
      acc22_1 = fmaf(q1, Y10_b, acc22_1);
      acc21_1 = fmaf(-q2, Y11_b, acc21_1);
      acc24_1 = fmaf(-q3, Y12_b, acc24_1);
      acc23_1 = fmaf(q4, Y13_b, acc23_1);
      acc25_1 = fmaf(-q2, Y13_b, acc25_1);
      acc24_1 = fmaf(q1, Y14_b, acc24_1);
      acc25_1 = fmaf(q0, Y15_b, acc25_1);
    }
    { const float q = W8_0_b * X0_0_b;
      acc26_0 = fmaf(q, Y9_b, acc26_0);
      acc27_0 = fmaf(q, Y10_b, acc27_0);
      acc28_0 = fmaf(q, Y11_b, acc28_0);
      acc29_0 = fmaf(q, Y12_b, acc29_0);
      acc30_0 = fmaf(q, Y13_b, acc30_0);
      acc31_0 = fmaf(q, Y14_b, acc31_0);
      acc32_0 = fmaf(q, Y15_b, acc32_0);
    }
    { const float q = W8_1_b * X0_1_b;
      acc26_1 = fmaf(q, Y9_b, acc26_1);
      acc27_1 = fmaf(q, Y10_b, acc27_1);
      acc28_1 = fmaf(q, Y11_b, acc28_1);
      acc29_1 = fmaf(q, Y12_b, acc29_1);
      acc30_1 = fmaf(q, Y13_b, acc30_1);
      acc31_1 = fmaf(q, Y14_b, acc31_1);
      acc32_1 = fmaf(q, Y15_b, acc32_1);
    }
    { const float q = W9_0_b * X1_0_b;
      const float q0 = 0.18257418583505539f * q;
      const float q1 = 0.7071067811865476f * q;
      const float q2 = 0.447213595499958f * q;
      const float q3 = 0.5773502691896256f * q;
      const float q4 = 0.632455532033676f * q;
      acc37_0 = fmaf(q0, Y4_b, acc37_0);
      acc39_0 = fmaf(q1, Y4_b, acc39_0);
      acc36_0 = fmaf(q2, Y5_b, acc36_0);
      acc38_0 = fmaf(q3, Y5_b, acc38_0);
      acc35_0 = fmaf(-q4, Y6_b, acc35_0);
      acc34_0 = fmaf(-q3, Y7_b, acc34_0);
      acc33_0 = fmaf(-q1, Y8_b, acc33_0);
      acc35_0 = fmaf(-q0, Y8_b, acc35_0);
    }
    { const float q = W9_1_b * X1_1_b;
      const float q0 = 0.18257418583505539f * q;
      const float q1 = 0.7071067811865476f * q;
      const float q2 = 0.447213595499958f * q;
      const float q3 = 0.5773502691896256f * q;
      const float q4 = 0.632455532033676f * q;
      acc37_1 = fmaf(q0, Y4_b, acc37_1);
      acc39_1 = fmaf(q1, Y4_b, acc39_1);
      acc36_1 = fmaf(q2, Y5_b, acc36_1);
      acc38_1 = fmaf(q3, Y5_b, acc38_1);
      acc35_1 = fmaf(-q4, Y6_b, acc35_1);
      acc34_1 = fmaf(-q3, Y7_b, acc34_1);
      acc33_1 = fmaf(-q1, Y8_b, acc33_1);
      acc35_1 = fmaf(-q0, Y8_b, acc35_1);
    }
    { const float q = W9_0_b * X2_0_b;
      const float q0 = 0.5773502691896258f * q;
      const float q1 = 0.7302967433402215f * q;
      const float q2 = 0.7745966692414836f * q;
      acc34_0 = fmaf(-q0, Y4_b, acc34_0);
      acc35_0 = fmaf(-q1, Y5_b, acc35_0);
      acc36_0 = fmaf(-q2, Y6_b, acc36_0);
      acc37_0 = fmaf(-q1, Y7_b, acc37_0);
      acc38_0 = fmaf(-q0, Y8_b, acc38_0);
    }
    { const float q = W9_1_b * X2_1_b;
      const float q0 = 0.5773502691896258f * q;
      const float q1 = 0.7302967433402215f * q;
      const float q2 = 0.7745966692414836f * q;
      acc34_1 = fmaf(-q0, Y4_b, acc34_1);
      acc35_1 = fmaf(-q1, Y5_b, acc35_1);
      acc36_1 = fmaf(-q2, Y6_b, acc36_1);
      acc37_1 = fmaf(-q1, Y7_b, acc37_1);
      acc38_1 = fmaf(-q0, Y8_b, acc38_1);
    }
    { const float q = W9_0_b * X3_0_b;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.18257418583505539f * q;
      const float q2 = 0.5773502691896256f * q;
      const float q3 = 0.632455532033676f * q;
      const float q4 = 0.447213595499958f * q;
      acc33_0 = fmaf(-q0, Y4_b, acc33_0);
      acc35_0 = fmaf(q1, Y4_b, acc35_0);
      acc34_0 = fmaf(-q2, Y5_b, acc34_0);
      acc37_0 = fmaf(-q3, Y6_b, acc37_0);
      acc36_0 = fmaf(q4, Y7_b, acc36_0);
      acc38_0 = fmaf(-q2, Y7_b, acc38_0);
      acc37_0 = fmaf(q1, Y8_b, acc37_0);
      acc39_0 = fmaf(-q0, Y8_b, acc39_0);
    }
    { const float q = W9_1_b * X3_1_b;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.18257418583505539f * q;
      const float q2 = 0.5773502691896256f * q;
      const float q3 = 0.632455532033676f * q;
      const float q4 = 0.447213595499958f * q;
      acc33_1 = fmaf(-q0, Y4_b, acc33_1);
      acc35_1 = fmaf(q1, Y4_b, acc35_1);
      acc34_1 = fmaf(-q2, Y5_b, acc34_1);
      acc37_1 = fmaf(-q3, Y6_b, acc37_1);
      acc36_1 = fmaf(q4, Y7_b, acc36_1);
      acc38_1 = fmaf(-q2, Y7_b, acc38_1);
      acc37_1 = fmaf(q1, Y8_b, acc37_1);
      acc39_1 = fmaf(-q0, Y8_b, acc39_1);
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
      red[2048 + lane] = acc16_0;
      red[2112 + lane] = acc16_1;
      red[2176 + lane] = acc17_0;
      red[2240 + lane] = acc17_1;
      red[2304 + lane] = acc18_0;
      red[2368 + lane] = acc18_1;
      red[2432 + lane] = acc19_0;
      red[2496 + lane] = acc19_1;
      red[2560 + lane] = acc20_0;
      red[2624 + lane] = acc20_1;
      red[2688 + lane] = acc21_0;
      red[2752 + lane] = acc21_1;
      red[2816 + lane] = acc22_0;
      red[2880 + lane] = acc22_1;
      red[2944 + lane] = acc23_0;
      red[3008 + lane] = acc23_1;
      red[3072 + lane] = acc24_0;
      red[3136 + lane] = acc24_1;
      red[3200 + lane] = acc25_0;
      red[3264 + lane] = acc25_1;
      red[3328 + lane] = acc26_0;
      red[3392 + lane] = acc26_1;
      red[3456 + lane] = acc27_0;
      red[3520 + lane] = acc27_1;
      red[3584 + lane] = acc28_0;
      red[3648 + lane] = acc28_1;
      red[3712 + lane] = acc29_0;
      red[3776 + lane] = acc29_1;
      red[3840 + lane] = acc30_0;
      red[3904 + lane] = acc30_1;
      red[3968 + lane] = acc31_0;
      red[4032 + lane] = acc31_1;
      red[4096 + lane] = acc32_0;
      red[4160 + lane] = acc32_1;
      red[4224 + lane] = acc33_0;
      red[4288 + lane] = acc33_1;
      red[4352 + lane] = acc34_0;
      red[4416 + lane] = acc34_1;
      red[4480 + lane] = acc35_0;
      red[4544 + lane] = acc35_1;
      red[4608 + lane] = acc36_0;
      red[4672 + lane] = acc36_1;
      red[4736 + lane] = acc37_0;
      red[4800 + lane] = acc37_1;
      red[4864 + lane] = acc38_0;
      red[4928 + lane] = acc38_1;
      red[4992 + lane] = acc39_0;
      red[5056 + lane] = acc39_1;
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
      acc16_0 += red[2048 + lane];
      acc16_1 += red[2112 + lane];
      acc17_0 += red[2176 + lane];
      acc17_1 += red[2240 + lane];
      acc18_0 += red[2304 + lane];
      acc18_1 += red[2368 + lane];
      acc19_0 += red[2432 + lane];
      acc19_1 += red[2496 + lane];
      acc20_0 += red[2560 + lane];
      acc20_1 += red[2624 + lane];
      acc21_0 += red[2688 + lane];
      acc21_1 += red[2752 + lane];
      acc22_0 += red[2816 + lane];
      acc22_1 += red[2880 + lane];
      acc23_0 += red[2944 + lane];
      acc23_1 += red[3008 + lane];
      acc24_0 += red[3072 + lane];
      acc24_1 += red[3136 + lane];
      acc25_0 += red[3200 + lane];
      acc25_1 += red[3264 + lane];
      acc26_0 += red[3328 + lane];
      acc26_1 += red[3392 + lane];
      acc27_0 += red[3456 + lane];
      acc27_1 += red[3520 + lane];
      acc28_0 += red[3584 + lane];
      acc28_1 += red[3648 + lane];
      acc29_0 += red[3712 + lane];
      acc29_1 += red[3776 + lane];
      acc30_0 += red[3840 + lane];
      acc30_1 += red[3904 + lane];
      acc31_0 += red[3968 + lane];
      acc31_1 += red[4032 + lane];
      acc32_0 += red[4096 + lane];
      acc32_1 += red[4160 + lane];
      acc33_0 += red[4224 + lane];
      acc33_1 += red[4288 + lane];
      acc34_0 += red[4352 + lane];
      acc34_1 += red[4416 + lane];
      acc35_0 += red[4480 + lane];
      acc35_1 += red[4544 + lane];
      acc36_0 += red[4608 + lane];
      acc36_1 += red[4672 + lane];
      acc37_0 += red[4736 + lane];
      acc37_1 += red[4800 + lane];
      acc38_0 += red[4864 + lane];
      acc38_1 += red[4928 + lane];
      acc39_0 += red[4992 + lane];
      acc39_1 += red[5056 + lane];
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
  op[2048] = acc16_0;
  op[2112] = acc16_1;
  op[2176] = acc17_0;
  op[2240] = acc17_1;
  op[2304] = acc18_0;
  op[2368] = acc18_1;
  op[2432] = acc19_0;
  op[2496] = acc19_1;
  op[2560] = acc20_0;
  op[2624] = acc20_1;
  op[2688] = acc21_0;
  op[2752] = acc21_1;
  op[2816] = acc22_0;
  op[2880] = acc22_1;
  op[2944] = acc23_0;
  op[3008] = acc23_1;
  op[3072] = acc24_0;
  op[3136] = acc24_1;
  op[3200] = acc25_0;
  op[3264] = acc25_1;
  op[3328] = acc26_0;
  op[3392] = acc26_1;
  op[3456] = acc27_0;
  op[3520] = acc27_1;
  op[3584] = acc28_0;
  op[3648] = acc28_1;
  op[3712] = acc29_0;
  op[3776] = acc29_1;
  op[3840] = acc30_0;
  op[3904] = acc30_1;
  op[3968] = acc31_0;
  op[4032] = acc31_1;
  op[4096] = acc32_0;
  op[4160] = acc32_1;
  op[4224] = acc33_0;
  op[4288] = acc33_1;
  op[4352] = acc34_0;
  op[4416] = acc34_1;
  op[4480] = acc35_0;
  op[4544] = acc35_1;
  op[4608] = acc36_0;
  op[4672] = acc36_1;
  op[4736] = acc37_0;
  op[4800] = acc37_1;
  op[4864] = acc38_0;
  op[4928] = acc38_1;
  op[4992] = acc39_0;
  op[5056] = acc39_1;
}

// Backward from gO = dL/dout: gW[e, w, c] (written), gYp[part][e][m] = partial sums of dL/dY[e, m] over
// the channels and paths of one wave (2 partial(s): channel half h x path group g, part
// h * 1 + g; summed by the caller), gX[send, k, c] (atomic adds).  Null outputs are skipped.
extern "C" __global__ void __launch_bounds__(256)
mm_tpw_l2_bwd_kernel(const int* __restrict__ rowptr, int nR, const int* __restrict__ eid,
    const int* __restrict__ send, const float* __restrict__ Y, long y_stride, const float* __restrict__ W,
    long w_stride, const float* __restrict__ X, long x_stride, const float* __restrict__ gO, long g_stride,
    float* __restrict__ gW, long gw_stride, float* __restrict__ gYp, long gy_cb_stride,
    float* __restrict__ gX, long gx_stride) {
  const int gw = blockIdx.x * 4 + (threadIdx.x >> 6);   // global wave: receiver i, sub-wave h
  const int i = gw / 2, h = gw % 2;
  if (i >= nR) return;
  const int lane = threadIdx.x & 63;
  const int c = h * 64 + lane;
  const int p0 = rowptr[i], p1 = rowptr[i + 1];
  const int part = h;
  const int cl = lane & 15;
  const bool b3 = cl & 8, b2 = cl & 4, b1 = cl & 2, b0 = cl & 1;
  const float* __restrict__ gp = gO + (size_t)i * g_stride + c;
  const float g0_0 = gp[0];
  const float g1_0 = gp[128];
  const float g2_0 = gp[256];
  const float g3_0 = gp[384];
  const float g4_0 = gp[512];
  const float g5_0 = gp[640];
  const float g6_0 = gp[768];
  const float g7_0 = gp[896];
  const float g8_0 = gp[1024];
  const float g9_0 = gp[1152];
  const float g10_0 = gp[1280];
  const float g11_0 = gp[1408];
  const float g12_0 = gp[1536];
  const float g13_0 = gp[1664];
  const float g14_0 = gp[1792];
  const float g15_0 = gp[1920];
  const float g16_0 = gp[2048];
  const float g17_0 = gp[2176];
  const float g18_0 = gp[2304];
  const float g19_0 = gp[2432];
  const float g20_0 = gp[2560];
  const float g21_0 = gp[2688];
  const float g22_0 = gp[2816];
  const float g23_0 = gp[2944];
  const float g24_0 = gp[3072];
  const float g25_0 = gp[3200];
  const float g26_0 = gp[3328];
  const float g27_0 = gp[3456];
  const float g28_0 = gp[3584];
  const float g29_0 = gp[3712];
  const float g30_0 = gp[3840];
  const float g31_0 = gp[3968];
  const float g32_0 = gp[4096];
  const float g33_0 = gp[4224];
  const float g34_0 = gp[4352];
  const float g35_0 = gp[4480];
  const float g36_0 = gp[4608];
  const float g37_0 = gp[4736];
  const float g38_0 = gp[4864];
  const float g39_0 = gp[4992];
  const float G0_0 = g0_0;
  const float G1_0 = 0.5773502691896257f * g1_0;
  const float G2_0 = 0.5773502691896258f * g1_0;
  const float G3_0 = 0.5773502691896257f * g1_0;
  const float G4_0 = g2_0;
  const float G5_0 = g3_0;
  const float G6_0 = g4_0;
  const float G7_0 = g5_0;
  const float G8_0 = g6_0;
  const float G9_0 = g7_0;
  const float G10_0 = 0.547722557505166f * g10_0;
  const float G11_0 = 0.547722557505166f * g9_0;
  const float G12_0 = -0.31622776601683794f * g8_0;
  const float G13_0 = -0.547722557505166f * g8_0;
  const float G14_0 = 0.547722557505166f * g8_0;
  const float G15_0 = 0.632455532033676f * g9_0;
  const float G16_0 = 0.547722557505166f * g10_0;
  const float G17_0 = 0.547722557505166f * g8_0;
  const float G18_0 = -0.31622776601683794f * g10_0;
  const float G19_0 = 0.547722557505166f * g9_0;
  const float G20_0 = 0.547722557505166f * g10_0;
  const float G21_0 = g11_0;
  const float G22_0 = g12_0;
  const float G23_0 = g13_0;
  const float G24_0 = g14_0;
  const float G25_0 = g15_0;
  const float G26_0 = fmaf(0.7071067811865475f, g20_0, 0.408248290463863f * g18_0);
  const float G27_0 = -0.7071067811865476f * g17_0;
  const float G28_0 = -0.7071067811865475f * g16_0;
  const float G29_0 = -0.7071067811865476f * g17_0;
  const float G30_0 = -0.8164965809277261f * g18_0;
  const float G31_0 = -0.7071067811865476f * g19_0;
  const float G32_0 = -0.7071067811865475f * g16_0;
  const float G33_0 = -0.7071067811865476f * g19_0;
  const float G34_0 = fmaf(-0.7071067811865475f, g20_0, 0.408248290463863f * g18_0);
  const float G35_0 = 0.5976143046671967f * g25_0;
  const float G36_0 = 0.48795003647426655f * g24_0;
  const float G37_0 = fmaf(0.15430334996209188f, g25_0, 0.5345224838248488f * g23_0);
  const float G38_0 = -0.3779644730092272f * g22_0;
  const float G39_0 = -0.15430334996209188f * g21_0;
  const float G40_0 = -0.48795003647426655f * g22_0;
  const float G41_0 = -0.5976143046671967f * g21_0;
  const float G42_0 = 0.48795003647426655f * g21_0;
  const float G43_0 = 0.6172133998483676f * g22_0;
  const float G44_0 = 0.6546536707079772f * g23_0;
  const float G45_0 = 0.6172133998483676f * g24_0;
  const float G46_0 = 0.48795003647426655f * g25_0;
  const float G47_0 = 0.5976143046671967f * g21_0;
  const float G48_0 = 0.48795003647426655f * g22_0;
  const float G49_0 = -0.15430334996209188f * g21_0;
  const float G50_0 = -0.3779644730092272f * g24_0;
  const float G51_0 = fmaf(-0.15430334996209188f, g25_0, 0.5345224838248488f * g23_0);
  const float G52_0 = 0.48795003647426655f * g24_0;
  const float G53_0 = 0.5976143046671967f * g25_0;
  const float G54_0 = g26_0;
  const float G55_0 = g27_0;
  const float G56_0 = g28_0;
  const float G57_0 = g29_0;
  const float G58_0 = g30_0;
  const float G59_0 = g31_0;
  const float G60_0 = g32_0;
  const float G61_0 = fmaf(0.7071067811865476f, g39_0, 0.18257418583505539f * g37_0);
  const float G62_0 = fmaf(0.5773502691896256f, g38_0, 0.447213595499958f * g36_0);
  const float G63_0 = -0.632455532033676f * g35_0;
  const float G64_0 = -0.5773502691896256f * g34_0;
  const float G65_0 = fmaf(-0.18257418583505539f, g35_0, -0.7071067811865476f * g33_0);
  const float G66_0 = -0.5773502691896258f * g34_0;
  const float G67_0 = -0.7302967433402215f * g35_0;
  const float G68_0 = -0.7745966692414836f * g36_0;
  const float G69_0 = -0.7302967433402215f * g37_0;
  const float G70_0 = -0.5773502691896258f * g38_0;
  const float G71_0 = fmaf(0.18257418583505539f, g35_0, -0.7071067811865476f * g33_0);
  const float G72_0 = -0.5773502691896256f * g34_0;
  const float G73_0 = -0.632455532033676f * g37_0;
  const float G74_0 = fmaf(-0.5773502691896256f, g38_0, 0.447213595499958f * g36_0);
  const float G75_0 = fmaf(-0.7071067811865476f, g39_0, 0.18257418583505539f * g37_0);
  for (int p = p0; p < p1; p += 2) {
    const bool two = p + 1 < p1;   // wave-uniform
    const int ea = __builtin_amdgcn_readfirstlane(eid ? eid[p] : p);
    const int sa = __builtin_amdgcn_readfirstlane(send[ea]);
    const float* __restrict__ wpa = W + (size_t)ea * w_stride + c;
    const float W0_0_a = wpa[0];
    const float W1_0_a = wpa[128];
    const float W2_0_a = wpa[256];
    const float W3_0_a = wpa[384];
    const float W4_0_a = wpa[512];
    const float W5_0_a = wpa[640];
    const float W6_0_a = wpa[768];
    const float W7_0_a = wpa[896];
    const float W8_0_a = wpa[1024];
    const float W9_0_a = wpa[1152];
    const float* __restrict__ xpa = X + (size_t)sa * x_stride + c;
    const float X0_0_a = xpa[0];
    const float X1_0_a = xpa[128];
    const float X2_0_a = xpa[256];
    const float X3_0_a = xpa[384];
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
    const float W1_0_b = wpb[128];
    const float W2_0_b = wpb[256];
    const float W3_0_b = wpb[384];
    const float W4_0_b = wpb[512];
    const float W5_0_b = wpb[640];
    const float W6_0_b = wpb[768];
    const float W7_0_b = wpb[896];
    const float W8_0_b = wpb[1024];
    const float W9_0_b = wpb[1152];
    const float* __restrict__ xpb = X + (size_t)sb * x_stride + c;
    const float X0_0_b = xpb[0];
    const float X1_0_b = xpb[128];
    const float X2_0_b = xpb[256];
    const float X3_0_b = xpb[384];
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
    float gx1_0 = 0.f;
    float gx2_0 = 0.f;
    float gx3_0 = 0.f;
    float* __restrict__ gwp = gW ? gW + (size_t)ea * gw_stride + c : nullptr;
    {
      float gw0 = 0.f;
      { const float q = W0_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y0_a, G0_0, u); gy0 = fmaf(q, G0_0, gy0);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W0_0_a, u, gx0_0);
      }
      if (gwp) gwp[0] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W1_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y1_a, G1_0, u); gy1 = fmaf(q, G1_0, gy1);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W1_0_a, u, gx1_0);
      }
      { const float q = W1_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y2_a, G2_0, u); gy2 = fmaf(q, G2_0, gy2);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W1_0_a, u, gx2_0);
      }
      { const float q = W1_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y3_a, G3_0, u); gy3 = fmaf(q, G3_0, gy3);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W1_0_a, u, gx3_0);
      }
      if (gwp) gwp[128] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W2_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y1_a, G4_0, u); gy1 = fmaf(q, G4_0, gy1);
        u = fmaf(Y2_a, G5_0, u); gy2 = fmaf(q, G5_0, gy2);
        u = fmaf(Y3_a, G6_0, u); gy3 = fmaf(q, G6_0, gy3);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W2_0_a, u, gx0_0);
      }
      if (gwp) gwp[256] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W3_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y0_a, G7_0, u); gy0 = fmaf(q, G7_0, gy0);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W3_0_a, u, gx1_0);
      }
      { const float q = W3_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y0_a, G8_0, u); gy0 = fmaf(q, G8_0, gy0);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W3_0_a, u, gx2_0);
      }
      { const float q = W3_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y0_a, G9_0, u); gy0 = fmaf(q, G9_0, gy0);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W3_0_a, u, gx3_0);
      }
      if (gwp) gwp[384] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W4_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y4_a, G10_0, u); gy4 = fmaf(q, G10_0, gy4);
        u = fmaf(Y5_a, G11_0, u); gy5 = fmaf(q, G11_0, gy5);
        u = fmaf(Y6_a, G12_0, u); gy6 = fmaf(q, G12_0, gy6);
        u = fmaf(Y8_a, G13_0, u); gy8 = fmaf(q, G13_0, gy8);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W4_0_a, u, gx1_0);
      }
      { const float q = W4_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y5_a, G14_0, u); gy5 = fmaf(q, G14_0, gy5);
        u = fmaf(Y6_a, G15_0, u); gy6 = fmaf(q, G15_0, gy6);
        u = fmaf(Y7_a, G16_0, u); gy7 = fmaf(q, G16_0, gy7);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W4_0_a, u, gx2_0);
      }
      { const float q = W4_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y4_a, G17_0, u); gy4 = fmaf(q, G17_0, gy4);
        u = fmaf(Y6_a, G18_0, u); gy6 = fmaf(q, G18_0, gy6);
        u = fmaf(Y7_a, G19_0, u); gy7 = fmaf(q, G19_0, gy7);
        u = fmaf(Y8_a, G20_0, u); gy8 = fmaf(q, G20_0, gy8);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W4_0_a, u, gx3_0);
      }
      if (gwp) gwp[512] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W5_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y4_a, G21_0, u); gy4 = fmaf(q, G21_0, gy4);
        u = fmaf(Y5_a, G22_0, u); gy5 = fmaf(q, G22_0, gy5);
        u = fmaf(Y6_a, G23_0, u); gy6 = fmaf(q, G23_0, gy6);
        u = fmaf(Y7_a, G24_0, u); gy7 = fmaf(q, G24_0, gy7);
        u = fmaf(Y8_a, G25_0, u); gy8 = fmaf(q, G25_0, gy8);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W5_0_a, u, gx0_0);
      }
      if (gwp) gwp[640] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W6_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y1_a, G26_0, u); gy1 = fmaf(q, G26_0, gy1);
        u = fmaf(Y2_a, G27_0, u); gy2 = fmaf(q, G27_0, gy2);
        u = fmaf(Y3_a, G28_0, u); gy3 = fmaf(q, G28_0, gy3);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W6_0_a, u, gx1_0);
      }
      { const float q = W6_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y1_a, G29_0, u); gy1 = fmaf(q, G29_0, gy1);
        u = fmaf(Y2_a, G30_0, u); gy2 = fmaf(q, G30_0, gy2);
        u = fmaf(Y3_a, G31_0, u); gy3 = fmaf(q, G31_0, gy3);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W6_0_a, u, gx2_0);
      }
      { const float q = W6_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y1_a, G32_0, u); gy1 = fmaf(q, G32_0, gy1);
        u = fmaf(Y2_a, G33_0, u); gy2 = fmaf(q, G33_0, gy2);
        u = fmaf(Y3_a, G34_0, u); gy3 = fmaf(q, G34_0, gy3);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W6_0_a, u, gx3_0);
      }
      if (gwp) gwp[768] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W7_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y9_a, G35_0, u); gy9 = fmaf(q, G35_0, gy9);
        u = fmaf(Y10_a, G36_0, u); gy10 = fmaf(q, G36_0, gy10);
        u = fmaf(Y11_a, G37_0, u); gy11 = fmaf(q, G37_0, gy11);
        u = fmaf(Y12_a, G38_0, u); gy12 = fmaf(q, G38_0, gy12);
        u = fmaf(Y13_a, G39_0, u); gy13 = fmaf(q, G39_0, gy13);
        u = fmaf(Y14_a, G40_0, u); gy14 = fmaf(q, G40_0, gy14);
        u = fmaf(Y15_a, G41_0, u); gy15 = fmaf(q, G41_0, gy15);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W7_0_a, u, gx1_0);
      }
      { const float q = W7_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y10_a, G42_0, u); gy10 = fmaf(q, G42_0, gy10);
        u = fmaf(Y11_a, G43_0, u); gy11 = fmaf(q, G43_0, gy11);
        u = fmaf(Y12_a, G44_0, u); gy12 = fmaf(q, G44_0, gy12);
        u = fmaf(Y13_a, G45_0, u); gy13 = fmaf(q, G45_0, gy13);
        u = fmaf(Y14_a, G46_0, u); gy14 = fmaf(q, G46_0, gy14);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W7_0_a, u, gx2_0);
      }
      { const float q = W7_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y9_a, G47_0, u); gy9 = fmaf(q, G47_0, gy9);
        u = fmaf(Y10_a, G48_0, u); gy10 = fmaf(q, G48_0, gy10);
        u = fmaf(Y11_a, G49_0, u); gy11 = fmaf(q, G49_0, gy11);
        u = fmaf(Y12_a, G50_0, u); gy12 = fmaf(q, G50_0, gy12);
        u = fmaf(Y13_a, G51_0, u); gy13 = fmaf(q, G51_0, gy13);
        u = fmaf(Y14_a, G52_0, u); gy14 = fmaf(q, G52_0, gy14);
        u = fmaf(Y15_a, G53_0, u); gy15 = fmaf(q, G53_0, gy15);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W7_0_a, u, gx3_0);
      }
      if (gwp) gwp[896] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W8_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y9_a, G54_0, u); gy9 = fmaf(q, G54_0, gy9);
        u = fmaf(Y10_a, G55_0, u); gy10 = fmaf(q, G55_0, gy10);
        u = fmaf(Y11_a, G56_0, u); gy11 = fmaf(q, G56_0, gy11);
        u = fmaf(Y12_a, G57_0, u); gy12 = fmaf(q, G57_0, gy12);
        u = fmaf(Y13_a, G58_0, u); gy13 = fmaf(q, G58_0, gy13);
        u = fmaf(Y14_a, G59_0, u); gy14 = fmaf(q, G59_0, gy14);
        u = fmaf(Y15_a, G60_0, u); gy15 = fmaf(q, G60_0, gy15);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W8_0_a, u, gx0_0);
      }
      if (gwp) gwp[1024] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W9_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y4_a, G61_0, u); gy4 = fmaf(q, G61_0, gy4);
        u = fmaf(Y5_a, G62_0, u); gy5 = fmaf(q, G62_0, gy5);
        u = fmaf(Y6_a, G63_0, u); gy6 = fmaf(q, G63_0, gy6);
        u = fmaf(Y7_a, G64_0, u); gy7 = fmaf(q, G64_0, gy7);
        u = fmaf(Y8_a, G65_0, u); gy8 = fmaf(q, G65_0, gy8);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W9_0_a, u, gx1_0);
      }
      { const float q = W9_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y4_a, G66_0, u); gy4 = fmaf(q, G66_0, gy4);
        u = fmaf(Y5_a, G67_0, u); gy5 = fmaf(q, G67_0, gy5);
        u = fmaf(Y6_a, G68_0, u); gy6 = fmaf(q, G68_0, gy6);
        u = fmaf(Y7_a, G69_0, u); gy7 = fmaf(q, G69_0, gy7);
        u = fmaf(Y8_a, G70_0, u); gy8 = fmaf(q, G70_0, gy8);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W9_0_a, u, gx2_0);
      }
      { const float q = W9_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y4_a, G71_0, u); gy4 = fmaf(q, G71_0, gy4);
        u = fmaf(Y5_a, G72_0, u); gy5 = fmaf(q, G72_0, gy5);
        u = fmaf(Y6_a, G73_0, u); gy6 = fmaf(q, G73_0, gy6);
        u = fmaf(Y7_a, G74_0, u); gy7 = fmaf(q, G74_0, gy7);
        u = fmaf(Y8_a, G75_0, u); gy8 = fmaf(q, G75_0, gy8);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W9_0_a, u, gx3_0);
      }
      if (gwp) gwp[1152] = gw0;
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
      atomicAdd(gxp + 128, gx1_0);
      atomicAdd(gxp + 256, gx2_0);
      atomicAdd(gxp + 384, gx3_0);
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
    float gx1_0 = 0.f;
    float gx2_0 = 0.f;
    float gx3_0 = 0.f;
    float* __restrict__ gwp = gW ? gW + (size_t)eb * gw_stride + c : nullptr;
    {
      float gw0 = 0.f;
      { const float q = W0_0_b * X0_0_b; float u = 0.f;
        u = fmaf(Y0_b, G0_0, u); gy0 = fmaf(q, G0_0, gy0);
        gw0 = fmaf(X0_0_b, u, gw0); gx0_0 = fmaf(W0_0_b, u, gx0_0);
      }
      if (gwp) gwp[0] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W1_0_b * X1_0_b; float u = 0.f;
        u = fmaf(Y1_b, G1_0, u); gy1 = fmaf(q, G1_0, gy1);
        gw0 = fmaf(X1_0_b, u, gw0); gx1_0 = fmaf(W1_0_b, u, gx1_0);
      }
      { const float q = W1_0_b * X2_0_b; float u = 0.f;
        u = fmaf(Y2_b, G2_0, u); gy2 = fmaf(q, G2_0, gy2);
        gw0 = fmaf(X2_0_b, u, gw0); gx2_0 = fmaf(W1_0_b, u, gx2_0);
      }
      { const float q = W1_0_b * X3_0_b; float u = 0.f;
        u = fmaf(Y3_b, G3_0, u); gy3 = fmaf(q, G3_0, gy3);
        gw0 = fmaf(X3_0_b, u, gw0); gx3_0 = fmaf(W1_0_b, u, gx3_0);
      }
      if (gwp) gwp[128] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W2_0_b * X0_0_b; float u = 0.f;
        u = fmaf(Y1_b, G4_0, u); gy1 = fmaf(q, G4_0, gy1);
        u = fmaf(Y2_b, G5_0, u); gy2 = fmaf(q, G5_0, gy2);
        u = fmaf(Y3_b, G6_0, u); gy3 = fmaf(q, G6_0, gy3);
        gw0 = fmaf(X0_0_b, u, gw0); gx0_0 = fmaf(W2_0_b, u, gx0_0);
      }
      if (gwp) gwp[256] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W3_0_b * X1_0_b; float u = 0.f;
        u = fmaf(Y0_b, G7_0, u); gy0 = fmaf(q, G7_0, gy0);
        gw0 = fmaf(X1_0_b, u, gw0); gx1_0 = fmaf(W3_0_b, u, gx1_0);
      }
      { const float q = W3_0_b * X2_0_b; float u = 0.f;
        u = fmaf(Y0_b, G8_0, u); gy0 = fmaf(q, G8_0, gy0);
        gw0 = fmaf(X2_0_b, u, gw0); gx2_0 = fmaf(W3_0_b, u, gx2_0);
      }
      { const float q = W3_0_b * X3_0_b; float u = 0.f;
        u = fmaf(Y0_b, G9_0, u); gy0 = fmaf(q, G9_0, gy0);
        gw0 = fmaf(X3_0_b, u, gw0); gx3_0 = fmaf(W3_0_b, u, gx3_0);
      }
      if (gwp) gwp[384] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W4_0_b * X1_0_b; float u = 0.f;
        u = fmaf(Y4_b, G10_0, u); gy4 = fmaf(q, G10_0, gy4);
        u = fmaf(Y5_b, G11_0, u); gy5 = fmaf(q, G11_0, gy5);
        u = fmaf(Y6_b, G12_0, u); gy6 = fmaf(q, G12_0, gy6);
        u = fmaf(Y8_b, G13_0, u); gy8 = fmaf(q, G13_0, gy8);
        gw0 = fmaf(X1_0_b, u, gw0); gx1_0 = fmaf(W4_0_b, u, gx1_0);
      }
      { const float q = W4_0_b * X2_0_b; float u = 0.f;
        u = fmaf(Y5_b, G14_0, u); gy5 = fmaf(q, G14_0, gy5);
        u = fmaf(Y6_b, G15_0, u); gy6 = fmaf(q, G15_0, gy6);
        u = fmaf(Y7_b, G16_0, u); gy7 = fmaf(q, G16_0, gy7);
        gw0 = fmaf(X2_0_b, u, gw0); gx2_0 = fmaf(W4_0_b, u, gx2_0);
      }
      { const float q = W4_0_b * X3_0_b; float u = 0.f;
        u = fmaf(Y4_b, G17_0, u); gy4 = fmaf(q, G17_0, gy4);
        u = fmaf(Y6_b, G18_0, u); gy6 = fmaf(q, G18_0, gy6);
        u = fmaf(Y7_b, G19_0, u); gy7 = fmaf(q, G19_0, gy7);
        u = fmaf(Y8_b, G20_0, u); gy8 = fmaf(q, G20_0, gy8);
        gw0 = fmaf(X3_0_b, u, gw0); gx3_0 = fmaf(W4_0_b, u, gx3_0);
      }
      if (gwp) gwp[512] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W5_0_b * X0_0_b; float u = 0.f;
        u = fmaf(Y4_b, G21_0, u); gy4 = fmaf(q, G21_0, gy4);
        u = fmaf(Y5_b, G22_0, u); gy5 = fmaf(q, G22_0, gy5);
        u = fmaf(Y6_b, G23_0, u); gy6 = fmaf(q, G23_0, gy6);
        u = fmaf(Y7_b, G24_0, u); gy7 = fmaf(q, G24_0, gy7);
        u = fmaf(Y8_b, G25_0, u); gy8 = fmaf(q, G25_0, gy8);
        gw0 = fmaf(X0_0_b, u, gw0); gx0_0 = fmaf(W5_0_b, u, gx0_0);
      }
      if (gwp) gwp[640] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W6_0_b * X1_0_b; float u = 0.f;
        u = fmaf(Y1_b, G26_0, u); gy1 = fmaf(q, G26_0, gy1);
        u = fmaf(Y2_b, G27_0, u); gy2 = fmaf(q, G27_0, gy2);
        u = fmaf(Y3_b, G28_0, u); gy3 = fmaf(q, G28_0, gy3);
        gw0 = fmaf(X1_0_b, u, gw0); gx1_0 = fmaf(W6_0_b, u, gx1_0);
      }
      { const float q = W6_0_b * X2_0_b; float u = 0.f;
        u = fmaf(Y1_b, G29_0, u); gy1 = fmaf(q, G29_0, gy1);
        u = fmaf(Y2_b, G30_0, u); gy2 = fmaf(q, G30_0, gy2);
        u = fmaf(Y3_b, G31_0, u); gy3 = fmaf(q, G31_0, gy3);
        gw0 = fmaf(X2_0_b, u, gw0); gx2_0 = fmaf(W6_0_b, u, gx2_0);
      }
      { const float q = W6_0_b * X3_0_b; float u = 0.f;
        u = fmaf(Y1_b, G32_0, u); gy1 = fmaf(q, G32_0, gy1);
        u = fmaf(Y2_b, G33_0, u); gy2 = fmaf(q, G33_0, gy2);
        u = fmaf(Y3_b, G34_0, u); gy3 = fmaf(q, G34_0, gy3);
        gw0 = fmaf(X3_0_b, u, gw0); gx3_0 = fmaf(W6_0_b, u, gx3_0);
      }
      if (gwp) gwp[768] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W7_0_b * X1_0_b; float u = 0.f;
        u = fmaf(Y9_b, G35_0, u); gy9 = fmaf(q, G35_0, gy9);
        u = fmaf(Y10_b, G36_0, u); gy10 = fmaf(q, G36_0, gy10);
        u = fmaf(Y11_b, G37_0, u); gy11 = fmaf(q, G37_0, gy11);
        u = fmaf(Y12_b, G38_0, u); gy12 = fmaf(q, G38_0, gy12);
        u = fmaf(Y13_b, G39_0, u); gy13 = fmaf(q, G39_0, gy13);
        u = fmaf(Y14_b, G40_0, u); gy14 = fmaf(q, G40_0, gy14);
        u = fmaf(Y15_b, G41_0, u); gy15 = fmaf(q, G41_0, gy15);
        gw0 = fmaf(X1_0_b, u, gw0); gx1_0 = fmaf(W7_0_b, u, gx1_0);
      }
      { const float q = W7_0_b * X2_0_b; float u = 0.f;
        u = fmaf(Y10_b, G42_0, u); gy10 = fmaf(q, G42_0, gy10);
        u = fmaf(Y11_b, G43_0, u); gy11 = fmaf(q, G43_0, gy11);
        u = fmaf(Y12_b, G44_0, u); gy12 = fmaf(q, G44_0, gy12);
        u = fmaf(Y13_b, G45_0, u); gy13 = fmaf(q, G45_0, gy13);
        u = fmaf(Y14_b, G46_0, u); gy14 = fmaf(q, G46_0, gy14);
        gw0 = fmaf(X2_0_b, u, gw0); gx2_0 = fmaf(W7_0_b, u, gx2_0);
      }
      { const float q = W7_0_b * X3_0_b; float u = 0.f;
        u = fmaf(Y9_b, G47_0, u); gy9 = fmaf(q, G47_0, gy9);
        u = fmaf(Y10_b, G48_0, u); gy10 = fmaf(q, G48_0, gy10);
        u = fmaf(Y11_b, G49_0, u); gy11 = fmaf(q, G49_0, gy11);
        u = fmaf(Y12_b, G50_0, u); gy12 = fmaf(q, G50_0, gy12);
        u = fmaf(Y13_b, G51_0, u); gy13 = fmaf(q, G51_0, gy13);
        u = fmaf(Y14_b, G52_0, u); gy14 = fmaf(q, G52_0, gy14);
        u = fmaf(Y15_b, G53_0, u); gy15 = fmaf(q, G53_0, gy15);
        gw0 = fmaf(X3_0_b, u, gw0); gx3_0 = fmaf(W7_0_b, u, gx3_0);
      }
      if (gwp) gwp[896] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W8_0_b * X0_0_b; float u = 0.f;
        u = fmaf(Y9_b, G54_0, u); gy9 = fmaf(q, G54_0, gy9);
        u = fmaf(Y10_b, G55_0, u); gy10 = fmaf(q, G55_0, gy10);
        u = fmaf(Y11_b, G56_0, u); gy11 = fmaf(q, G56_0, gy11);
        u = fmaf(Y12_b, G57_0, u); gy12 = fmaf(q, G57_0, gy12);
        u = fmaf(Y13_b, G58_0, u); gy13 = fmaf(q, G58_0, gy13);
        u = fmaf(Y14_b, G59_0, u); gy14 = fmaf(q, G59_0, gy14);
        u = fmaf(Y15_b, G60_0, u); gy15 = fmaf(q, G60_0, gy15);
        gw0 = fmaf(X0_0_b, u, gw0); gx0_0 = fmaf(W8_0_b, u, gx0_0);
      }
      if (gwp) gwp[1024] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W9_0_b * X1_0_b; float u = 0.f;
        u = fmaf(Y4_b, G61_0, u); gy4 = fmaf(q, G61_0, gy4);
        u = fmaf(Y5_b, G62_0, u); gy5 = fmaf(q, G62_0, gy5);
        u = fmaf(Y6_b, G63_0, u); gy6 = fmaf(q, G63_0, gy6);
        u = fmaf(Y7_b, G64_0, u); gy7 = fmaf(q, G64_0, gy7);
        u = fmaf(Y8_b, G65_0, u); gy8 = fmaf(q, G65_0, gy8);
        gw0 = fmaf(X1_0_b, u, gw0); gx1_0 = fmaf(W9_0_b, u, gx1_0);
      }
      { const float q = W9_0_b * X2_0_b; float u = 0.f;
        u = fmaf(Y4_b, G66_0, u); gy4 = fmaf(q, G66_0, gy4);
        u = fmaf(Y5_b, G67_0, u); gy5 = fmaf(q, G67_0, gy5);
        u = fmaf(Y6_b, G68_0, u); gy6 = fmaf(q, G68_0, gy6);
        u = fmaf(Y7_b, G69_0, u); gy7 = fmaf(q, G69_0, gy7);
        u = fmaf(Y8_b, G70_0, u); gy8 = fmaf(q, G70_0, gy8);
        gw0 = fmaf(X2_0_b, u, gw0); gx2_0 = fmaf(W9_0_b, u, gx2_0);
      }
      { const float q = W9_0_b * X3_0_b; float u = 0.f;
        u = fmaf(Y4_b, G71_0, u); gy4 = fmaf(q, G71_0, gy4);
        u = fmaf(Y5_b, G72_0, u); gy5 = fmaf(q, G72_0, gy5);
        u = fmaf(Y6_b, G73_0, u); gy6 = fmaf(q, G73_0, gy6);
        u = fmaf(Y7_b, G74_0, u); gy7 = fmaf(q, G74_0, gy7);
        u = fmaf(Y8_b, G75_0, u); gy8 = fmaf(q, G75_0, gy8);
        gw0 = fmaf(X3_0_b, u, gw0); gx3_0 = fmaf(W9_0_b, u, gx3_0);
      }
      if (gwp) gwp[1152] = gw0;
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
      atomicAdd(gxp + 128, gx1_0);
      atomicAdd(gxp + 256, gx2_0);
      atomicAdd(gxp + 384, gx3_0);
    }
    }
  }
}

// Backward from gO = dL/dout: gW[e, w, c] (written), gYp[part][e][m] = partial sums of dL/dY[e, m] over
// the channels and paths of one wave (2 partial(s): channel half h x path group g, part
// h * 1 + g; summed by the caller), gX[send, k, c] (atomic adds).  Null outputs are skipped.
extern "C" __global__ void __launch_bounds__(256)
mm_tpw_l2_bwd_shared_kernel(const int* __restrict__ rowptr, int nR, const int* __restrict__ eid,
    const int* __restrict__ send, const float* __restrict__ Y, long y_stride, const float* __restrict__ W,
    long w_stride, const float* __restrict__ X, long x_stride, const float* __restrict__ gO, long g_stride,
    float* __restrict__ gW, long gw_stride, float* __restrict__ gYp, long gy_cb_stride,
    float* __restrict__ gX, long gx_stride) {
  const int wave = threadIdx.x >> 6;
  const int gw = blockIdx.x;   // receiver i, sub-wave h
  const int i = gw / 2, h = gw % 2;
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
  const float g1_0 = gp[128];
  const float g2_0 = gp[256];
  const float g3_0 = gp[384];
  const float g4_0 = gp[512];
  const float g5_0 = gp[640];
  const float g6_0 = gp[768];
  const float g7_0 = gp[896];
  const float g8_0 = gp[1024];
  const float g9_0 = gp[1152];
  const float g10_0 = gp[1280];
  const float g11_0 = gp[1408];
  const float g12_0 = gp[1536];
  const float g13_0 = gp[1664];
  const float g14_0 = gp[1792];
  const float g15_0 = gp[1920];
  const float g16_0 = gp[2048];
  const float g17_0 = gp[2176];
  const float g18_0 = gp[2304];
  const float g19_0 = gp[2432];
  const float g20_0 = gp[2560];
  const float g21_0 = gp[2688];
  const float g22_0 = gp[2816];
  const float g23_0 = gp[2944];
  const float g24_0 = gp[3072];
  const float g25_0 = gp[3200];
  const float g26_0 = gp[3328];
  const float g27_0 = gp[3456];
  const float g28_0 = gp[3584];
  const float g29_0 = gp[3712];
  const float g30_0 = gp[3840];
  const float g31_0 = gp[3968];
  const float g32_0 = gp[4096];
  const float g33_0 = gp[4224];
  const float g34_0 = gp[4352];
  const float g35_0 = gp[4480];
  const float g36_0 = gp[4608];
  const float g37_0 = gp[4736];
  const float g38_0 = gp[4864];
  const float g39_0 = gp[4992];
  const float G0_0 = g0_0;
  const float G1_0 = 0.5773502691896257f * g1_0;
  const float G2_0 = 0.5773502691896258f * g1_0;
  const float G3_0 = 0.5773502691896257f * g1_0;
  const float G4_0 = g2_0;
  const float G5_0 = g3_0;
  const float G6_0 = g4_0;
  const float G7_0 = g5_0;
  const float G8_0 = g6_0;
  const float G9_0 = g7_0;
  const float G10_0 = 0.547722557505166f * g10_0;
  const float G11_0 = 0.547722557505166f * g9_0;
  const float G12_0 = -0.31622776601683794f * g8_0;
  const float G13_0 = -0.547722557505166f * g8_0;
  const float G14_0 = 0.547722557505166f * g8_0;
  const float G15_0 = 0.632455532033676f * g9_0;
  const float G16_0 = 0.547722557505166f * g10_0;
  const float G17_0 = 0.547722557505166f * g8_0;
  const float G18_0 = -0.31622776601683794f * g10_0;
  const float G19_0 = 0.547722557505166f * g9_0;
  const float G20_0 = 0.547722557505166f * g10_0;
  const float G21_0 = g11_0;
  const float G22_0 = g12_0;
  const float G23_0 = g13_0;
  const float G24_0 = g14_0;
  const float G25_0 = g15_0;
  const float G26_0 = fmaf(0.7071067811865475f, g20_0, 0.408248290463863f * g18_0);
  const float G27_0 = -0.7071067811865476f * g17_0;
  const float G28_0 = -0.7071067811865475f * g16_0;
  const float G29_0 = -0.7071067811865476f * g17_0;
  const float G30_0 = -0.8164965809277261f * g18_0;
  const float G31_0 = -0.7071067811865476f * g19_0;
  const float G32_0 = -0.7071067811865475f * g16_0;
  const float G33_0 = -0.7071067811865476f * g19_0;
  const float G34_0 = fmaf(-0.7071067811865475f, g20_0, 0.408248290463863f * g18_0);
  const float G35_0 = 0.5976143046671967f * g25_0;
  const float G36_0 = 0.48795003647426655f * g24_0;
  const float G37_0 = fmaf(0.15430334996209188f, g25_0, 0.5345224838248488f * g23_0);
  const float G38_0 = -0.3779644730092272f * g22_0;
  const float G39_0 = -0.15430334996209188f * g21_0;
  const float G40_0 = -0.48795003647426655f * g22_0;
  const float G41_0 = -0.5976143046671967f * g21_0;
  const float G42_0 = 0.48795003647426655f * g21_0;
  const float G43_0 = 0.6172133998483676f * g22_0;
  const float G44_0 = 0.6546536707079772f * g23_0;
  const float G45_0 = 0.6172133998483676f * g24_0;
  const float G46_0 = 0.48795003647426655f * g25_0;
  const float G47_0 = 0.5976143046671967f * g21_0;
  const float G48_0 = 0.48795003647426655f * g22_0;
  const float G49_0 = -0.15430334996209188f * g21_0;
  const float G50_0 = -0.3779644730092272f * g24_0;
  const float G51_0 = fmaf(-0.15430334996209188f, g25_0, 0.5345224838248488f * g23_0);
  const float G52_0 = 0.48795003647426655f * g24_0;
  const float G53_0 = 0.5976143046671967f * g25_0;
  const float G54_0 = g26_0;
  const float G55_0 = g27_0;
  const float G56_0 = g28_0;
  const float G57_0 = g29_0;
  const float G58_0 = g30_0;
  const float G59_0 = g31_0;
  const float G60_0 = g32_0;
  const float G61_0 = fmaf(0.7071067811865476f, g39_0, 0.18257418583505539f * g37_0);
  const float G62_0 = fmaf(0.5773502691896256f, g38_0, 0.447213595499958f * g36_0);
  const float G63_0 = -0.632455532033676f * g35_0;
  const float G64_0 = -0.5773502691896256f * g34_0;
  const float G65_0 = fmaf(-0.18257418583505539f, g35_0, -0.7071067811865476f * g33_0);
  const float G66_0 = -0.5773502691896258f * g34_0;
  const float G67_0 = -0.7302967433402215f * g35_0;
  const float G68_0 = -0.7745966692414836f * g36_0;
  const float G69_0 = -0.7302967433402215f * g37_0;
  const float G70_0 = -0.5773502691896258f * g38_0;
  const float G71_0 = fmaf(0.18257418583505539f, g35_0, -0.7071067811865476f * g33_0);
  const float G72_0 = -0.5773502691896256f * g34_0;
  const float G73_0 = -0.632455532033676f * g37_0;
  const float G74_0 = fmaf(-0.5773502691896256f, g38_0, 0.447213595499958f * g36_0);
  const float G75_0 = fmaf(-0.7071067811865476f, g39_0, 0.18257418583505539f * g37_0);
  for (int p = p0; p < p1; p += 2) {
    const bool two = p + 1 < p1;   // wave-uniform
    const int ea = __builtin_amdgcn_readfirstlane(eid ? eid[p] : p);
    const int sa = __builtin_amdgcn_readfirstlane(send[ea]);
    const float* __restrict__ wpa = W + (size_t)ea * w_stride + c;
    const float W0_0_a = wpa[0];
    const float W1_0_a = wpa[128];
    const float W2_0_a = wpa[256];
    const float W3_0_a = wpa[384];
    const float W4_0_a = wpa[512];
    const float W5_0_a = wpa[640];
    const float W6_0_a = wpa[768];
    const float W7_0_a = wpa[896];
    const float W8_0_a = wpa[1024];
    const float W9_0_a = wpa[1152];
    const float* __restrict__ xpa = X + (size_t)sa * x_stride + c;
    const float X0_0_a = xpa[0];
    const float X1_0_a = xpa[128];
    const float X2_0_a = xpa[256];
    const float X3_0_a = xpa[384];
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
    const float W1_0_b = wpb[128];
    const float W2_0_b = wpb[256];
    const float W3_0_b = wpb[384];
    const float W4_0_b = wpb[512];
    const float W5_0_b = wpb[640];
    const float W6_0_b = wpb[768];
    const float W7_0_b = wpb[896];
    const float W8_0_b = wpb[1024];
    const float W9_0_b = wpb[1152];
    const float* __restrict__ xpb = X + (size_t)sb * x_stride + c;
    const float X0_0_b = xpb[0];
    const float X1_0_b = xpb[128];
    const float X2_0_b = xpb[256];
    const float X3_0_b = xpb[384];
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
    float gx1_0 = 0.f;
    float gx2_0 = 0.f;
    float gx3_0 = 0.f;
    float* __restrict__ gwp = gW ? gW + (size_t)ea * gw_stride + c : nullptr;
    {
      float gw0 = 0.f;
      { const float q = W0_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y0_a, G0_0, u); gy0 = fmaf(q, G0_0, gy0);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W0_0_a, u, gx0_0);
      }
      if (gwp) gwp[0] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W1_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y1_a, G1_0, u); gy1 = fmaf(q, G1_0, gy1);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W1_0_a, u, gx1_0);
      }
      { const float q = W1_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y2_a, G2_0, u); gy2 = fmaf(q, G2_0, gy2);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W1_0_a, u, gx2_0);
      }
      { const float q = W1_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y3_a, G3_0, u); gy3 = fmaf(q, G3_0, gy3);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W1_0_a, u, gx3_0);
      }
      if (gwp) gwp[128] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W2_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y1_a, G4_0, u); gy1 = fmaf(q, G4_0, gy1);
        u = fmaf(Y2_a, G5_0, u); gy2 = fmaf(q, G5_0, gy2);
        u = fmaf(Y3_a, G6_0, u); gy3 = fmaf(q, G6_0, gy3);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W2_0_a, u, gx0_0);
      }
      if (gwp) gwp[256] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W3_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y0_a, G7_0, u); gy0 = fmaf(q, G7_0, gy0);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W3_0_a, u, gx1_0);
      }
      { const float q = W3_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y0_a, G8_0, u); gy0 = fmaf(q, G8_0, gy0);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W3_0_a, u, gx2_0);
      }
      { const float q = W3_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y0_a, G9_0, u); gy0 = fmaf(q, G9_0, gy0);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W3_0_a, u, gx3_0);
      }
      if (gwp) gwp[384] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W4_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y4_a, G10_0, u); gy4 = fmaf(q, G10_0, gy4);
        u = fmaf(Y5_a, G11_0, u); gy5 = fmaf(q, G11_0, gy5);
        u = fmaf(Y6_a, G12_0, u); gy6 = fmaf(q, G12_0, gy6);
        u = fmaf(Y8_a, G13_0, u); gy8 = fmaf(q, G13_0, gy8);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W4_0_a, u, gx1_0);
      }
      { const float q = W4_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y5_a, G14_0, u); gy5 = fmaf(q, G14_0, gy5);
        u = fmaf(Y6_a, G15_0, u); gy6 = fmaf(q, G15_0, gy6);
        u = fmaf(Y7_a, G16_0, u); gy7 = fmaf(q, G16_0, gy7);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W4_0_a, u, gx2_0);
      }
      { const float q = W4_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y4_a, G17_0, u); gy4 = fmaf(q, G17_0, gy4);
        u = fmaf(Y6_a, G18_0, u); gy6 = fmaf(q, G18_0, gy6);
        u = fmaf(Y7_a, G19_0, u); gy7 = fmaf(q, G19_0, gy7);
        u = fmaf(Y8_a, G20_0, u); gy8 = fmaf(q, G20_0, gy8);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W4_0_a, u, gx3_0);
      }
      if (gwp) gwp[512] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W5_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y4_a, G21_0, u); gy4 = fmaf(q, G21_0, gy4);
        u = fmaf(Y5_a, G22_0, u); gy5 = fmaf(q, G22_0, gy5);
        u = fmaf(Y6_a, G23_0, u); gy6 = fmaf(q, G23_0, gy6);
        u = fmaf(Y7_a, G24_0, u); gy7 = fmaf(q, G24_0, gy7);
        u = fmaf(Y8_a, G25_0, u); gy8 = fmaf(q, G25_0, gy8);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W5_0_a, u, gx0_0);
      }
      if (gwp) gwp[640] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W6_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y1_a, G26_0, u); gy1 = fmaf(q, G26_0, gy1);
        u = fmaf(Y2_a, G27_0, u); gy2 = fmaf(q, G27_0, gy2);
        u = fmaf(Y3_a, G28_0, u); gy3 = fmaf(q, G28_0, gy3);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W6_0_a, u, gx1_0);
      }
      { const float q = W6_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y1_a, G29_0, u); gy1 = fmaf(q, G29_0, gy1);
        u = fmaf(Y2_a, G30_0, u); gy2 = fmaf(q, G30_0, gy2);
        u = fmaf(Y3_a, G31_0, u); gy3 = fmaf(q, G31_0, gy3);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W6_0_a, u, gx2_0);
      }
      { const float q = W6_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y1_a, G32_0, u); gy1 = fmaf(q, G32_0, gy1);
        u = fmaf(Y2_a, G33_0, u); gy2 = fmaf(q, G33_0, gy2);
        u = fmaf(Y3_a, G34_0, u); gy3 = fmaf(q, G34_0, gy3);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W6_0_a, u, gx3_0);
      }
      if (gwp) gwp[768] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W7_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y9_a, G35_0, u); gy9 = fmaf(q, G35_0, gy9);
        u = fmaf(Y10_a, G36_0, u); gy10 = fmaf(q, G36_0, gy10);
        u = fmaf(Y11_a, G37_0, u); gy11 = fmaf(q, G37_0, gy11);
        u = fmaf(Y12_a, G38_0, u); gy12 = fmaf(q, G38_0, gy12);
        u = fmaf(Y13_a, G39_0, u); gy13 = fmaf(q, G39_0, gy13);
        u = fmaf(Y14_a, G40_0, u); gy14 = fmaf(q, G40_0, gy14);
        u = fmaf(Y15_a, G41_0, u); gy15 = fmaf(q, G41_0, gy15);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W7_0_a, u, gx1_0);
      }
      { const float q = W7_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y10_a, G42_0, u); gy10 = fmaf(q, G42_0, gy10);
        u = fmaf(Y11_a, G43_0, u); gy11 = fmaf(q, G43_0, gy11);
        u = fmaf(Y12_a, G44_0, u); gy12 = fmaf(q, G44_0, gy12);
        u = fmaf(Y13_a, G45_0, u); gy13 = fmaf(q, G45_0, gy13);
        u = fmaf(Y14_a, G46_0, u); gy14 = fmaf(q, G46_0, gy14);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W7_0_a, u, gx2_0);
      }
      { const float q = W7_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y9_a, G47_0, u); gy9 = fmaf(q, G47_0, gy9);
        u = fmaf(Y10_a, G48_0, u); gy10 = fmaf(q, G48_0, gy10);
        u = fmaf(Y11_a, G49_0, u); gy11 = fmaf(q, G49_0, gy11);
        u = fmaf(Y12_a, G50_0, u); gy12 = fmaf(q, G50_0, gy12);
        u = fmaf(Y13_a, G51_0, u); gy13 = fmaf(q, G51_0, gy13);
        u = fmaf(Y14_a, G52_0, u); gy14 = fmaf(q, G52_0, gy14);
        u = fmaf(Y15_a, G53_0, u); gy15 = fmaf(q, G53_0, gy15);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W7_0_a, u, gx3_0);
      }
      if (gwp) gwp[896] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W8_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y9_a, G54_0, u); gy9 = fmaf(q, G54_0, gy9);
        u = fmaf(Y10_a, G55_0, u); gy10 = fmaf(q, G55_0, gy10);
        u = fmaf(Y11_a, G56_0, u); gy11 = fmaf(q, G56_0, gy11);
        u = fmaf(Y12_a, G57_0, u); gy12 = fmaf(q, G57_0, gy12);
        u = fmaf(Y13_a, G58_0, u); gy13 = fmaf(q, G58_0, gy13);
        u = fmaf(Y14_a, G59_0, u); gy14 = fmaf(q, G59_0, gy14);
        u = fmaf(Y15_a, G60_0, u); gy15 = fmaf(q, G60_0, gy15);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W8_0_a, u, gx0_0);
      }
      if (gwp) gwp[1024] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W9_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y4_a, G61_0, u); gy4 = fmaf(q, G61_0, gy4);
        u = fmaf(Y5_a, G62_0, u); gy5 = fmaf(q, G62_0, gy5);
        u = fmaf(Y6_a, G63_0, u); gy6 = fmaf(q, G63_0, gy6);
        u = fmaf(Y7_a, G64_0, u); gy7 = fmaf(q, G64_0, gy7);
        u = fmaf(Y8_a, G65_0, u); gy8 = fmaf(q, G65_0, gy8);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W9_0_a, u, gx1_0);
      }
      { const float q = W9_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y4_a, G66_0, u); gy4 = fmaf(q, G66_0, gy4);
        u = fmaf(Y5_a, G67_0, u); gy5 = fmaf(q, G67_0, gy5);
        u = fmaf(Y6_a, G68_0, u); gy6 = fmaf(q, G68_0, gy6);
        u = fmaf(Y7_a, G69_0, u); gy7 = fmaf(q, G69_0, gy7);
        u = fmaf(Y8_a, G70_0, u); gy8 = fmaf(q, G70_0, gy8);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W9_0_a, u, gx2_0);
      }
      { const float q = W9_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y4_a, G71_0, u); gy4 = fmaf(q, G71_0, gy4);
        u = fmaf(Y5_a, G72_0, u); gy5 = fmaf(q, G72_0, gy5);
        u = fmaf(Y6_a, G73_0, u); gy6 = fmaf(q, G73_0, gy6);
        u = fmaf(Y7_a, G74_0, u); gy7 = fmaf(q, G74_0, gy7);
        u = fmaf(Y8_a, G75_0, u); gy8 = fmaf(q, G75_0, gy8);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W9_0_a, u, gx3_0);
      }
      if (gwp) gwp[1152] = gw0;
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
      atomicAdd(gxp + 128, gx1_0);
      atomicAdd(gxp + 256, gx2_0);
      atomicAdd(gxp + 384, gx3_0);
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
    float gx1_0 = 0.f;
    float gx2_0 = 0.f;
    float gx3_0 = 0.f;
    float* __restrict__ gwp = gW ? gW + (size_t)eb * gw_stride + c : nullptr;
    {
      float gw0 = 0.f;
      { const float q = W0_0_b * X0_0_b; float u = 0.f;
        u = fmaf(Y0_b, G0_0, u); gy0 = fmaf(q, G0_0, gy0);
        gw0 = fmaf(X0_0_b, u, gw0); gx0_0 = fmaf(W0_0_b, u, gx0_0);
      }
      if (gwp) gwp[0] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W1_0_b * X1_0_b; float u = 0.f;
        u = fmaf(Y1_b, G1_0, u); gy1 = fmaf(q, G1_0, gy1);
        gw0 = fmaf(X1_0_b, u, gw0); gx1_0 = fmaf(W1_0_b, u, gx1_0);
      }
      { const float q = W1_0_b * X2_0_b; float u = 0.f;
        u = fmaf(Y2_b, G2_0, u); gy2 = fmaf(q, G2_0, gy2);
        gw0 = fmaf(X2_0_b, u, gw0); gx2_0 = fmaf(W1_0_b, u, gx2_0);
      }
      { const float q = W1_0_b * X3_0_b; float u = 0.f;
        u = fmaf(Y3_b, G3_0, u); gy3 = fmaf(q, G3_0, gy3);
        gw0 = fmaf(X3_0_b, u, gw0); gx3_0 = fmaf(W1_0_b, u, gx3_0);
      }
      if (gwp) gwp[128] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W2_0_b * X0_0_b; float u = 0.f;
        u = fmaf(Y1_b, G4_0, u); gy1 = fmaf(q, G4_0, gy1);
        u = fmaf(Y2_b, G5_0, u); gy2 = fmaf(q, G5_0, gy2);
        u = fmaf(Y3_b, G6_0, u); gy3 = fmaf(q, G6_0, gy3);
        gw0 = fmaf(X0_0_b, u, gw0); gx0_0 = fmaf(W2_0_b, u, gx0_0);
      }
      if (gwp) gwp[256] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W3_0_b * X1_0_b; float u = 0.f;
        u = fmaf(Y0_b, G7_0, u); gy0 = fmaf(q, G7_0, gy0);
        gw0 = fmaf(X1_0_b, u, gw0); gx1_0 = fmaf(W3_0_b, u, gx1_0);
      }
      { const float q = W3_0_b * X2_0_b; float u = 0.f;
        u = fmaf(Y0_b, G8_0, u); gy0 = fmaf(q, G8_0, gy0);
        gw0 = fmaf(X2_0_b, u, gw0); gx2_0 = fmaf(W3_0_b, u, gx2_0);
      }
      { const float q = W3_0_b * X3_0_b; float u = 0.f;
        u = fmaf(Y0_b, G9_0, u); gy0 = fmaf(q, G9_0, gy0);
        gw0 = fmaf(X3_0_b, u, gw0); gx3_0 = fmaf(W3_0_b, u, gx3_0);
      }
      if (gwp) gwp[384] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W4_0_b * X1_0_b; float u = 0.f;
        u = fmaf(Y4_b, G10_0, u); gy4 = fmaf(q, G10_0, gy4);
        u = fmaf(Y5_b, G11_0, u); gy5 = fmaf(q, G11_0, gy5);
        u = fmaf(Y6_b, G12_0, u); gy6 = fmaf(q, G12_0, gy6);
        u = fmaf(Y8_b, G13_0, u); gy8 = fmaf(q, G13_0, gy8);
        gw0 = fmaf(X1_0_b, u, gw0); gx1_0 = fmaf(W4_0_b, u, gx1_0);
      }
      { const float q = W4_0_b * X2_0_b; float u = 0.f;
        u = fmaf(Y5_b, G14_0, u); gy5 = fmaf(q, G14_0, gy5);
        u = fmaf(Y6_b, G15_0, u); gy6 = fmaf(q, G15_0, gy6);
        u = fmaf(Y7_b, G16_0, u); gy7 = fmaf(q, G16_0, gy7);
        gw0 = fmaf(X2_0_b, u, gw0); gx2_0 = fmaf(W4_0_b, u, gx2_0);
      }
      { const float q = W4_0_b * X3_0_b; float u = 0.f;
        u = fmaf(Y4_b, G17_0, u); gy4 = fmaf(q, G17_0, gy4);
        u = fmaf(Y6_b, G18_0, u); gy6 = fmaf(q, G18_0, gy6);
        u = fmaf(Y7_b, G19_0, u); gy7 = fmaf(q, G19_0, gy7);
        u = fmaf(Y8_b, G20_0, u); gy8 = fmaf(q, G20_0, gy8);
        gw0 = fmaf(X3_0_b, u, gw0); gx3_0 = fmaf(W4_0_b, u, gx3_0);
      }
      if (gwp) gwp[512] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W5_0_b * X0_0_b; float u = 0.f;
        u = fmaf(Y4_b, G21_0, u); gy4 = fmaf(q, G21_0, gy4);
        u = fmaf(Y5_b, G22_0, u); gy5 = fmaf(q, G22_0, gy5);
        u = fmaf(Y6_b, G23_0, u); gy6 = fmaf(q, G23_0, gy6);
        u = fmaf(Y7_b, G24_0, u); gy7 = fmaf(q, G24_0, gy7);
        u = fmaf(Y8_b, G25_0, u); gy8 = fmaf(q, G25_0, gy8);
        gw0 = fmaf(X0_0_b, u, gw0); gx0_0 = fmaf(W5_0_b, u, gx0_0);
      }
      if (gwp) gwp[640] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W6_0_b * X1_0_b; float u = 0.f;
        u = fmaf(Y1_b, G26_0, u); gy1 = fmaf(q, G26_0, gy1);
        u = fmaf(Y2_b, G27_0, u); gy2 = fmaf(q, G27_0, gy2);
        u = fmaf(Y3_b, G28_0, u); gy3 = fmaf(q, G28_0, gy3);
        gw0 = fmaf(X1_0_b, u, gw0); gx1_0 = fmaf(W6_0_b, u, gx1_0);
      }
      { const float q = W6_0_b * X2_0_b; float u = 0.f;
        u = fmaf(Y1_b, G29_0, u); gy1 = fmaf(q, G29_0, gy1);
        u = fmaf(Y2_b, G30_0, u); gy2 = fmaf(q, G30_0, gy2);
        u = fmaf(Y3_b, G31_0, u); gy3 = fmaf(q, G31_0, gy3);
        gw0 = fmaf(X2_0_b, u, gw0); gx2_0 = fmaf(W6_0_b, u, gx2_0);
      }
      { const float q = W6_0_b * X3_0_b; float u = 0.f;
        u = fmaf(Y1_b, G32_0, u); gy1 = fmaf(q, G32_0, gy1);
        u = fmaf(Y2_b, G33_0, u); gy2 = fmaf(q, G33_0, gy2);
        u = fmaf(Y3_b, G34_0, u); gy3 = fmaf(q, G34_0, gy3);
        gw0 = fmaf(X3_0_b, u, gw0); gx3_0 = fmaf(W6_0_b, u, gx3_0);
      }
      if (gwp) gwp[768] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W7_0_b * X1_0_b; float u = 0.f;
        u = fmaf(Y9_b, G35_0, u); gy9 = fmaf(q, G35_0, gy9);
        u = fmaf(Y10_b, G36_0, u); gy10 = fmaf(q, G36_0, gy10);
        u = fmaf(Y11_b, G37_0, u); gy11 = fmaf(q, G37_0, gy11);
        u = fmaf(Y12_b, G38_0, u); gy12 = fmaf(q, G38_0, gy12);
        u = fmaf(Y13_b, G39_0, u); gy13 = fmaf(q, G39_0, gy13);
        u = fmaf(Y14_b, G40_0, u); gy14 = fmaf(q, G40_0, gy14);
        u = fmaf(Y15_b, G41_0, u); gy15 = fmaf(q, G41_0, gy15);
        gw0 = fmaf(X1_0_b, u, gw0); gx1_0 = fmaf(W7_0_b, u, gx1_0);
      }
      { const float q = W7_0_b * X2_0_b; float u = 0.f;
        u = fmaf(Y10_b, G42_0, u); gy10 = fmaf(q, G42_0, gy10);
        u = fmaf(Y11_b, G43_0, u); gy11 = fmaf(q, G43_0, gy11);
        u = fmaf(Y12_b, G44_0, u); gy12 = fmaf(q, G44_0, gy12);
        u = fmaf(Y13_b, G45_0, u); gy13 = fmaf(q, G45_0, gy13);
        u = fmaf(Y14_b, G46_0, u); gy14 = fmaf(q, G46_0, gy14);
        gw0 = fmaf(X2_0_b, u, gw0); gx2_0 = fmaf(W7_0_b, u, gx2_0);
      }
      { const float q = W7_0_b * X3_0_b; float u = 0.f;
        u = fmaf(Y9_b, G47_0, u); gy9 = fmaf(q, G47_0, gy9);
        u = fmaf(Y10_b, G48_0, u); gy10 = fmaf(q, G48_0, gy10);
        u = fmaf(Y11_b, G49_0, u); gy11 = fmaf(q, G49_0, gy11);
        u = fmaf(Y12_b, G50_0, u); gy12 = fmaf(q, G50_0, gy12);
        u = fmaf(Y13_b, G51_0, u); gy13 = fmaf(q, G51_0, gy13);
        u = fmaf(Y14_b, G52_0, u); gy14 = fmaf(q, G52_0, gy14);
        u = fmaf(Y15_b, G53_0, u); gy15 = fmaf(q, G53_0, gy15);
        gw0 = fmaf(X3_0_b, u, gw0); gx3_0 = fmaf(W7_0_b, u, gx3_0);
      }
      if (gwp) gwp[896] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W8_0_b * X0_0_b; float u = 0.f;
        u = fmaf(Y9_b, G54_0, u); gy9 = fmaf(q, G54_0, gy9);
        u = fmaf(Y10_b, G55_0, u); gy10 = fmaf(q, G55_0, gy10);
        u = fmaf(Y11_b, G56_0, u); gy11 = fmaf(q, G56_0, gy11);
        u = fmaf(Y12_b, G57_0, u); gy12 = fmaf(q, G57_0, gy12);
        u = fmaf(Y13_b, G58_0, u); gy13 = fmaf(q, G58_0, gy13);
        u = fmaf(Y14_b, G59_0, u); gy14 = fmaf(q, G59_0, gy14);
        u = fmaf(Y15_b, G60_0, u); gy15 = fmaf(q, G60_0, gy15);
        gw0 = fmaf(X0_0_b, u, gw0); gx0_0 = fmaf(W8_0_b, u, gx0_0);
      }
      if (gwp) gwp[1024] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W9_0_b * X1_0_b; float u = 0.f;
        u = fmaf(Y4_b, G61_0, u); gy4 = fmaf(q, G61_0, gy4);
        u = fmaf(Y5_b, G62_0, u); gy5 = fmaf(q, G62_0, gy5);
        u = fmaf(Y6_b, G63_0, u); gy6 = fmaf(q, G63_0, gy6);
        u = fmaf(Y7_b, G64_0, u); gy7 = fmaf(q, G64_0, gy7);
        u = fmaf(Y8_b, G65_0, u); gy8 = fmaf(q, G65_0, gy8);
        gw0 = fmaf(X1_0_b, u, gw0); gx1_0 = fmaf(W9_0_b, u, gx1_0);
      }
      { const float q = W9_0_b * X2_0_b; float u = 0.f;
        u = fmaf(Y4_b, G66_0, u); gy4 = fmaf(q, G66_0, gy4);
        u = fmaf(Y5_b, G67_0, u); gy5 = fmaf(q, G67_0, gy5);
        u = fmaf(Y6_b, G68_0, u); gy6 = fmaf(q, G68_0, gy6);
        u = fmaf(Y7_b, G69_0, u); gy7 = fmaf(q, G69_0, gy7);
        u = fmaf(Y8_b, G70_0, u); gy8 = fmaf(q, G70_0, gy8);
        gw0 = fmaf(X2_0_b, u, gw0); gx2_0 = fmaf(W9_0_b, u, gx2_0);
      }
      { const float q = W9_0_b * X3_0_b; float u = 0.f;
        u = fmaf(Y4_b, G71_0, u); gy4 = fmaf(q, G71_0, gy4);
        u = fmaf(Y5_b, G72_0, u); gy5 = fmaf(q, G72_0, gy5);
        u = fmaf(Y6_b, G73_0, u); gy6 = fmaf(q, G73_0, gy6);
        u = fmaf(Y7_b, G74_0, u); gy7 = fmaf(q, G74_0, gy7);
        u = fmaf(Y8_b, G75_0, u); gy8 = fmaf(q, G75_0, gy8);
        gw0 = fmaf(X3_0_b, u, gw0); gx3_0 = fmaf(W9_0_b, u, gx3_0);
      }
      if (gwp) gwp[1152] = gw0;
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
      atomicAdd(gxp + 128, gx1_0);
      atomicAdd(gxp + 256, gx2_0);
      atomicAdd(gxp + 384, gx3_0);
    }
    }
  }
}

extern "C" int mm_tpw_l2_fwd_n(long E, const int* rowptr, int nR, const int* eid, const int* send, const float* Y,
    long y_stride, const float* W, long w_stride, const float* X, long x_stride, float* out, long out_stride,
    hipStream_t stream) {
  MM_CHECK_ARG(nR >= 0, "bad sizes");
  MM_CHECK_ARG(y_stride >= 16 && w_stride >= 1280 && x_stride >= 512 && out_stride >= 5120,
               "row strides smaller than the path table's widths");
  if (nR == 0) return MM_OK;
  const long waves = (long)nR * 1;
  // E < 0: unknown, shared where the receivers alone leave most of the chip idle
  // (a launch takes fewer than 2^32 threads)
  const bool shared = E < 0 ? waves <= 2048 : true && waves < (1L << 24) && E >= 10L * nR;
  dim3 grid((unsigned)(shared ? waves : (waves + 3) / 4)), block(256);
  hipLaunchKernelGGL(shared ? mm_tpw_l2_fwd_shared_kernel : mm_tpw_l2_fwd_kernel, grid, block, 0, stream, rowptr, nR, eid, send, Y, y_stride, W,
                     w_stride, X, x_stride, out, out_stride);
  return mm::launch_status("mm_tpw_l2_fwd");
}

extern "C" int mm_tpw_l2_fwd(const int* rowptr, int nR, const int* eid, const int* send, const float* Y,
    long y_stride, const float* W, long w_stride, const float* X, long x_stride,
    float* out, long out_stride, hipStream_t stream) {
  return mm_tpw_l2_fwd_n(-1, rowptr, nR, eid, send, Y, y_stride, W, w_stride, X, x_stride, out, out_stride, stream);
}

extern "C" int mm_tpw_l2_bwd_n(long E, const int* rowptr, int nR, const int* eid, const int* send, const float* Y,
    long y_stride, const float* W, long w_stride, const float* X, long x_stride, const float* gO, long g_stride,
    float* gW, long gw_stride, float* gYp, long gy_cb_stride, float* gX, long gx_stride, hipStream_t stream) {
  MM_CHECK_ARG(nR >= 0, "bad sizes");
  MM_CHECK_ARG(y_stride >= 16 && w_stride >= 1280 && x_stride >= 512 && g_stride >= 5120,
               "row strides smaller than the path table's widths");
  MM_CHECK_ARG(!gW || gw_stride >= 1280, "gW row stride");
  MM_CHECK_ARG(!gX || gx_stride >= 512, "gX row stride");
  if (nR == 0) return MM_OK;
  const long waves = (long)nR * 2;
  // E < 0: unknown, shared where the receivers alone leave most of the chip idle
  // (a launch takes fewer than 2^32 threads)
  const bool shared = E < 0 ? waves <= 2048 : true && waves < (1L << 24) && E >= 10L * nR;
  dim3 grid((unsigned)(shared ? waves : (waves + 3) / 4)), block(256);
  hipLaunchKernelGGL(shared ? mm_tpw_l2_bwd_shared_kernel : mm_tpw_l2_bwd_kernel, grid, block, 0, stream, rowptr, nR, eid, send, Y, y_stride, W,
                     w_stride, X, x_stride, gO, g_stride, gW, gw_stride, gYp, gy_cb_stride, gX, gx_stride);
  return mm::launch_status("mm_tpw_l2_bwd");
}

extern "C" int mm_tpw_l2_bwd(const int* rowptr, int nR, const int* eid, const int* send, const float* Y,
    long y_stride, const float* W, long w_stride, const float* X, long x_stride,
    const float* gO, long g_stride, float* gW, long gw_stride, float* gYp, long gy_cb_stride, float* gX,
    long gx_stride, hipStream_t stream) {
  return mm_tpw_l2_bwd_n(-1, rowptr, nR, eid, send, Y, y_stride, W, w_stride, X, x_stride, gO, g_stride, gW, gw_stride, gYp, gy_cb_stride, gX, gx_stride, stream);
}
