// generated by mace_onegpu/codegen.py -- explicit-weight channelwise TP 'l0123'
// nX=16, nW=23, nO=99, terms=353
//
// out[i, o, c] = sum_{p in [rowptr[i], rowptr[i+1])} sum_terms coef * W[e, w, c] * X[send[e], k, c] * Y[e, m],
// e = eid[p] (or p when eid is null): receiver-CSR over a permutation, so edges need not be stored sorted.
// Forward: one wave per receiver and channel half, 1 channel(s) per lane (c = 64 h + lane + 64 j),
// 2 wave(s) per receiver, 1 edge(s) loaded together.  Backward: 1 channel(s) per lane, 2 wave(s)
// per receiver, 1 edge(s) loaded together; dL/dY partials: 6 per edge (one per channel half).
#include "../common.h"

extern "C" __global__ void __launch_bounds__(256)
mm_tpw_l0123_fwd_kernel(const int* __restrict__ rowptr, int nR, const int* __restrict__ eid,
    const int* __restrict__ send, const float* __restrict__ Y, long y_stride, const float* __restrict__ W,
    long w_stride, const float* __restrict__ X, long x_stride, float* __restrict__ out, long out_stride) {
  const int gw = blockIdx.x * 4 + (threadIdx.x >> 6);   // global wave: receiver i, sub-wave h
  const int i = gw / 2, h = gw % 2;
  if (i >= nR) return;
  const int lane = threadIdx.x & 63;
  const int c = h * 64 + lane;
  const int p0 = rowptr[i], p1 = rowptr[i + 1];
  float acc0_0 = 0.f;
  float acc1_0 = 0.f;
  float acc2_0 = 0.f;
  float acc3_0 = 0.f;
  float acc4_0 = 0.f;
  float acc5_0 = 0.f;
  float acc6_0 = 0.f;
  float acc7_0 = 0.f;
  float acc8_0 = 0.f;
  float acc9_0 = 0.f;
  float acc10_0 = 0.f;
  float acc11_0 = 0.f;
  float acc12_0 = 0.f;
  float acc13_0 = 0.f;
  float acc14_0 = 0.f;
  float acc15_0 = 0.f;
  float acc16_0 = 0.f;
  float acc17_0 = 0.f;
  float acc18_0 = 0.f;
  float acc19_0 = 0.f;
  float acc20_0 = 0.f;
  float acc21_0 = 0.f;
  float acc22_0 = 0.f;
  float acc23_0 = 0.f;
  float acc24_0 = 0.f;
  float acc25_0 = 0.f;
  float acc26_0 = 0.f;
  float acc27_0 = 0.f;
  float acc28_0 = 0.f;
  float acc29_0 = 0.f;
  float acc30_0 = 0.f;
  float acc31_0 = 0.f;
  float acc32_0 = 0.f;
  float acc33_0 = 0.f;
  float acc34_0 = 0.f;
  float acc35_0 = 0.f;
  float acc36_0 = 0.f;
  float acc37_0 = 0.f;
  float acc38_0 = 0.f;
  float acc39_0 = 0.f;
  float acc40_0 = 0.f;
  float acc41_0 = 0.f;
  float acc42_0 = 0.f;
  float acc43_0 = 0.f;
  float acc44_0 = 0.f;
  float acc45_0 = 0.f;
  float acc46_0 = 0.f;
  float acc47_0 = 0.f;
  float acc48_0 = 0.f;
  float acc49_0 = 0.f;
  float acc50_0 = 0.f;
  float acc51_0 = 0.f;
  float acc52_0 = 0.f;
  float acc53_0 = 0.f;
  float acc54_0 = 0.f;
  float acc55_0 = 0.f;
  float acc56_0 = 0.f;
  float acc57_0 = 0.f;
  float acc58_0 = 0.f;
  float acc59_0 = 0.f;
  float acc60_0 = 0.f;
  float acc61_0 = 0.f;
  float acc62_0 = 0.f;
  float acc63_0 = 0.f;
  float acc64_0 = 0.f;
  float acc65_0 = 0.f;
  float acc66_0 = 0.f;
  float acc67_0 = 0.f;
  float acc68_0 = 0.f;
  float acc69_0 = 0.f;
  float acc70_0 = 0.f;
  float acc71_0 = 0.f;
  float acc72_0 = 0.f;
  float acc73_0 = 0.f;
  float acc74_0 = 0.f;
  float acc75_0 = 0.f;
  float acc76_0 = 0.f;
  float acc77_0 = 0.f;
  float acc78_0 = 0.f;
  float acc79_0 = 0.f;
  float acc80_0 = 0.f;
  float acc81_0 = 0.f;
  float acc82_0 = 0.f;
  float acc83_0 = 0.f;
  float acc84_0 = 0.f;
  float acc85_0 = 0.f;
  float acc86_0 = 0.f;
  float acc87_0 = 0.f;
  float acc88_0 = 0.f;
  float acc89_0 = 0.f;
  float acc90_0 = 0.f;
  float acc91_0 = 0.f;
  float acc92_0 = 0.f;
  float acc93_0 = 0.f;
  float acc94_0 = 0.f;
  float acc95_0 = 0.f;
  float acc96_0 = 0.f;
  float acc97_0 = 0.f;
  float acc98_0 = 0.f;
  for (int p = p0; p < p1; ++p) {
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
    const float W10_0_a = wpa[1280];
    const float W11_0_a = wpa[1408];
    const float W12_0_a = wpa[1536];
    const float W13_0_a = wpa[1664];
    const float W14_0_a = wpa[1792];
    const float W15_0_a = wpa[1920];
    const float W16_0_a = wpa[2048];
    const float W17_0_a = wpa[2176];
    const float W18_0_a = wpa[2304];
    const float W19_0_a = wpa[2432];
    const float W20_0_a = wpa[2560];
    const float W21_0_a = wpa[2688];
    const float W22_0_a = wpa[2816];
    const float* __restrict__ xpa = X + (size_t)sa * x_stride + c;
    const float X0_0_a = xpa[0];
    const float X1_0_a = xpa[128];
    const float X2_0_a = xpa[256];
    const float X3_0_a = xpa[384];
    const float X4_0_a = xpa[512];
    const float X5_0_a = xpa[640];
    const float X6_0_a = xpa[768];
    const float X7_0_a = xpa[896];
    const float X8_0_a = xpa[1024];
    const float X9_0_a = xpa[1152];
    const float X10_0_a = xpa[1280];
    const float X11_0_a = xpa[1408];
    const float X12_0_a = xpa[1536];
    const float X13_0_a = xpa[1664];
    const float X14_0_a = xpa[1792];
    const float X15_0_a = xpa[1920];
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
    { const float q = W0_0_a * X0_0_a;
      acc0_0 = fmaf(q, Y0_a, acc0_0);
    }
    { const float q = W1_0_a * X1_0_a;
      const float q0 = 0.5773502691896257f * q;
      acc1_0 = fmaf(q0, Y1_a, acc1_0);
    }
    { const float q = W1_0_a * X2_0_a;
      const float q0 = 0.5773502691896258f * q;
      acc1_0 = fmaf(q0, Y2_a, acc1_0);
    }
    { const float q = W1_0_a * X3_0_a;
      const float q0 = 0.5773502691896257f * q;
      acc1_0 = fmaf(q0, Y3_a, acc1_0);
    }
    { const float q = W2_0_a * X4_0_a;
      const float q0 = 0.4472135954999579f * q;
      acc2_0 = fmaf(q0, Y4_a, acc2_0);
    }
    { const float q = W2_0_a * X5_0_a;
      const float q0 = 0.4472135954999579f * q;
      acc2_0 = fmaf(q0, Y5_a, acc2_0);
    }
    { const float q = W2_0_a * X6_0_a;
      const float q0 = 0.44721359549995804f * q;
      acc2_0 = fmaf(q0, Y6_a, acc2_0);
    }
    { const float q = W2_0_a * X7_0_a;
      const float q0 = 0.4472135954999579f * q;
      acc2_0 = fmaf(q0, Y7_a, acc2_0);
    }
    { const float q = W2_0_a * X8_0_a;
      const float q0 = 0.4472135954999579f * q;
      acc2_0 = fmaf(q0, Y8_a, acc2_0);
    }
    { const float q = W3_0_a * X9_0_a;
      const float q0 = 0.3779644730092272f * q;
      acc3_0 = fmaf(q0, Y9_a, acc3_0);
    }
    { const float q = W3_0_a * X10_0_a;
      const float q0 = 0.3779644730092272f * q;
      acc3_0 = fmaf(q0, Y10_a, acc3_0);
    }
    { const float q = W3_0_a * X11_0_a;
      const float q0 = 0.3779644730092272f * q;
      acc3_0 = fmaf(q0, Y11_a, acc3_0);
    }
    { const float q = W3_0_a * X12_0_a;
      const float q0 = 0.3779644730092273f * q;
      acc3_0 = fmaf(q0, Y12_a, acc3_0);
    }
    { const float q = W3_0_a * X13_0_a;
      const float q0 = 0.3779644730092272f * q;
      acc3_0 = fmaf(q0, Y13_a, acc3_0);
    }
    { const float q = W3_0_a * X14_0_a;
      const float q0 = 0.3779644730092272f * q;
      acc3_0 = fmaf(q0, Y14_a, acc3_0);
    }
    { const float q = W3_0_a * X15_0_a;
      const float q0 = 0.3779644730092272f * q;
      acc3_0 = fmaf(q0, Y15_a, acc3_0);
    }
    { const float q = W4_0_a * X0_0_a;
      acc4_0 = fmaf(q, Y1_a, acc4_0);
      acc5_0 = fmaf(q, Y2_a, acc5_0);
      acc6_0 = fmaf(q, Y3_a, acc6_0);
    }
    { const float q = W5_0_a * X1_0_a;
      acc7_0 = fmaf(q, Y0_a, acc7_0);
    }
    { const float q = W5_0_a * X2_0_a;
      acc8_0 = fmaf(q, Y0_a, acc8_0);
    }
    { const float q = W5_0_a * X3_0_a;
      acc9_0 = fmaf(q, Y0_a, acc9_0);
    }
    { const float q = W6_0_a * X1_0_a;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc12_0 = fmaf(q0, Y4_a, acc12_0);
      acc11_0 = fmaf(q0, Y5_a, acc11_0);
      acc10_0 = fmaf(-q1, Y6_a, acc10_0);
      acc10_0 = fmaf(-q0, Y8_a, acc10_0);
    }
    { const float q = W6_0_a * X2_0_a;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.632455532033676f * q;
      acc10_0 = fmaf(q0, Y5_a, acc10_0);
      acc11_0 = fmaf(q1, Y6_a, acc11_0);
      acc12_0 = fmaf(q0, Y7_a, acc12_0);
    }
    { const float q = W6_0_a * X3_0_a;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc10_0 = fmaf(q0, Y4_a, acc10_0);
      acc12_0 = fmaf(-q1, Y6_a, acc12_0);
      acc11_0 = fmaf(q0, Y7_a, acc11_0);
      acc12_0 = fmaf(q0, Y8_a, acc12_0);
    }
    { const float q = W7_0_a * X4_0_a;
      const float q0 = 0.547722557505166f * q;
      acc15_0 = fmaf(q0, Y1_a, acc15_0);
      acc13_0 = fmaf(q0, Y3_a, acc13_0);
    }
    { const float q = W7_0_a * X5_0_a;
      const float q0 = 0.547722557505166f * q;
      acc14_0 = fmaf(q0, Y1_a, acc14_0);
      acc13_0 = fmaf(q0, Y2_a, acc13_0);
    }
    { const float q = W7_0_a * X6_0_a;
      const float q0 = 0.31622776601683794f * q;
      const float q1 = 0.632455532033676f * q;
      acc13_0 = fmaf(-q0, Y1_a, acc13_0);
      acc14_0 = fmaf(q1, Y2_a, acc14_0);
      acc15_0 = fmaf(-q0, Y3_a, acc15_0);
    }
    { const float q = W7_0_a * X7_0_a;
      const float q0 = 0.547722557505166f * q;
      acc15_0 = fmaf(q0, Y2_a, acc15_0);
      acc14_0 = fmaf(q0, Y3_a, acc14_0);
    }
    { const float q = W7_0_a * X8_0_a;
      const float q0 = 0.547722557505166f * q;
      acc13_0 = fmaf(-q0, Y1_a, acc13_0);
      acc15_0 = fmaf(q0, Y3_a, acc15_0);
    }
    { const float q = W8_0_a * X4_0_a;
      const float q0 = 0.4629100498862757f * q;
      const float q1 = 0.3779644730092272f * q;
      const float q2 = 0.11952286093343936f * q;
      acc18_0 = fmaf(q0, Y9_a, acc18_0);
      acc17_0 = fmaf(q1, Y10_a, acc17_0);
      acc18_0 = fmaf(-q2, Y11_a, acc18_0);
      acc16_0 = fmaf(-q2, Y13_a, acc16_0);
      acc16_0 = fmaf(-q0, Y15_a, acc16_0);
    }
    { const float q = W8_0_a * X5_0_a;
      const float q0 = 0.3779644730092272f * q;
      const float q1 = 0.47809144373375745f * q;
      const float q2 = 0.29277002188456f * q;
      acc18_0 = fmaf(q0, Y10_a, acc18_0);
      acc17_0 = fmaf(q1, Y11_a, acc17_0);
      acc16_0 = fmaf(-q2, Y12_a, acc16_0);
      acc16_0 = fmaf(-q0, Y14_a, acc16_0);
    }
    { const float q = W8_0_a * X6_0_a;
      const float q0 = 0.41403933560541256f * q;
      const float q1 = 0.5070925528371102f * q;
      acc16_0 = fmaf(q0, Y11_a, acc16_0);
      acc17_0 = fmaf(q1, Y12_a, acc17_0);
      acc18_0 = fmaf(q0, Y13_a, acc18_0);
    }
    { const float q = W8_0_a * X7_0_a;
      const float q0 = 0.3779644730092272f * q;
      const float q1 = 0.29277002188456f * q;
      const float q2 = 0.47809144373375745f * q;
      acc16_0 = fmaf(q0, Y10_a, acc16_0);
      acc18_0 = fmaf(-q1, Y12_a, acc18_0);
      acc17_0 = fmaf(q2, Y13_a, acc17_0);
      acc18_0 = fmaf(q0, Y14_a, acc18_0);
    }
    { const float q = W8_0_a * X8_0_a;
      const float q0 = 0.4629100498862757f * q;
      const float q1 = 0.11952286093343936f * q;
      const float q2 = 0.3779644730092272f * q;
      acc16_0 = fmaf(q0, Y9_a, acc16_0);
      acc16_0 = fmaf(q1, Y11_a, acc16_0);
      acc18_0 = fmaf(-q1, Y13_a, acc18_0);
      acc17_0 = fmaf(q2, Y14_a, acc17_0);
      acc18_0 = fmaf(q0, Y15_a, acc18_0);
    }
    { const float q = W9_0_a * X9_0_a;
      const float q0 = 0.4629100498862757f * q;
      acc21_0 = fmaf(q0, Y4_a, acc21_0);
      acc19_0 = fmaf(q0, Y8_a, acc19_0);
    }
    { const float q = W9_0_a * X10_0_a;
      const float q0 = 0.3779644730092272f * q;
      acc20_0 = fmaf(q0, Y4_a, acc20_0);
      acc21_0 = fmaf(q0, Y5_a, acc21_0);
      acc19_0 = fmaf(q0, Y7_a, acc19_0);
    }
    { const float q = W9_0_a * X11_0_a;
      const float q0 = 0.11952286093343936f * q;
      const float q1 = 0.47809144373375745f * q;
      const float q2 = 0.41403933560541256f * q;
      acc21_0 = fmaf(-q0, Y4_a, acc21_0);
      acc20_0 = fmaf(q1, Y5_a, acc20_0);
      acc19_0 = fmaf(q2, Y6_a, acc19_0);
      acc19_0 = fmaf(q0, Y8_a, acc19_0);
    }
    { const float q = W9_0_a * X12_0_a;
      const float q0 = 0.29277002188456f * q;
      const float q1 = 0.5070925528371102f * q;
      acc19_0 = fmaf(-q0, Y5_a, acc19_0);
      acc20_0 = fmaf(q1, Y6_a, acc20_0);
      acc21_0 = fmaf(-q0, Y7_a, acc21_0);
    }
    { const float q = W9_0_a * X13_0_a;
      const float q0 = 0.11952286093343936f * q;
      const float q1 = 0.41403933560541256f * q;
      const float q2 = 0.47809144373375745f * q;
      acc19_0 = fmaf(-q0, Y4_a, acc19_0);
      acc21_0 = fmaf(q1, Y6_a, acc21_0);
      acc20_0 = fmaf(q2, Y7_a, acc20_0);
      acc21_0 = fmaf(-q0, Y8_a, acc21_0);
    }
    { const float q = W9_0_a * X14_0_a;
      const float q0 = 0.3779644730092272f * q;
      acc19_0 = fmaf(-q0, Y5_a, acc19_0);
      acc21_0 = fmaf(q0, Y7_a, acc21_0);
      acc20_0 = fmaf(q0, Y8_a, acc20_0);
    }
    { const float q = W9_0_a * X15_0_a;
      const float q0 = 0.4629100498862757f * q;
      acc19_0 = fmaf(-q0, Y4_a, acc19_0);
      acc21_0 = fmaf(q0, Y8_a, acc21_0);
    }
    { const float q = W10_0_a * X0_0_a;
      acc22_0 = fmaf(q, Y4_a, acc22_0);
      acc23_0 = fmaf(q, Y5_a, acc23_0);
      acc24_0 = fmaf(q, Y6_a, acc24_0);
      acc25_0 = fmaf(q, Y7_a, acc25_0);
      acc26_0 = fmaf(q, Y8_a, acc26_0);
    }
    { const float q = W11_0_a * X1_0_a;
      const float q0 = 0.408248290463863f * q;
      const float q1 = 0.7071067811865475f * q;
      acc29_0 = fmaf(q0, Y1_a, acc29_0);
      acc31_0 = fmaf(q1, Y1_a, acc31_0);
      acc28_0 = fmaf(-q1, Y2_a, acc28_0);
      acc27_0 = fmaf(-q1, Y3_a, acc27_0);
    }
    { const float q = W11_0_a * X2_0_a;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.8164965809277261f * q;
      acc28_0 = fmaf(-q0, Y1_a, acc28_0);
      acc29_0 = fmaf(-q1, Y2_a, acc29_0);
      acc30_0 = fmaf(-q0, Y3_a, acc30_0);
    }
    { const float q = W11_0_a * X3_0_a;
      const float q0 = 0.7071067811865475f * q;
      const float q1 = 0.408248290463863f * q;
      acc27_0 = fmaf(-q0, Y1_a, acc27_0);
      acc30_0 = fmaf(-q0, Y2_a, acc30_0);
      acc29_0 = fmaf(q1, Y3_a, acc29_0);
      acc31_0 = fmaf(-q0, Y3_a, acc31_0);
    }
    { const float q = W12_0_a * X1_0_a;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.5345224838248488f * q;
      const float q3 = 0.15430334996209188f * q;
      const float q4 = 0.3779644730092272f * q;
      acc36_0 = fmaf(q0, Y9_a, acc36_0);
      acc35_0 = fmaf(q1, Y10_a, acc35_0);
      acc34_0 = fmaf(q2, Y11_a, acc34_0);
      acc36_0 = fmaf(q3, Y11_a, acc36_0);
      acc33_0 = fmaf(-q4, Y12_a, acc33_0);
      acc32_0 = fmaf(-q3, Y13_a, acc32_0);
      acc33_0 = fmaf(-q1, Y14_a, acc33_0);
      acc32_0 = fmaf(-q0, Y15_a, acc32_0);
    }
    { const float q = W12_0_a * X2_0_a;
      const float q0 = 0.48795003647426655f * q;
      const float q1 = 0.6172133998483676f * q;
      const float q2 = 0.6546536707079772f * q;
      acc32_0 = fmaf(q0, Y10_a, acc32_0);
      acc33_0 = fmaf(q1, Y11_a, acc33_0);
      acc34_0 = fmaf(q2, Y12_a, acc34_0);
      acc35_0 = fmaf(q1, Y13_a, acc35_0);
      acc36_0 = fmaf(q0, Y14_a, acc36_0);
    }
    { const float q = W12_0_a * X3_0_a;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.15430334996209188f * q;
      const float q3 = 0.3779644730092272f * q;
      const float q4 = 0.5345224838248488f * q;
      acc32_0 = fmaf(q0, Y9_a, acc32_0);
      acc33_0 = fmaf(q1, Y10_a, acc33_0);
      acc32_0 = fmaf(-q2, Y11_a, acc32_0);
      acc35_0 = fmaf(-q3, Y12_a, acc35_0);
      acc34_0 = fmaf(q4, Y13_a, acc34_0);
      acc36_0 = fmaf(-q2, Y13_a, acc36_0);
      acc35_0 = fmaf(q1, Y14_a, acc35_0);
      acc36_0 = fmaf(q0, Y15_a, acc36_0);
    }
    { const float q = W13_0_a * X4_0_a;
      acc37_0 = fmaf(q, Y0_a, acc37_0);
    }
    { const float q = W13_0_a * X5_0_a;
      acc38_0 = fmaf(q, Y0_a, acc38_0);
    }
    { const float q = W13_0_a * X6_0_a;
      acc39_0 = fmaf(q, Y0_a, acc39_0);
    }
    { const float q = W13_0_a * X7_0_a;
      acc40_0 = fmaf(q, Y0_a, acc40_0);
    }
    { const float q = W13_0_a * X8_0_a;
      acc41_0 = fmaf(q, Y0_a, acc41_0);
    }
    { const float q = W14_0_a * X4_0_a;
      const float q0 = 0.5345224838248488f * q;
      const float q1 = 0.46291004988627565f * q;
      acc44_0 = fmaf(q0, Y4_a, acc44_0);
      acc45_0 = fmaf(-q1, Y5_a, acc45_0);
      acc42_0 = fmaf(q0, Y6_a, acc42_0);
      acc43_0 = fmaf(-q1, Y7_a, acc43_0);
    }
    { const float q = W14_0_a * X5_0_a;
      const float q0 = 0.46291004988627565f * q;
      const float q1 = 0.2672612419124244f * q;
      acc45_0 = fmaf(-q0, Y4_a, acc45_0);
      acc44_0 = fmaf(-q1, Y5_a, acc44_0);
      acc46_0 = fmaf(q0, Y5_a, acc46_0);
      acc43_0 = fmaf(-q1, Y6_a, acc43_0);
      acc42_0 = fmaf(-q0, Y7_a, acc42_0);
      acc43_0 = fmaf(q0, Y8_a, acc43_0);
    }
    { const float q = W14_0_a * X6_0_a;
      const float q0 = 0.5345224838248488f * q;
      const float q1 = 0.2672612419124244f * q;
      acc42_0 = fmaf(q0, Y4_a, acc42_0);
      acc43_0 = fmaf(-q1, Y5_a, acc43_0);
      acc44_0 = fmaf(-q0, Y6_a, acc44_0);
      acc45_0 = fmaf(-q1, Y7_a, acc45_0);
      acc46_0 = fmaf(q0, Y8_a, acc46_0);
    }
    { const float q = W14_0_a * X7_0_a;
      const float q0 = 0.46291004988627565f * q;
      const float q1 = 0.2672612419124244f * q;
      acc43_0 = fmaf(-q0, Y4_a, acc43_0);
      acc42_0 = fmaf(-q0, Y5_a, acc42_0);
      acc45_0 = fmaf(-q1, Y6_a, acc45_0);
      acc44_0 = fmaf(-q1, Y7_a, acc44_0);
      acc46_0 = fmaf(-q0, Y7_a, acc46_0);
      acc45_0 = fmaf(-q0, Y8_a, acc45_0);
    }
    { const float q = W14_0_a * X8_0_a;
      const float q0 = 0.46291004988627565f * q;
      const float q1 = 0.5345224838248488f * q;
      acc43_0 = fmaf(q0, Y5_a, acc43_0);
      acc46_0 = fmaf(q1, Y6_a, acc46_0);
      acc45_0 = fmaf(-q0, Y7_a, acc45_0);
      acc44_0 = fmaf(q1, Y8_a, acc44_0);
    }
    { const float q = W15_0_a * X9_0_a;
      const float q0 = 0.5976143046671968f * q;
      acc51_0 = fmaf(q0, Y1_a, acc51_0);
      acc47_0 = fmaf(q0, Y3_a, acc47_0);
    }
    { const float q = W15_0_a * X10_0_a;
      const float q0 = 0.4879500364742667f * q;
      acc50_0 = fmaf(q0, Y1_a, acc50_0);
      acc47_0 = fmaf(q0, Y2_a, acc47_0);
      acc48_0 = fmaf(q0, Y3_a, acc48_0);
    }
    { const float q = W15_0_a * X11_0_a;
      const float q0 = 0.5345224838248489f * q;
      const float q1 = 0.1543033499620919f * q;
      const float q2 = 0.6172133998483678f * q;
      acc49_0 = fmaf(q0, Y1_a, acc49_0);
      acc51_0 = fmaf(q1, Y1_a, acc51_0);
      acc48_0 = fmaf(q2, Y2_a, acc48_0);
      acc47_0 = fmaf(-q1, Y3_a, acc47_0);
    }
    { const float q = W15_0_a * X12_0_a;
      const float q0 = 0.3779644730092273f * q;
      const float q1 = 0.6546536707079773f * q;
      acc48_0 = fmaf(-q0, Y1_a, acc48_0);
      acc49_0 = fmaf(q1, Y2_a, acc49_0);
      acc50_0 = fmaf(-q0, Y3_a, acc50_0);
    }
    { const float q = W15_0_a * X13_0_a;
      const float q0 = 0.1543033499620919f * q;
      const float q1 = 0.6172133998483678f * q;
      const float q2 = 0.5345224838248489f * q;
      acc47_0 = fmaf(-q0, Y1_a, acc47_0);
      acc50_0 = fmaf(q1, Y2_a, acc50_0);
      acc49_0 = fmaf(q2, Y3_a, acc49_0);
      acc51_0 = fmaf(-q0, Y3_a, acc51_0);
    }
    { const float q = W15_0_a * X14_0_a;
      const float q0 = 0.4879500364742667f * q;
      acc48_0 = fmaf(-q0, Y1_a, acc48_0);
      acc51_0 = fmaf(q0, Y2_a, acc51_0);
      acc50_0 = fmaf(q0, Y3_a, acc50_0);
    }
    { const float q = W15_0_a * X15_0_a;
      const float q0 = 0.5976143046671968f * q;
      acc47_0 = fmaf(-q0, Y1_a, acc47_0);
      acc51_0 = fmaf(q0, Y3_a, acc51_0);
    }
    { const float q = W16_0_a * X9_0_a;
      const float q0 = 0.545544725589981f * q;
      const float q1 = 0.38575837490522974f * q;
      const float q2 = 0.24397501823713336f * q;
      acc54_0 = fmaf(q0, Y9_a, acc54_0);
      acc55_0 = fmaf(-q1, Y10_a, acc55_0);
      acc56_0 = fmaf(q2, Y11_a, acc56_0);
      acc52_0 = fmaf(q2, Y13_a, acc52_0);
      acc53_0 = fmaf(-q1, Y14_a, acc53_0);
    }
    { const float q = W16_0_a * X10_0_a;
      const float q0 = 0.38575837490522974f * q;
      const float q1 = 0.2988071523335984f * q;
      const float q2 = 0.4879500364742667f * q;
      acc55_0 = fmaf(-q0, Y9_a, acc55_0);
      acc55_0 = fmaf(-q1, Y11_a, acc55_0);
      acc52_0 = fmaf(q2, Y12_a, acc52_0);
      acc53_0 = fmaf(-q1, Y13_a, acc53_0);
      acc53_0 = fmaf(q0, Y15_a, acc53_0);
    }
    { const float q = W16_0_a * X11_0_a;
      const float q0 = 0.24397501823713336f * q;
      const float q1 = 0.2988071523335984f * q;
      const float q2 = 0.3273268353539886f * q;
      const float q3 = 0.3779644730092273f * q;
      const float q4 = 0.15430334996209194f * q;
      acc56_0 = fmaf(q0, Y9_a, acc56_0);
      acc55_0 = fmaf(-q1, Y10_a, acc55_0);
      acc54_0 = fmaf(-q2, Y11_a, acc54_0);
      acc56_0 = fmaf(q3, Y11_a, acc56_0);
      acc53_0 = fmaf(-q4, Y12_a, acc53_0);
      acc52_0 = fmaf(-q3, Y13_a, acc52_0);
      acc53_0 = fmaf(q1, Y14_a, acc53_0);
      acc52_0 = fmaf(-q0, Y15_a, acc52_0);
    }
    { const float q = W16_0_a * X12_0_a;
      const float q0 = 0.4879500364742667f * q;
      const float q1 = 0.15430334996209194f * q;
      const float q2 = 0.4364357804719849f * q;
      acc52_0 = fmaf(q0, Y10_a, acc52_0);
      acc53_0 = fmaf(-q1, Y11_a, acc53_0);
      acc54_0 = fmaf(-q2, Y12_a, acc54_0);
      acc55_0 = fmaf(-q1, Y13_a, acc55_0);
      acc56_0 = fmaf(q0, Y14_a, acc56_0);
    }
    { const float q = W16_0_a * X13_0_a;
      const float q0 = 0.24397501823713336f * q;
      const float q1 = 0.2988071523335984f * q;
      const float q2 = 0.3779644730092273f * q;
      const float q3 = 0.15430334996209194f * q;
      const float q4 = 0.3273268353539886f * q;
      acc52_0 = fmaf(q0, Y9_a, acc52_0);
      acc53_0 = fmaf(-q1, Y10_a, acc53_0);
      acc52_0 = fmaf(-q2, Y11_a, acc52_0);
      acc55_0 = fmaf(-q3, Y12_a, acc55_0);
      acc54_0 = fmaf(-q4, Y13_a, acc54_0);
      acc56_0 = fmaf(-q2, Y13_a, acc56_0);
      acc55_0 = fmaf(-q1, Y14_a, acc55_0);
      acc56_0 = fmaf(q0, Y15_a, acc56_0);
    }
    { const float q = W16_0_a * X14_0_a;
      const float q0 = 0.38575837490522974f * q;
      const float q1 = 0.2988071523335984f * q;
      const float q2 = 0.4879500364742667f * q;
      acc53_0 = fmaf(-q0, Y9_a, acc53_0);
      acc53_0 = fmaf(q1, Y11_a, acc53_0);
      acc56_0 = fmaf(q2, Y12_a, acc56_0);
      acc55_0 = fmaf(-q1, Y13_a, acc55_0);
      acc55_0 = fmaf(-q0, Y15_a, acc55_0);
    }
    { const float q = W16_0_a * X15_0_a;
      const float q0 = 0.38575837490522974f * q;
      const float q1 = 0.24397501823713336f * q;
      const float q2 = 0.545544725589981f * q;
      acc53_0 = fmaf(q0, Y10_a, acc53_0);
      acc52_0 = fmaf(-q1, Y11_a, acc52_0);
      acc56_0 = fmaf(q1, Y13_a, acc56_0);
      acc55_0 = fmaf(-q0, Y14_a, acc55_0);
      acc54_0 = fmaf(q2, Y15_a, acc54_0);
    }
    { const float q = W17_0_a * X0_0_a;
      acc57_0 = fmaf(q, Y9_a, acc57_0);
      acc58_0 = fmaf(q, Y10_a, acc58_0);
      acc59_0 = fmaf(q, Y11_a, acc59_0);
      acc60_0 = fmaf(q, Y12_a, acc60_0);
      acc61_0 = fmaf(q, Y13_a, acc61_0);
      acc62_0 = fmaf(q, Y14_a, acc62_0);
      acc63_0 = fmaf(q, Y15_a, acc63_0);
    }
    { const float q = W18_0_a * X1_0_a;
      const float q0 = 0.18257418583505539f * q;
      const float q1 = 0.7071067811865476f * q;
      const float q2 = 0.447213595499958f * q;
      const float q3 = 0.5773502691896256f * q;
      const float q4 = 0.632455532033676f * q;
      acc68_0 = fmaf(q0, Y4_a, acc68_0);
      acc70_0 = fmaf(q1, Y4_a, acc70_0);
      acc67_0 = fmaf(q2, Y5_a, acc67_0);
      acc69_0 = fmaf(q3, Y5_a, acc69_0);
      acc66_0 = fmaf(-q4, Y6_a, acc66_0);
      acc65_0 = fmaf(-q3, Y7_a, acc65_0);
      acc64_0 = fmaf(-q1, Y8_a, acc64_0);
      acc66_0 = fmaf(-q0, Y8_a, acc66_0);
    }
    { const float q = W18_0_a * X2_0_a;
      const float q0 = 0.5773502691896258f * q;
      const float q1 = 0.7302967433402215f * q;
      const float q2 = 0.7745966692414836f * q;
      acc65_0 = fmaf(-q0, Y4_a, acc65_0);
      acc66_0 = fmaf(-q1, Y5_a, acc66_0);
      acc67_0 = fmaf(-q2, Y6_a, acc67_0);
      acc68_0 = fmaf(-q1, Y7_a, acc68_0);
      acc69_0 = fmaf(-q0, Y8_a, acc69_0);
    }
    { const float q = W18_0_a * X3_0_a;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.18257418583505539f * q;
      const float q2 = 0.5773502691896256f * q;
      const float q3 = 0.632455532033676f * q;
      const float q4 = 0.447213595499958f * q;
      acc64_0 = fmaf(-q0, Y4_a, acc64_0);
      acc66_0 = fmaf(q1, Y4_a, acc66_0);
      acc65_0 = fmaf(-q2, Y5_a, acc65_0);
      acc68_0 = fmaf(-q3, Y6_a, acc68_0);
      acc67_0 = fmaf(q4, Y7_a, acc67_0);
      acc69_0 = fmaf(-q2, Y7_a, acc69_0);
      acc68_0 = fmaf(q1, Y8_a, acc68_0);
      acc70_0 = fmaf(-q0, Y8_a, acc70_0);
    }
    { const float q = W19_0_a * X4_0_a;
      const float q0 = 0.18257418583505539f * q;
      const float q1 = 0.7071067811865476f * q;
      const float q2 = 0.5773502691896258f * q;
      acc75_0 = fmaf(q0, Y1_a, acc75_0);
      acc77_0 = fmaf(q1, Y1_a, acc77_0);
      acc72_0 = fmaf(-q2, Y2_a, acc72_0);
      acc71_0 = fmaf(-q1, Y3_a, acc71_0);
      acc73_0 = fmaf(q0, Y3_a, acc73_0);
    }
    { const float q = W19_0_a * X5_0_a;
      const float q0 = 0.447213595499958f * q;
      const float q1 = 0.5773502691896256f * q;
      const float q2 = 0.7302967433402215f * q;
      acc74_0 = fmaf(q0, Y1_a, acc74_0);
      acc76_0 = fmaf(q1, Y1_a, acc76_0);
      acc73_0 = fmaf(-q2, Y2_a, acc73_0);
      acc72_0 = fmaf(-q1, Y3_a, acc72_0);
    }
    { const float q = W19_0_a * X6_0_a;
      const float q0 = 0.632455532033676f * q;
      const float q1 = 0.7745966692414836f * q;
      acc73_0 = fmaf(-q0, Y1_a, acc73_0);
      acc74_0 = fmaf(-q1, Y2_a, acc74_0);
      acc75_0 = fmaf(-q0, Y3_a, acc75_0);
    }
    { const float q = W19_0_a * X7_0_a;
      const float q0 = 0.5773502691896256f * q;
      const float q1 = 0.7302967433402215f * q;
      const float q2 = 0.447213595499958f * q;
      acc72_0 = fmaf(-q0, Y1_a, acc72_0);
      acc75_0 = fmaf(-q1, Y2_a, acc75_0);
      acc74_0 = fmaf(q2, Y3_a, acc74_0);
      acc76_0 = fmaf(-q0, Y3_a, acc76_0);
    }
    { const float q = W19_0_a * X8_0_a;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.18257418583505539f * q;
      const float q2 = 0.5773502691896258f * q;
      acc71_0 = fmaf(-q0, Y1_a, acc71_0);
      acc73_0 = fmaf(-q1, Y1_a, acc73_0);
      acc76_0 = fmaf(-q2, Y2_a, acc76_0);
      acc75_0 = fmaf(q1, Y3_a, acc75_0);
      acc77_0 = fmaf(-q0, Y3_a, acc77_0);
    }
    { const float q = W20_0_a * X4_0_a;
      const float q0 = 0.2886751345948128f * q;
      const float q1 = 0.5773502691896258f * q;
      const float q2 = 0.447213595499958f * q;
      acc82_0 = fmaf(q0, Y9_a, acc82_0);
      acc81_0 = fmaf(q1, Y10_a, acc81_0);
      acc82_0 = fmaf(-q2, Y11_a, acc82_0);
      acc84_0 = fmaf(-q0, Y11_a, acc84_0);
      acc79_0 = fmaf(q1, Y12_a, acc79_0);
      acc78_0 = fmaf(q0, Y13_a, acc78_0);
      acc80_0 = fmaf(-q2, Y13_a, acc80_0);
      acc80_0 = fmaf(-q0, Y15_a, acc80_0);
    }
    { const float q = W20_0_a * X5_0_a;
      const float q0 = 0.45643546458763845f * q;
      const float q1 = 0.3535533905932738f * q;
      const float q2 = 0.18257418583505539f * q;
      acc83_0 = fmaf(-q0, Y9_a, acc83_0);
      acc82_0 = fmaf(-q1, Y10_a, acc82_0);
      acc84_0 = fmaf(q0, Y10_a, acc84_0);
      acc81_0 = fmaf(-q2, Y11_a, acc81_0);
      acc83_0 = fmaf(q1, Y11_a, acc83_0);
      acc80_0 = fmaf(-q2, Y12_a, acc80_0);
      acc79_0 = fmaf(-q1, Y13_a, acc79_0);
      acc78_0 = fmaf(-q0, Y14_a, acc78_0);
      acc80_0 = fmaf(q1, Y14_a, acc80_0);
      acc79_0 = fmaf(q0, Y15_a, acc79_0);
    }
    { const float q = W20_0_a * X6_0_a;
      const float q0 = 0.6454972243679029f * q;
      const float q1 = 0.3872983346207418f * q;
      const float q2 = 0.5163977794943223f * q;
      acc78_0 = fmaf(q0, Y9_a, acc78_0);
      acc80_0 = fmaf(-q1, Y11_a, acc80_0);
      acc81_0 = fmaf(-q2, Y12_a, acc81_0);
      acc82_0 = fmaf(-q1, Y13_a, acc82_0);
      acc84_0 = fmaf(q0, Y15_a, acc84_0);
    }
    { const float q = W20_0_a * X7_0_a;
      const float q0 = 0.45643546458763845f * q;
      const float q1 = 0.3535533905932738f * q;
      const float q2 = 0.18257418583505539f * q;
      acc79_0 = fmaf(-q0, Y9_a, acc79_0);
      acc78_0 = fmaf(-q0, Y10_a, acc78_0);
      acc80_0 = fmaf(-q1, Y10_a, acc80_0);
      acc79_0 = fmaf(-q1, Y11_a, acc79_0);
      acc82_0 = fmaf(-q2, Y12_a, acc82_0);
      acc81_0 = fmaf(-q2, Y13_a, acc81_0);
      acc83_0 = fmaf(-q1, Y13_a, acc83_0);
      acc82_0 = fmaf(-q1, Y14_a, acc82_0);
      acc84_0 = fmaf(-q0, Y14_a, acc84_0);
      acc83_0 = fmaf(-q0, Y15_a, acc83_0);
    }
    { const float q = W20_0_a * X8_0_a;
      const float q0 = 0.2886751345948128f * q;
      const float q1 = 0.447213595499958f * q;
      const float q2 = 0.5773502691896258f * q;
      acc80_0 = fmaf(q0, Y9_a, acc80_0);
      acc78_0 = fmaf(q0, Y11_a, acc78_0);
      acc80_0 = fmaf(q1, Y11_a, acc80_0);
      acc83_0 = fmaf(q2, Y12_a, acc83_0);
      acc82_0 = fmaf(-q1, Y13_a, acc82_0);
      acc84_0 = fmaf(q0, Y13_a, acc84_0);
      acc81_0 = fmaf(q2, Y14_a, acc81_0);
      acc82_0 = fmaf(q0, Y15_a, acc82_0);
    }
    { const float q = W21_0_a * X9_0_a;
      acc85_0 = fmaf(q, Y0_a, acc85_0);
    }
    { const float q = W21_0_a * X10_0_a;
      acc86_0 = fmaf(q, Y0_a, acc86_0);
    }
    { const float q = W21_0_a * X11_0_a;
      acc87_0 = fmaf(q, Y0_a, acc87_0);
    }
    { const float q = W21_0_a * X12_0_a;
      acc88_0 = fmaf(q, Y0_a, acc88_0);
    }
    { const float q = W21_0_a * X13_0_a;
      acc89_0 = fmaf(q, Y0_a, acc89_0);
    }
    { const float q = W21_0_a * X14_0_a;
      acc90_0 = fmaf(q, Y0_a, acc90_0);
    }
    { const float q = W21_0_a * X15_0_a;
      acc91_0 = fmaf(q, Y0_a, acc91_0);
    }
    { const float q = W22_0_a * X9_0_a;
      const float q0 = 0.2886751345948128f * q;
      const float q1 = 0.45643546458763845f * q;
      const float q2 = 0.6454972243679029f * q;
      acc96_0 = fmaf(q0, Y4_a, acc96_0);
      acc97_0 = fmaf(-q1, Y5_a, acc97_0);
      acc92_0 = fmaf(q2, Y6_a, acc92_0);
      acc93_0 = fmaf(-q1, Y7_a, acc93_0);
      acc94_0 = fmaf(q0, Y8_a, acc94_0);
    }
    { const float q = W22_0_a * X10_0_a;
      const float q0 = 0.5773502691896258f * q;
      const float q1 = 0.3535533905932738f * q;
      const float q2 = 0.45643546458763845f * q;
      acc95_0 = fmaf(q0, Y4_a, acc95_0);
      acc96_0 = fmaf(-q1, Y5_a, acc96_0);
      acc98_0 = fmaf(q2, Y5_a, acc98_0);
      acc92_0 = fmaf(-q2, Y7_a, acc92_0);
      acc94_0 = fmaf(-q1, Y7_a, acc94_0);
    }
    { const float q = W22_0_a * X11_0_a;
      const float q0 = 0.447213595499958f * q;
      const float q1 = 0.2886751345948128f * q;
      const float q2 = 0.18257418583505539f * q;
      const float q3 = 0.3535533905932738f * q;
      const float q4 = 0.3872983346207418f * q;
      acc96_0 = fmaf(-q0, Y4_a, acc96_0);
      acc98_0 = fmaf(-q1, Y4_a, acc98_0);
      acc95_0 = fmaf(-q2, Y5_a, acc95_0);
      acc97_0 = fmaf(q3, Y5_a, acc97_0);
      acc94_0 = fmaf(-q4, Y6_a, acc94_0);
      acc93_0 = fmaf(-q3, Y7_a, acc93_0);
      acc92_0 = fmaf(q1, Y8_a, acc92_0);
      acc94_0 = fmaf(q0, Y8_a, acc94_0);
    }
    { const float q = W22_0_a * X12_0_a;
      const float q0 = 0.5773502691896258f * q;
      const float q1 = 0.18257418583505539f * q;
      const float q2 = 0.5163977794943223f * q;
      acc93_0 = fmaf(q0, Y4_a, acc93_0);
      acc94_0 = fmaf(-q1, Y5_a, acc94_0);
      acc95_0 = fmaf(-q2, Y6_a, acc95_0);
      acc96_0 = fmaf(-q1, Y7_a, acc96_0);
      acc97_0 = fmaf(q0, Y8_a, acc97_0);
    }
    { const float q = W22_0_a * X13_0_a;
      const float q0 = 0.2886751345948128f * q;
      const float q1 = 0.447213595499958f * q;
      const float q2 = 0.3535533905932738f * q;
      const float q3 = 0.3872983346207418f * q;
      const float q4 = 0.18257418583505539f * q;
      acc92_0 = fmaf(q0, Y4_a, acc92_0);
      acc94_0 = fmaf(-q1, Y4_a, acc94_0);
      acc93_0 = fmaf(-q2, Y5_a, acc93_0);
      acc96_0 = fmaf(-q3, Y6_a, acc96_0);
      acc95_0 = fmaf(-q4, Y7_a, acc95_0);
      acc97_0 = fmaf(-q2, Y7_a, acc97_0);
      acc96_0 = fmaf(-q1, Y8_a, acc96_0);
      acc98_0 = fmaf(q0, Y8_a, acc98_0);
    }
    { const float q = W22_0_a * X14_0_a;
      const float q0 = 0.45643546458763845f * q;
      const float q1 = 0.3535533905932738f * q;
      const float q2 = 0.5773502691896258f * q;
      acc92_0 = fmaf(-q0, Y5_a, acc92_0);
      acc94_0 = fmaf(q1, Y5_a, acc94_0);
      acc96_0 = fmaf(-q1, Y7_a, acc96_0);
      acc98_0 = fmaf(-q0, Y7_a, acc98_0);
      acc95_0 = fmaf(q2, Y8_a, acc95_0);
    }
    { const float q = W22_0_a * X15_0_a;
      const float q0 = 0.2886751345948128f * q;
      const float q1 = 0.45643546458763845f * q;
      const float q2 = 0.6454972243679029f * q;
      acc94_0 = fmaf(-q0, Y4_a, acc94_0);
      acc93_0 = fmaf(q1, Y5_a, acc93_0);
      acc98_0 = fmaf(q2, Y6_a, acc98_0);
      acc97_0 = fmaf(-q1, Y7_a, acc97_0);
      acc96_0 = fmaf(q0, Y8_a, acc96_0);
    }
  }
  float* __restrict__ op = out + (size_t)i * out_stride + c;
  op[0] = acc0_0;
  op[128] = acc1_0;
  op[256] = acc2_0;
  op[384] = acc3_0;
  op[512] = acc4_0;
  op[640] = acc5_0;
  op[768] = acc6_0;
  op[896] = acc7_0;
  op[1024] = acc8_0;
  op[1152] = acc9_0;
  op[1280] = acc10_0;
  op[1408] = acc11_0;
  op[1536] = acc12_0;
  op[1664] = acc13_0;
  op[1792] = acc14_0;
  op[1920] = acc15_0;
  op[2048] = acc16_0;
  op[2176] = acc17_0;
  op[2304] = acc18_0;
  op[2432] = acc19_0;
  op[2560] = acc20_0;
  op[2688] = acc21_0;
  op[2816] = acc22_0;
  op[2944] = acc23_0;
  op[3072] = acc24_0;
  op[3200] = acc25_0;
  op[3328] = acc26_0;
  op[3456] = acc27_0;
  op[3584] = acc28_0;
  op[3712] = acc29_0;
  op[3840] = acc30_0;
  op[3968] = acc31_0;
  op[4096] = acc32_0;
  op[4224] = acc33_0;
  op[4352] = acc34_0;
  op[4480] = acc35_0;
  op[4608] = acc36_0;
  op[4736] = acc37_0;
  op[4864] = acc38_0;
  op[4992] = acc39_0;
  op[5120] = acc40_0;
  op[5248] = acc41_0;
  op[5376] = acc42_0;
  op[5504] = acc43_0;
  op[5632] = acc44_0;
  op[5760] = acc45_0;
  op[5888] = acc46_0;
  op[6016] = acc47_0;
  op[6144] = acc48_0;
  op[6272] = acc49_0;
  op[6400] = acc50_0;
  op[6528] = acc51_0;
  op[6656] = acc52_0;
  op[6784] = acc53_0;
  op[6912] = acc54_0;
  op[7040] = acc55_0;
  op[7168] = acc56_0;
  op[7296] = acc57_0;
  op[7424] = acc58_0;
  op[7552] = acc59_0;
  op[7680] = acc60_0;
  op[7808] = acc61_0;
  op[7936] = acc62_0;
  op[8064] = acc63_0;
  op[8192] = acc64_0;
  op[8320] = acc65_0;
  op[8448] = acc66_0;
  op[8576] = acc67_0;
  op[8704] = acc68_0;
  op[8832] = acc69_0;
  op[8960] = acc70_0;
  op[9088] = acc71_0;
  op[9216] = acc72_0;
  op[9344] = acc73_0;
  op[9472] = acc74_0;
  op[9600] = acc75_0;
  op[9728] = acc76_0;
  op[9856] = acc77_0;
  op[9984] = acc78_0;
  op[10112] = acc79_0;
  op[10240] = acc80_0;
  op[10368] = acc81_0;
  op[10496] = acc82_0;
  op[10624] = acc83_0;
  op[10752] = acc84_0;
  op[10880] = acc85_0;
  op[11008] = acc86_0;
  op[11136] = acc87_0;
  op[11264] = acc88_0;
  op[11392] = acc89_0;
  op[11520] = acc90_0;
  op[11648] = acc91_0;
  op[11776] = acc92_0;
  op[11904] = acc93_0;
  op[12032] = acc94_0;
  op[12160] = acc95_0;
  op[12288] = acc96_0;
  op[12416] = acc97_0;
  op[12544] = acc98_0;
}

extern "C" __global__ void __launch_bounds__(256)
mm_tpw_l0123_fwd_shared_kernel(const int* __restrict__ rowptr, int nR, const int* __restrict__ eid,
    const int* __restrict__ send, const float* __restrict__ Y, long y_stride, const float* __restrict__ W,
    long w_stride, const float* __restrict__ X, long x_stride, float* __restrict__ out, long out_stride) {
  __shared__ float red[99 * 64];   // one wave's sums [accumulator][lane]
  const int wave = threadIdx.x >> 6;
  const int gw = blockIdx.x;   // receiver i, sub-wave h
  const int i = gw / 2, h = gw % 2;
  if (i >= nR) return;
  const int lane = threadIdx.x & 63;
  const int c = h * 64 + lane;
  const int r0 = rowptr[i], nr = rowptr[i + 1] - r0;
  const int p0 = r0 + (int)((long)nr * wave / 4), p1 = r0 + (int)((long)nr * (wave + 1) / 4);
  float acc0_0 = 0.f;
  float acc1_0 = 0.f;
  float acc2_0 = 0.f;
  float acc3_0 = 0.f;
  float acc4_0 = 0.f;
  float acc5_0 = 0.f;
  float acc6_0 = 0.f;
  float acc7_0 = 0.f;
  float acc8_0 = 0.f;
  float acc9_0 = 0.f;
  float acc10_0 = 0.f;
  float acc11_0 = 0.f;
  float acc12_0 = 0.f;
  float acc13_0 = 0.f;
  float acc14_0 = 0.f;
  float acc15_0 = 0.f;
  float acc16_0 = 0.f;
  float acc17_0 = 0.f;
  float acc18_0 = 0.f;
  float acc19_0 = 0.f;
  float acc20_0 = 0.f;
  float acc21_0 = 0.f;
  float acc22_0 = 0.f;
  float acc23_0 = 0.f;
  float acc24_0 = 0.f;
  float acc25_0 = 0.f;
  float acc26_0 = 0.f;
  float acc27_0 = 0.f;
  float acc28_0 = 0.f;
  float acc29_0 = 0.f;
  float acc30_0 = 0.f;
  float acc31_0 = 0.f;
  float acc32_0 = 0.f;
  float acc33_0 = 0.f;
  float acc34_0 = 0.f;
  float acc35_0 = 0.f;
  float acc36_0 = 0.f;
  float acc37_0 = 0.f;
  float acc38_0 = 0.f;
  float acc39_0 = 0.f;
  float acc40_0 = 0.f;
  float acc41_0 = 0.f;
  float acc42_0 = 0.f;
  float acc43_0 = 0.f;
  float acc44_0 = 0.f;
  float acc45_0 = 0.f;
  float acc46_0 = 0.f;
  float acc47_0 = 0.f;
  float acc48_0 = 0.f;
  float acc49_0 = 0.f;
  float acc50_0 = 0.f;
  float acc51_0 = 0.f;
  float acc52_0 = 0.f;
  float acc53_0 = 0.f;
  float acc54_0 = 0.f;
  float acc55_0 = 0.f;
  float acc56_0 = 0.f;
  float acc57_0 = 0.f;
  float acc58_0 = 0.f;
  float acc59_0 = 0.f;
  float acc60_0 = 0.f;
  float acc61_0 = 0.f;
  float acc62_0 = 0.f;
  float acc63_0 = 0.f;
  float acc64_0 = 0.f;
  float acc65_0 = 0.f;
  float acc66_0 = 0.f;
  float acc67_0 = 0.f;
  float acc68_0 = 0.f;
  float acc69_0 = 0.f;
  float acc70_0 = 0.f;
  float acc71_0 = 0.f;
  float acc72_0 = 0.f;
  float acc73_0 = 0.f;
  float acc74_0 = 0.f;
  float acc75_0 = 0.f;
  float acc76_0 = 0.f;
  float acc77_0 = 0.f;
  float acc78_0 = 0.f;
  float acc79_0 = 0.f;
  float acc80_0 = 0.f;
  float acc81_0 = 0.f;
  float acc82_0 = 0.f;
  float acc83_0 = 0.f;
  float acc84_0 = 0.f;
  float acc85_0 = 0.f;
  float acc86_0 = 0.f;
  float acc87_0 = 0.f;
  float acc88_0 = 0.f;
  float acc89_0 = 0.f;
  float acc90_0 = 0.f;
  float acc91_0 = 0.f;
  float acc92_0 = 0.f;
  float acc93_0 = 0.f;
  float acc94_0 = 0.f;
  float acc95_0 = 0.f;
  float acc96_0 = 0.f;
  float acc97_0 = 0.f;
  float acc98_0 = 0.f;
  for (int p = p0; p < p1; ++p) {
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
    const float W10_0_a = wpa[1280];
    const float W11_0_a = wpa[1408];
    const float W12_0_a = wpa[1536];
    const float W13_0_a = wpa[1664];
    const float W14_0_a = wpa[1792];
    const float W15_0_a = wpa[1920];
    const float W16_0_a = wpa[2048];
    const float W17_0_a = wpa[2176];
    const float W18_0_a = wpa[2304];
    const float W19_0_a = wpa[2432];
    const float W20_0_a = wpa[2560];
    const float W21_0_a = wpa[2688];
    const float W22_0_a = wpa[2816];
    const float* __restrict__ xpa = X + (size_t)sa * x_stride + c;
    const float X0_0_a = xpa[0];
    const float X1_0_a = xpa[128];
    const float X2_0_a = xpa[256];
    const float X3_0_a = xpa[384];
    const float X4_0_a = xpa[512];
    const float X5_0_a = xpa[640];
    const float X6_0_a = xpa[768];
    const float X7_0_a = xpa[896];
    const float X8_0_a = xpa[1024];
    const float X9_0_a = xpa[1152];
    const float X10_0_a = xpa[1280];
    const float X11_0_a = xpa[1408];
    const float X12_0_a = xpa[1536];
    const float X13_0_a = xpa[1664];
    const float X14_0_a = xpa[1792];
    const float X15_0_a = xpa[1920];
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
    { const float q = W0_0_a * X0_0_a;
      acc0_0 = fmaf(q, Y0_a, acc0_0);
    }
    { const float q = W1_0_a * X1_0_a;
      const float q0 = 0.5773502691896257f * q;
      acc1_0 = fmaf(q0, Y1_a, acc1_0);
    }
    { const float q = W1_0_a * X2_0_a;
      const float q0 = 0.5773502691896258f * q;
      acc1_0 = fmaf(q0, Y2_a, acc1_0);
    }
    { const float q = W1_0_a * X3_0_a;
      const float q0 = 0.5773502691896257f * q;
      acc1_0 = fmaf(q0, Y3_a, acc1_0);
    }
    { const float q = W2_0_a * X4_0_a;
      const float q0 = 0.4472135954999579f * q;
      acc2_0 = fmaf(q0, Y4_a, acc2_0);
    }
    { const float q = W2_0_a * X5_0_a;
      const float q0 = 0.4472135954999579f * q;
      acc2_0 = fmaf(q0, Y5_a, acc2_0);
    }
    { const float q = W2_0_a * X6_0_a;
      const float q0 = 0.44721359549995804f * q;
      acc2_0 = fmaf(q0, Y6_a, acc2_0);
    }
    { const float q = W2_0_a * X7_0_a;
      const float q0 = 0.4472135954999579f * q;
      acc2_0 = fmaf(q0, Y7_a, acc2_0);
    }
    { const float q = W2_0_a * X8_0_a;
      const float q0 = 0.4472135954999579f * q;
      acc2_0 = fmaf(q0, Y8_a, acc2_0);
    }
    { const float q = W3_0_a * X9_0_a;
      const float q0 = 0.3779644730092272f * q;
      acc3_0 = fmaf(q0, Y9_a, acc3_0);
    }
    { const float q = W3_0_a * X10_0_a;
      const float q0 = 0.3779644730092272f * q;
      acc3_0 = fmaf(q0, Y10_a, acc3_0);
    }
    { const float q = W3_0_a * X11_0_a;
      const float q0 = 0.3779644730092272f * q;
      acc3_0 = fmaf(q0, Y11_a, acc3_0);
    }
    { const float q = W3_0_a * X12_0_a;
      const float q0 = 0.3779644730092273f * q;
      acc3_0 = fmaf(q0, Y12_a, acc3_0);
    }
    { const float q = W3_0_a * X13_0_a;
      const float q0 = 0.3779644730092272f * q;
      acc3_0 = fmaf(q0, Y13_a, acc3_0);
    }
    { const float q = W3_0_a * X14_0_a;
      const float q0 = 0.3779644730092272f * q;
      acc3_0 = fmaf(q0, Y14_a, acc3_0);
    }
    { const float q = W3_0_a * X15_0_a;
      const float q0 = 0.3779644730092272f * q;
      acc3_0 = fmaf(q0, Y15_a, acc3_0);
    }
    { const float q = W4_0_a * X0_0_a;
      acc4_0 = fmaf(q, Y1_a, acc4_0);
      acc5_0 = fmaf(q, Y2_a, acc5_0);
      acc6_0 = fmaf(q, Y3_a, acc6_0);
    }
    { const float q = W5_0_a * X1_0_a;
      acc7_0 = fmaf(q, Y0_a, acc7_0);
    }
    { const float q = W5_0_a * X2_0_a;
      acc8_0 = fmaf(q, Y0_a, acc8_0);
    }
    { const float q = W5_0_a * X3_0_a;
      acc9_0 = fmaf(q, Y0_a, acc9_0);
    }
    { const float q = W6_0_a * X1_0_a;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc12_0 = fmaf(q0, Y4_a, acc12_0);
      acc11_0 = fmaf(q0, Y5_a, acc11_0);
      acc10_0 = fmaf(-q1, Y6_a, acc10_0);
      acc10_0 = fmaf(-q0, Y8_a, acc10_0);
    }
    { const float q = W6_0_a * X2_0_a;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.632455532033676f * q;
      acc10_0 = fmaf(q0, Y5_a, acc10_0);
      acc11_0 = fmaf(q1, Y6_a, acc11_0);
      acc12_0 = fmaf(q0, Y7_a, acc12_0);
    }
    { const float q = W6_0_a * X3_0_a;
      const float q0 = 0.547722557505166f * q;
      const float q1 = 0.31622776601683794f * q;
      acc10_0 = fmaf(q0, Y4_a, acc10_0);
      acc12_0 = fmaf(-q1, Y6_a, acc12_0);
      acc11_0 = fmaf(q0, Y7_a, acc11_0);
      acc12_0 = fmaf(q0, Y8_a, acc12_0);
    }
    { const float q = W7_0_a * X4_0_a;
      const float q0 = 0.547722557505166f * q;
      acc15_0 = fmaf(q0, Y1_a, acc15_0);
      acc13_0 = fmaf(q0, Y3_a, acc13_0);
    }
    { const float q = W7_0_a * X5_0_a;
      const float q0 = 0.547722557505166f * q;
      acc14_0 = fmaf(q0, Y1_a, acc14_0);
      acc13_0 = fmaf(q0, Y2_a, acc13_0);
    }
    { const float q = W7_0_a * X6_0_a;
      const float q0 = 0.31622776601683794f * q;
      const float q1 = 0.632455532033676f * q;
      acc13_0 = fmaf(-q0, Y1_a, acc13_0);
      acc14_0 = fmaf(q1, Y2_a, acc14_0);
      acc15_0 = fmaf(-q0, Y3_a, acc15_0);
    }
    { const float q = W7_0_a * X7_0_a;
      const float q0 = 0.547722557505166f * q;
      acc15_0 = fmaf(q0, Y2_a, acc15_0);
      acc14_0 = fmaf(q0, Y3_a, acc14_0);
    }
    { const float q = W7_0_a * X8_0_a;
      const float q0 = 0.547722557505166f * q;
      acc13_0 = fmaf(-q0, Y1_a, acc13_0);
      acc15_0 = fmaf(q0, Y3_a, acc15_0);
    }
    { const float q = W8_0_a * X4_0_a;
      const float q0 = 0.4629100498862757f * q;
      const float q1 = 0.3779644730092272f * q;
      const float q2 = 0.11952286093343936f * q;
      acc18_0 = fmaf(q0, Y9_a, acc18_0);
      acc17_0 = fmaf(q1, Y10_a, acc17_0);
      acc18_0 = fmaf(-q2, Y11_a, acc18_0);
      acc16_0 = fmaf(-q2, Y13_a, acc16_0);
      acc16_0 = fmaf(-q0, Y15_a, acc16_0);
    }
    { const float q = W8_0_a * X5_0_a;
      const float q0 = 0.3779644730092272f * q;
      const float q1 = 0.47809144373375745f * q;
      const float q2 = 0.29277002188456f * q;
      acc18_0 = fmaf(q0, Y10_a, acc18_0);
      acc17_0 = fmaf(q1, Y11_a, acc17_0);
      acc16_0 = fmaf(-q2, Y12_a, acc16_0);
      acc16_0 = fmaf(-q0, Y14_a, acc16_0);
    }
    { const float q = W8_0_a * X6_0_a;
      const float q0 = 0.41403933560541256f * q;
      const float q1 = 0.5070925528371102f * q;
      acc16_0 = fmaf(q0, Y11_a, acc16_0);
      acc17_0 = fmaf(q1, Y12_a, acc17_0);
      acc18_0 = fmaf(q0, Y13_a, acc18_0);
    }
    { const float q = W8_0_a * X7_0_a;
      const float q0 = 0.3779644730092272f * q;
      const float q1 = 0.29277002188456f * q;
      const float q2 = 0.47809144373375745f * q;
      acc16_0 = fmaf(q0, Y10_a, acc16_0);
      acc18_0 = fmaf(-q1, Y12_a, acc18_0);
      acc17_0 = fmaf(q2, Y13_a, acc17_0);
      acc18_0 = fmaf(q0, Y14_a, acc18_0);
    }
    { const float q = W8_0_a * X8_0_a;
      const float q0 = 0.4629100498862757f * q;
      const float q1 = 0.11952286093343936f * q;
      const float q2 = 0.3779644730092272f * q;
      acc16_0 = fmaf(q0, Y9_a, acc16_0);
      acc16_0 = fmaf(q1, Y11_a, acc16_0);
      acc18_0 = fmaf(-q1, Y13_a, acc18_0);
      acc17_0 = fmaf(q2, Y14_a, acc17_0);
      acc18_0 = fmaf(q0, Y15_a, acc18_0);
    }
    { const float q = W9_0_a * X9_0_a;
      const float q0 = 0.4629100498862757f * q;
      acc21_0 = fmaf(q0, Y4_a, acc21_0);
      acc19_0 = fmaf(q0, Y8_a, acc19_0);
    }
    { const float q = W9_0_a * X10_0_a;
      const float q0 = 0.3779644730092272f * q;
      acc20_0 = fmaf(q0, Y4_a, acc20_0);
      acc21_0 = fmaf(q0, Y5_a, acc21_0);
      acc19_0 = fmaf(q0, Y7_a, acc19_0);
    }
    { const float q = W9_0_a * X11_0_a;
      const float q0 = 0.11952286093343936f * q;
      const float q1 = 0.47809144373375745f * q;
      const float q2 = 0.41403933560541256f * q;
      acc21_0 = fmaf(-q0, Y4_a, acc21_0);
      acc20_0 = fmaf(q1, Y5_a, acc20_0);
      acc19_0 = fmaf(q2, Y6_a, acc19_0);
      acc19_0 = fmaf(q0, Y8_a, acc19_0);
    }
    { const float q = W9_0_a * X12_0_a;
      const float q0 = 0.29277002188456f * q;
      const float q1 = 0.5070925528371102f * q;
      acc19_0 = fmaf(-q0, Y5_a, acc19_0);
      acc20_0 = fmaf(q1, Y6_a, acc20_0);
      acc21_0 = fmaf(-q0, Y7_a, acc21_0);
    }
    { const float q = W9_0_a * X13_0_a;
      const float q0 = 0.11952286093343936f * q;
      const float q1 = 0.41403933560541256f * q;
      const float q2 = 0.47809144373375745f * q;
      acc19_0 = fmaf(-q0, Y4_a, acc19_0);
      acc21_0 = fmaf(q1, Y6_a, acc21_0);
      acc20_0 = fmaf(q2, Y7_a, acc20_0);
      acc21_0 = fmaf(-q0, Y8_a, acc21_0);
    }
    { const float q = W9_0_a * X14_0_a;
      const float q0 = 0.3779644730092272f * q;
      acc19_0 = fmaf(-q0, Y5_a, acc19_0);
      acc21_0 = fmaf(q0, Y7_a, acc21_0);
      acc20_0 = fmaf(q0, Y8_a, acc20_0);
    }
    { const float q = W9_0_a * X15_0_a;
      const float q0 = 0.4629100498862757f * q;
      acc19_0 = fmaf(-q0, Y4_a, acc19_0);
      acc21_0 = fmaf(q0, Y8_a, acc21_0);
    }
    { const float q = W10_0_a * X0_0_a;
      acc22_0 = fmaf(q, Y4_a, acc22_0);
      acc23_0 = fmaf(q, Y5_a, acc23_0);
      acc24_0 = fmaf(q, Y6_a, acc24_0);
      acc25_0 = fmaf(q, Y7_a, acc25_0);
      acc26_0 = fmaf(q, Y8_a, acc26_0);
    }
    { const float q = W11_0_a * X1_0_a;
      const float q0 = 0.408248290463863f * q;
      const float q1 = 0.7071067811865475f * q;
      acc29_0 = fmaf(q0, Y1_a, acc29_0);
      acc31_0 = fmaf(q1, Y1_a, acc31_0);
      acc28_0 = fmaf(-q1, Y2_a, acc28_0);
      acc27_0 = fmaf(-q1, Y3_a, acc27_0);
    }
    { const float q = W11_0_a * X2_0_a;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.8164965809277261f * q;
      acc28_0 = fmaf(-q0, Y1_a, acc28_0);
      acc29_0 = fmaf(-q1, Y2_a, acc29_0);
      acc30_0 = fmaf(-q0, Y3_a, acc30_0);
    }
    { const float q = W11_0_a * X3_0_a;
      const float q0 = 0.7071067811865475f * q;
      const float q1 = 0.408248290463863f * q;
      acc27_0 = fmaf(-q0, Y1_a, acc27_0);
      acc30_0 = fmaf(-q0, Y2_a, acc30_0);
      acc29_0 = fmaf(q1, Y3_a, acc29_0);
      acc31_0 = fmaf(-q0, Y3_a, acc31_0);
    }
    { const float q = W12_0_a * X1_0_a;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.5345224838248488f * q;
      const float q3 = 0.15430334996209188f * q;
      const float q4 = 0.3779644730092272f * q;
      acc36_0 = fmaf(q0, Y9_a, acc36_0);
      acc35_0 = fmaf(q1, Y10_a, acc35_0);
      acc34_0 = fmaf(q2, Y11_a, acc34_0);
      acc36_0 = fmaf(q3, Y11_a, acc36_0);
      acc33_0 = fmaf(-q4, Y12_a, acc33_0);
      acc32_0 = fmaf(-q3, Y13_a, acc32_0);
      acc33_0 = fmaf(-q1, Y14_a, acc33_0);
      acc32_0 = fmaf(-q0, Y15_a, acc32_0);
    }
    { const float q = W12_0_a * X2_0_a;
      const float q0 = 0.48795003647426655f * q;
      const float q1 = 0.6172133998483676f * q;
      const float q2 = 0.6546536707079772f * q;
      acc32_0 = fmaf(q0, Y10_a, acc32_0);
      acc33_0 = fmaf(q1, Y11_a, acc33_0);
      acc34_0 = fmaf(q2, Y12_a, acc34_0);
      acc35_0 = fmaf(q1, Y13_a, acc35_0);
      acc36_0 = fmaf(q0, Y14_a, acc36_0);
    }
    { const float q = W12_0_a * X3_0_a;
      const float q0 = 0.5976143046671967f * q;
      const float q1 = 0.48795003647426655f * q;
      const float q2 = 0.15430334996209188f * q;
      const float q3 = 0.3779644730092272f * q;
      const float q4 = 0.5345224838248488f * q;
      acc32_0 = fmaf(q0, Y9_a, acc32_0);
      acc33_0 = fmaf(q1, Y10_a, acc33_0);
      acc32_0 = fmaf(-q2, Y11_a, acc32_0);
      acc35_0 = fmaf(-q3, Y12_a, acc35_0);
      acc34_0 = fmaf(q4, Y13_a, acc34_0);
      acc36_0 = fmaf(-q2, Y13_a, acc36_0);
      acc35_0 = fmaf(q1, Y14_a, acc35_0);
      acc36_0 = fmaf(q0, Y15_a, acc36_0);
    }
    { const float q = W13_0_a * X4_0_a;
      acc37_0 = fmaf(q, Y0_a, acc37_0);
    }
    { const float q = W13_0_a * X5_0_a;
      acc38_0 = fmaf(q, Y0_a, acc38_0);
    }
    { const float q = W13_0_a * X6_0_a;
      acc39_0 = fmaf(q, Y0_a, acc39_0);
    }
    { const float q = W13_0_a * X7_0_a;
      acc40_0 = fmaf(q, Y0_a, acc40_0);
    }
    { const float q = W13_0_a * X8_0_a;
      acc41_0 = fmaf(q, Y0_a, acc41_0);
    }
    { const float q = W14_0_a * X4_0_a;
      const float q0 = 0.5345224838248488f * q;
      const float q1 = 0.46291004988627565f * q;
      acc44_0 = fmaf(q0, Y4_a, acc44_0);
      acc45_0 = fmaf(-q1, Y5_a, acc45_0);
      acc42_0 = fmaf(q0, Y6_a, acc42_0);
      acc43_0 = fmaf(-q1, Y7_a, acc43_0);
    }
    { const float q = W14_0_a * X5_0_a;
      const float q0 = 0.46291004988627565f * q;
      const float q1 = 0.2672612419124244f * q;
      acc45_0 = fmaf(-q0, Y4_a, acc45_0);
      acc44_0 = fmaf(-q1, Y5_a, acc44_0);
      acc46_0 = fmaf(q0, Y5_a, acc46_0);
      acc43_0 = fmaf(-q1, Y6_a, acc43_0);
      acc42_0 = fmaf(-q0, Y7_a, acc42_0);
      acc43_0 = fmaf(q0, Y8_a, acc43_0);
    }
    { const float q = W14_0_a * X6_0_a;
      const float q0 = 0.5345224838248488f * q;
      const float q1 = 0.2672612419124244f * q;
      acc42_0 = fmaf(q0, Y4_a, acc42_0);
      acc43_0 = fmaf(-q1, Y5_a, acc43_0);
      acc44_0 = fmaf(-q0, Y6_a, acc44_0);
      acc45_0 = fmaf(-q1, Y7_a, acc45_0);
      acc46_0 = fmaf(q0, Y8_a, acc46_0);
    }
    { const float q = W14_0_a * X7_0_a;
      const float q0 = 0.46291004988627565f * q;
      const float q1 = 0.2672612419124244f * q;
      acc43_0 = fmaf(-q0, Y4_a, acc43_0);
      acc42_0 = fmaf(-q0, Y5_a, acc42_0);
      acc45_0 = fmaf(-q1, Y6_a, acc45_0);
      acc44_0 = fmaf(-q1, Y7_a, acc44_0);
      acc46_0 = fmaf(-q0, Y7_a, acc46_0);
      acc45_0 = fmaf(-q0, Y8_a, acc45_0);
    }
    { const float q = W14_0_a * X8_0_a;
      const float q0 = 0.46291004988627565f * q;
      const float q1 = 0.5345224838248488f * q;
      acc43_0 = fmaf(q0, Y5_a, acc43_0);
      acc46_0 = fmaf(q1, Y6_a, acc46_0);
      acc45_0 = fmaf(-q0, Y7_a, acc45_0);
      acc44_0 = fmaf(q1, Y8_a, acc44_0);
    }
    { const float q = W15_0_a * X9_0_a;
      const float q0 = 0.5976143046671968f * q;
      acc51_0 = fmaf(q0, Y1_a, acc51_0);
      acc47_0 = fmaf(q0, Y3_a, acc47_0);
    }
    { const float q = W15_0_a * X10_0_a;
      const float q0 = 0.4879500364742667f * q;
      acc50_0 = fmaf(q0, Y1_a, acc50_0);
      acc47_0 = fmaf(q0, Y2_a, acc47_0);
      acc48_0 = fmaf(q0, Y3_a, acc48_0);
    }
    { const float q = W15_0_a * X11_0_a;
      const float q0 = 0.5345224838248489f * q;
      const float q1 = 0.1543033499620919f * q;
      const float q2 = 0.6172133998483678f * q;
      acc49_0 = fmaf(q0, Y1_a, acc49_0);
      acc51_0 = fmaf(q1, Y1_a, acc51_0);
      acc48_0 = fmaf(q2, Y2_a, acc48_0);
      acc47_0 = fmaf(-q1, Y3_a, acc47_0);
    }
    { const float q = W15_0_a * X12_0_a;
      const float q0 = 0.3779644730092273f * q;
      const float q1 = 0.6546536707079773f * q;
      acc48_0 = fmaf(-q0, Y1_a, acc48_0);
      acc49_0 = fmaf(q1, Y2_a, acc49_0);
      acc50_0 = fmaf(-q0, Y3_a, acc50_0);
    }
    { const float q = W15_0_a * X13_0_a;
      const float q0 = 0.1543033499620919f * q;
      const float q1 = 0.6172133998483678f * q;
      const float q2 = 0.5345224838248489f * q;
      acc47_0 = fmaf(-q0, Y1_a, acc47_0);
      acc50_0 = fmaf(q1, Y2_a, acc50_0);
      acc49_0 = fmaf(q2, Y3_a, acc49_0);
      acc51_0 = fmaf(-q0, Y3_a, acc51_0);
    }
    { const float q = W15_0_a * X14_0_a;
      const float q0 = 0.4879500364742667f * q;
      acc48_0 = fmaf(-q0, Y1_a, acc48_0);
      acc51_0 = fmaf(q0, Y2_a, acc51_0);
      acc50_0 = fmaf(q0, Y3_a, acc50_0);
    }
    { const float q = W15_0_a * X15_0_a;
      const float q0 = 0.5976143046671968f * q;
      acc47_0 = fmaf(-q0, Y1_a, acc47_0);
      acc51_0 = fmaf(q0, Y3_a, acc51_0);
    }
    { const float q = W16_0_a * X9_0_a;
      const float q0 = 0.545544725589981f * q;
      const float q1 = 0.38575837490522974f * q;
      const float q2 = 0.24397501823713336f * q;
      acc54_0 = fmaf(q0, Y9_a, acc54_0);
      acc55_0 = fmaf(-q1, Y10_a, acc55_0);
      acc56_0 = fmaf(q2, Y11_a, acc56_0);
      acc52_0 = fmaf(q2, Y13_a, acc52_0);
      acc53_0 = fmaf(-q1, Y14_a, acc53_0);
    }
    { const float q = W16_0_a * X10_0_a;
      const float q0 = 0.38575837490522974f * q;
      const float q1 = 0.2988071523335984f * q;
      const float q2 = 0.4879500364742667f * q;
      acc55_0 = fmaf(-q0, Y9_a, acc55_0);
      acc55_0 = fmaf(-q1, Y11_a, acc55_0);
      acc52_0 = fmaf(q2, Y12_a, acc52_0);
      acc53_0 = fmaf(-q1, Y13_a, acc53_0);
      acc53_0 = fmaf(q0, Y15_a, acc53_0);
    }
    { const float q = W16_0_a * X11_0_a;
      const float q0 = 0.24397501823713336f * q;
      const float q1 = 0.2988071523335984f * q;
      const float q2 = 0.3273268353539886f * q;
      const float q3 = 0.3779644730092273f * q;
      const float q4 = 0.15430334996209194f * q;
      acc56_0 = fmaf(q0, Y9_a, acc56_0);
      acc55_0 = fmaf(-q1, Y10_a, acc55_0);
      acc54_0 = fmaf(-q2, Y11_a, acc54_0);
      acc56_0 = fmaf(q3, Y11_a, acc56_0);
      acc53_0 = fmaf(-q4, Y12_a, acc53_0);
      acc52_0 = fmaf(-q3, Y13_a, acc52_0);
      acc53_0 = fmaf(q1, Y14_a, acc53_0);
      acc52_0 = fmaf(-q0, Y15_a, acc52_0);
    }
    { const float q = W16_0_a * X12_0_a;
      const float q0 = 0.4879500364742667f * q;
      const float q1 = 0.15430334996209194f * q;
      const float q2 = 0.4364357804719849f * q;
      acc52_0 = fmaf(q0, Y10_a, acc52_0);
      acc53_0 = fmaf(-q1, Y11_a, acc53_0);
      acc54_0 = fmaf(-q2, Y12_a, acc54_0);
      acc55_0 = fmaf(-q1, Y13_a, acc55_0);
      acc56_0 = fmaf(q0, Y14_a, acc56_0);
    }
    { const float q = W16_0_a * X13_0_a;
      const float q0 = 0.24397501823713336f * q;
      const float q1 = 0.2988071523335984f * q;
      const float q2 = 0.3779644730092273f * q;
      const float q3 = 0.15430334996209194f * q;
      const float q4 = 0.3273268353539886f * q;
      acc52_0 = fmaf(q0, Y9_a, acc52_0);
      acc53_0 = fmaf(-q1, Y10_a, acc53_0);
      acc52_0 = fmaf(-q2, Y11_a, acc52_0);
      acc55_0 = fmaf(-q3, Y12_a, acc55_0);
      acc54_0 = fmaf(-q4, Y13_a, acc54_0);
      acc56_0 = fmaf(-q2, Y13_a, acc56_0);
      acc55_0 = fmaf(-q1, Y14_a, acc55_0);
      acc56_0 = fmaf(q0, Y15_a, acc56_0);
    }
    { const float q = W16_0_a * X14_0_a;
      const float q0 = 0.38575837490522974f * q;
      const float q1 = 0.2988071523335984f * q;
      const float q2 = 0.4879500364742667f * q;
      acc53_0 = fmaf(-q0, Y9_a, acc53_0);
      acc53_0 = fmaf(q1, Y11_a, acc53_0);
      acc56_0 = fmaf(q2, Y12_a, acc56_0);
      acc55_0 = fmaf(-q1, Y13_a, acc55_0);
      acc55_0 = fmaf(-q0, Y15_a, acc55_0);
    }
    { const float q = W16_0_a * X15_0_a;
      const float q0 = 0.38575837490522974f * q;
      const float q1 = 0.24397501823713336f * q;
      const float q2 = 0.545544725589981f * q;
      acc53_0 = fmaf(q0, Y10_a, acc53_0);
      acc52_0 = fmaf(-q1, Y11_a, acc52_0);
      acc56_0 = fmaf(q1, Y13_a, acc56_0);
      acc55_0 = fmaf(-q0, Y14_a, acc55_0);
      acc54_0 = fmaf(q2, Y15_a, acc54_0);
    }
    { const float q = W17_0_a * X0_0_a;
      acc57_0 = fmaf(q, Y9_a, acc57_0);
      acc58_0 = fmaf(q, Y10_a, acc58_0);
      acc59_0 = fmaf(q, Y11_a, acc59_0);
      acc60_0 = fmaf(q, Y12_a, acc60_0);
      acc61_0 = fmaf(q, Y13_a, acc61_0);
      acc62_0 = fmaf(q, Y14_a, acc62_0);
      acc63_0 = fmaf(q, Y15_a, acc63_0);
    }
    { const float q = W18_0_a * X1_0_a;
      const float q0 = 0.18257418583505539f * q;
      const float q1 = 0.7071067811865476f * q;
      const float q2 = 0.447213595499958f * q;
      const float q3 = 0.5773502691896256f * q;
      const float q4 = 0.632455532033676f * q;
      acc68_0 = fmaf(q0, Y4_a, acc68_0);
      acc70_0 = fmaf(q1, Y4_a, acc70_0);
      acc67_0 = fmaf(q2, Y5_a, acc67_0);
      acc69_0 = fmaf(q3, Y5_a, acc69_0);
      acc66_0 = fmaf(-q4, Y6_a, acc66_0);
      acc65_0 = fmaf(-q3, Y7_a, acc65_0);
      acc64_0 = fmaf(-q1, Y8_a, acc64_0);
      acc66_0 = fmaf(-q0, Y8_a, acc66_0);
    }
    { const float q = W18_0_a * X2_0_a;
      const float q0 = 0.5773502691896258f * q;
      const float q1 = 0.7302967433402215f * q;
      const float q2 = 0.7745966692414836f * q;
      acc65_0 = fmaf(-q0, Y4_a, acc65_0);
      acc66_0 = fmaf(-q1, Y5_a, acc66_0);
      acc67_0 = fmaf(-q2, Y6_a, acc67_0);
      acc68_0 = fmaf(-q1, Y7_a, acc68_0);
      acc69_0 = fmaf(-q0, Y8_a, acc69_0);
    }
    { const float q = W18_0_a * X3_0_a;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.18257418583505539f * q;
      const float q2 = 0.5773502691896256f * q;
      const float q3 = 0.632455532033676f * q;
      const float q4 = 0.447213595499958f * q;
      acc64_0 = fmaf(-q0, Y4_a, acc64_0);
      acc66_0 = fmaf(q1, Y4_a, acc66_0);
      acc65_0 = fmaf(-q2, Y5_a, acc65_0);
      acc68_0 = fmaf(-q3, Y6_a, acc68_0);
      acc67_0 = fmaf(q4, Y7_a, acc67_0);
      acc69_0 = fmaf(-q2, Y7_a, acc69_0);
      acc68_0 = fmaf(q1, Y8_a, acc68_0);
      acc70_0 = fmaf(-q0, Y8_a, acc70_0);
    }
    { const float q = W19_0_a * X4_0_a;
      const float q0 = 0.18257418583505539f * q;
      const float q1 = 0.7071067811865476f * q;
      const float q2 = 0.5773502691896258f * q;
      acc75_0 = fmaf(q0, Y1_a, acc75_0);
      acc77_0 = fmaf(q1, Y1_a, acc77_0);
      acc72_0 = fmaf(-q2, Y2_a, acc72_0);
      acc71_0 = fmaf(-q1, Y3_a, acc71_0);
      acc73_0 = fmaf(q0, Y3_a, acc73_0);
    }
    { const float q = W19_0_a * X5_0_a;
      const float q0 = 0.447213595499958f * q;
      const float q1 = 0.5773502691896256f * q;
      const float q2 = 0.7302967433402215f * q;
      acc74_0 = fmaf(q0, Y1_a, acc74_0);
      acc76_0 = fmaf(q1, Y1_a, acc76_0);
      acc73_0 = fmaf(-q2, Y2_a, acc73_0);
      acc72_0 = fmaf(-q1, Y3_a, acc72_0);
    }
    { const float q = W19_0_a * X6_0_a;
      const float q0 = 0.632455532033676f * q;
      const float q1 = 0.7745966692414836f * q;
      acc73_0 = fmaf(-q0, Y1_a, acc73_0);
      acc74_0 = fmaf(-q1, Y2_a, acc74_0);
      acc75_0 = fmaf(-q0, Y3_a, acc75_0);
    }
    { const float q = W19_0_a * X7_0_a;
      const float q0 = 0.5773502691896256f * q;
      const float q1 = 0.7302967433402215f * q;
      const float q2 = 0.447213595499958f * q;
      acc72_0 = fmaf(-q0, Y1_a, acc72_0);
      acc75_0 = fmaf(-q1, Y2_a, acc75_0);
      acc74_0 = fmaf(q2, Y3_a, acc74_0);
      acc76_0 = fmaf(-q0, Y3_a, acc76_0);
    }
    { const float q = W19_0_a * X8_0_a;
      const float q0 = 0.7071067811865476f * q;
      const float q1 = 0.18257418583505539f * q;
      const float q2 = 0.5773502691896258f * q;
      acc71_0 = fmaf(-q0, Y1_a, acc71_0);
      acc73_0 = fmaf(-q1, Y1_a, acc73_0);
      acc76_0 = fmaf(-q2, Y2_a, acc76_0);
      acc75_0 = fmaf(q1, Y3_a, acc75_0);
      acc77_0 = fmaf(-q0, Y3_a, acc77_0);
    }
    { const float q = W20_0_a * X4_0_a;
      const float q0 = 0.2886751345948128f * q;
      const float q1 = 0.5773502691896258f * q;
      const float q2 = 0.447213595499958f * q;
      acc82_0 = fmaf(q0, Y9_a, acc82_0);
      acc81_0 = fmaf(q1, Y10_a, acc81_0);
      acc82_0 = fmaf(-q2, Y11_a, acc82_0);
      acc84_0 = fmaf(-q0, Y11_a, acc84_0);
      acc79_0 = fmaf(q1, Y12_a, acc79_0);
      acc78_0 = fmaf(q0, Y13_a, acc78_0);
      acc80_0 = fmaf(-q2, Y13_a, acc80_0);
      acc80_0 = fmaf(-q0, Y15_a, acc80_0);
    }
    { const float q = W20_0_a * X5_0_a;
      const float q0 = 0.45643546458763845f * q;
      const float q1 = 0.3535533905932738f * q;
      const float q2 = 0.18257418583505539f * q;
      acc83_0 = fmaf(-q0, Y9_a, acc83_0);
      acc82_0 = fmaf(-q1, Y10_a, acc82_0);
      acc84_0 = fmaf(q0, Y10_a, acc84_0);
      acc81_0 = fmaf(-q2, Y11_a, acc81_0);
      acc83_0 = fmaf(q1, Y11_a, acc83_0);
      acc80_0 = fmaf(-q2, Y12_a, acc80_0);
      acc79_0 = fmaf(-q1, Y13_a, acc79_0);
      acc78_0 = fmaf(-q0, Y14_a, acc78_0);
      acc80_0 = fmaf(q1, Y14_a, acc80_0);
      acc79_0 = fmaf(q0, Y15_a, acc79_0);
    }
    { const float q = W20_0_a * X6_0_a;
      const float q0 = 0.6454972243679029f * q;
      const float q1 = 0.3872983346207418f * q;
      const float q2 = 0.5163977794943223f * q;
      acc78_0 = fmaf(q0, Y9_a, acc78_0);
      acc80_0 = fmaf(-q1, Y11_a, acc80_0);
      acc81_0 = fmaf(-q2, Y12_a, acc81_0);
      acc82_0 = fmaf(-q1, Y13_a, acc82_0);
      acc84_0 = fmaf(q0, Y15_a, acc84_0);
    }
    { const float q = W20_0_a * X7_0_a;
      const float q0 = 0.45643546458763845f * q;
      const float q1 = 0.3535533905932738f * q;
      const float q2 = 0.18257418583505539f * q;
      acc79_0 = fmaf(-q0, Y9_a, acc79_0);
      acc78_0 = fmaf(-q0, Y10_a, acc78_0);
      acc80_0 = fmaf(-q1, Y10_a, acc80_0);
      acc79_0 = fmaf(-q1, Y11_a, acc79_0);
      acc82_0 = fmaf(-q2, Y12_a, acc82_0);
      acc81_0 = fmaf(-q2, Y13_a, acc81_0);
      acc83_0 = fmaf(-q1, Y13_a, acc83_0);
      acc82_0 = fmaf(-q1, Y14_a, acc82_0);
      acc84_0 = fmaf(-q0, Y14_a, acc84_0);
      acc83_0 = fmaf(-q0, Y15_a, acc83_0);
    }
    { const float q = W20_0_a * X8_0_a;
      const float q0 = 0.2886751345948128f * q;
      const float q1 = 0.447213595499958f * q;
      const float q2 = 0.5773502691896258f * q;
      acc80_0 = fmaf(q0, Y9_a, acc80_0);
      acc78_0 = fmaf(q0, Y11_a, acc78_0);
      acc80_0 = fmaf(q1, Y11_a, acc80_0);
      acc83_0 = fmaf(q2, Y12_a, acc83_0);
      acc82_0 = fmaf(-q1, Y13_a, acc82_0);
      acc84_0 = fmaf(q0, Y13_a, acc84_0);
      acc81_0 = fmaf(q2, Y14_a, acc81_0);
      acc82_0 = fmaf(q0, Y15_a, acc82_0);
    }
    { const float q = W21_0_a * X9_0_a;
      acc85_0 = fmaf(q, Y0_a, acc85_0);
    }
    { const float q = W21_0_a * X10_0_a;
      acc86_0 = fmaf(q, Y0_a, acc86_0);
    }
    { const float q = W21_0_a * X11_0_a;
      acc87_0 = fmaf(q, Y0_a, acc87_0);
    }
    { const float q = W21_0_a * X12_0_a;
      acc88_0 = fmaf(q, Y0_a, acc88_0);
    }
    { const float q = W21_0_a * X13_0_a;
      acc89_0 = fmaf(q, Y0_a, acc89_0);
    }
    { const float q = W21_0_a * X14_0_a;
      acc90_0 = fmaf(q, Y0_a, acc90_0);
    }
    { const float q = W21_0_a * X15_0_a;
      acc91_0 = fmaf(q, Y0_a, acc91_0);
    }
    { const float q = W22_0_a * X9_0_a;
      const float q0 = 0.2886751345948128f * q;
      const float q1 = 0.45643546458763845f * q;
      const float q2 = 0.6454972243679029f * q;
      acc96_0 = fmaf(q0, Y4_a, acc96_0);
      acc97_0 = fmaf(-q1, Y5_a, acc97_0);
      acc92_0 = fmaf(q2, Y6_a, acc92_0);
      acc93_0 = fmaf(-q1, Y7_a, acc93_0);
      acc94_0 = fmaf(q0, Y8_a, acc94_0);
    }
    { const float q = W22_0_a * X10_0_a;
      const float q0 = 0.5773502691896258f * q;
      const float q1 = 0.3535533905932738f * q;
      const float q2 = 0.45643546458763845f * q;
      acc95_0 = fmaf(q0, Y4_a, acc95_0);
      acc96_0 = fmaf(-q1, Y5_a, acc96_0);
      acc98_0 = fmaf(q2, Y5_a, acc98_0);
      acc92_0 = fmaf(-q2, Y7_a, acc92_0);
      acc94_0 = fmaf(-q1, Y7_a, acc94_0);
    }
    { const float q = W22_0_a * X11_0_a;
      const float q0 = 0.447213595499958f * q;
      const float q1 = 0.2886751345948128f * q;
      const float q2 = 0.18257418583505539f * q;
      const float q3 = 0.3535533905932738f * q;
      const float q4 = 0.3872983346207418f * q;
      acc96_0 = fmaf(-q0, Y4_a, acc96_0);
      acc98_0 = fmaf(-q1, Y4_a, acc98_0);
      acc95_0 = fmaf(-q2, Y5_a, acc95_0);
      acc97_0 = fmaf(q3, Y5_a, acc97_0);
      acc94_0 = fmaf(-q4, Y6_a, acc94_0);
      acc93_0 = fmaf(-q3, Y7_a, acc93_0);
      acc92_0 = fmaf(q1, Y8_a, acc92_0);
      acc94_0 = fmaf(q0, Y8_a, acc94_0);
    }
    { const float q = W22_0_a * X12_0_a;
      const float q0 = 0.5773502691896258f * q;
      const float q1 = 0.18257418583505539f * q;
      const float q2 = 0.5163977794943223f * q;
      acc93_0 = fmaf(q0, Y4_a, acc93_0);
      acc94_0 = fmaf(-q1, Y5_a, acc94_0);
      acc95_0 = fmaf(-q2, Y6_a, acc95_0);
      acc96_0 = fmaf(-q1, Y7_a, acc96_0);
      acc97_0 = fmaf(q0, Y8_a, acc97_0);
    }
    { const float q = W22_0_a * X13_0_a;
      const float q0 = 0.2886751345948128f * q;
      const float q1 = 0.447213595499958f * q;
      const float q2 = 0.3535533905932738f * q;
      const float q3 = 0.3872983346207418f * q;
      const float q4 = 0.18257418583505539f * q;
      acc92_0 = fmaf(q0, Y4_a, acc92_0);
      acc94_0 = fmaf(-q1, Y4_a, acc94_0);
      acc93_0 = fmaf(-q2, Y5_a, acc93_0);
      acc96_0 = fmaf(-q3, Y6_a, acc96_0);
      acc95_0 = fmaf(-q4, Y7_a, acc95_0);
      acc97_0 = fmaf(-q2, Y7_a, acc97_0);
      acc96_0 = fmaf(-q1, Y8_a, acc96_0);
      acc98_0 = fmaf(q0, Y8_a, acc98_0);
    }
    { const float q = W22_0_a * X14_0_a;
      const float q0 = 0.45643546458763845f * q;
      const float q1 = 0.3535533905932738f * q;
      const float q2 = 0.5773502691896258f * q;
      acc92_0 = fmaf(-q0, Y5_a, acc92_0);
      acc94_0 = fmaf(q1, Y5_a, acc94_0);
      acc96_0 = fmaf(-q1, Y7_a, acc96_0);
      acc98_0 = fmaf(-q0, Y7_a, acc98_0);
      acc95_0 = fmaf(q2, Y8_a, acc95_0);
    }
    { const float q = W22_0_a * X15_0_a;
      const float q0 = 0.2886751345948128f * q;
      const float q1 = 0.45643546458763845f * q;
      const float q2 = 0.6454972243679029f * q;
      acc94_0 = fmaf(-q0, Y4_a, acc94_0);
      acc93_0 = fmaf(q1, Y5_a, acc93_0);
      acc98_0 = fmaf(q2, Y6_a, acc98_0);
      acc97_0 = fmaf(-q1, Y7_a, acc97_0);
      acc96_0 = fmaf(q0, Y8_a, acc96_0);
    }
  }
  for (int s = 1; s < 4; ++s) {   // the waves' sums in wave order
    if (wave == s) {
      red[0 + lane] = acc0_0;
      red[64 + lane] = acc1_0;
      red[128 + lane] = acc2_0;
      red[192 + lane] = acc3_0;
      red[256 + lane] = acc4_0;
      red[320 + lane] = acc5_0;
      red[384 + lane] = acc6_0;
      red[448 + lane] = acc7_0;
      red[512 + lane] = acc8_0;
      red[576 + lane] = acc9_0;
      red[640 + lane] = acc10_0;
      red[704 + lane] = acc11_0;
      red[768 + lane] = acc12_0;
      red[832 + lane] = acc13_0;
      red[896 + lane] = acc14_0;
      red[960 + lane] = acc15_0;
      red[1024 + lane] = acc16_0;
      red[1088 + lane] = acc17_0;
      red[1152 + lane] = acc18_0;
      red[1216 + lane] = acc19_0;
      red[1280 + lane] = acc20_0;
      red[1344 + lane] = acc21_0;
      red[1408 + lane] = acc22_0;
      red[1472 + lane] = acc23_0;
      red[1536 + lane] = acc24_0;
      red[1600 + lane] = acc25_0;
      red[1664 + lane] = acc26_0;
      red[1728 + lane] = acc27_0;
      red[1792 + lane] = acc28_0;
      red[1856 + lane] = acc29_0;
      red[1920 + lane] = acc30_0;
      red[1984 + lane] = acc31_0;
      red[2048 + lane] = acc32_0;
      red[2112 + lane] = acc33_0;
      red[2176 + lane] = acc34_0;
      red[2240 + lane] = acc35_0;
      red[2304 + lane] = acc36_0;
      red[2368 + lane] = acc37_0;
      red[2432 + lane] = acc38_0;
      red[2496 + lane] = acc39_0;
      red[2560 + lane] = acc40_0;
      red[2624 + lane] = acc41_0;
      red[2688 + lane] = acc42_0;
      red[2752 + lane] = acc43_0;
      red[2816 + lane] = acc44_0;
      red[2880 + lane] = acc45_0;
      red[2944 + lane] = acc46_0;
      red[3008 + lane] = acc47_0;
      red[3072 + lane] = acc48_0;
      red[3136 + lane] = acc49_0;
      red[3200 + lane] = acc50_0;
      red[3264 + lane] = acc51_0;
      red[3328 + lane] = acc52_0;
      red[3392 + lane] = acc53_0;
      red[3456 + lane] = acc54_0;
      red[3520 + lane] = acc55_0;
      red[3584 + lane] = acc56_0;
      red[3648 + lane] = acc57_0;
      red[3712 + lane] = acc58_0;
      red[3776 + lane] = acc59_0;
      red[3840 + lane] = acc60_0;
      red[3904 + lane] = acc61_0;
      red[3968 + lane] = acc62_0;
      red[4032 + lane] = acc63_0;
      red[4096 + lane] = acc64_0;
      red[4160 + lane] = acc65_0;
      red[4224 + lane] = acc66_0;
      red[4288 + lane] = acc67_0;
      red[4352 + lane] = acc68_0;
      red[4416 + lane] = acc69_0;
      red[4480 + lane] = acc70_0;
      red[4544 + lane] = acc71_0;
      red[4608 + lane] = acc72_0;
      red[4672 + lane] = acc73_0;
      red[4736 + lane] = acc74_0;
      red[4800 + lane] = acc75_0;
      red[4864 + lane] = acc76_0;
      red[4928 + lane] = acc77_0;
      red[4992 + lane] = acc78_0;
      red[5056 + lane] = acc79_0;
      red[5120 + lane] = acc80_0;
      red[5184 + lane] = acc81_0;
      red[5248 + lane] = acc82_0;
      red[5312 + lane] = acc83_0;
      red[5376 + lane] = acc84_0;
      red[5440 + lane] = acc85_0;
      red[5504 + lane] = acc86_0;
      red[5568 + lane] = acc87_0;
      red[5632 + lane] = acc88_0;
      red[5696 + lane] = acc89_0;
      red[5760 + lane] = acc90_0;
      red[5824 + lane] = acc91_0;
      red[5888 + lane] = acc92_0;
      red[5952 + lane] = acc93_0;
      red[6016 + lane] = acc94_0;
      red[6080 + lane] = acc95_0;
      red[6144 + lane] = acc96_0;
      red[6208 + lane] = acc97_0;
      red[6272 + lane] = acc98_0;
    }
    __syncthreads();
    if (wave == 0) {
      acc0_0 += red[0 + lane];
      acc1_0 += red[64 + lane];
      acc2_0 += red[128 + lane];
      acc3_0 += red[192 + lane];
      acc4_0 += red[256 + lane];
      acc5_0 += red[320 + lane];
      acc6_0 += red[384 + lane];
      acc7_0 += red[448 + lane];
      acc8_0 += red[512 + lane];
      acc9_0 += red[576 + lane];
      acc10_0 += red[640 + lane];
      acc11_0 += red[704 + lane];
      acc12_0 += red[768 + lane];
      acc13_0 += red[832 + lane];
      acc14_0 += red[896 + lane];
      acc15_0 += red[960 + lane];
      acc16_0 += red[1024 + lane];
      acc17_0 += red[1088 + lane];
      acc18_0 += red[1152 + lane];
      acc19_0 += red[1216 + lane];
      acc20_0 += red[1280 + lane];
      acc21_0 += red[1344 + lane];
      acc22_0 += red[1408 + lane];
      acc23_0 += red[1472 + lane];
      acc24_0 += red[1536 + lane];
      acc25_0 += red[1600 + lane];
      acc26_0 += red[1664 + lane];
      acc27_0 += red[1728 + lane];
      acc28_0 += red[1792 + lane];
      acc29_0 += red[1856 + lane];
      acc30_0 += red[1920 + lane];
      acc31_0 += red[1984 + lane];
      acc32_0 += red[2048 + lane];
      acc33_0 += red[2112 + lane];
      acc34_0 += red[2176 + lane];
      acc35_0 += red[2240 + lane];
      acc36_0 += red[2304 + lane];
      acc37_0 += red[2368 + lane];
      acc38_0 += red[2432 + lane];
      acc39_0 += red[2496 + lane];
      acc40_0 += red[2560 + lane];
      acc41_0 += red[2624 + lane];
      acc42_0 += red[2688 + lane];
      acc43_0 += red[2752 + lane];
      acc44_0 += red[2816 + lane];
      acc45_0 += red[2880 + lane];
      acc46_0 += red[2944 + lane];
      acc47_0 += red[3008 + lane];
      acc48_0 += red[3072 + lane];
      acc49_0 += red[3136 + lane];
      acc50_0 += red[3200 + lane];
      acc51_0 += red[3264 + lane];
      acc52_0 += red[3328 + lane];
      acc53_0 += red[3392 + lane];
      acc54_0 += red[3456 + lane];
      acc55_0 += red[3520 + lane];
      acc56_0 += red[3584 + lane];
      acc57_0 += red[3648 + lane];
      acc58_0 += red[3712 + lane];
      acc59_0 += red[3776 + lane];
      acc60_0 += red[3840 + lane];
      acc61_0 += red[3904 + lane];
      acc62_0 += red[3968 + lane];
      acc63_0 += red[4032 + lane];
      acc64_0 += red[4096 + lane];
      acc65_0 += red[4160 + lane];
      acc66_0 += red[4224 + lane];
      acc67_0 += red[4288 + lane];
      acc68_0 += red[4352 + lane];
      acc69_0 += red[4416 + lane];
      acc70_0 += red[4480 + lane];
      acc71_0 += red[4544 + lane];
      acc72_0 += red[4608 + lane];
      acc73_0 += red[4672 + lane];
      acc74_0 += red[4736 + lane];
      acc75_0 += red[4800 + lane];
      acc76_0 += red[4864 + lane];
      acc77_0 += red[4928 + lane];
      acc78_0 += red[4992 + lane];
      acc79_0 += red[5056 + lane];
      acc80_0 += red[5120 + lane];
      acc81_0 += red[5184 + lane];
      acc82_0 += red[5248 + lane];
      acc83_0 += red[5312 + lane];
      acc84_0 += red[5376 + lane];
      acc85_0 += red[5440 + lane];
      acc86_0 += red[5504 + lane];
      acc87_0 += red[5568 + lane];
      acc88_0 += red[5632 + lane];
      acc89_0 += red[5696 + lane];
      acc90_0 += red[5760 + lane];
      acc91_0 += red[5824 + lane];
      acc92_0 += red[5888 + lane];
      acc93_0 += red[5952 + lane];
      acc94_0 += red[6016 + lane];
      acc95_0 += red[6080 + lane];
      acc96_0 += red[6144 + lane];
      acc97_0 += red[6208 + lane];
      acc98_0 += red[6272 + lane];
    }
    __syncthreads();
  }
  if (wave) return;
  float* __restrict__ op = out + (size_t)i * out_stride + c;
  op[0] = acc0_0;
  op[128] = acc1_0;
  op[256] = acc2_0;
  op[384] = acc3_0;
  op[512] = acc4_0;
  op[640] = acc5_0;
  op[768] = acc6_0;
  op[896] = acc7_0;
  op[1024] = acc8_0;
  op[1152] = acc9_0;
  op[1280] = acc10_0;
  op[1408] = acc11_0;
  op[1536] = acc12_0;
  op[1664] = acc13_0;
  op[1792] = acc14_0;
  op[1920] = acc15_0;
  op[2048] = acc16_0;
  op[2176] = acc17_0;
  op[2304] = acc18_0;
  op[2432] = acc19_0;
  op[2560] = acc20_0;
  op[2688] = acc21_0;
  op[2816] = acc22_0;
  op[2944] = acc23_0;
  op[3072] = acc24_0;
  op[3200] = acc25_0;
  op[3328] = acc26_0;
  op[3456] = acc27_0;
  op[3584] = acc28_0;
  op[3712] = acc29_0;
  op[3840] = acc30_0;
  op[3968] = acc31_0;
  op[4096] = acc32_0;
  op[4224] = acc33_0;
  op[4352] = acc34_0;
  op[4480] = acc35_0;
  op[4608] = acc36_0;
  op[4736] = acc37_0;
  op[4864] = acc38_0;
  op[4992] = acc39_0;
  op[5120] = acc40_0;
  op[5248] = acc41_0;
  op[5376] = acc42_0;
  op[5504] = acc43_0;
  op[5632] = acc44_0;
  op[5760] = acc45_0;
  op[5888] = acc46_0;
  op[6016] = acc47_0;
  op[6144] = acc48_0;
  op[6272] = acc49_0;
  op[6400] = acc50_0;
  op[6528] = acc51_0;
  op[6656] = acc52_0;
  op[6784] = acc53_0;
  op[6912] = acc54_0;
  op[7040] = acc55_0;
  op[7168] = acc56_0;
  op[7296] = acc57_0;
  op[7424] = acc58_0;
  op[7552] = acc59_0;
  op[7680] = acc60_0;
  op[7808] = acc61_0;
  op[7936] = acc62_0;
  op[8064] = acc63_0;
  op[8192] = acc64_0;
  op[8320] = acc65_0;
  op[8448] = acc66_0;
  op[8576] = acc67_0;
  op[8704] = acc68_0;
  op[8832] = acc69_0;
  op[8960] = acc70_0;
  op[9088] = acc71_0;
  op[9216] = acc72_0;
  op[9344] = acc73_0;
  op[9472] = acc74_0;
  op[9600] = acc75_0;
  op[9728] = acc76_0;
  op[9856] = acc77_0;
  op[9984] = acc78_0;
  op[10112] = acc79_0;
  op[10240] = acc80_0;
  op[10368] = acc81_0;
  op[10496] = acc82_0;
  op[10624] = acc83_0;
  op[10752] = acc84_0;
  op[10880] = acc85_0;
  op[11008] = acc86_0;
  op[11136] = acc87_0;
  op[11264] = acc88_0;
  op[11392] = acc89_0;
  op[11520] = acc90_0;
  op[11648] = acc91_0;
  op[11776] = acc92_0;
  op[11904] = acc93_0;
  op[12032] = acc94_0;
  op[12160] = acc95_0;
  op[12288] = acc96_0;
  op[12416] = acc97_0;
  op[12544] = acc98_0;
}

// Backward from gO = dL/dout: gW[e, w, c] (written), gYp[part][e][m] = partial sums of dL/dY[e, m] over
// the channels and paths of one wave (6 partial(s): channel half h x path group g, part
// h * 3 + g; summed by the caller), gX[send, k, c] (atomic adds).  Null outputs are skipped.
// Path groups (one wave each): [[0, 1, 4, 5, 6, 10, 11, 12, 17, 18], [2, 7, 8, 13, 14, 19, 20], [3, 9, 15, 16, 21, 22]].
extern "C" __global__ void __launch_bounds__(256)
mm_tpw_l0123_bwd_kernel(const int* __restrict__ rowptr, int nR, const int* __restrict__ eid,
    const int* __restrict__ send, const float* __restrict__ Y, long y_stride, const float* __restrict__ W,
    long w_stride, const float* __restrict__ X, long x_stride, const float* __restrict__ gO, long g_stride,
    float* __restrict__ gW, long gw_stride, float* __restrict__ gYp, long gy_cb_stride,
    float* __restrict__ gX, long gx_stride) {
  const int gw = blockIdx.x * 4 + (threadIdx.x >> 6);   // global wave: receiver i, sub-wave h
  const int i = gw / 6, h = gw % 6;
  if (i >= nR) return;
  const int lane = threadIdx.x & 63;
  const int c = (h / 3) * 64 + lane;
  const int p0 = rowptr[i], p1 = rowptr[i + 1];
  const int pg = h % 3;   // path group; channel half h / 3
  const int part = h;
  const int cl = lane & 15;
  const bool b3 = cl & 8, b2 = cl & 4, b1 = cl & 2, b0 = cl & 1;
  if (pg == 0) {
  const float* __restrict__ gp = gO + (size_t)i * g_stride + c;
  const float g0_0 = gp[0];
  const float g1_0 = gp[128];
  const float g4_0 = gp[512];
  const float g5_0 = gp[640];
  const float g6_0 = gp[768];
  const float g7_0 = gp[896];
  const float g8_0 = gp[1024];
  const float g9_0 = gp[1152];
  const float g10_0 = gp[1280];
  const float g11_0 = gp[1408];
  const float g12_0 = gp[1536];
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
  const float g57_0 = gp[7296];
  const float g58_0 = gp[7424];
  const float g59_0 = gp[7552];
  const float g60_0 = gp[7680];
  const float g61_0 = gp[7808];
  const float g62_0 = gp[7936];
  const float g63_0 = gp[8064];
  const float g64_0 = gp[8192];
  const float g65_0 = gp[8320];
  const float g66_0 = gp[8448];
  const float g67_0 = gp[8576];
  const float g68_0 = gp[8704];
  const float g69_0 = gp[8832];
  const float g70_0 = gp[8960];
  const float G0_0 = g0_0;
  const float G1_0 = 0.5773502691896257f * g1_0;
  const float G2_0 = 0.5773502691896258f * g1_0;
  const float G3_0 = 0.5773502691896257f * g1_0;
  const float G4_0 = g4_0;
  const float G5_0 = g5_0;
  const float G6_0 = g6_0;
  const float G7_0 = g7_0;
  const float G8_0 = g8_0;
  const float G9_0 = g9_0;
  const float G10_0 = 0.547722557505166f * g12_0;
  const float G11_0 = 0.547722557505166f * g11_0;
  const float G12_0 = -0.31622776601683794f * g10_0;
  const float G13_0 = -0.547722557505166f * g10_0;
  const float G14_0 = 0.547722557505166f * g10_0;
  const float G15_0 = 0.632455532033676f * g11_0;
  const float G16_0 = 0.547722557505166f * g12_0;
  const float G17_0 = 0.547722557505166f * g10_0;
  const float G18_0 = -0.31622776601683794f * g12_0;
  const float G19_0 = 0.547722557505166f * g11_0;
  const float G20_0 = 0.547722557505166f * g12_0;
  const float G21_0 = g22_0;
  const float G22_0 = g23_0;
  const float G23_0 = g24_0;
  const float G24_0 = g25_0;
  const float G25_0 = g26_0;
  const float G26_0 = fmaf(0.7071067811865475f, g31_0, 0.408248290463863f * g29_0);
  const float G27_0 = -0.7071067811865476f * g28_0;
  const float G28_0 = -0.7071067811865475f * g27_0;
  const float G29_0 = -0.7071067811865476f * g28_0;
  const float G30_0 = -0.8164965809277261f * g29_0;
  const float G31_0 = -0.7071067811865476f * g30_0;
  const float G32_0 = -0.7071067811865475f * g27_0;
  const float G33_0 = -0.7071067811865476f * g30_0;
  const float G34_0 = fmaf(-0.7071067811865475f, g31_0, 0.408248290463863f * g29_0);
  const float G35_0 = 0.5976143046671967f * g36_0;
  const float G36_0 = 0.48795003647426655f * g35_0;
  const float G37_0 = fmaf(0.15430334996209188f, g36_0, 0.5345224838248488f * g34_0);
  const float G38_0 = -0.3779644730092272f * g33_0;
  const float G39_0 = -0.15430334996209188f * g32_0;
  const float G40_0 = -0.48795003647426655f * g33_0;
  const float G41_0 = -0.5976143046671967f * g32_0;
  const float G42_0 = 0.48795003647426655f * g32_0;
  const float G43_0 = 0.6172133998483676f * g33_0;
  const float G44_0 = 0.6546536707079772f * g34_0;
  const float G45_0 = 0.6172133998483676f * g35_0;
  const float G46_0 = 0.48795003647426655f * g36_0;
  const float G47_0 = 0.5976143046671967f * g32_0;
  const float G48_0 = 0.48795003647426655f * g33_0;
  const float G49_0 = -0.15430334996209188f * g32_0;
  const float G50_0 = -0.3779644730092272f * g35_0;
  const float G51_0 = fmaf(-0.15430334996209188f, g36_0, 0.5345224838248488f * g34_0);
  const float G52_0 = 0.48795003647426655f * g35_0;
  const float G53_0 = 0.5976143046671967f * g36_0;
  const float G54_0 = g57_0;
  const float G55_0 = g58_0;
  const float G56_0 = g59_0;
  const float G57_0 = g60_0;
  const float G58_0 = g61_0;
  const float G59_0 = g62_0;
  const float G60_0 = g63_0;
  const float G61_0 = fmaf(0.7071067811865476f, g70_0, 0.18257418583505539f * g68_0);
  const float G62_0 = fmaf(0.5773502691896256f, g69_0, 0.447213595499958f * g67_0);
  const float G63_0 = -0.632455532033676f * g66_0;
  const float G64_0 = -0.5773502691896256f * g65_0;
  const float G65_0 = fmaf(-0.18257418583505539f, g66_0, -0.7071067811865476f * g64_0);
  const float G66_0 = -0.5773502691896258f * g65_0;
  const float G67_0 = -0.7302967433402215f * g66_0;
  const float G68_0 = -0.7745966692414836f * g67_0;
  const float G69_0 = -0.7302967433402215f * g68_0;
  const float G70_0 = -0.5773502691896258f * g69_0;
  const float G71_0 = fmaf(0.18257418583505539f, g66_0, -0.7071067811865476f * g64_0);
  const float G72_0 = -0.5773502691896256f * g65_0;
  const float G73_0 = -0.632455532033676f * g68_0;
  const float G74_0 = fmaf(-0.5773502691896256f, g69_0, 0.447213595499958f * g67_0);
  const float G75_0 = fmaf(-0.7071067811865476f, g70_0, 0.18257418583505539f * g68_0);
  for (int p = p0; p < p1; ++p) {
    const int ea = __builtin_amdgcn_readfirstlane(eid ? eid[p] : p);
    const int sa = __builtin_amdgcn_readfirstlane(send[ea]);
    const float* __restrict__ wpa = W + (size_t)ea * w_stride + c;
    const float W0_0_a = wpa[0];
    const float W1_0_a = wpa[128];
    const float W4_0_a = wpa[512];
    const float W5_0_a = wpa[640];
    const float W6_0_a = wpa[768];
    const float W10_0_a = wpa[1280];
    const float W11_0_a = wpa[1408];
    const float W12_0_a = wpa[1536];
    const float W17_0_a = wpa[2176];
    const float W18_0_a = wpa[2304];
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
      { const float q = W4_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y1_a, G4_0, u); gy1 = fmaf(q, G4_0, gy1);
        u = fmaf(Y2_a, G5_0, u); gy2 = fmaf(q, G5_0, gy2);
        u = fmaf(Y3_a, G6_0, u); gy3 = fmaf(q, G6_0, gy3);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W4_0_a, u, gx0_0);
      }
      if (gwp) gwp[512] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W5_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y0_a, G7_0, u); gy0 = fmaf(q, G7_0, gy0);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W5_0_a, u, gx1_0);
      }
      { const float q = W5_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y0_a, G8_0, u); gy0 = fmaf(q, G8_0, gy0);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W5_0_a, u, gx2_0);
      }
      { const float q = W5_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y0_a, G9_0, u); gy0 = fmaf(q, G9_0, gy0);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W5_0_a, u, gx3_0);
      }
      if (gwp) gwp[640] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W6_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y4_a, G10_0, u); gy4 = fmaf(q, G10_0, gy4);
        u = fmaf(Y5_a, G11_0, u); gy5 = fmaf(q, G11_0, gy5);
        u = fmaf(Y6_a, G12_0, u); gy6 = fmaf(q, G12_0, gy6);
        u = fmaf(Y8_a, G13_0, u); gy8 = fmaf(q, G13_0, gy8);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W6_0_a, u, gx1_0);
      }
      { const float q = W6_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y5_a, G14_0, u); gy5 = fmaf(q, G14_0, gy5);
        u = fmaf(Y6_a, G15_0, u); gy6 = fmaf(q, G15_0, gy6);
        u = fmaf(Y7_a, G16_0, u); gy7 = fmaf(q, G16_0, gy7);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W6_0_a, u, gx2_0);
      }
      { const float q = W6_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y4_a, G17_0, u); gy4 = fmaf(q, G17_0, gy4);
        u = fmaf(Y6_a, G18_0, u); gy6 = fmaf(q, G18_0, gy6);
        u = fmaf(Y7_a, G19_0, u); gy7 = fmaf(q, G19_0, gy7);
        u = fmaf(Y8_a, G20_0, u); gy8 = fmaf(q, G20_0, gy8);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W6_0_a, u, gx3_0);
      }
      if (gwp) gwp[768] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W10_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y4_a, G21_0, u); gy4 = fmaf(q, G21_0, gy4);
        u = fmaf(Y5_a, G22_0, u); gy5 = fmaf(q, G22_0, gy5);
        u = fmaf(Y6_a, G23_0, u); gy6 = fmaf(q, G23_0, gy6);
        u = fmaf(Y7_a, G24_0, u); gy7 = fmaf(q, G24_0, gy7);
        u = fmaf(Y8_a, G25_0, u); gy8 = fmaf(q, G25_0, gy8);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W10_0_a, u, gx0_0);
      }
      if (gwp) gwp[1280] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W11_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y1_a, G26_0, u); gy1 = fmaf(q, G26_0, gy1);
        u = fmaf(Y2_a, G27_0, u); gy2 = fmaf(q, G27_0, gy2);
        u = fmaf(Y3_a, G28_0, u); gy3 = fmaf(q, G28_0, gy3);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W11_0_a, u, gx1_0);
      }
      { const float q = W11_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y1_a, G29_0, u); gy1 = fmaf(q, G29_0, gy1);
        u = fmaf(Y2_a, G30_0, u); gy2 = fmaf(q, G30_0, gy2);
        u = fmaf(Y3_a, G31_0, u); gy3 = fmaf(q, G31_0, gy3);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W11_0_a, u, gx2_0);
      }
      { const float q = W11_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y1_a, G32_0, u); gy1 = fmaf(q, G32_0, gy1);
        u = fmaf(Y2_a, G33_0, u); gy2 = fmaf(q, G33_0, gy2);
        u = fmaf(Y3_a, G34_0, u); gy3 = fmaf(q, G34_0, gy3);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W11_0_a, u, gx3_0);
      }
      if (gwp) gwp[1408] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W12_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y9_a, G35_0, u); gy9 = fmaf(q, G35_0, gy9);
        u = fmaf(Y10_a, G36_0, u); gy10 = fmaf(q, G36_0, gy10);
        u = fmaf(Y11_a, G37_0, u); gy11 = fmaf(q, G37_0, gy11);
        u = fmaf(Y12_a, G38_0, u); gy12 = fmaf(q, G38_0, gy12);
        u = fmaf(Y13_a, G39_0, u); gy13 = fmaf(q, G39_0, gy13);
        u = fmaf(Y14_a, G40_0, u); gy14 = fmaf(q, G40_0, gy14);
        u = fmaf(Y15_a, G41_0, u); gy15 = fmaf(q, G41_0, gy15);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W12_0_a, u, gx1_0);
      }
      { const float q = W12_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y10_a, G42_0, u); gy10 = fmaf(q, G42_0, gy10);
        u = fmaf(Y11_a, G43_0, u); gy11 = fmaf(q, G43_0, gy11);
        u = fmaf(Y12_a, G44_0, u); gy12 = fmaf(q, G44_0, gy12);
        u = fmaf(Y13_a, G45_0, u); gy13 = fmaf(q, G45_0, gy13);
        u = fmaf(Y14_a, G46_0, u); gy14 = fmaf(q, G46_0, gy14);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W12_0_a, u, gx2_0);
      }
      { const float q = W12_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y9_a, G47_0, u); gy9 = fmaf(q, G47_0, gy9);
        u = fmaf(Y10_a, G48_0, u); gy10 = fmaf(q, G48_0, gy10);
        u = fmaf(Y11_a, G49_0, u); gy11 = fmaf(q, G49_0, gy11);
        u = fmaf(Y12_a, G50_0, u); gy12 = fmaf(q, G50_0, gy12);
        u = fmaf(Y13_a, G51_0, u); gy13 = fmaf(q, G51_0, gy13);
        u = fmaf(Y14_a, G52_0, u); gy14 = fmaf(q, G52_0, gy14);
        u = fmaf(Y15_a, G53_0, u); gy15 = fmaf(q, G53_0, gy15);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W12_0_a, u, gx3_0);
      }
      if (gwp) gwp[1536] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W17_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y9_a, G54_0, u); gy9 = fmaf(q, G54_0, gy9);
        u = fmaf(Y10_a, G55_0, u); gy10 = fmaf(q, G55_0, gy10);
        u = fmaf(Y11_a, G56_0, u); gy11 = fmaf(q, G56_0, gy11);
        u = fmaf(Y12_a, G57_0, u); gy12 = fmaf(q, G57_0, gy12);
        u = fmaf(Y13_a, G58_0, u); gy13 = fmaf(q, G58_0, gy13);
        u = fmaf(Y14_a, G59_0, u); gy14 = fmaf(q, G59_0, gy14);
        u = fmaf(Y15_a, G60_0, u); gy15 = fmaf(q, G60_0, gy15);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W17_0_a, u, gx0_0);
      }
      if (gwp) gwp[2176] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W18_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y4_a, G61_0, u); gy4 = fmaf(q, G61_0, gy4);
        u = fmaf(Y5_a, G62_0, u); gy5 = fmaf(q, G62_0, gy5);
        u = fmaf(Y6_a, G63_0, u); gy6 = fmaf(q, G63_0, gy6);
        u = fmaf(Y7_a, G64_0, u); gy7 = fmaf(q, G64_0, gy7);
        u = fmaf(Y8_a, G65_0, u); gy8 = fmaf(q, G65_0, gy8);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W18_0_a, u, gx1_0);
      }
      { const float q = W18_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y4_a, G66_0, u); gy4 = fmaf(q, G66_0, gy4);
        u = fmaf(Y5_a, G67_0, u); gy5 = fmaf(q, G67_0, gy5);
        u = fmaf(Y6_a, G68_0, u); gy6 = fmaf(q, G68_0, gy6);
        u = fmaf(Y7_a, G69_0, u); gy7 = fmaf(q, G69_0, gy7);
        u = fmaf(Y8_a, G70_0, u); gy8 = fmaf(q, G70_0, gy8);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W18_0_a, u, gx2_0);
      }
      { const float q = W18_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y4_a, G71_0, u); gy4 = fmaf(q, G71_0, gy4);
        u = fmaf(Y5_a, G72_0, u); gy5 = fmaf(q, G72_0, gy5);
        u = fmaf(Y6_a, G73_0, u); gy6 = fmaf(q, G73_0, gy6);
        u = fmaf(Y7_a, G74_0, u); gy7 = fmaf(q, G74_0, gy7);
        u = fmaf(Y8_a, G75_0, u); gy8 = fmaf(q, G75_0, gy8);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W18_0_a, u, gx3_0);
      }
      if (gwp) gwp[2304] = gw0;
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
  }
  }
  else if (pg == 1) {
  const float* __restrict__ gp = gO + (size_t)i * g_stride + c;
  const float g2_0 = gp[256];
  const float g13_0 = gp[1664];
  const float g14_0 = gp[1792];
  const float g15_0 = gp[1920];
  const float g16_0 = gp[2048];
  const float g17_0 = gp[2176];
  const float g18_0 = gp[2304];
  const float g37_0 = gp[4736];
  const float g38_0 = gp[4864];
  const float g39_0 = gp[4992];
  const float g40_0 = gp[5120];
  const float g41_0 = gp[5248];
  const float g42_0 = gp[5376];
  const float g43_0 = gp[5504];
  const float g44_0 = gp[5632];
  const float g45_0 = gp[5760];
  const float g46_0 = gp[5888];
  const float g71_0 = gp[9088];
  const float g72_0 = gp[9216];
  const float g73_0 = gp[9344];
  const float g74_0 = gp[9472];
  const float g75_0 = gp[9600];
  const float g76_0 = gp[9728];
  const float g77_0 = gp[9856];
  const float g78_0 = gp[9984];
  const float g79_0 = gp[10112];
  const float g80_0 = gp[10240];
  const float g81_0 = gp[10368];
  const float g82_0 = gp[10496];
  const float g83_0 = gp[10624];
  const float g84_0 = gp[10752];
  const float G0_0 = 0.4472135954999579f * g2_0;
  const float G1_0 = 0.4472135954999579f * g2_0;
  const float G2_0 = 0.44721359549995804f * g2_0;
  const float G3_0 = 0.4472135954999579f * g2_0;
  const float G4_0 = 0.4472135954999579f * g2_0;
  const float G5_0 = 0.547722557505166f * g15_0;
  const float G6_0 = 0.547722557505166f * g13_0;
  const float G7_0 = 0.547722557505166f * g14_0;
  const float G8_0 = 0.547722557505166f * g13_0;
  const float G9_0 = -0.31622776601683794f * g13_0;
  const float G10_0 = 0.632455532033676f * g14_0;
  const float G11_0 = -0.31622776601683794f * g15_0;
  const float G12_0 = 0.547722557505166f * g15_0;
  const float G13_0 = 0.547722557505166f * g14_0;
  const float G14_0 = -0.547722557505166f * g13_0;
  const float G15_0 = 0.547722557505166f * g15_0;
  const float G16_0 = 0.4629100498862757f * g18_0;
  const float G17_0 = 0.3779644730092272f * g17_0;
  const float G18_0 = -0.11952286093343936f * g18_0;
  const float G19_0 = -0.11952286093343936f * g16_0;
  const float G20_0 = -0.4629100498862757f * g16_0;
  const float G21_0 = 0.3779644730092272f * g18_0;
  const float G22_0 = 0.47809144373375745f * g17_0;
  const float G23_0 = -0.29277002188456f * g16_0;
  const float G24_0 = -0.3779644730092272f * g16_0;
  const float G25_0 = 0.41403933560541256f * g16_0;
  const float G26_0 = 0.5070925528371102f * g17_0;
  const float G27_0 = 0.41403933560541256f * g18_0;
  const float G28_0 = 0.3779644730092272f * g16_0;
  const float G29_0 = -0.29277002188456f * g18_0;
  const float G30_0 = 0.47809144373375745f * g17_0;
  const float G31_0 = 0.3779644730092272f * g18_0;
  const float G32_0 = 0.4629100498862757f * g16_0;
  const float G33_0 = 0.11952286093343936f * g16_0;
  const float G34_0 = -0.11952286093343936f * g18_0;
  const float G35_0 = 0.3779644730092272f * g17_0;
  const float G36_0 = 0.4629100498862757f * g18_0;
  const float G37_0 = g37_0;
  const float G38_0 = g38_0;
  const float G39_0 = g39_0;
  const float G40_0 = g40_0;
  const float G41_0 = g41_0;
  const float G42_0 = 0.5345224838248488f * g44_0;
  const float G43_0 = -0.46291004988627565f * g45_0;
  const float G44_0 = 0.5345224838248488f * g42_0;
  const float G45_0 = -0.46291004988627565f * g43_0;
  const float G46_0 = -0.46291004988627565f * g45_0;
  const float G47_0 = fmaf(0.46291004988627565f, g46_0, -0.2672612419124244f * g44_0);
  const float G48_0 = -0.2672612419124244f * g43_0;
  const float G49_0 = -0.46291004988627565f * g42_0;
  const float G50_0 = 0.46291004988627565f * g43_0;
  const float G51_0 = 0.5345224838248488f * g42_0;
  const float G52_0 = -0.2672612419124244f * g43_0;
  const float G53_0 = -0.5345224838248489f * g44_0;
  const float G54_0 = -0.2672612419124244f * g45_0;
  const float G55_0 = 0.5345224838248488f * g46_0;
  const float G56_0 = -0.46291004988627565f * g43_0;
  const float G57_0 = -0.46291004988627565f * g42_0;
  const float G58_0 = -0.2672612419124244f * g45_0;
  const float G59_0 = fmaf(-0.46291004988627565f, g46_0, -0.2672612419124244f * g44_0);
  const float G60_0 = -0.46291004988627565f * g45_0;
  const float G61_0 = 0.46291004988627565f * g43_0;
  const float G62_0 = 0.5345224838248488f * g46_0;
  const float G63_0 = -0.46291004988627565f * g45_0;
  const float G64_0 = 0.5345224838248488f * g44_0;
  const float G65_0 = fmaf(0.7071067811865476f, g77_0, 0.18257418583505539f * g75_0);
  const float G66_0 = -0.5773502691896258f * g72_0;
  const float G67_0 = fmaf(0.18257418583505539f, g73_0, -0.7071067811865476f * g71_0);
  const float G68_0 = fmaf(0.5773502691896256f, g76_0, 0.447213595499958f * g74_0);
  const float G69_0 = -0.7302967433402215f * g73_0;
  const float G70_0 = -0.5773502691896256f * g72_0;
  const float G71_0 = -0.632455532033676f * g73_0;
  const float G72_0 = -0.7745966692414836f * g74_0;
  const float G73_0 = -0.632455532033676f * g75_0;
  const float G74_0 = -0.5773502691896256f * g72_0;
  const float G75_0 = -0.7302967433402215f * g75_0;
  const float G76_0 = fmaf(-0.5773502691896256f, g76_0, 0.447213595499958f * g74_0);
  const float G77_0 = fmaf(-0.18257418583505539f, g73_0, -0.7071067811865476f * g71_0);
  const float G78_0 = -0.5773502691896258f * g76_0;
  const float G79_0 = fmaf(-0.7071067811865476f, g77_0, 0.18257418583505539f * g75_0);
  const float G80_0 = 0.2886751345948128f * g82_0;
  const float G81_0 = 0.5773502691896258f * g81_0;
  const float G82_0 = fmaf(-0.2886751345948128f, g84_0, -0.447213595499958f * g82_0);
  const float G83_0 = 0.5773502691896258f * g79_0;
  const float G84_0 = fmaf(-0.447213595499958f, g80_0, 0.2886751345948128f * g78_0);
  const float G85_0 = -0.2886751345948128f * g80_0;
  const float G86_0 = -0.45643546458763845f * g83_0;
  const float G87_0 = fmaf(0.45643546458763845f, g84_0, -0.3535533905932738f * g82_0);
  const float G88_0 = fmaf(0.3535533905932738f, g83_0, -0.18257418583505539f * g81_0);
  const float G89_0 = -0.18257418583505539f * g80_0;
  const float G90_0 = -0.3535533905932738f * g79_0;
  const float G91_0 = fmaf(0.3535533905932738f, g80_0, -0.45643546458763845f * g78_0);
  const float G92_0 = 0.45643546458763845f * g79_0;
  const float G93_0 = 0.6454972243679029f * g78_0;
  const float G94_0 = -0.3872983346207418f * g80_0;
  const float G95_0 = -0.5163977794943223f * g81_0;
  const float G96_0 = -0.3872983346207418f * g82_0;
  const float G97_0 = 0.6454972243679029f * g84_0;
  const float G98_0 = -0.45643546458763845f * g79_0;
  const float G99_0 = fmaf(-0.3535533905932738f, g80_0, -0.45643546458763845f * g78_0);
  const float G100_0 = -0.3535533905932738f * g79_0;
  const float G101_0 = -0.18257418583505539f * g82_0;
  const float G102_0 = fmaf(-0.3535533905932738f, g83_0, -0.18257418583505539f * g81_0);
  const float G103_0 = fmaf(-0.45643546458763845f, g84_0, -0.3535533905932738f * g82_0);
  const float G104_0 = -0.45643546458763845f * g83_0;
  const float G105_0 = 0.2886751345948128f * g80_0;
  const float G106_0 = fmaf(0.447213595499958f, g80_0, 0.2886751345948128f * g78_0);
  const float G107_0 = 0.5773502691896258f * g83_0;
  const float G108_0 = fmaf(0.2886751345948128f, g84_0, -0.447213595499958f * g82_0);
  const float G109_0 = 0.5773502691896258f * g81_0;
  const float G110_0 = 0.2886751345948128f * g82_0;
  for (int p = p0; p < p1; ++p) {
    const int ea = __builtin_amdgcn_readfirstlane(eid ? eid[p] : p);
    const int sa = __builtin_amdgcn_readfirstlane(send[ea]);
    const float* __restrict__ wpa = W + (size_t)ea * w_stride + c;
    const float W2_0_a = wpa[256];
    const float W7_0_a = wpa[896];
    const float W8_0_a = wpa[1024];
    const float W13_0_a = wpa[1664];
    const float W14_0_a = wpa[1792];
    const float W19_0_a = wpa[2432];
    const float W20_0_a = wpa[2560];
    const float* __restrict__ xpa = X + (size_t)sa * x_stride + c;
    const float X4_0_a = xpa[512];
    const float X5_0_a = xpa[640];
    const float X6_0_a = xpa[768];
    const float X7_0_a = xpa[896];
    const float X8_0_a = xpa[1024];
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
    float gx4_0 = 0.f;
    float gx5_0 = 0.f;
    float gx6_0 = 0.f;
    float gx7_0 = 0.f;
    float gx8_0 = 0.f;
    float* __restrict__ gwp = gW ? gW + (size_t)ea * gw_stride + c : nullptr;
    {
      float gw0 = 0.f;
      { const float q = W2_0_a * X4_0_a; float u = 0.f;
        u = fmaf(Y4_a, G0_0, u); gy4 = fmaf(q, G0_0, gy4);
        gw0 = fmaf(X4_0_a, u, gw0); gx4_0 = fmaf(W2_0_a, u, gx4_0);
      }
      { const float q = W2_0_a * X5_0_a; float u = 0.f;
        u = fmaf(Y5_a, G1_0, u); gy5 = fmaf(q, G1_0, gy5);
        gw0 = fmaf(X5_0_a, u, gw0); gx5_0 = fmaf(W2_0_a, u, gx5_0);
      }
      { const float q = W2_0_a * X6_0_a; float u = 0.f;
        u = fmaf(Y6_a, G2_0, u); gy6 = fmaf(q, G2_0, gy6);
        gw0 = fmaf(X6_0_a, u, gw0); gx6_0 = fmaf(W2_0_a, u, gx6_0);
      }
      { const float q = W2_0_a * X7_0_a; float u = 0.f;
        u = fmaf(Y7_a, G3_0, u); gy7 = fmaf(q, G3_0, gy7);
        gw0 = fmaf(X7_0_a, u, gw0); gx7_0 = fmaf(W2_0_a, u, gx7_0);
      }
      { const float q = W2_0_a * X8_0_a; float u = 0.f;
        u = fmaf(Y8_a, G4_0, u); gy8 = fmaf(q, G4_0, gy8);
        gw0 = fmaf(X8_0_a, u, gw0); gx8_0 = fmaf(W2_0_a, u, gx8_0);
      }
      if (gwp) gwp[256] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W7_0_a * X4_0_a; float u = 0.f;
        u = fmaf(Y1_a, G5_0, u); gy1 = fmaf(q, G5_0, gy1);
        u = fmaf(Y3_a, G6_0, u); gy3 = fmaf(q, G6_0, gy3);
        gw0 = fmaf(X4_0_a, u, gw0); gx4_0 = fmaf(W7_0_a, u, gx4_0);
      }
      { const float q = W7_0_a * X5_0_a; float u = 0.f;
        u = fmaf(Y1_a, G7_0, u); gy1 = fmaf(q, G7_0, gy1);
        u = fmaf(Y2_a, G8_0, u); gy2 = fmaf(q, G8_0, gy2);
        gw0 = fmaf(X5_0_a, u, gw0); gx5_0 = fmaf(W7_0_a, u, gx5_0);
      }
      { const float q = W7_0_a * X6_0_a; float u = 0.f;
        u = fmaf(Y1_a, G9_0, u); gy1 = fmaf(q, G9_0, gy1);
        u = fmaf(Y2_a, G10_0, u); gy2 = fmaf(q, G10_0, gy2);
        u = fmaf(Y3_a, G11_0, u); gy3 = fmaf(q, G11_0, gy3);
        gw0 = fmaf(X6_0_a, u, gw0); gx6_0 = fmaf(W7_0_a, u, gx6_0);
      }
      { const float q = W7_0_a * X7_0_a; float u = 0.f;
        u = fmaf(Y2_a, G12_0, u); gy2 = fmaf(q, G12_0, gy2);
        u = fmaf(Y3_a, G13_0, u); gy3 = fmaf(q, G13_0, gy3);
        gw0 = fmaf(X7_0_a, u, gw0); gx7_0 = fmaf(W7_0_a, u, gx7_0);
      }
      { const float q = W7_0_a * X8_0_a; float u = 0.f;
        u = fmaf(Y1_a, G14_0, u); gy1 = fmaf(q, G14_0, gy1);
        u = fmaf(Y3_a, G15_0, u); gy3 = fmaf(q, G15_0, gy3);
        gw0 = fmaf(X8_0_a, u, gw0); gx8_0 = fmaf(W7_0_a, u, gx8_0);
      }
      if (gwp) gwp[896] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W8_0_a * X4_0_a; float u = 0.f;
        u = fmaf(Y9_a, G16_0, u); gy9 = fmaf(q, G16_0, gy9);
        u = fmaf(Y10_a, G17_0, u); gy10 = fmaf(q, G17_0, gy10);
        u = fmaf(Y11_a, G18_0, u); gy11 = fmaf(q, G18_0, gy11);
        u = fmaf(Y13_a, G19_0, u); gy13 = fmaf(q, G19_0, gy13);
        u = fmaf(Y15_a, G20_0, u); gy15 = fmaf(q, G20_0, gy15);
        gw0 = fmaf(X4_0_a, u, gw0); gx4_0 = fmaf(W8_0_a, u, gx4_0);
      }
      { const float q = W8_0_a * X5_0_a; float u = 0.f;
        u = fmaf(Y10_a, G21_0, u); gy10 = fmaf(q, G21_0, gy10);
        u = fmaf(Y11_a, G22_0, u); gy11 = fmaf(q, G22_0, gy11);
        u = fmaf(Y12_a, G23_0, u); gy12 = fmaf(q, G23_0, gy12);
        u = fmaf(Y14_a, G24_0, u); gy14 = fmaf(q, G24_0, gy14);
        gw0 = fmaf(X5_0_a, u, gw0); gx5_0 = fmaf(W8_0_a, u, gx5_0);
      }
      { const float q = W8_0_a * X6_0_a; float u = 0.f;
        u = fmaf(Y11_a, G25_0, u); gy11 = fmaf(q, G25_0, gy11);
        u = fmaf(Y12_a, G26_0, u); gy12 = fmaf(q, G26_0, gy12);
        u = fmaf(Y13_a, G27_0, u); gy13 = fmaf(q, G27_0, gy13);
        gw0 = fmaf(X6_0_a, u, gw0); gx6_0 = fmaf(W8_0_a, u, gx6_0);
      }
      { const float q = W8_0_a * X7_0_a; float u = 0.f;
        u = fmaf(Y10_a, G28_0, u); gy10 = fmaf(q, G28_0, gy10);
        u = fmaf(Y12_a, G29_0, u); gy12 = fmaf(q, G29_0, gy12);
        u = fmaf(Y13_a, G30_0, u); gy13 = fmaf(q, G30_0, gy13);
        u = fmaf(Y14_a, G31_0, u); gy14 = fmaf(q, G31_0, gy14);
        gw0 = fmaf(X7_0_a, u, gw0); gx7_0 = fmaf(W8_0_a, u, gx7_0);
      }
      { const float q = W8_0_a * X8_0_a; float u = 0.f;
        u = fmaf(Y9_a, G32_0, u); gy9 = fmaf(q, G32_0, gy9);
        u = fmaf(Y11_a, G33_0, u); gy11 = fmaf(q, G33_0, gy11);
        u = fmaf(Y13_a, G34_0, u); gy13 = fmaf(q, G34_0, gy13);
        u = fmaf(Y14_a, G35_0, u); gy14 = fmaf(q, G35_0, gy14);
        u = fmaf(Y15_a, G36_0, u); gy15 = fmaf(q, G36_0, gy15);
        gw0 = fmaf(X8_0_a, u, gw0); gx8_0 = fmaf(W8_0_a, u, gx8_0);
      }
      if (gwp) gwp[1024] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W13_0_a * X4_0_a; float u = 0.f;
        u = fmaf(Y0_a, G37_0, u); gy0 = fmaf(q, G37_0, gy0);
        gw0 = fmaf(X4_0_a, u, gw0); gx4_0 = fmaf(W13_0_a, u, gx4_0);
      }
      { const float q = W13_0_a * X5_0_a; float u = 0.f;
        u = fmaf(Y0_a, G38_0, u); gy0 = fmaf(q, G38_0, gy0);
        gw0 = fmaf(X5_0_a, u, gw0); gx5_0 = fmaf(W13_0_a, u, gx5_0);
      }
      { const float q = W13_0_a * X6_0_a; float u = 0.f;
        u = fmaf(Y0_a, G39_0, u); gy0 = fmaf(q, G39_0, gy0);
        gw0 = fmaf(X6_0_a, u, gw0); gx6_0 = fmaf(W13_0_a, u, gx6_0);
      }
      { const float q = W13_0_a * X7_0_a; float u = 0.f;
        u = fmaf(Y0_a, G40_0, u); gy0 = fmaf(q, G40_0, gy0);
        gw0 = fmaf(X7_0_a, u, gw0); gx7_0 = fmaf(W13_0_a, u, gx7_0);
      }
      { const float q = W13_0_a * X8_0_a; float u = 0.f;
        u = fmaf(Y0_a, G41_0, u); gy0 = fmaf(q, G41_0, gy0);
        gw0 = fmaf(X8_0_a, u, gw0); gx8_0 = fmaf(W13_0_a, u, gx8_0);
      }
      if (gwp) gwp[1664] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W14_0_a * X4_0_a; float u = 0.f;
        u = fmaf(Y4_a, G42_0, u); gy4 = fmaf(q, G42_0, gy4);
        u = fmaf(Y5_a, G43_0, u); gy5 = fmaf(q, G43_0, gy5);
        u = fmaf(Y6_a, G44_0, u); gy6 = fmaf(q, G44_0, gy6);
        u = fmaf(Y7_a, G45_0, u); gy7 = fmaf(q, G45_0, gy7);
        gw0 = fmaf(X4_0_a, u, gw0); gx4_0 = fmaf(W14_0_a, u, gx4_0);
      }
      { const float q = W14_0_a * X5_0_a; float u = 0.f;
        u = fmaf(Y4_a, G46_0, u); gy4 = fmaf(q, G46_0, gy4);
        u = fmaf(Y5_a, G47_0, u); gy5 = fmaf(q, G47_0, gy5);
        u = fmaf(Y6_a, G48_0, u); gy6 = fmaf(q, G48_0, gy6);
        u = fmaf(Y7_a, G49_0, u); gy7 = fmaf(q, G49_0, gy7);
        u = fmaf(Y8_a, G50_0, u); gy8 = fmaf(q, G50_0, gy8);
        gw0 = fmaf(X5_0_a, u, gw0); gx5_0 = fmaf(W14_0_a, u, gx5_0);
      }
      { const float q = W14_0_a * X6_0_a; float u = 0.f;
        u = fmaf(Y4_a, G51_0, u); gy4 = fmaf(q, G51_0, gy4);
        u = fmaf(Y5_a, G52_0, u); gy5 = fmaf(q, G52_0, gy5);
        u = fmaf(Y6_a, G53_0, u); gy6 = fmaf(q, G53_0, gy6);
        u = fmaf(Y7_a, G54_0, u); gy7 = fmaf(q, G54_0, gy7);
        u = fmaf(Y8_a, G55_0, u); gy8 = fmaf(q, G55_0, gy8);
        gw0 = fmaf(X6_0_a, u, gw0); gx6_0 = fmaf(W14_0_a, u, gx6_0);
      }
      { const float q = W14_0_a * X7_0_a; float u = 0.f;
        u = fmaf(Y4_a, G56_0, u); gy4 = fmaf(q, G56_0, gy4);
        u = fmaf(Y5_a, G57_0, u); gy5 = fmaf(q, G57_0, gy5);
        u = fmaf(Y6_a, G58_0, u); gy6 = fmaf(q, G58_0, gy6);
        u = fmaf(Y7_a, G59_0, u); gy7 = fmaf(q, G59_0, gy7);
        u = fmaf(Y8_a, G60_0, u); gy8 = fmaf(q, G60_0, gy8);
        gw0 = fmaf(X7_0_a, u, gw0); gx7_0 = fmaf(W14_0_a, u, gx7_0);
      }
      { const float q = W14_0_a * X8_0_a; float u = 0.f;
        u = fmaf(Y5_a, G61_0, u); gy5 = fmaf(q, G61_0, gy5);
        u = fmaf(Y6_a, G62_0, u); gy6 = fmaf(q, G62_0, gy6);
        u = fmaf(Y7_a, G63_0, u); gy7 = fmaf(q, G63_0, gy7);
        u = fmaf(Y8_a, G64_0, u); gy8 = fmaf(q, G64_0, gy8);
        gw0 = fmaf(X8_0_a, u, gw0); gx8_0 = fmaf(W14_0_a, u, gx8_0);
      }
      if (gwp) gwp[1792] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W19_0_a * X4_0_a; float u = 0.f;
        u = fmaf(Y1_a, G65_0, u); gy1 = fmaf(q, G65_0, gy1);
        u = fmaf(Y2_a, G66_0, u); gy2 = fmaf(q, G66_0, gy2);
        u = fmaf(Y3_a, G67_0, u); gy3 = fmaf(q, G67_0, gy3);
        gw0 = fmaf(X4_0_a, u, gw0); gx4_0 = fmaf(W19_0_a, u, gx4_0);
      }
      { const float q = W19_0_a * X5_0_a; float u = 0.f;
        u = fmaf(Y1_a, G68_0, u); gy1 = fmaf(q, G68_0, gy1);
        u = fmaf(Y2_a, G69_0, u); gy2 = fmaf(q, G69_0, gy2);
        u = fmaf(Y3_a, G70_0, u); gy3 = fmaf(q, G70_0, gy3);
        gw0 = fmaf(X5_0_a, u, gw0); gx5_0 = fmaf(W19_0_a, u, gx5_0);
      }
      { const float q = W19_0_a * X6_0_a; float u = 0.f;
        u = fmaf(Y1_a, G71_0, u); gy1 = fmaf(q, G71_0, gy1);
        u = fmaf(Y2_a, G72_0, u); gy2 = fmaf(q, G72_0, gy2);
        u = fmaf(Y3_a, G73_0, u); gy3 = fmaf(q, G73_0, gy3);
        gw0 = fmaf(X6_0_a, u, gw0); gx6_0 = fmaf(W19_0_a, u, gx6_0);
      }
      { const float q = W19_0_a * X7_0_a; float u = 0.f;
        u = fmaf(Y1_a, G74_0, u); gy1 = fmaf(q, G74_0, gy1);
        u = fmaf(Y2_a, G75_0, u); gy2 = fmaf(q, G75_0, gy2);
        u = fmaf(Y3_a, G76_0, u); gy3 = fmaf(q, G76_0, gy3);
        gw0 = fmaf(X7_0_a, u, gw0); gx7_0 = fmaf(W19_0_a, u, gx7_0);
      }
      { const float q = W19_0_a * X8_0_a; float u = 0.f;
        u = fmaf(Y1_a, G77_0, u); gy1 = fmaf(q, G77_0, gy1);
        u = fmaf(Y2_a, G78_0, u); gy2 = fmaf(q, G78_0, gy2);
        u = fmaf(Y3_a, G79_0, u); gy3 = fmaf(q, G79_0, gy3);
        gw0 = fmaf(X8_0_a, u, gw0); gx8_0 = fmaf(W19_0_a, u, gx8_0);
      }
      if (gwp) gwp[2432] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W20_0_a * X4_0_a; float u = 0.f;
        u = fmaf(Y9_a, G80_0, u); gy9 = fmaf(q, G80_0, gy9);
        u = fmaf(Y10_a, G81_0, u); gy10 = fmaf(q, G81_0, gy10);
        u = fmaf(Y11_a, G82_0, u); gy11 = fmaf(q, G82_0, gy11);
        u = fmaf(Y12_a, G83_0, u); gy12 = fmaf(q, G83_0, gy12);
        u = fmaf(Y13_a, G84_0, u); gy13 = fmaf(q, G84_0, gy13);
        u = fmaf(Y15_a, G85_0, u); gy15 = fmaf(q, G85_0, gy15);
        gw0 = fmaf(X4_0_a, u, gw0); gx4_0 = fmaf(W20_0_a, u, gx4_0);
      }
      { const float q = W20_0_a * X5_0_a; float u = 0.f;
        u = fmaf(Y9_a, G86_0, u); gy9 = fmaf(q, G86_0, gy9);
        u = fmaf(Y10_a, G87_0, u); gy10 = fmaf(q, G87_0, gy10);
        u = fmaf(Y11_a, G88_0, u); gy11 = fmaf(q, G88_0, gy11);
        u = fmaf(Y12_a, G89_0, u); gy12 = fmaf(q, G89_0, gy12);
        u = fmaf(Y13_a, G90_0, u); gy13 = fmaf(q, G90_0, gy13);
        u = fmaf(Y14_a, G91_0, u); gy14 = fmaf(q, G91_0, gy14);
        u = fmaf(Y15_a, G92_0, u); gy15 = fmaf(q, G92_0, gy15);
        gw0 = fmaf(X5_0_a, u, gw0); gx5_0 = fmaf(W20_0_a, u, gx5_0);
      }
      { const float q = W20_0_a * X6_0_a; float u = 0.f;
        u = fmaf(Y9_a, G93_0, u); gy9 = fmaf(q, G93_0, gy9);
        u = fmaf(Y11_a, G94_0, u); gy11 = fmaf(q, G94_0, gy11);
        u = fmaf(Y12_a, G95_0, u); gy12 = fmaf(q, G95_0, gy12);
        u = fmaf(Y13_a, G96_0, u); gy13 = fmaf(q, G96_0, gy13);
        u = fmaf(Y15_a, G97_0, u); gy15 = fmaf(q, G97_0, gy15);
        gw0 = fmaf(X6_0_a, u, gw0); gx6_0 = fmaf(W20_0_a, u, gx6_0);
      }
      { const float q = W20_0_a * X7_0_a; float u = 0.f;
        u = fmaf(Y9_a, G98_0, u); gy9 = fmaf(q, G98_0, gy9);
        u = fmaf(Y10_a, G99_0, u); gy10 = fmaf(q, G99_0, gy10);
        u = fmaf(Y11_a, G100_0, u); gy11 = fmaf(q, G100_0, gy11);
        u = fmaf(Y12_a, G101_0, u); gy12 = fmaf(q, G101_0, gy12);
        u = fmaf(Y13_a, G102_0, u); gy13 = fmaf(q, G102_0, gy13);
        u = fmaf(Y14_a, G103_0, u); gy14 = fmaf(q, G103_0, gy14);
        u = fmaf(Y15_a, G104_0, u); gy15 = fmaf(q, G104_0, gy15);
        gw0 = fmaf(X7_0_a, u, gw0); gx7_0 = fmaf(W20_0_a, u, gx7_0);
      }
      { const float q = W20_0_a * X8_0_a; float u = 0.f;
        u = fmaf(Y9_a, G105_0, u); gy9 = fmaf(q, G105_0, gy9);
        u = fmaf(Y11_a, G106_0, u); gy11 = fmaf(q, G106_0, gy11);
        u = fmaf(Y12_a, G107_0, u); gy12 = fmaf(q, G107_0, gy12);
        u = fmaf(Y13_a, G108_0, u); gy13 = fmaf(q, G108_0, gy13);
        u = fmaf(Y14_a, G109_0, u); gy14 = fmaf(q, G109_0, gy14);
        u = fmaf(Y15_a, G110_0, u); gy15 = fmaf(q, G110_0, gy15);
        gw0 = fmaf(X8_0_a, u, gw0); gx8_0 = fmaf(W20_0_a, u, gx8_0);
      }
      if (gwp) gwp[2560] = gw0;
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
      atomicAdd(gxp + 512, gx4_0);
      atomicAdd(gxp + 640, gx5_0);
      atomicAdd(gxp + 768, gx6_0);
      atomicAdd(gxp + 896, gx7_0);
      atomicAdd(gxp + 1024, gx8_0);
    }
  }
  }
  else if (pg == 2) {
  const float* __restrict__ gp = gO + (size_t)i * g_stride + c;
  const float g3_0 = gp[384];
  const float g19_0 = gp[2432];
  const float g20_0 = gp[2560];
  const float g21_0 = gp[2688];
  const float g47_0 = gp[6016];
  const float g48_0 = gp[6144];
  const float g49_0 = gp[6272];
  const float g50_0 = gp[6400];
  const float g51_0 = gp[6528];
  const float g52_0 = gp[6656];
  const float g53_0 = gp[6784];
  const float g54_0 = gp[6912];
  const float g55_0 = gp[7040];
  const float g56_0 = gp[7168];
  const float g85_0 = gp[10880];
  const float g86_0 = gp[11008];
  const float g87_0 = gp[11136];
  const float g88_0 = gp[11264];
  const float g89_0 = gp[11392];
  const float g90_0 = gp[11520];
  const float g91_0 = gp[11648];
  const float g92_0 = gp[11776];
  const float g93_0 = gp[11904];
  const float g94_0 = gp[12032];
  const float g95_0 = gp[12160];
  const float g96_0 = gp[12288];
  const float g97_0 = gp[12416];
  const float g98_0 = gp[12544];
  const float G0_0 = 0.3779644730092272f * g3_0;
  const float G1_0 = 0.3779644730092272f * g3_0;
  const float G2_0 = 0.3779644730092272f * g3_0;
  const float G3_0 = 0.3779644730092273f * g3_0;
  const float G4_0 = 0.3779644730092272f * g3_0;
  const float G5_0 = 0.3779644730092272f * g3_0;
  const float G6_0 = 0.3779644730092272f * g3_0;
  const float G7_0 = 0.4629100498862757f * g21_0;
  const float G8_0 = 0.4629100498862757f * g19_0;
  const float G9_0 = 0.3779644730092272f * g20_0;
  const float G10_0 = 0.3779644730092272f * g21_0;
  const float G11_0 = 0.3779644730092272f * g19_0;
  const float G12_0 = -0.11952286093343936f * g21_0;
  const float G13_0 = 0.47809144373375745f * g20_0;
  const float G14_0 = 0.41403933560541256f * g19_0;
  const float G15_0 = 0.11952286093343936f * g19_0;
  const float G16_0 = -0.29277002188456f * g19_0;
  const float G17_0 = 0.5070925528371102f * g20_0;
  const float G18_0 = -0.29277002188456f * g21_0;
  const float G19_0 = -0.11952286093343936f * g19_0;
  const float G20_0 = 0.41403933560541256f * g21_0;
  const float G21_0 = 0.47809144373375745f * g20_0;
  const float G22_0 = -0.11952286093343936f * g21_0;
  const float G23_0 = -0.3779644730092272f * g19_0;
  const float G24_0 = 0.3779644730092272f * g21_0;
  const float G25_0 = 0.3779644730092272f * g20_0;
  const float G26_0 = -0.4629100498862757f * g19_0;
  const float G27_0 = 0.4629100498862757f * g21_0;
  const float G28_0 = 0.5976143046671968f * g51_0;
  const float G29_0 = 0.5976143046671968f * g47_0;
  const float G30_0 = 0.4879500364742667f * g50_0;
  const float G31_0 = 0.4879500364742667f * g47_0;
  const float G32_0 = 0.4879500364742667f * g48_0;
  const float G33_0 = fmaf(0.1543033499620919f, g51_0, 0.5345224838248489f * g49_0);
  const float G34_0 = 0.6172133998483678f * g48_0;
  const float G35_0 = -0.1543033499620919f * g47_0;
  const float G36_0 = -0.3779644730092273f * g48_0;
  const float G37_0 = 0.6546536707079773f * g49_0;
  const float G38_0 = -0.3779644730092273f * g50_0;
  const float G39_0 = -0.1543033499620919f * g47_0;
  const float G40_0 = 0.6172133998483678f * g50_0;
  const float G41_0 = fmaf(-0.1543033499620919f, g51_0, 0.5345224838248489f * g49_0);
  const float G42_0 = -0.4879500364742667f * g48_0;
  const float G43_0 = 0.4879500364742667f * g51_0;
  const float G44_0 = 0.4879500364742667f * g50_0;
  const float G45_0 = -0.5976143046671968f * g47_0;
  const float G46_0 = 0.5976143046671968f * g51_0;
  const float G47_0 = 0.545544725589981f * g54_0;
  const float G48_0 = -0.38575837490522974f * g55_0;
  const float G49_0 = 0.24397501823713336f * g56_0;
  const float G50_0 = 0.24397501823713336f * g52_0;
  const float G51_0 = -0.38575837490522974f * g53_0;
  const float G52_0 = -0.38575837490522974f * g55_0;
  const float G53_0 = -0.2988071523335984f * g55_0;
  const float G54_0 = 0.4879500364742667f * g52_0;
  const float G55_0 = -0.2988071523335984f * g53_0;
  const float G56_0 = 0.38575837490522974f * g53_0;
  const float G57_0 = 0.24397501823713336f * g56_0;
  const float G58_0 = -0.2988071523335984f * g55_0;
  const float G59_0 = fmaf(0.3779644730092273f, g56_0, -0.3273268353539886f * g54_0);
  const float G60_0 = -0.15430334996209194f * g53_0;
  const float G61_0 = -0.3779644730092273f * g52_0;
  const float G62_0 = 0.2988071523335984f * g53_0;
  const float G63_0 = -0.24397501823713336f * g52_0;
  const float G64_0 = 0.4879500364742667f * g52_0;
  const float G65_0 = -0.15430334996209194f * g53_0;
  const float G66_0 = -0.4364357804719849f * g54_0;
  const float G67_0 = -0.15430334996209194f * g55_0;
  const float G68_0 = 0.4879500364742667f * g56_0;
  const float G69_0 = 0.24397501823713336f * g52_0;
  const float G70_0 = -0.2988071523335984f * g53_0;
  const float G71_0 = -0.3779644730092273f * g52_0;
  const float G72_0 = -0.15430334996209194f * g55_0;
  const float G73_0 = fmaf(-0.3779644730092273f, g56_0, -0.3273268353539886f * g54_0);
  const float G74_0 = -0.2988071523335984f * g55_0;
  const float G75_0 = 0.24397501823713336f * g56_0;
  const float G76_0 = -0.38575837490522974f * g53_0;
  const float G77_0 = 0.2988071523335984f * g53_0;
  const float G78_0 = 0.4879500364742667f * g56_0;
  const float G79_0 = -0.2988071523335984f * g55_0;
  const float G80_0 = -0.38575837490522974f * g55_0;
  const float G81_0 = 0.38575837490522974f * g53_0;
  const float G82_0 = -0.24397501823713336f * g52_0;
  const float G83_0 = 0.24397501823713336f * g56_0;
  const float G84_0 = -0.38575837490522974f * g55_0;
  const float G85_0 = 0.545544725589981f * g54_0;
  const float G86_0 = g85_0;
  const float G87_0 = g86_0;
  const float G88_0 = g87_0;
  const float G89_0 = g88_0;
  const float G90_0 = g89_0;
  const float G91_0 = g90_0;
  const float G92_0 = g91_0;
  const float G93_0 = 0.2886751345948128f * g96_0;
  const float G94_0 = -0.45643546458763845f * g97_0;
  const float G95_0 = 0.6454972243679029f * g92_0;
  const float G96_0 = -0.45643546458763845f * g93_0;
  const float G97_0 = 0.2886751345948128f * g94_0;
  const float G98_0 = 0.5773502691896258f * g95_0;
  const float G99_0 = fmaf(0.45643546458763845f, g98_0, -0.3535533905932738f * g96_0);
  const float G100_0 = fmaf(-0.3535533905932738f, g94_0, -0.45643546458763845f * g92_0);
  const float G101_0 = fmaf(-0.2886751345948128f, g98_0, -0.447213595499958f * g96_0);
  const float G102_0 = fmaf(0.3535533905932738f, g97_0, -0.18257418583505539f * g95_0);
  const float G103_0 = -0.3872983346207418f * g94_0;
  const float G104_0 = -0.3535533905932738f * g93_0;
  const float G105_0 = fmaf(0.447213595499958f, g94_0, 0.2886751345948128f * g92_0);
  const float G106_0 = 0.5773502691896258f * g93_0;
  const float G107_0 = -0.18257418583505539f * g94_0;
  const float G108_0 = -0.5163977794943223f * g95_0;
  const float G109_0 = -0.18257418583505539f * g96_0;
  const float G110_0 = 0.5773502691896258f * g97_0;
  const float G111_0 = fmaf(-0.447213595499958f, g94_0, 0.2886751345948128f * g92_0);
  const float G112_0 = -0.3535533905932738f * g93_0;
  const float G113_0 = -0.3872983346207418f * g96_0;
  const float G114_0 = fmaf(-0.3535533905932738f, g97_0, -0.18257418583505539f * g95_0);
  const float G115_0 = fmaf(0.2886751345948128f, g98_0, -0.447213595499958f * g96_0);
  const float G116_0 = fmaf(0.3535533905932738f, g94_0, -0.45643546458763845f * g92_0);
  const float G117_0 = fmaf(-0.45643546458763845f, g98_0, -0.3535533905932738f * g96_0);
  const float G118_0 = 0.5773502691896258f * g95_0;
  const float G119_0 = -0.2886751345948128f * g94_0;
  const float G120_0 = 0.45643546458763845f * g93_0;
  const float G121_0 = 0.6454972243679029f * g98_0;
  const float G122_0 = -0.45643546458763845f * g97_0;
  const float G123_0 = 0.2886751345948128f * g96_0;
  for (int p = p0; p < p1; ++p) {
    const int ea = __builtin_amdgcn_readfirstlane(eid ? eid[p] : p);
    const int sa = __builtin_amdgcn_readfirstlane(send[ea]);
    const float* __restrict__ wpa = W + (size_t)ea * w_stride + c;
    const float W3_0_a = wpa[384];
    const float W9_0_a = wpa[1152];
    const float W15_0_a = wpa[1920];
    const float W16_0_a = wpa[2048];
    const float W21_0_a = wpa[2688];
    const float W22_0_a = wpa[2816];
    const float* __restrict__ xpa = X + (size_t)sa * x_stride + c;
    const float X9_0_a = xpa[1152];
    const float X10_0_a = xpa[1280];
    const float X11_0_a = xpa[1408];
    const float X12_0_a = xpa[1536];
    const float X13_0_a = xpa[1664];
    const float X14_0_a = xpa[1792];
    const float X15_0_a = xpa[1920];
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
    float gx9_0 = 0.f;
    float gx10_0 = 0.f;
    float gx11_0 = 0.f;
    float gx12_0 = 0.f;
    float gx13_0 = 0.f;
    float gx14_0 = 0.f;
    float gx15_0 = 0.f;
    float* __restrict__ gwp = gW ? gW + (size_t)ea * gw_stride + c : nullptr;
    {
      float gw0 = 0.f;
      { const float q = W3_0_a * X9_0_a; float u = 0.f;
        u = fmaf(Y9_a, G0_0, u); gy9 = fmaf(q, G0_0, gy9);
        gw0 = fmaf(X9_0_a, u, gw0); gx9_0 = fmaf(W3_0_a, u, gx9_0);
      }
      { const float q = W3_0_a * X10_0_a; float u = 0.f;
        u = fmaf(Y10_a, G1_0, u); gy10 = fmaf(q, G1_0, gy10);
        gw0 = fmaf(X10_0_a, u, gw0); gx10_0 = fmaf(W3_0_a, u, gx10_0);
      }
      { const float q = W3_0_a * X11_0_a; float u = 0.f;
        u = fmaf(Y11_a, G2_0, u); gy11 = fmaf(q, G2_0, gy11);
        gw0 = fmaf(X11_0_a, u, gw0); gx11_0 = fmaf(W3_0_a, u, gx11_0);
      }
      { const float q = W3_0_a * X12_0_a; float u = 0.f;
        u = fmaf(Y12_a, G3_0, u); gy12 = fmaf(q, G3_0, gy12);
        gw0 = fmaf(X12_0_a, u, gw0); gx12_0 = fmaf(W3_0_a, u, gx12_0);
      }
      { const float q = W3_0_a * X13_0_a; float u = 0.f;
        u = fmaf(Y13_a, G4_0, u); gy13 = fmaf(q, G4_0, gy13);
        gw0 = fmaf(X13_0_a, u, gw0); gx13_0 = fmaf(W3_0_a, u, gx13_0);
      }
      { const float q = W3_0_a * X14_0_a; float u = 0.f;
        u = fmaf(Y14_a, G5_0, u); gy14 = fmaf(q, G5_0, gy14);
        gw0 = fmaf(X14_0_a, u, gw0); gx14_0 = fmaf(W3_0_a, u, gx14_0);
      }
      { const float q = W3_0_a * X15_0_a; float u = 0.f;
        u = fmaf(Y15_a, G6_0, u); gy15 = fmaf(q, G6_0, gy15);
        gw0 = fmaf(X15_0_a, u, gw0); gx15_0 = fmaf(W3_0_a, u, gx15_0);
      }
      if (gwp) gwp[384] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W9_0_a * X9_0_a; float u = 0.f;
        u = fmaf(Y4_a, G7_0, u); gy4 = fmaf(q, G7_0, gy4);
        u = fmaf(Y8_a, G8_0, u); gy8 = fmaf(q, G8_0, gy8);
        gw0 = fmaf(X9_0_a, u, gw0); gx9_0 = fmaf(W9_0_a, u, gx9_0);
      }
      { const float q = W9_0_a * X10_0_a; float u = 0.f;
        u = fmaf(Y4_a, G9_0, u); gy4 = fmaf(q, G9_0, gy4);
        u = fmaf(Y5_a, G10_0, u); gy5 = fmaf(q, G10_0, gy5);
        u = fmaf(Y7_a, G11_0, u); gy7 = fmaf(q, G11_0, gy7);
        gw0 = fmaf(X10_0_a, u, gw0); gx10_0 = fmaf(W9_0_a, u, gx10_0);
      }
      { const float q = W9_0_a * X11_0_a; float u = 0.f;
        u = fmaf(Y4_a, G12_0, u); gy4 = fmaf(q, G12_0, gy4);
        u = fmaf(Y5_a, G13_0, u); gy5 = fmaf(q, G13_0, gy5);
        u = fmaf(Y6_a, G14_0, u); gy6 = fmaf(q, G14_0, gy6);
        u = fmaf(Y8_a, G15_0, u); gy8 = fmaf(q, G15_0, gy8);
        gw0 = fmaf(X11_0_a, u, gw0); gx11_0 = fmaf(W9_0_a, u, gx11_0);
      }
      { const float q = W9_0_a * X12_0_a; float u = 0.f;
        u = fmaf(Y5_a, G16_0, u); gy5 = fmaf(q, G16_0, gy5);
        u = fmaf(Y6_a, G17_0, u); gy6 = fmaf(q, G17_0, gy6);
        u = fmaf(Y7_a, G18_0, u); gy7 = fmaf(q, G18_0, gy7);
        gw0 = fmaf(X12_0_a, u, gw0); gx12_0 = fmaf(W9_0_a, u, gx12_0);
      }
      { const float q = W9_0_a * X13_0_a; float u = 0.f;
        u = fmaf(Y4_a, G19_0, u); gy4 = fmaf(q, G19_0, gy4);
        u = fmaf(Y6_a, G20_0, u); gy6 = fmaf(q, G20_0, gy6);
        u = fmaf(Y7_a, G21_0, u); gy7 = fmaf(q, G21_0, gy7);
        u = fmaf(Y8_a, G22_0, u); gy8 = fmaf(q, G22_0, gy8);
        gw0 = fmaf(X13_0_a, u, gw0); gx13_0 = fmaf(W9_0_a, u, gx13_0);
      }
      { const float q = W9_0_a * X14_0_a; float u = 0.f;
        u = fmaf(Y5_a, G23_0, u); gy5 = fmaf(q, G23_0, gy5);
        u = fmaf(Y7_a, G24_0, u); gy7 = fmaf(q, G24_0, gy7);
        u = fmaf(Y8_a, G25_0, u); gy8 = fmaf(q, G25_0, gy8);
        gw0 = fmaf(X14_0_a, u, gw0); gx14_0 = fmaf(W9_0_a, u, gx14_0);
      }
      { const float q = W9_0_a * X15_0_a; float u = 0.f;
        u = fmaf(Y4_a, G26_0, u); gy4 = fmaf(q, G26_0, gy4);
        u = fmaf(Y8_a, G27_0, u); gy8 = fmaf(q, G27_0, gy8);
        gw0 = fmaf(X15_0_a, u, gw0); gx15_0 = fmaf(W9_0_a, u, gx15_0);
      }
      if (gwp) gwp[1152] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W15_0_a * X9_0_a; float u = 0.f;
        u = fmaf(Y1_a, G28_0, u); gy1 = fmaf(q, G28_0, gy1);
        u = fmaf(Y3_a, G29_0, u); gy3 = fmaf(q, G29_0, gy3);
        gw0 = fmaf(X9_0_a, u, gw0); gx9_0 = fmaf(W15_0_a, u, gx9_0);
      }
      { const float q = W15_0_a * X10_0_a; float u = 0.f;
        u = fmaf(Y1_a, G30_0, u); gy1 = fmaf(q, G30_0, gy1);
        u = fmaf(Y2_a, G31_0, u); gy2 = fmaf(q, G31_0, gy2);
        u = fmaf(Y3_a, G32_0, u); gy3 = fmaf(q, G32_0, gy3);
        gw0 = fmaf(X10_0_a, u, gw0); gx10_0 = fmaf(W15_0_a, u, gx10_0);
      }
      { const float q = W15_0_a * X11_0_a; float u = 0.f;
        u = fmaf(Y1_a, G33_0, u); gy1 = fmaf(q, G33_0, gy1);
        u = fmaf(Y2_a, G34_0, u); gy2 = fmaf(q, G34_0, gy2);
        u = fmaf(Y3_a, G35_0, u); gy3 = fmaf(q, G35_0, gy3);
        gw0 = fmaf(X11_0_a, u, gw0); gx11_0 = fmaf(W15_0_a, u, gx11_0);
      }
      { const float q = W15_0_a * X12_0_a; float u = 0.f;
        u = fmaf(Y1_a, G36_0, u); gy1 = fmaf(q, G36_0, gy1);
        u = fmaf(Y2_a, G37_0, u); gy2 = fmaf(q, G37_0, gy2);
        u = fmaf(Y3_a, G38_0, u); gy3 = fmaf(q, G38_0, gy3);
        gw0 = fmaf(X12_0_a, u, gw0); gx12_0 = fmaf(W15_0_a, u, gx12_0);
      }
      { const float q = W15_0_a * X13_0_a; float u = 0.f;
        u = fmaf(Y1_a, G39_0, u); gy1 = fmaf(q, G39_0, gy1);
        u = fmaf(Y2_a, G40_0, u); gy2 = fmaf(q, G40_0, gy2);
        u = fmaf(Y3_a, G41_0, u); gy3 = fmaf(q, G41_0, gy3);
        gw0 = fmaf(X13_0_a, u, gw0); gx13_0 = fmaf(W15_0_a, u, gx13_0);
      }
      { const float q = W15_0_a * X14_0_a; float u = 0.f;
        u = fmaf(Y1_a, G42_0, u); gy1 = fmaf(q, G42_0, gy1);
        u = fmaf(Y2_a, G43_0, u); gy2 = fmaf(q, G43_0, gy2);
        u = fmaf(Y3_a, G44_0, u); gy3 = fmaf(q, G44_0, gy3);
        gw0 = fmaf(X14_0_a, u, gw0); gx14_0 = fmaf(W15_0_a, u, gx14_0);
      }
      { const float q = W15_0_a * X15_0_a; float u = 0.f;
        u = fmaf(Y1_a, G45_0, u); gy1 = fmaf(q, G45_0, gy1);
        u = fmaf(Y3_a, G46_0, u); gy3 = fmaf(q, G46_0, gy3);
        gw0 = fmaf(X15_0_a, u, gw0); gx15_0 = fmaf(W15_0_a, u, gx15_0);
      }
      if (gwp) gwp[1920] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W16_0_a * X9_0_a; float u = 0.f;
        u = fmaf(Y9_a, G47_0, u); gy9 = fmaf(q, G47_0, gy9);
        u = fmaf(Y10_a, G48_0, u); gy10 = fmaf(q, G48_0, gy10);
        u = fmaf(Y11_a, G49_0, u); gy11 = fmaf(q, G49_0, gy11);
        u = fmaf(Y13_a, G50_0, u); gy13 = fmaf(q, G50_0, gy13);
        u = fmaf(Y14_a, G51_0, u); gy14 = fmaf(q, G51_0, gy14);
        gw0 = fmaf(X9_0_a, u, gw0); gx9_0 = fmaf(W16_0_a, u, gx9_0);
      }
      { const float q = W16_0_a * X10_0_a; float u = 0.f;
        u = fmaf(Y9_a, G52_0, u); gy9 = fmaf(q, G52_0, gy9);
        u = fmaf(Y11_a, G53_0, u); gy11 = fmaf(q, G53_0, gy11);
        u = fmaf(Y12_a, G54_0, u); gy12 = fmaf(q, G54_0, gy12);
        u = fmaf(Y13_a, G55_0, u); gy13 = fmaf(q, G55_0, gy13);
        u = fmaf(Y15_a, G56_0, u); gy15 = fmaf(q, G56_0, gy15);
        gw0 = fmaf(X10_0_a, u, gw0); gx10_0 = fmaf(W16_0_a, u, gx10_0);
      }
      { const float q = W16_0_a * X11_0_a; float u = 0.f;
        u = fmaf(Y9_a, G57_0, u); gy9 = fmaf(q, G57_0, gy9);
        u = fmaf(Y10_a, G58_0, u); gy10 = fmaf(q, G58_0, gy10);
        u = fmaf(Y11_a, G59_0, u); gy11 = fmaf(q, G59_0, gy11);
        u = fmaf(Y12_a, G60_0, u); gy12 = fmaf(q, G60_0, gy12);
        u = fmaf(Y13_a, G61_0, u); gy13 = fmaf(q, G61_0, gy13);
        u = fmaf(Y14_a, G62_0, u); gy14 = fmaf(q, G62_0, gy14);
        u = fmaf(Y15_a, G63_0, u); gy15 = fmaf(q, G63_0, gy15);
        gw0 = fmaf(X11_0_a, u, gw0); gx11_0 = fmaf(W16_0_a, u, gx11_0);
      }
      { const float q = W16_0_a * X12_0_a; float u = 0.f;
        u = fmaf(Y10_a, G64_0, u); gy10 = fmaf(q, G64_0, gy10);
        u = fmaf(Y11_a, G65_0, u); gy11 = fmaf(q, G65_0, gy11);
        u = fmaf(Y12_a, G66_0, u); gy12 = fmaf(q, G66_0, gy12);
        u = fmaf(Y13_a, G67_0, u); gy13 = fmaf(q, G67_0, gy13);
        u = fmaf(Y14_a, G68_0, u); gy14 = fmaf(q, G68_0, gy14);
        gw0 = fmaf(X12_0_a, u, gw0); gx12_0 = fmaf(W16_0_a, u, gx12_0);
      }
      { const float q = W16_0_a * X13_0_a; float u = 0.f;
        u = fmaf(Y9_a, G69_0, u); gy9 = fmaf(q, G69_0, gy9);
        u = fmaf(Y10_a, G70_0, u); gy10 = fmaf(q, G70_0, gy10);
        u = fmaf(Y11_a, G71_0, u); gy11 = fmaf(q, G71_0, gy11);
        u = fmaf(Y12_a, G72_0, u); gy12 = fmaf(q, G72_0, gy12);
        u = fmaf(Y13_a, G73_0, u); gy13 = fmaf(q, G73_0, gy13);
        u = fmaf(Y14_a, G74_0, u); gy14 = fmaf(q, G74_0, gy14);
        u = fmaf(Y15_a, G75_0, u); gy15 = fmaf(q, G75_0, gy15);
        gw0 = fmaf(X13_0_a, u, gw0); gx13_0 = fmaf(W16_0_a, u, gx13_0);
      }
      { const float q = W16_0_a * X14_0_a; float u = 0.f;
        u = fmaf(Y9_a, G76_0, u); gy9 = fmaf(q, G76_0, gy9);
        u = fmaf(Y11_a, G77_0, u); gy11 = fmaf(q, G77_0, gy11);
        u = fmaf(Y12_a, G78_0, u); gy12 = fmaf(q, G78_0, gy12);
        u = fmaf(Y13_a, G79_0, u); gy13 = fmaf(q, G79_0, gy13);
        u = fmaf(Y15_a, G80_0, u); gy15 = fmaf(q, G80_0, gy15);
        gw0 = fmaf(X14_0_a, u, gw0); gx14_0 = fmaf(W16_0_a, u, gx14_0);
      }
      { const float q = W16_0_a * X15_0_a; float u = 0.f;
        u = fmaf(Y10_a, G81_0, u); gy10 = fmaf(q, G81_0, gy10);
        u = fmaf(Y11_a, G82_0, u); gy11 = fmaf(q, G82_0, gy11);
        u = fmaf(Y13_a, G83_0, u); gy13 = fmaf(q, G83_0, gy13);
        u = fmaf(Y14_a, G84_0, u); gy14 = fmaf(q, G84_0, gy14);
        u = fmaf(Y15_a, G85_0, u); gy15 = fmaf(q, G85_0, gy15);
        gw0 = fmaf(X15_0_a, u, gw0); gx15_0 = fmaf(W16_0_a, u, gx15_0);
      }
      if (gwp) gwp[2048] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W21_0_a * X9_0_a; float u = 0.f;
        u = fmaf(Y0_a, G86_0, u); gy0 = fmaf(q, G86_0, gy0);
        gw0 = fmaf(X9_0_a, u, gw0); gx9_0 = fmaf(W21_0_a, u, gx9_0);
      }
      { const float q = W21_0_a * X10_0_a; float u = 0.f;
        u = fmaf(Y0_a, G87_0, u); gy0 = fmaf(q, G87_0, gy0);
        gw0 = fmaf(X10_0_a, u, gw0); gx10_0 = fmaf(W21_0_a, u, gx10_0);
      }
      { const float q = W21_0_a * X11_0_a; float u = 0.f;
        u = fmaf(Y0_a, G88_0, u); gy0 = fmaf(q, G88_0, gy0);
        gw0 = fmaf(X11_0_a, u, gw0); gx11_0 = fmaf(W21_0_a, u, gx11_0);
      }
      { const float q = W21_0_a * X12_0_a; float u = 0.f;
        u = fmaf(Y0_a, G89_0, u); gy0 = fmaf(q, G89_0, gy0);
        gw0 = fmaf(X12_0_a, u, gw0); gx12_0 = fmaf(W21_0_a, u, gx12_0);
      }
      { const float q = W21_0_a * X13_0_a; float u = 0.f;
        u = fmaf(Y0_a, G90_0, u); gy0 = fmaf(q, G90_0, gy0);
        gw0 = fmaf(X13_0_a, u, gw0); gx13_0 = fmaf(W21_0_a, u, gx13_0);
      }
      { const float q = W21_0_a * X14_0_a; float u = 0.f;
        u = fmaf(Y0_a, G91_0, u); gy0 = fmaf(q, G91_0, gy0);
        gw0 = fmaf(X14_0_a, u, gw0); gx14_0 = fmaf(W21_0_a, u, gx14_0);
      }
      { const float q = W21_0_a * X15_0_a; float u = 0.f;
        u = fmaf(Y0_a, G92_0, u); gy0 = fmaf(q, G92_0, gy0);
        gw0 = fmaf(X15_0_a, u, gw0); gx15_0 = fmaf(W21_0_a, u, gx15_0);
      }
      if (gwp) gwp[2688] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W22_0_a * X9_0_a; float u = 0.f;
        u = fmaf(Y4_a, G93_0, u); gy4 = fmaf(q, G93_0, gy4);
        u = fmaf(Y5_a, G94_0, u); gy5 = fmaf(q, G94_0, gy5);
        u = fmaf(Y6_a, G95_0, u); gy6 = fmaf(q, G95_0, gy6);
        u = fmaf(Y7_a, G96_0, u); gy7 = fmaf(q, G96_0, gy7);
        u = fmaf(Y8_a, G97_0, u); gy8 = fmaf(q, G97_0, gy8);
        gw0 = fmaf(X9_0_a, u, gw0); gx9_0 = fmaf(W22_0_a, u, gx9_0);
      }
      { const float q = W22_0_a * X10_0_a; float u = 0.f;
        u = fmaf(Y4_a, G98_0, u); gy4 = fmaf(q, G98_0, gy4);
        u = fmaf(Y5_a, G99_0, u); gy5 = fmaf(q, G99_0, gy5);
        u = fmaf(Y7_a, G100_0, u); gy7 = fmaf(q, G100_0, gy7);
        gw0 = fmaf(X10_0_a, u, gw0); gx10_0 = fmaf(W22_0_a, u, gx10_0);
      }
      { const float q = W22_0_a * X11_0_a; float u = 0.f;
        u = fmaf(Y4_a, G101_0, u); gy4 = fmaf(q, G101_0, gy4);
        u = fmaf(Y5_a, G102_0, u); gy5 = fmaf(q, G102_0, gy5);
        u = fmaf(Y6_a, G103_0, u); gy6 = fmaf(q, G103_0, gy6);
        u = fmaf(Y7_a, G104_0, u); gy7 = fmaf(q, G104_0, gy7);
        u = fmaf(Y8_a, G105_0, u); gy8 = fmaf(q, G105_0, gy8);
        gw0 = fmaf(X11_0_a, u, gw0); gx11_0 = fmaf(W22_0_a, u, gx11_0);
      }
      { const float q = W22_0_a * X12_0_a; float u = 0.f;
        u = fmaf(Y4_a, G106_0, u); gy4 = fmaf(q, G106_0, gy4);
        u = fmaf(Y5_a, G107_0, u); gy5 = fmaf(q, G107_0, gy5);
        u = fmaf(Y6_a, G108_0, u); gy6 = fmaf(q, G108_0, gy6);
        u = fmaf(Y7_a, G109_0, u); gy7 = fmaf(q, G109_0, gy7);
        u = fmaf(Y8_a, G110_0, u); gy8 = fmaf(q, G110_0, gy8);
        gw0 = fmaf(X12_0_a, u, gw0); gx12_0 = fmaf(W22_0_a, u, gx12_0);
      }
      { const float q = W22_0_a * X13_0_a; float u = 0.f;
        u = fmaf(Y4_a, G111_0, u); gy4 = fmaf(q, G111_0, gy4);
        u = fmaf(Y5_a, G112_0, u); gy5 = fmaf(q, G112_0, gy5);
        u = fmaf(Y6_a, G113_0, u); gy6 = fmaf(q, G113_0, gy6);
        u = fmaf(Y7_a, G114_0, u); gy7 = fmaf(q, G114_0, gy7);
        u = fmaf(Y8_a, G115_0, u); gy8 = fmaf(q, G115_0, gy8);
        gw0 = fmaf(X13_0_a, u, gw0); gx13_0 = fmaf(W22_0_a, u, gx13_0);
      }
      { const float q = W22_0_a * X14_0_a; float u = 0.f;
        u = fmaf(Y5_a, G116_0, u); gy5 = fmaf(q, G116_0, gy5);
        u = fmaf(Y7_a, G117_0, u); gy7 = fmaf(q, G117_0, gy7);
        u = fmaf(Y8_a, G118_0, u); gy8 = fmaf(q, G118_0, gy8);
        gw0 = fmaf(X14_0_a, u, gw0); gx14_0 = fmaf(W22_0_a, u, gx14_0);
      }
      { const float q = W22_0_a * X15_0_a; float u = 0.f;
        u = fmaf(Y4_a, G119_0, u); gy4 = fmaf(q, G119_0, gy4);
        u = fmaf(Y5_a, G120_0, u); gy5 = fmaf(q, G120_0, gy5);
        u = fmaf(Y6_a, G121_0, u); gy6 = fmaf(q, G121_0, gy6);
        u = fmaf(Y7_a, G122_0, u); gy7 = fmaf(q, G122_0, gy7);
        u = fmaf(Y8_a, G123_0, u); gy8 = fmaf(q, G123_0, gy8);
        gw0 = fmaf(X15_0_a, u, gw0); gx15_0 = fmaf(W22_0_a, u, gx15_0);
      }
      if (gwp) gwp[2816] = gw0;
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
      atomicAdd(gxp + 1152, gx9_0);
      atomicAdd(gxp + 1280, gx10_0);
      atomicAdd(gxp + 1408, gx11_0);
      atomicAdd(gxp + 1536, gx12_0);
      atomicAdd(gxp + 1664, gx13_0);
      atomicAdd(gxp + 1792, gx14_0);
      atomicAdd(gxp + 1920, gx15_0);
    }
  }
  }
}

// Backward from gO = dL/dout: gW[e, w, c] (written), gYp[part][e][m] = partial sums of dL/dY[e, m] over
// the channels and paths of one wave (6 partial(s): channel half h x path group g, part
// h * 3 + g; summed by the caller), gX[send, k, c] (atomic adds).  Null outputs are skipped.
// Path groups (one wave each): [[0, 1, 4, 5, 6, 10, 11, 12, 17, 18], [2, 7, 8, 13, 14, 19, 20], [3, 9, 15, 16, 21, 22]].
extern "C" __global__ void __launch_bounds__(256)
mm_tpw_l0123_bwd_shared_kernel(const int* __restrict__ rowptr, int nR, const int* __restrict__ eid,
    const int* __restrict__ send, const float* __restrict__ Y, long y_stride, const float* __restrict__ W,
    long w_stride, const float* __restrict__ X, long x_stride, const float* __restrict__ gO, long g_stride,
    float* __restrict__ gW, long gw_stride, float* __restrict__ gYp, long gy_cb_stride,
    float* __restrict__ gX, long gx_stride) {
  const int wave = threadIdx.x >> 6;
  const int gw = blockIdx.x;   // receiver i, sub-wave h
  const int i = gw / 6, h = gw % 6;
  if (i >= nR) return;
  const int lane = threadIdx.x & 63;
  const int c = (h / 3) * 64 + lane;
  const int r0 = rowptr[i], nr = rowptr[i + 1] - r0;
  const int p0 = r0 + (int)((long)nr * wave / 4), p1 = r0 + (int)((long)nr * (wave + 1) / 4);
  const int pg = h % 3;   // path group; channel half h / 3
  const int part = h;
  const int cl = lane & 15;
  const bool b3 = cl & 8, b2 = cl & 4, b1 = cl & 2, b0 = cl & 1;
  if (pg == 0) {
  const float* __restrict__ gp = gO + (size_t)i * g_stride + c;
  const float g0_0 = gp[0];
  const float g1_0 = gp[128];
  const float g4_0 = gp[512];
  const float g5_0 = gp[640];
  const float g6_0 = gp[768];
  const float g7_0 = gp[896];
  const float g8_0 = gp[1024];
  const float g9_0 = gp[1152];
  const float g10_0 = gp[1280];
  const float g11_0 = gp[1408];
  const float g12_0 = gp[1536];
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
  const float g57_0 = gp[7296];
  const float g58_0 = gp[7424];
  const float g59_0 = gp[7552];
  const float g60_0 = gp[7680];
  const float g61_0 = gp[7808];
  const float g62_0 = gp[7936];
  const float g63_0 = gp[8064];
  const float g64_0 = gp[8192];
  const float g65_0 = gp[8320];
  const float g66_0 = gp[8448];
  const float g67_0 = gp[8576];
  const float g68_0 = gp[8704];
  const float g69_0 = gp[8832];
  const float g70_0 = gp[8960];
  const float G0_0 = g0_0;
  const float G1_0 = 0.5773502691896257f * g1_0;
  const float G2_0 = 0.5773502691896258f * g1_0;
  const float G3_0 = 0.5773502691896257f * g1_0;
  const float G4_0 = g4_0;
  const float G5_0 = g5_0;
  const float G6_0 = g6_0;
  const float G7_0 = g7_0;
  const float G8_0 = g8_0;
  const float G9_0 = g9_0;
  const float G10_0 = 0.547722557505166f * g12_0;
  const float G11_0 = 0.547722557505166f * g11_0;
  const float G12_0 = -0.31622776601683794f * g10_0;
  const float G13_0 = -0.547722557505166f * g10_0;
  const float G14_0 = 0.547722557505166f * g10_0;
  const float G15_0 = 0.632455532033676f * g11_0;
  const float G16_0 = 0.547722557505166f * g12_0;
  const float G17_0 = 0.547722557505166f * g10_0;
  const float G18_0 = -0.31622776601683794f * g12_0;
  const float G19_0 = 0.547722557505166f * g11_0;
  const float G20_0 = 0.547722557505166f * g12_0;
  const float G21_0 = g22_0;
  const float G22_0 = g23_0;
  const float G23_0 = g24_0;
  const float G24_0 = g25_0;
  const float G25_0 = g26_0;
  const float G26_0 = fmaf(0.7071067811865475f, g31_0, 0.408248290463863f * g29_0);
  const float G27_0 = -0.7071067811865476f * g28_0;
  const float G28_0 = -0.7071067811865475f * g27_0;
  const float G29_0 = -0.7071067811865476f * g28_0;
  const float G30_0 = -0.8164965809277261f * g29_0;
  const float G31_0 = -0.7071067811865476f * g30_0;
  const float G32_0 = -0.7071067811865475f * g27_0;
  const float G33_0 = -0.7071067811865476f * g30_0;
  const float G34_0 = fmaf(-0.7071067811865475f, g31_0, 0.408248290463863f * g29_0);
  const float G35_0 = 0.5976143046671967f * g36_0;
  const float G36_0 = 0.48795003647426655f * g35_0;
  const float G37_0 = fmaf(0.15430334996209188f, g36_0, 0.5345224838248488f * g34_0);
  const float G38_0 = -0.3779644730092272f * g33_0;
  const float G39_0 = -0.15430334996209188f * g32_0;
  const float G40_0 = -0.48795003647426655f * g33_0;
  const float G41_0 = -0.5976143046671967f * g32_0;
  const float G42_0 = 0.48795003647426655f * g32_0;
  const float G43_0 = 0.6172133998483676f * g33_0;
  const float G44_0 = 0.6546536707079772f * g34_0;
  const float G45_0 = 0.6172133998483676f * g35_0;
  const float G46_0 = 0.48795003647426655f * g36_0;
  const float G47_0 = 0.5976143046671967f * g32_0;
  const float G48_0 = 0.48795003647426655f * g33_0;
  const float G49_0 = -0.15430334996209188f * g32_0;
  const float G50_0 = -0.3779644730092272f * g35_0;
  const float G51_0 = fmaf(-0.15430334996209188f, g36_0, 0.5345224838248488f * g34_0);
  const float G52_0 = 0.48795003647426655f * g35_0;
  const float G53_0 = 0.5976143046671967f * g36_0;
  const float G54_0 = g57_0;
  const float G55_0 = g58_0;
  const float G56_0 = g59_0;
  const float G57_0 = g60_0;
  const float G58_0 = g61_0;
  const float G59_0 = g62_0;
  const float G60_0 = g63_0;
  const float G61_0 = fmaf(0.7071067811865476f, g70_0, 0.18257418583505539f * g68_0);
  const float G62_0 = fmaf(0.5773502691896256f, g69_0, 0.447213595499958f * g67_0);
  const float G63_0 = -0.632455532033676f * g66_0;
  const float G64_0 = -0.5773502691896256f * g65_0;
  const float G65_0 = fmaf(-0.18257418583505539f, g66_0, -0.7071067811865476f * g64_0);
  const float G66_0 = -0.5773502691896258f * g65_0;
  const float G67_0 = -0.7302967433402215f * g66_0;
  const float G68_0 = -0.7745966692414836f * g67_0;
  const float G69_0 = -0.7302967433402215f * g68_0;
  const float G70_0 = -0.5773502691896258f * g69_0;
  const float G71_0 = fmaf(0.18257418583505539f, g66_0, -0.7071067811865476f * g64_0);
  const float G72_0 = -0.5773502691896256f * g65_0;
  const float G73_0 = -0.632455532033676f * g68_0;
  const float G74_0 = fmaf(-0.5773502691896256f, g69_0, 0.447213595499958f * g67_0);
  const float G75_0 = fmaf(-0.7071067811865476f, g70_0, 0.18257418583505539f * g68_0);
  for (int p = p0; p < p1; ++p) {
    const int ea = __builtin_amdgcn_readfirstlane(eid ? eid[p] : p);
    const int sa = __builtin_amdgcn_readfirstlane(send[ea]);
    const float* __restrict__ wpa = W + (size_t)ea * w_stride + c;
    const float W0_0_a = wpa[0];
    const float W1_0_a = wpa[128];
    const float W4_0_a = wpa[512];
    const float W5_0_a = wpa[640];
    const float W6_0_a = wpa[768];
    const float W10_0_a = wpa[1280];
    const float W11_0_a = wpa[1408];
    const float W12_0_a = wpa[1536];
    const float W17_0_a = wpa[2176];
    const float W18_0_a = wpa[2304];
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
      { const float q = W4_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y1_a, G4_0, u); gy1 = fmaf(q, G4_0, gy1);
        u = fmaf(Y2_a, G5_0, u); gy2 = fmaf(q, G5_0, gy2);
        u = fmaf(Y3_a, G6_0, u); gy3 = fmaf(q, G6_0, gy3);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W4_0_a, u, gx0_0);
      }
      if (gwp) gwp[512] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W5_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y0_a, G7_0, u); gy0 = fmaf(q, G7_0, gy0);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W5_0_a, u, gx1_0);
      }
      { const float q = W5_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y0_a, G8_0, u); gy0 = fmaf(q, G8_0, gy0);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W5_0_a, u, gx2_0);
      }
      { const float q = W5_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y0_a, G9_0, u); gy0 = fmaf(q, G9_0, gy0);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W5_0_a, u, gx3_0);
      }
      if (gwp) gwp[640] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W6_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y4_a, G10_0, u); gy4 = fmaf(q, G10_0, gy4);
        u = fmaf(Y5_a, G11_0, u); gy5 = fmaf(q, G11_0, gy5);
        u = fmaf(Y6_a, G12_0, u); gy6 = fmaf(q, G12_0, gy6);
        u = fmaf(Y8_a, G13_0, u); gy8 = fmaf(q, G13_0, gy8);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W6_0_a, u, gx1_0);
      }
      { const float q = W6_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y5_a, G14_0, u); gy5 = fmaf(q, G14_0, gy5);
        u = fmaf(Y6_a, G15_0, u); gy6 = fmaf(q, G15_0, gy6);
        u = fmaf(Y7_a, G16_0, u); gy7 = fmaf(q, G16_0, gy7);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W6_0_a, u, gx2_0);
      }
      { const float q = W6_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y4_a, G17_0, u); gy4 = fmaf(q, G17_0, gy4);
        u = fmaf(Y6_a, G18_0, u); gy6 = fmaf(q, G18_0, gy6);
        u = fmaf(Y7_a, G19_0, u); gy7 = fmaf(q, G19_0, gy7);
        u = fmaf(Y8_a, G20_0, u); gy8 = fmaf(q, G20_0, gy8);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W6_0_a, u, gx3_0);
      }
      if (gwp) gwp[768] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W10_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y4_a, G21_0, u); gy4 = fmaf(q, G21_0, gy4);
        u = fmaf(Y5_a, G22_0, u); gy5 = fmaf(q, G22_0, gy5);
        u = fmaf(Y6_a, G23_0, u); gy6 = fmaf(q, G23_0, gy6);
        u = fmaf(Y7_a, G24_0, u); gy7 = fmaf(q, G24_0, gy7);
        u = fmaf(Y8_a, G25_0, u); gy8 = fmaf(q, G25_0, gy8);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W10_0_a, u, gx0_0);
      }
      if (gwp) gwp[1280] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W11_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y1_a, G26_0, u); gy1 = fmaf(q, G26_0, gy1);
        u = fmaf(Y2_a, G27_0, u); gy2 = fmaf(q, G27_0, gy2);
        u = fmaf(Y3_a, G28_0, u); gy3 = fmaf(q, G28_0, gy3);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W11_0_a, u, gx1_0);
      }
      { const float q = W11_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y1_a, G29_0, u); gy1 = fmaf(q, G29_0, gy1);
        u = fmaf(Y2_a, G30_0, u); gy2 = fmaf(q, G30_0, gy2);
        u = fmaf(Y3_a, G31_0, u); gy3 = fmaf(q, G31_0, gy3);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W11_0_a, u, gx2_0);
      }
      { const float q = W11_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y1_a, G32_0, u); gy1 = fmaf(q, G32_0, gy1);
        u = fmaf(Y2_a, G33_0, u); gy2 = fmaf(q, G33_0, gy2);
        u = fmaf(Y3_a, G34_0, u); gy3 = fmaf(q, G34_0, gy3);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W11_0_a, u, gx3_0);
      }
      if (gwp) gwp[1408] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W12_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y9_a, G35_0, u); gy9 = fmaf(q, G35_0, gy9);
        u = fmaf(Y10_a, G36_0, u); gy10 = fmaf(q, G36_0, gy10);
        u = fmaf(Y11_a, G37_0, u); gy11 = fmaf(q, G37_0, gy11);
        u = fmaf(Y12_a, G38_0, u); gy12 = fmaf(q, G38_0, gy12);
        u = fmaf(Y13_a, G39_0, u); gy13 = fmaf(q, G39_0, gy13);
        u = fmaf(Y14_a, G40_0, u); gy14 = fmaf(q, G40_0, gy14);
        u = fmaf(Y15_a, G41_0, u); gy15 = fmaf(q, G41_0, gy15);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W12_0_a, u, gx1_0);
      }
      { const float q = W12_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y10_a, G42_0, u); gy10 = fmaf(q, G42_0, gy10);
        u = fmaf(Y11_a, G43_0, u); gy11 = fmaf(q, G43_0, gy11);
        u = fmaf(Y12_a, G44_0, u); gy12 = fmaf(q, G44_0, gy12);
        u = fmaf(Y13_a, G45_0, u); gy13 = fmaf(q, G45_0, gy13);
        u = fmaf(Y14_a, G46_0, u); gy14 = fmaf(q, G46_0, gy14);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W12_0_a, u, gx2_0);
      }
      { const float q = W12_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y9_a, G47_0, u); gy9 = fmaf(q, G47_0, gy9);
        u = fmaf(Y10_a, G48_0, u); gy10 = fmaf(q, G48_0, gy10);
        u = fmaf(Y11_a, G49_0, u); gy11 = fmaf(q, G49_0, gy11);
        u = fmaf(Y12_a, G50_0, u); gy12 = fmaf(q, G50_0, gy12);
        u = fmaf(Y13_a, G51_0, u); gy13 = fmaf(q, G51_0, gy13);
        u = fmaf(Y14_a, G52_0, u); gy14 = fmaf(q, G52_0, gy14);
        u = fmaf(Y15_a, G53_0, u); gy15 = fmaf(q, G53_0, gy15);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W12_0_a, u, gx3_0);
      }
      if (gwp) gwp[1536] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W17_0_a * X0_0_a; float u = 0.f;
        u = fmaf(Y9_a, G54_0, u); gy9 = fmaf(q, G54_0, gy9);
        u = fmaf(Y10_a, G55_0, u); gy10 = fmaf(q, G55_0, gy10);
        u = fmaf(Y11_a, G56_0, u); gy11 = fmaf(q, G56_0, gy11);
        u = fmaf(Y12_a, G57_0, u); gy12 = fmaf(q, G57_0, gy12);
        u = fmaf(Y13_a, G58_0, u); gy13 = fmaf(q, G58_0, gy13);
        u = fmaf(Y14_a, G59_0, u); gy14 = fmaf(q, G59_0, gy14);
        u = fmaf(Y15_a, G60_0, u); gy15 = fmaf(q, G60_0, gy15);
        gw0 = fmaf(X0_0_a, u, gw0); gx0_0 = fmaf(W17_0_a, u, gx0_0);
      }
      if (gwp) gwp[2176] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W18_0_a * X1_0_a; float u = 0.f;
        u = fmaf(Y4_a, G61_0, u); gy4 = fmaf(q, G61_0, gy4);
        u = fmaf(Y5_a, G62_0, u); gy5 = fmaf(q, G62_0, gy5);
        u = fmaf(Y6_a, G63_0, u); gy6 = fmaf(q, G63_0, gy6);
        u = fmaf(Y7_a, G64_0, u); gy7 = fmaf(q, G64_0, gy7);
        u = fmaf(Y8_a, G65_0, u); gy8 = fmaf(q, G65_0, gy8);
        gw0 = fmaf(X1_0_a, u, gw0); gx1_0 = fmaf(W18_0_a, u, gx1_0);
      }
      { const float q = W18_0_a * X2_0_a; float u = 0.f;
        u = fmaf(Y4_a, G66_0, u); gy4 = fmaf(q, G66_0, gy4);
        u = fmaf(Y5_a, G67_0, u); gy5 = fmaf(q, G67_0, gy5);
        u = fmaf(Y6_a, G68_0, u); gy6 = fmaf(q, G68_0, gy6);
        u = fmaf(Y7_a, G69_0, u); gy7 = fmaf(q, G69_0, gy7);
        u = fmaf(Y8_a, G70_0, u); gy8 = fmaf(q, G70_0, gy8);
        gw0 = fmaf(X2_0_a, u, gw0); gx2_0 = fmaf(W18_0_a, u, gx2_0);
      }
      { const float q = W18_0_a * X3_0_a; float u = 0.f;
        u = fmaf(Y4_a, G71_0, u); gy4 = fmaf(q, G71_0, gy4);
        u = fmaf(Y5_a, G72_0, u); gy5 = fmaf(q, G72_0, gy5);
        u = fmaf(Y6_a, G73_0, u); gy6 = fmaf(q, G73_0, gy6);
        u = fmaf(Y7_a, G74_0, u); gy7 = fmaf(q, G74_0, gy7);
        u = fmaf(Y8_a, G75_0, u); gy8 = fmaf(q, G75_0, gy8);
        gw0 = fmaf(X3_0_a, u, gw0); gx3_0 = fmaf(W18_0_a, u, gx3_0);
      }
      if (gwp) gwp[2304] = gw0;
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
  }
  }
  else if (pg == 1) {
  const float* __restrict__ gp = gO + (size_t)i * g_stride + c;
  const float g2_0 = gp[256];
  const float g13_0 = gp[1664];
  const float g14_0 = gp[1792];
  const float g15_0 = gp[1920];
  const float g16_0 = gp[2048];
  const float g17_0 = gp[2176];
  const float g18_0 = gp[2304];
  const float g37_0 = gp[4736];
  const float g38_0 = gp[4864];
  const float g39_0 = gp[4992];
  const float g40_0 = gp[5120];
  const float g41_0 = gp[5248];
  const float g42_0 = gp[5376];
  const float g43_0 = gp[5504];
  const float g44_0 = gp[5632];
  const float g45_0 = gp[5760];
  const float g46_0 = gp[5888];
  const float g71_0 = gp[9088];
  const float g72_0 = gp[9216];
  const float g73_0 = gp[9344];
  const float g74_0 = gp[9472];
  const float g75_0 = gp[9600];
  const float g76_0 = gp[9728];
  const float g77_0 = gp[9856];
  const float g78_0 = gp[9984];
  const float g79_0 = gp[10112];
  const float g80_0 = gp[10240];
  const float g81_0 = gp[10368];
  const float g82_0 = gp[10496];
  const float g83_0 = gp[10624];
  const float g84_0 = gp[10752];
  const float G0_0 = 0.4472135954999579f * g2_0;
  const float G1_0 = 0.4472135954999579f * g2_0;
  const float G2_0 = 0.44721359549995804f * g2_0;
  const float G3_0 = 0.4472135954999579f * g2_0;
  const float G4_0 = 0.4472135954999579f * g2_0;
  const float G5_0 = 0.547722557505166f * g15_0;
  const float G6_0 = 0.547722557505166f * g13_0;
  const float G7_0 = 0.547722557505166f * g14_0;
  const float G8_0 = 0.547722557505166f * g13_0;
  const float G9_0 = -0.31622776601683794f * g13_0;
  const float G10_0 = 0.632455532033676f * g14_0;
  const float G11_0 = -0.31622776601683794f * g15_0;
  const float G12_0 = 0.547722557505166f * g15_0;
  const float G13_0 = 0.547722557505166f * g14_0;
  const float G14_0 = -0.547722557505166f * g13_0;
  const float G15_0 = 0.547722557505166f * g15_0;
  const float G16_0 = 0.4629100498862757f * g18_0;
  const float G17_0 = 0.3779644730092272f * g17_0;
  const float G18_0 = -0.11952286093343936f * g18_0;
  const float G19_0 = -0.11952286093343936f * g16_0;
  const float G20_0 = -0.4629100498862757f * g16_0;
  const float G21_0 = 0.3779644730092272f * g18_0;
  const float G22_0 = 0.47809144373375745f * g17_0;
  const float G23_0 = -0.29277002188456f * g16_0;
  const float G24_0 = -0.3779644730092272f * g16_0;
  const float G25_0 = 0.41403933560541256f * g16_0;
  const float G26_0 = 0.5070925528371102f * g17_0;
  const float G27_0 = 0.41403933560541256f * g18_0;
  const float G28_0 = 0.3779644730092272f * g16_0;
  const float G29_0 = -0.29277002188456f * g18_0;
  const float G30_0 = 0.47809144373375745f * g17_0;
  const float G31_0 = 0.3779644730092272f * g18_0;
  const float G32_0 = 0.4629100498862757f * g16_0;
  const float G33_0 = 0.11952286093343936f * g16_0;
  const float G34_0 = -0.11952286093343936f * g18_0;
  const float G35_0 = 0.3779644730092272f * g17_0;
  const float G36_0 = 0.4629100498862757f * g18_0;
  const float G37_0 = g37_0;
  const float G38_0 = g38_0;
  const float G39_0 = g39_0;
  const float G40_0 = g40_0;
  const float G41_0 = g41_0;
  const float G42_0 = 0.5345224838248488f * g44_0;
  const float G43_0 = -0.46291004988627565f * g45_0;
  const float G44_0 = 0.5345224838248488f * g42_0;
  const float G45_0 = -0.46291004988627565f * g43_0;
  const float G46_0 = -0.46291004988627565f * g45_0;
  const float G47_0 = fmaf(0.46291004988627565f, g46_0, -0.2672612419124244f * g44_0);
  const float G48_0 = -0.2672612419124244f * g43_0;
  const float G49_0 = -0.46291004988627565f * g42_0;
  const float G50_0 = 0.46291004988627565f * g43_0;
  const float G51_0 = 0.5345224838248488f * g42_0;
  const float G52_0 = -0.2672612419124244f * g43_0;
  const float G53_0 = -0.5345224838248489f * g44_0;
  const float G54_0 = -0.2672612419124244f * g45_0;
  const float G55_0 = 0.5345224838248488f * g46_0;
  const float G56_0 = -0.46291004988627565f * g43_0;
  const float G57_0 = -0.46291004988627565f * g42_0;
  const float G58_0 = -0.2672612419124244f * g45_0;
  const float G59_0 = fmaf(-0.46291004988627565f, g46_0, -0.2672612419124244f * g44_0);
  const float G60_0 = -0.46291004988627565f * g45_0;
  const float G61_0 = 0.46291004988627565f * g43_0;
  const float G62_0 = 0.5345224838248488f * g46_0;
  const float G63_0 = -0.46291004988627565f * g45_0;
  const float G64_0 = 0.5345224838248488f * g44_0;
  const float G65_0 = fmaf(0.7071067811865476f, g77_0, 0.18257418583505539f * g75_0);
  const float G66_0 = -0.5773502691896258f * g72_0;
  const float G67_0 = fmaf(0.18257418583505539f, g73_0, -0.7071067811865476f * g71_0);
  const float G68_0 = fmaf(0.5773502691896256f, g76_0, 0.447213595499958f * g74_0);
  const float G69_0 = -0.7302967433402215f * g73_0;
  const float G70_0 = -0.5773502691896256f * g72_0;
  const float G71_0 = -0.632455532033676f * g73_0;
  const float G72_0 = -0.7745966692414836f * g74_0;
  const float G73_0 = -0.632455532033676f * g75_0;
  const float G74_0 = -0.5773502691896256f * g72_0;
  const float G75_0 = -0.7302967433402215f * g75_0;
  const float G76_0 = fmaf(-0.5773502691896256f, g76_0, 0.447213595499958f * g74_0);
  const float G77_0 = fmaf(-0.18257418583505539f, g73_0, -0.7071067811865476f * g71_0);
  const float G78_0 = -0.5773502691896258f * g76_0;
  const float G79_0 = fmaf(-0.7071067811865476f, g77_0, 0.18257418583505539f * g75_0);
  const float G80_0 = 0.2886751345948128f * g82_0;
  const float G81_0 = 0.5773502691896258f * g81_0;
  const float G82_0 = fmaf(-0.2886751345948128f, g84_0, -0.447213595499958f * g82_0);
  const float G83_0 = 0.5773502691896258f * g79_0;
  const float G84_0 = fmaf(-0.447213595499958f, g80_0, 0.2886751345948128f * g78_0);
  const float G85_0 = -0.2886751345948128f * g80_0;
  const float G86_0 = -0.45643546458763845f * g83_0;
  const float G87_0 = fmaf(0.45643546458763845f, g84_0, -0.3535533905932738f * g82_0);
  const float G88_0 = fmaf(0.3535533905932738f, g83_0, -0.18257418583505539f * g81_0);
  const float G89_0 = -0.18257418583505539f * g80_0;
  const float G90_0 = -0.3535533905932738f * g79_0;
  const float G91_0 = fmaf(0.3535533905932738f, g80_0, -0.45643546458763845f * g78_0);
  const float G92_0 = 0.45643546458763845f * g79_0;
  const float G93_0 = 0.6454972243679029f * g78_0;
  const float G94_0 = -0.3872983346207418f * g80_0;
  const float G95_0 = -0.5163977794943223f * g81_0;
  const float G96_0 = -0.3872983346207418f * g82_0;
  const float G97_0 = 0.6454972243679029f * g84_0;
  const float G98_0 = -0.45643546458763845f * g79_0;
  const float G99_0 = fmaf(-0.3535533905932738f, g80_0, -0.45643546458763845f * g78_0);
  const float G100_0 = -0.3535533905932738f * g79_0;
  const float G101_0 = -0.18257418583505539f * g82_0;
  const float G102_0 = fmaf(-0.3535533905932738f, g83_0, -0.18257418583505539f * g81_0);
  const float G103_0 = fmaf(-0.45643546458763845f, g84_0, -0.3535533905932738f * g82_0);
  const float G104_0 = -0.45643546458763845f * g83_0;
  const float G105_0 = 0.2886751345948128f * g80_0;
  const float G106_0 = fmaf(0.447213595499958f, g80_0, 0.2886751345948128f * g78_0);
  const float G107_0 = 0.5773502691896258f * g83_0;
  const float G108_0 = fmaf(0.2886751345948128f, g84_0, -0.447213595499958f * g82_0);
  const float G109_0 = 0.5773502691896258f * g81_0;
  const float G110_0 = 0.2886751345948128f * g82_0;
  for (int p = p0; p < p1; ++p) {
    const int ea = __builtin_amdgcn_readfirstlane(eid ? eid[p] : p);
    const int sa = __builtin_amdgcn_readfirstlane(send[ea]);
    const float* __restrict__ wpa = W + (size_t)ea * w_stride + c;
    const float W2_0_a = wpa[256];
    const float W7_0_a = wpa[896];
    const float W8_0_a = wpa[1024];
    const float W13_0_a = wpa[1664];
    const float W14_0_a = wpa[1792];
    const float W19_0_a = wpa[2432];
    const float W20_0_a = wpa[2560];
    const float* __restrict__ xpa = X + (size_t)sa * x_stride + c;
    const float X4_0_a = xpa[512];
    const float X5_0_a = xpa[640];
    const float X6_0_a = xpa[768];
    const float X7_0_a = xpa[896];
    const float X8_0_a = xpa[1024];
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
    float gx4_0 = 0.f;
    float gx5_0 = 0.f;
    float gx6_0 = 0.f;
    float gx7_0 = 0.f;
    float gx8_0 = 0.f;
    float* __restrict__ gwp = gW ? gW + (size_t)ea * gw_stride + c : nullptr;
    {
      float gw0 = 0.f;
      { const float q = W2_0_a * X4_0_a; float u = 0.f;
        u = fmaf(Y4_a, G0_0, u); gy4 = fmaf(q, G0_0, gy4);
        gw0 = fmaf(X4_0_a, u, gw0); gx4_0 = fmaf(W2_0_a, u, gx4_0);
      }
      { const float q = W2_0_a * X5_0_a; float u = 0.f;
        u = fmaf(Y5_a, G1_0, u); gy5 = fmaf(q, G1_0, gy5);
        gw0 = fmaf(X5_0_a, u, gw0); gx5_0 = fmaf(W2_0_a, u, gx5_0);
      }
      { const float q = W2_0_a * X6_0_a; float u = 0.f;
        u = fmaf(Y6_a, G2_0, u); gy6 = fmaf(q, G2_0, gy6);
        gw0 = fmaf(X6_0_a, u, gw0); gx6_0 = fmaf(W2_0_a, u, gx6_0);
      }
      { const float q = W2_0_a * X7_0_a; float u = 0.f;
        u = fmaf(Y7_a, G3_0, u); gy7 = fmaf(q, G3_0, gy7);
        gw0 = fmaf(X7_0_a, u, gw0); gx7_0 = fmaf(W2_0_a, u, gx7_0);
      }
      { const float q = W2_0_a * X8_0_a; float u = 0.f;
        u = fmaf(Y8_a, G4_0, u); gy8 = fmaf(q, G4_0, gy8);
        gw0 = fmaf(X8_0_a, u, gw0); gx8_0 = fmaf(W2_0_a, u, gx8_0);
      }
      if (gwp) gwp[256] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W7_0_a * X4_0_a; float u = 0.f;
        u = fmaf(Y1_a, G5_0, u); gy1 = fmaf(q, G5_0, gy1);
        u = fmaf(Y3_a, G6_0, u); gy3 = fmaf(q, G6_0, gy3);
        gw0 = fmaf(X4_0_a, u, gw0); gx4_0 = fmaf(W7_0_a, u, gx4_0);
      }
      { const float q = W7_0_a * X5_0_a; float u = 0.f;
        u = fmaf(Y1_a, G7_0, u); gy1 = fmaf(q, G7_0, gy1);
        u = fmaf(Y2_a, G8_0, u); gy2 = fmaf(q, G8_0, gy2);
        gw0 = fmaf(X5_0_a, u, gw0); gx5_0 = fmaf(W7_0_a, u, gx5_0);
      }
      { const float q = W7_0_a * X6_0_a; float u = 0.f;
        u = fmaf(Y1_a, G9_0, u); gy1 = fmaf(q, G9_0, gy1);
        u = fmaf(Y2_a, G10_0, u); gy2 = fmaf(q, G10_0, gy2);
        u = fmaf(Y3_a, G11_0, u); gy3 = fmaf(q, G11_0, gy3);
        gw0 = fmaf(X6_0_a, u, gw0); gx6_0 = fmaf(W7_0_a, u, gx6_0);
      }
      { const float q = W7_0_a * X7_0_a; float u = 0.f;
        u = fmaf(Y2_a, G12_0, u); gy2 = fmaf(q, G12_0, gy2);
        u = fmaf(Y3_a, G13_0, u); gy3 = fmaf(q, G13_0, gy3);
        gw0 = fmaf(X7_0_a, u, gw0); gx7_0 = fmaf(W7_0_a, u, gx7_0);
      }
      { const float q = W7_0_a * X8_0_a; float u = 0.f;
        u = fmaf(Y1_a, G14_0, u); gy1 = fmaf(q, G14_0, gy1);
        u = fmaf(Y3_a, G15_0, u); gy3 = fmaf(q, G15_0, gy3);
        gw0 = fmaf(X8_0_a, u, gw0); gx8_0 = fmaf(W7_0_a, u, gx8_0);
      }
      if (gwp) gwp[896] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W8_0_a * X4_0_a; float u = 0.f;
        u = fmaf(Y9_a, G16_0, u); gy9 = fmaf(q, G16_0, gy9);
        u = fmaf(Y10_a, G17_0, u); gy10 = fmaf(q, G17_0, gy10);
        u = fmaf(Y11_a, G18_0, u); gy11 = fmaf(q, G18_0, gy11);
        u = fmaf(Y13_a, G19_0, u); gy13 = fmaf(q, G19_0, gy13);
        u = fmaf(Y15_a, G20_0, u); gy15 = fmaf(q, G20_0, gy15);
        gw0 = fmaf(X4_0_a, u, gw0); gx4_0 = fmaf(W8_0_a, u, gx4_0);
      }
      { const float q = W8_0_a * X5_0_a; float u = 0.f;
        u = fmaf(Y10_a, G21_0, u); gy10 = fmaf(q, G21_0, gy10);
        u = fmaf(Y11_a, G22_0, u); gy11 = fmaf(q, G22_0, gy11);
        u = fmaf(Y12_a, G23_0, u); gy12 = fmaf(q, G23_0, gy12);
        u = fmaf(Y14_a, G24_0, u); gy14 = fmaf(q, G24_0, gy14);
        gw0 = fmaf(X5_0_a, u, gw0); gx5_0 = fmaf(W8_0_a, u, gx5_0);
      }
      { const float q = W8_0_a * X6_0_a; float u = 0.f;
        u = fmaf(Y11_a, G25_0, u); gy11 = fmaf(q, G25_0, gy11);
        u = fmaf(Y12_a, G26_0, u); gy12 = fmaf(q, G26_0, gy12);
        u = fmaf(Y13_a, G27_0, u); gy13 = fmaf(q, G27_0, gy13);
        gw0 = fmaf(X6_0_a, u, gw0); gx6_0 = fmaf(W8_0_a, u, gx6_0);
      }
      { const float q = W8_0_a * X7_0_a; float u = 0.f;
        u = fmaf(Y10_a, G28_0, u); gy10 = fmaf(q, G28_0, gy10);
        u = fmaf(Y12_a, G29_0, u); gy12 = fmaf(q, G29_0, gy12);
        u = fmaf(Y13_a, G30_0, u); gy13 = fmaf(q, G30_0, gy13);
        u = fmaf(Y14_a, G31_0, u); gy14 = fmaf(q, G31_0, gy14);
        gw0 = fmaf(X7_0_a, u, gw0); gx7_0 = fmaf(W8_0_a, u, gx7_0);
      }
      { const float q = W8_0_a * X8_0_a; float u = 0.f;
        u = fmaf(Y9_a, G32_0, u); gy9 = fmaf(q, G32_0, gy9);
        u = fmaf(Y11_a, G33_0, u); gy11 = fmaf(q, G33_0, gy11);
        u = fmaf(Y13_a, G34_0, u); gy13 = fmaf(q, G34_0, gy13);
        u = fmaf(Y14_a, G35_0, u); gy14 = fmaf(q, G35_0, gy14);
        u = fmaf(Y15_a, G36_0, u); gy15 = fmaf(q, G36_0, gy15);
        gw0 = fmaf(X8_0_a, u, gw0); gx8_0 = fmaf(W8_0_a, u, gx8_0);
      }
      if (gwp) gwp[1024] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W13_0_a * X4_0_a; float u = 0.f;
        u = fmaf(Y0_a, G37_0, u); gy0 = fmaf(q, G37_0, gy0);
        gw0 = fmaf(X4_0_a, u, gw0); gx4_0 = fmaf(W13_0_a, u, gx4_0);
      }
      { const float q = W13_0_a * X5_0_a; float u = 0.f;
        u = fmaf(Y0_a, G38_0, u); gy0 = fmaf(q, G38_0, gy0);
        gw0 = fmaf(X5_0_a, u, gw0); gx5_0 = fmaf(W13_0_a, u, gx5_0);
      }
      { const float q = W13_0_a * X6_0_a; float u = 0.f;
        u = fmaf(Y0_a, G39_0, u); gy0 = fmaf(q, G39_0, gy0);
        gw0 = fmaf(X6_0_a, u, gw0); gx6_0 = fmaf(W13_0_a, u, gx6_0);
      }
      { const float q = W13_0_a * X7_0_a; float u = 0.f;
        u = fmaf(Y0_a, G40_0, u); gy0 = fmaf(q, G40_0, gy0);
        gw0 = fmaf(X7_0_a, u, gw0); gx7_0 = fmaf(W13_0_a, u, gx7_0);
      }
      { const float q = W13_0_a * X8_0_a; float u = 0.f;
        u = fmaf(Y0_a, G41_0, u); gy0 = fmaf(q, G41_0, gy0);
        gw0 = fmaf(X8_0_a, u, gw0); gx8_0 = fmaf(W13_0_a, u, gx8_0);
      }
      if (gwp) gwp[1664] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W14_0_a * X4_0_a; float u = 0.f;
        u = fmaf(Y4_a, G42_0, u); gy4 = fmaf(q, G42_0, gy4);
        u = fmaf(Y5_a, G43_0, u); gy5 = fmaf(q, G43_0, gy5);
        u = fmaf(Y6_a, G44_0, u); gy6 = fmaf(q, G44_0, gy6);
        u = fmaf(Y7_a, G45_0, u); gy7 = fmaf(q, G45_0, gy7);
        gw0 = fmaf(X4_0_a, u, gw0); gx4_0 = fmaf(W14_0_a, u, gx4_0);
      }
      { const float q = W14_0_a * X5_0_a; float u = 0.f;
        u = fmaf(Y4_a, G46_0, u); gy4 = fmaf(q, G46_0, gy4);
        u = fmaf(Y5_a, G47_0, u); gy5 = fmaf(q, G47_0, gy5);
        u = fmaf(Y6_a, G48_0, u); gy6 = fmaf(q, G48_0, gy6);
        u = fmaf(Y7_a, G49_0, u); gy7 = fmaf(q, G49_0, gy7);
        u = fmaf(Y8_a, G50_0, u); gy8 = fmaf(q, G50_0, gy8);
        gw0 = fmaf(X5_0_a, u, gw0); gx5_0 = fmaf(W14_0_a, u, gx5_0);
      }
      { const float q = W14_0_a * X6_0_a; float u = 0.f;
        u = fmaf(Y4_a, G51_0, u); gy4 = fmaf(q, G51_0, gy4);
        u = fmaf(Y5_a, G52_0, u); gy5 = fmaf(q, G52_0, gy5);
        u = fmaf(Y6_a, G53_0, u); gy6 = fmaf(q, G53_0, gy6);
        u = fmaf(Y7_a, G54_0, u); gy7 = fmaf(q, G54_0, gy7);
        u = fmaf(Y8_a, G55_0, u); gy8 = fmaf(q, G55_0, gy8);
        gw0 = fmaf(X6_0_a, u, gw0); gx6_0 = fmaf(W14_0_a, u, gx6_0);
      }
      { const float q = W14_0_a * X7_0_a; float u = 0.f;
        u = fmaf(Y4_a, G56_0, u); gy4 = fmaf(q, G56_0, gy4);
        u = fmaf(Y5_a, G57_0, u); gy5 = fmaf(q, G57_0, gy5);
        u = fmaf(Y6_a, G58_0, u); gy6 = fmaf(q, G58_0, gy6);
        u = fmaf(Y7_a, G59_0, u); gy7 = fmaf(q, G59_0, gy7);
        u = fmaf(Y8_a, G60_0, u); gy8 = fmaf(q, G60_0, gy8);
        gw0 = fmaf(X7_0_a, u, gw0); gx7_0 = fmaf(W14_0_a, u, gx7_0);
      }
      { const float q = W14_0_a * X8_0_a; float u = 0.f;
        u = fmaf(Y5_a, G61_0, u); gy5 = fmaf(q, G61_0, gy5);
        u = fmaf(Y6_a, G62_0, u); gy6 = fmaf(q, G62_0, gy6);
        u = fmaf(Y7_a, G63_0, u); gy7 = fmaf(q, G63_0, gy7);
        u = fmaf(Y8_a, G64_0, u); gy8 = fmaf(q, G64_0, gy8);
        gw0 = fmaf(X8_0_a, u, gw0); gx8_0 = fmaf(W14_0_a, u, gx8_0);
      }
      if (gwp) gwp[1792] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W19_0_a * X4_0_a; float u = 0.f;
        u = fmaf(Y1_a, G65_0, u); gy1 = fmaf(q, G65_0, gy1);
        u = fmaf(Y2_a, G66_0, u); gy2 = fmaf(q, G66_0, gy2);
        u = fmaf(Y3_a, G67_0, u); gy3 = fmaf(q, G67_0, gy3);
        gw0 = fmaf(X4_0_a, u, gw0); gx4_0 = fmaf(W19_0_a, u, gx4_0);
      }
      { const float q = W19_0_a * X5_0_a; float u = 0.f;
        u = fmaf(Y1_a, G68_0, u); gy1 = fmaf(q, G68_0, gy1);
        u = fmaf(Y2_a, G69_0, u); gy2 = fmaf(q, G69_0, gy2);
        u = fmaf(Y3_a, G70_0, u); gy3 = fmaf(q, G70_0, gy3);
        gw0 = fmaf(X5_0_a, u, gw0); gx5_0 = fmaf(W19_0_a, u, gx5_0);
      }
      { const float q = W19_0_a * X6_0_a; float u = 0.f;
        u = fmaf(Y1_a, G71_0, u); gy1 = fmaf(q, G71_0, gy1);
        u = fmaf(Y2_a, G72_0, u); gy2 = fmaf(q, G72_0, gy2);
        u = fmaf(Y3_a, G73_0, u); gy3 = fmaf(q, G73_0, gy3);
        gw0 = fmaf(X6_0_a, u, gw0); gx6_0 = fmaf(W19_0_a, u, gx6_0);
      }
      { const float q = W19_0_a * X7_0_a; float u = 0.f;
        u = fmaf(Y1_a, G74_0, u); gy1 = fmaf(q, G74_0, gy1);
        u = fmaf(Y2_a, G75_0, u); gy2 = fmaf(q, G75_0, gy2);
        u = fmaf(Y3_a, G76_0, u); gy3 = fmaf(q, G76_0, gy3);
        gw0 = fmaf(X7_0_a, u, gw0); gx7_0 = fmaf(W19_0_a, u, gx7_0);
      }
      { const float q = W19_0_a * X8_0_a; float u = 0.f;
        u = fmaf(Y1_a, G77_0, u); gy1 = fmaf(q, G77_0, gy1);
        u = fmaf(Y2_a, G78_0, u); gy2 = fmaf(q, G78_0, gy2);
        u = fmaf(Y3_a, G79_0, u); gy3 = fmaf(q, G79_0, gy3);
        gw0 = fmaf(X8_0_a, u, gw0); gx8_0 = fmaf(W19_0_a, u, gx8_0);
      }
      if (gwp) gwp[2432] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W20_0_a * X4_0_a; float u = 0.f;
        u = fmaf(Y9_a, G80_0, u); gy9 = fmaf(q, G80_0, gy9);
        u = fmaf(Y10_a, G81_0, u); gy10 = fmaf(q, G81_0, gy10);
        u = fmaf(Y11_a, G82_0, u); gy11 = fmaf(q, G82_0, gy11);
        u = fmaf(Y12_a, G83_0, u); gy12 = fmaf(q, G83_0, gy12);
        u = fmaf(Y13_a, G84_0, u); gy13 = fmaf(q, G84_0, gy13);
        u = fmaf(Y15_a, G85_0, u); gy15 = fmaf(q, G85_0, gy15);
        gw0 = fmaf(X4_0_a, u, gw0); gx4_0 = fmaf(W20_0_a, u, gx4_0);
      }
      { const float q = W20_0_a * X5_0_a; float u = 0.f;
        u = fmaf(Y9_a, G86_0, u); gy9 = fmaf(q, G86_0, gy9);
        u = fmaf(Y10_a, G87_0, u); gy10 = fmaf(q, G87_0, gy10);
        u = fmaf(Y11_a, G88_0, u); gy11 = fmaf(q, G88_0, gy11);
        u = fmaf(Y12_a, G89_0, u); gy12 = fmaf(q, G89_0, gy12);
        u = fmaf(Y13_a, G90_0, u); gy13 = fmaf(q, G90_0, gy13);
        u = fmaf(Y14_a, G91_0, u); gy14 = fmaf(q, G91_0, gy14);
        u = fmaf(Y15_a, G92_0, u); gy15 = fmaf(q, G92_0, gy15);
        gw0 = fmaf(X5_0_a, u, gw0); gx5_0 = fmaf(W20_0_a, u, gx5_0);
      }
      { const float q = W20_0_a * X6_0_a; float u = 0.f;
        u = fmaf(Y9_a, G93_0, u); gy9 = fmaf(q, G93_0, gy9);
        u = fmaf(Y11_a, G94_0, u); gy11 = fmaf(q, G94_0, gy11);
        u = fmaf(Y12_a, G95_0, u); gy12 = fmaf(q, G95_0, gy12);
        u = fmaf(Y13_a, G96_0, u); gy13 = fmaf(q, G96_0, gy13);
        u = fmaf(Y15_a, G97_0, u); gy15 = fmaf(q, G97_0, gy15);
        gw0 = fmaf(X6_0_a, u, gw0); gx6_0 = fmaf(W20_0_a, u, gx6_0);
      }
      { const float q = W20_0_a * X7_0_a; float u = 0.f;
        u = fmaf(Y9_a, G98_0, u); gy9 = fmaf(q, G98_0, gy9);
        u = fmaf(Y10_a, G99_0, u); gy10 = fmaf(q, G99_0, gy10);
        u = fmaf(Y11_a, G100_0, u); gy11 = fmaf(q, G100_0, gy11);
        u = fmaf(Y12_a, G101_0, u); gy12 = fmaf(q, G101_0, gy12);
        u = fmaf(Y13_a, G102_0, u); gy13 = fmaf(q, G102_0, gy13);
        u = fmaf(Y14_a, G103_0, u); gy14 = fmaf(q, G103_0, gy14);
        u = fmaf(Y15_a, G104_0, u); gy15 = fmaf(q, G104_0, gy15);
        gw0 = fmaf(X7_0_a, u, gw0); gx7_0 = fmaf(W20_0_a, u, gx7_0);
      }
      { const float q = W20_0_a * X8_0_a; float u = 0.f;
        u = fmaf(Y9_a, G105_0, u); gy9 = fmaf(q, G105_0, gy9);
        u = fmaf(Y11_a, G106_0, u); gy11 = fmaf(q, G106_0, gy11);
        u = fmaf(Y12_a, G107_0, u); gy12 = fmaf(q, G107_0, gy12);
        u = fmaf(Y13_a, G108_0, u); gy13 = fmaf(q, G108_0, gy13);
        u = fmaf(Y14_a, G109_0, u); gy14 = fmaf(q, G109_0, gy14);
        u = fmaf(Y15_a, G110_0, u); gy15 = fmaf(q, G110_0, gy15);
        gw0 = fmaf(X8_0_a, u, gw0); gx8_0 = fmaf(W20_0_a, u, gx8_0);
      }
      if (gwp) gwp[2560] = gw0;
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
      atomicAdd(gxp + 512, gx4_0);
      atomicAdd(gxp + 640, gx5_0);
      atomicAdd(gxp + 768, gx6_0);
      atomicAdd(gxp + 896, gx7_0);
      atomicAdd(gxp + 1024, gx8_0);
    }
  }
  }
  else if (pg == 2) {
  const float* __restrict__ gp = gO + (size_t)i * g_stride + c;
  const float g3_0 = gp[384];
  const float g19_0 = gp[2432];
  const float g20_0 = gp[2560];
  const float g21_0 = gp[2688];
  const float g47_0 = gp[6016];
  const float g48_0 = gp[6144];
  const float g49_0 = gp[6272];
  const float g50_0 = gp[6400];
  const float g51_0 = gp[6528];
  const float g52_0 = gp[6656];
  const float g53_0 = gp[6784];
  const float g54_0 = gp[6912];
  const float g55_0 = gp[7040];
  const float g56_0 = gp[7168];
  const float g85_0 = gp[10880];
  const float g86_0 = gp[11008];
  const float g87_0 = gp[11136];
  const float g88_0 = gp[11264];
  const float g89_0 = gp[11392];
  const float g90_0 = gp[11520];
  const float g91_0 = gp[11648];
  const float g92_0 = gp[11776];
  const float g93_0 = gp[11904];
  const float g94_0 = gp[12032];
  const float g95_0 = gp[12160];
  const float g96_0 = gp[12288];
  const float g97_0 = gp[12416];
  const float g98_0 = gp[12544];
  const float G0_0 = 0.3779644730092272f * g3_0;
  const float G1_0 = 0.3779644730092272f * g3_0;
  const float G2_0 = 0.3779644730092272f * g3_0;
  const float G3_0 = 0.3779644730092273f * g3_0;
  const float G4_0 = 0.3779644730092272f * g3_0;
  const float G5_0 = 0.3779644730092272f * g3_0;
  const float G6_0 = 0.3779644730092272f * g3_0;
  const float G7_0 = 0.4629100498862757f * g21_0;
  const float G8_0 = 0.4629100498862757f * g19_0;
  const float G9_0 = 0.3779644730092272f * g20_0;
  const float G10_0 = 0.3779644730092272f * g21_0;
  const float G11_0 = 0.3779644730092272f * g19_0;
  const float G12_0 = -0.11952286093343936f * g21_0;
  const float G13_0 = 0.47809144373375745f * g20_0;
  const float G14_0 = 0.41403933560541256f * g19_0;
  const float G15_0 = 0.11952286093343936f * g19_0;
  const float G16_0 = -0.29277002188456f * g19_0;
  const float G17_0 = 0.5070925528371102f * g20_0;
  const float G18_0 = -0.29277002188456f * g21_0;
  const float G19_0 = -0.11952286093343936f * g19_0;
  const float G20_0 = 0.41403933560541256f * g21_0;
  const float G21_0 = 0.47809144373375745f * g20_0;
  const float G22_0 = -0.11952286093343936f * g21_0;
  const float G23_0 = -0.3779644730092272f * g19_0;
  const float G24_0 = 0.3779644730092272f * g21_0;
  const float G25_0 = 0.3779644730092272f * g20_0;
  const float G26_0 = -0.4629100498862757f * g19_0;
  const float G27_0 = 0.4629100498862757f * g21_0;
  const float G28_0 = 0.5976143046671968f * g51_0;
  const float G29_0 = 0.5976143046671968f * g47_0;
  const float G30_0 = 0.4879500364742667f * g50_0;
  const float G31_0 = 0.4879500364742667f * g47_0;
  const float G32_0 = 0.4879500364742667f * g48_0;
  const float G33_0 = fmaf(0.1543033499620919f, g51_0, 0.5345224838248489f * g49_0);
  const float G34_0 = 0.6172133998483678f * g48_0;
  const float G35_0 = -0.1543033499620919f * g47_0;
  const float G36_0 = -0.3779644730092273f * g48_0;
  const float G37_0 = 0.6546536707079773f * g49_0;
  const float G38_0 = -0.3779644730092273f * g50_0;
  const float G39_0 = -0.1543033499620919f * g47_0;
  const float G40_0 = 0.6172133998483678f * g50_0;
  const float G41_0 = fmaf(-0.1543033499620919f, g51_0, 0.5345224838248489f * g49_0);
  const float G42_0 = -0.4879500364742667f * g48_0;
  const float G43_0 = 0.4879500364742667f * g51_0;
  const float G44_0 = 0.4879500364742667f * g50_0;
  const float G45_0 = -0.5976143046671968f * g47_0;
  const float G46_0 = 0.5976143046671968f * g51_0;
  const float G47_0 = 0.545544725589981f * g54_0;
  const float G48_0 = -0.38575837490522974f * g55_0;
  const float G49_0 = 0.24397501823713336f * g56_0;
  const float G50_0 = 0.24397501823713336f * g52_0;
  const float G51_0 = -0.38575837490522974f * g53_0;
  const float G52_0 = -0.38575837490522974f * g55_0;
  const float G53_0 = -0.2988071523335984f * g55_0;
  const float G54_0 = 0.4879500364742667f * g52_0;
  const float G55_0 = -0.2988071523335984f * g53_0;
  const float G56_0 = 0.38575837490522974f * g53_0;
  const float G57_0 = 0.24397501823713336f * g56_0;
  const float G58_0 = -0.2988071523335984f * g55_0;
  const float G59_0 = fmaf(0.3779644730092273f, g56_0, -0.3273268353539886f * g54_0);
  const float G60_0 = -0.15430334996209194f * g53_0;
  const float G61_0 = -0.3779644730092273f * g52_0;
  const float G62_0 = 0.2988071523335984f * g53_0;
  const float G63_0 = -0.24397501823713336f * g52_0;
  const float G64_0 = 0.4879500364742667f * g52_0;
  const float G65_0 = -0.15430334996209194f * g53_0;
  const float G66_0 = -0.4364357804719849f * g54_0;
  const float G67_0 = -0.15430334996209194f * g55_0;
  const float G68_0 = 0.4879500364742667f * g56_0;
  const float G69_0 = 0.24397501823713336f * g52_0;
  const float G70_0 = -0.2988071523335984f * g53_0;
  const float G71_0 = -0.3779644730092273f * g52_0;
  const float G72_0 = -0.15430334996209194f * g55_0;
  const float G73_0 = fmaf(-0.3779644730092273f, g56_0, -0.3273268353539886f * g54_0);
  const float G74_0 = -0.2988071523335984f * g55_0;
  const float G75_0 = 0.24397501823713336f * g56_0;
  const float G76_0 = -0.38575837490522974f * g53_0;
  const float G77_0 = 0.2988071523335984f * g53_0;
  const float G78_0 = 0.4879500364742667f * g56_0;
  const float G79_0 = -0.2988071523335984f * g55_0;
  const float G80_0 = -0.38575837490522974f * g55_0;
  const float G81_0 = 0.38575837490522974f * g53_0;
  const float G82_0 = -0.24397501823713336f * g52_0;
  const float G83_0 = 0.24397501823713336f * g56_0;
  const float G84_0 = -0.38575837490522974f * g55_0;
  const float G85_0 = 0.545544725589981f * g54_0;
  const float G86_0 = g85_0;
  const float G87_0 = g86_0;
  const float G88_0 = g87_0;
  const float G89_0 = g88_0;
  const float G90_0 = g89_0;
  const float G91_0 = g90_0;
  const float G92_0 = g91_0;
  const float G93_0 = 0.2886751345948128f * g96_0;
  const float G94_0 = -0.45643546458763845f * g97_0;
  const float G95_0 = 0.6454972243679029f * g92_0;
  const float G96_0 = -0.45643546458763845f * g93_0;
  const float G97_0 = 0.2886751345948128f * g94_0;
  const float G98_0 = 0.5773502691896258f * g95_0;
  const float G99_0 = fmaf(0.45643546458763845f, g98_0, -0.3535533905932738f * g96_0);
  const float G100_0 = fmaf(-0.3535533905932738f, g94_0, -0.45643546458763845f * g92_0);
  const float G101_0 = fmaf(-0.2886751345948128f, g98_0, -0.447213595499958f * g96_0);
  const float G102_0 = fmaf(0.3535533905932738f, g97_0, -0.18257418583505539f * g95_0);
  const float G103_0 = -0.3872983346207418f * g94_0;
  const float G104_0 = -0.3535533905932738f * g93_0;
  const float G105_0 = fmaf(0.447213595499958f, g94_0, 0.2886751345948128f * g92_0);
  const float G106_0 = 0.5773502691896258f * g93_0;
  const float G107_0 = -0.18257418583505539f * g94_0;
  const float G108_0 = -0.5163977794943223f * g95_0;
  const float G109_0 = -0.18257418583505539f * g96_0;
  const float G110_0 = 0.5773502691896258f * g97_0;
  const float G111_0 = fmaf(-0.447213595499958f, g94_0, 0.2886751345948128f * g92_0);
  const float G112_0 = -0.3535533905932738f * g93_0;
  const float G113_0 = -0.3872983346207418f * g96_0;
  const float G114_0 = fmaf(-0.3535533905932738f, g97_0, -0.18257418583505539f * g95_0);
  const float G115_0 = fmaf(0.2886751345948128f, g98_0, -0.447213595499958f * g96_0);
  const float G116_0 = fmaf(0.3535533905932738f, g94_0, -0.45643546458763845f * g92_0);
  const float G117_0 = fmaf(-0.45643546458763845f, g98_0, -0.3535533905932738f * g96_0);
  const float G118_0 = 0.5773502691896258f * g95_0;
  const float G119_0 = -0.2886751345948128f * g94_0;
  const float G120_0 = 0.45643546458763845f * g93_0;
  const float G121_0 = 0.6454972243679029f * g98_0;
  const float G122_0 = -0.45643546458763845f * g97_0;
  const float G123_0 = 0.2886751345948128f * g96_0;
  for (int p = p0; p < p1; ++p) {
    const int ea = __builtin_amdgcn_readfirstlane(eid ? eid[p] : p);
    const int sa = __builtin_amdgcn_readfirstlane(send[ea]);
    const float* __restrict__ wpa = W + (size_t)ea * w_stride + c;
    const float W3_0_a = wpa[384];
    const float W9_0_a = wpa[1152];
    const float W15_0_a = wpa[1920];
    const float W16_0_a = wpa[2048];
    const float W21_0_a = wpa[2688];
    const float W22_0_a = wpa[2816];
    const float* __restrict__ xpa = X + (size_t)sa * x_stride + c;
    const float X9_0_a = xpa[1152];
    const float X10_0_a = xpa[1280];
    const float X11_0_a = xpa[1408];
    const float X12_0_a = xpa[1536];
    const float X13_0_a = xpa[1664];
    const float X14_0_a = xpa[1792];
    const float X15_0_a = xpa[1920];
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
    float gx9_0 = 0.f;
    float gx10_0 = 0.f;
    float gx11_0 = 0.f;
    float gx12_0 = 0.f;
    float gx13_0 = 0.f;
    float gx14_0 = 0.f;
    float gx15_0 = 0.f;
    float* __restrict__ gwp = gW ? gW + (size_t)ea * gw_stride + c : nullptr;
    {
      float gw0 = 0.f;
      { const float q = W3_0_a * X9_0_a; float u = 0.f;
        u = fmaf(Y9_a, G0_0, u); gy9 = fmaf(q, G0_0, gy9);
        gw0 = fmaf(X9_0_a, u, gw0); gx9_0 = fmaf(W3_0_a, u, gx9_0);
      }
      { const float q = W3_0_a * X10_0_a; float u = 0.f;
        u = fmaf(Y10_a, G1_0, u); gy10 = fmaf(q, G1_0, gy10);
        gw0 = fmaf(X10_0_a, u, gw0); gx10_0 = fmaf(W3_0_a, u, gx10_0);
      }
      { const float q = W3_0_a * X11_0_a; float u = 0.f;
        u = fmaf(Y11_a, G2_0, u); gy11 = fmaf(q, G2_0, gy11);
        gw0 = fmaf(X11_0_a, u, gw0); gx11_0 = fmaf(W3_0_a, u, gx11_0);
      }
      { const float q = W3_0_a * X12_0_a; float u = 0.f;
        u = fmaf(Y12_a, G3_0, u); gy12 = fmaf(q, G3_0, gy12);
        gw0 = fmaf(X12_0_a, u, gw0); gx12_0 = fmaf(W3_0_a, u, gx12_0);
      }
      { const float q = W3_0_a * X13_0_a; float u = 0.f;
        u = fmaf(Y13_a, G4_0, u); gy13 = fmaf(q, G4_0, gy13);
        gw0 = fmaf(X13_0_a, u, gw0); gx13_0 = fmaf(W3_0_a, u, gx13_0);
      }
      { const float q = W3_0_a * X14_0_a; float u = 0.f;
        u = fmaf(Y14_a, G5_0, u); gy14 = fmaf(q, G5_0, gy14);
        gw0 = fmaf(X14_0_a, u, gw0); gx14_0 = fmaf(W3_0_a, u, gx14_0);
      }
      { const float q = W3_0_a * X15_0_a; float u = 0.f;
        u = fmaf(Y15_a, G6_0, u); gy15 = fmaf(q, G6_0, gy15);
        gw0 = fmaf(X15_0_a, u, gw0); gx15_0 = fmaf(W3_0_a, u, gx15_0);
      }
      if (gwp) gwp[384] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W9_0_a * X9_0_a; float u = 0.f;
        u = fmaf(Y4_a, G7_0, u); gy4 = fmaf(q, G7_0, gy4);
        u = fmaf(Y8_a, G8_0, u); gy8 = fmaf(q, G8_0, gy8);
        gw0 = fmaf(X9_0_a, u, gw0); gx9_0 = fmaf(W9_0_a, u, gx9_0);
      }
      { const float q = W9_0_a * X10_0_a; float u = 0.f;
        u = fmaf(Y4_a, G9_0, u); gy4 = fmaf(q, G9_0, gy4);
        u = fmaf(Y5_a, G10_0, u); gy5 = fmaf(q, G10_0, gy5);
        u = fmaf(Y7_a, G11_0, u); gy7 = fmaf(q, G11_0, gy7);
        gw0 = fmaf(X10_0_a, u, gw0); gx10_0 = fmaf(W9_0_a, u, gx10_0);
      }
      { const float q = W9_0_a * X11_0_a; float u = 0.f;
        u = fmaf(Y4_a, G12_0, u); gy4 = fmaf(q, G12_0, gy4);
        u = fmaf(Y5_a, G13_0, u); gy5 = fmaf(q, G13_0, gy5);
        u = fmaf(Y6_a, G14_0, u); gy6 = fmaf(q, G14_0, gy6);
        u = fmaf(Y8_a, G15_0, u); gy8 = fmaf(q, G15_0, gy8);
        gw0 = fmaf(X11_0_a, u, gw0); gx11_0 = fmaf(W9_0_a, u, gx11_0);
      }
      { const float q = W9_0_a * X12_0_a; float u = 0.f;
        u = fmaf(Y5_a, G16_0, u); gy5 = fmaf(q, G16_0, gy5);
        u = fmaf(Y6_a, G17_0, u); gy6 = fmaf(q, G17_0, gy6);
        u = fmaf(Y7_a, G18_0, u); gy7 = fmaf(q, G18_0, gy7);
        gw0 = fmaf(X12_0_a, u, gw0); gx12_0 = fmaf(W9_0_a, u, gx12_0);
      }
      { const float q = W9_0_a * X13_0_a; float u = 0.f;
        u = fmaf(Y4_a, G19_0, u); gy4 = fmaf(q, G19_0, gy4);
        u = fmaf(Y6_a, G20_0, u); gy6 = fmaf(q, G20_0, gy6);
        u = fmaf(Y7_a, G21_0, u); gy7 = fmaf(q, G21_0, gy7);
        u = fmaf(Y8_a, G22_0, u); gy8 = fmaf(q, G22_0, gy8);
        gw0 = fmaf(X13_0_a, u, gw0); gx13_0 = fmaf(W9_0_a, u, gx13_0);
      }
      { const float q = W9_0_a * X14_0_a; float u = 0.f;
        u = fmaf(Y5_a, G23_0, u); gy5 = fmaf(q, G23_0, gy5);
        u = fmaf(Y7_a, G24_0, u); gy7 = fmaf(q, G24_0, gy7);
        u = fmaf(Y8_a, G25_0, u); gy8 = fmaf(q, G25_0, gy8);
        gw0 = fmaf(X14_0_a, u, gw0); gx14_0 = fmaf(W9_0_a, u, gx14_0);
      }
      { const float q = W9_0_a * X15_0_a; float u = 0.f;
        u = fmaf(Y4_a, G26_0, u); gy4 = fmaf(q, G26_0, gy4);
        u = fmaf(Y8_a, G27_0, u); gy8 = fmaf(q, G27_0, gy8);
        gw0 = fmaf(X15_0_a, u, gw0); gx15_0 = fmaf(W9_0_a, u, gx15_0);
      }
      if (gwp) gwp[1152] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W15_0_a * X9_0_a; float u = 0.f;
        u = fmaf(Y1_a, G28_0, u); gy1 = fmaf(q, G28_0, gy1);
        u = fmaf(Y3_a, G29_0, u); gy3 = fmaf(q, G29_0, gy3);
        gw0 = fmaf(X9_0_a, u, gw0); gx9_0 = fmaf(W15_0_a, u, gx9_0);
      }
      { const float q = W15_0_a * X10_0_a; float u = 0.f;
        u = fmaf(Y1_a, G30_0, u); gy1 = fmaf(q, G30_0, gy1);
        u = fmaf(Y2_a, G31_0, u); gy2 = fmaf(q, G31_0, gy2);
        u = fmaf(Y3_a, G32_0, u); gy3 = fmaf(q, G32_0, gy3);
        gw0 = fmaf(X10_0_a, u, gw0); gx10_0 = fmaf(W15_0_a, u, gx10_0);
      }
      { const float q = W15_0_a * X11_0_a; float u = 0.f;
        u = fmaf(Y1_a, G33_0, u); gy1 = fmaf(q, G33_0, gy1);
        u = fmaf(Y2_a, G34_0, u); gy2 = fmaf(q, G34_0, gy2);
        u = fmaf(Y3_a, G35_0, u); gy3 = fmaf(q, G35_0, gy3);
        gw0 = fmaf(X11_0_a, u, gw0); gx11_0 = fmaf(W15_0_a, u, gx11_0);
      }
      { const float q = W15_0_a * X12_0_a; float u = 0.f;
        u = fmaf(Y1_a, G36_0, u); gy1 = fmaf(q, G36_0, gy1);
        u = fmaf(Y2_a, G37_0, u); gy2 = fmaf(q, G37_0, gy2);
        u = fmaf(Y3_a, G38_0, u); gy3 = fmaf(q, G38_0, gy3);
        gw0 = fmaf(X12_0_a, u, gw0); gx12_0 = fmaf(W15_0_a, u, gx12_0);
      }
      { const float q = W15_0_a * X13_0_a; float u = 0.f;
        u = fmaf(Y1_a, G39_0, u); gy1 = fmaf(q, G39_0, gy1);
        u = fmaf(Y2_a, G40_0, u); gy2 = fmaf(q, G40_0, gy2);
        u = fmaf(Y3_a, G41_0, u); gy3 = fmaf(q, G41_0, gy3);
        gw0 = fmaf(X13_0_a, u, gw0); gx13_0 = fmaf(W15_0_a, u, gx13_0);
      }
      { const float q = W15_0_a * X14_0_a; float u = 0.f;
        u = fmaf(Y1_a, G42_0, u); gy1 = fmaf(q, G42_0, gy1);
        u = fmaf(Y2_a, G43_0, u); gy2 = fmaf(q, G43_0, gy2);
        u = fmaf(Y3_a, G44_0, u); gy3 = fmaf(q, G44_0, gy3);
        gw0 = fmaf(X14_0_a, u, gw0); gx14_0 = fmaf(W15_0_a, u, gx14_0);
      }
      { const float q = W15_0_a * X15_0_a; float u = 0.f;
        u = fmaf(Y1_a, G45_0, u); gy1 = fmaf(q, G45_0, gy1);
        u = fmaf(Y3_a, G46_0, u); gy3 = fmaf(q, G46_0, gy3);
        gw0 = fmaf(X15_0_a, u, gw0); gx15_0 = fmaf(W15_0_a, u, gx15_0);
      }
      if (gwp) gwp[1920] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W16_0_a * X9_0_a; float u = 0.f;
        u = fmaf(Y9_a, G47_0, u); gy9 = fmaf(q, G47_0, gy9);
        u = fmaf(Y10_a, G48_0, u); gy10 = fmaf(q, G48_0, gy10);
        u = fmaf(Y11_a, G49_0, u); gy11 = fmaf(q, G49_0, gy11);
        u = fmaf(Y13_a, G50_0, u); gy13 = fmaf(q, G50_0, gy13);
        u = fmaf(Y14_a, G51_0, u); gy14 = fmaf(q, G51_0, gy14);
        gw0 = fmaf(X9_0_a, u, gw0); gx9_0 = fmaf(W16_0_a, u, gx9_0);
      }
      { const float q = W16_0_a * X10_0_a; float u = 0.f;
        u = fmaf(Y9_a, G52_0, u); gy9 = fmaf(q, G52_0, gy9);
        u = fmaf(Y11_a, G53_0, u); gy11 = fmaf(q, G53_0, gy11);
        u = fmaf(Y12_a, G54_0, u); gy12 = fmaf(q, G54_0, gy12);
        u = fmaf(Y13_a, G55_0, u); gy13 = fmaf(q, G55_0, gy13);
        u = fmaf(Y15_a, G56_0, u); gy15 = fmaf(q, G56_0, gy15);
        gw0 = fmaf(X10_0_a, u, gw0); gx10_0 = fmaf(W16_0_a, u, gx10_0);
      }
      { const float q = W16_0_a * X11_0_a; float u = 0.f;
        u = fmaf(Y9_a, G57_0, u); gy9 = fmaf(q, G57_0, gy9);
        u = fmaf(Y10_a, G58_0, u); gy10 = fmaf(q, G58_0, gy10);
        u = fmaf(Y11_a, G59_0, u); gy11 = fmaf(q, G59_0, gy11);
        u = fmaf(Y12_a, G60_0, u); gy12 = fmaf(q, G60_0, gy12);
        u = fmaf(Y13_a, G61_0, u); gy13 = fmaf(q, G61_0, gy13);
        u = fmaf(Y14_a, G62_0, u); gy14 = fmaf(q, G62_0, gy14);
        u = fmaf(Y15_a, G63_0, u); gy15 = fmaf(q, G63_0, gy15);
        gw0 = fmaf(X11_0_a, u, gw0); gx11_0 = fmaf(W16_0_a, u, gx11_0);
      }
      { const float q = W16_0_a * X12_0_a; float u = 0.f;
        u = fmaf(Y10_a, G64_0, u); gy10 = fmaf(q, G64_0, gy10);
        u = fmaf(Y11_a, G65_0, u); gy11 = fmaf(q, G65_0, gy11);
        u = fmaf(Y12_a, G66_0, u); gy12 = fmaf(q, G66_0, gy12);
        u = fmaf(Y13_a, G67_0, u); gy13 = fmaf(q, G67_0, gy13);
        u = fmaf(Y14_a, G68_0, u); gy14 = fmaf(q, G68_0, gy14);
        gw0 = fmaf(X12_0_a, u, gw0); gx12_0 = fmaf(W16_0_a, u, gx12_0);
      }
      { const float q = W16_0_a * X13_0_a; float u = 0.f;
        u = fmaf(Y9_a, G69_0, u); gy9 = fmaf(q, G69_0, gy9);
        u = fmaf(Y10_a, G70_0, u); gy10 = fmaf(q, G70_0, gy10);
        u = fmaf(Y11_a, G71_0, u); gy11 = fmaf(q, G71_0, gy11);
        u = fmaf(Y12_a, G72_0, u); gy12 = fmaf(q, G72_0, gy12);
        u = fmaf(Y13_a, G73_0, u); gy13 = fmaf(q, G73_0, gy13);
        u = fmaf(Y14_a, G74_0, u); gy14 = fmaf(q, G74_0, gy14);
        u = fmaf(Y15_a, G75_0, u); gy15 = fmaf(q, G75_0, gy15);
        gw0 = fmaf(X13_0_a, u, gw0); gx13_0 = fmaf(W16_0_a, u, gx13_0);
      }
      { const float q = W16_0_a * X14_0_a; float u = 0.f;
        u = fmaf(Y9_a, G76_0, u); gy9 = fmaf(q, G76_0, gy9);
        u = fmaf(Y11_a, G77_0, u); gy11 = fmaf(q, G77_0, gy11);
        u = fmaf(Y12_a, G78_0, u); gy12 = fmaf(q, G78_0, gy12);
        u = fmaf(Y13_a, G79_0, u); gy13 = fmaf(q, G79_0, gy13);
        u = fmaf(Y15_a, G80_0, u); gy15 = fmaf(q, G80_0, gy15);
        gw0 = fmaf(X14_0_a, u, gw0); gx14_0 = fmaf(W16_0_a, u, gx14_0);
      }
      { const float q = W16_0_a * X15_0_a; float u = 0.f;
        u = fmaf(Y10_a, G81_0, u); gy10 = fmaf(q, G81_0, gy10);
        u = fmaf(Y11_a, G82_0, u); gy11 = fmaf(q, G82_0, gy11);
        u = fmaf(Y13_a, G83_0, u); gy13 = fmaf(q, G83_0, gy13);
        u = fmaf(Y14_a, G84_0, u); gy14 = fmaf(q, G84_0, gy14);
        u = fmaf(Y15_a, G85_0, u); gy15 = fmaf(q, G85_0, gy15);
        gw0 = fmaf(X15_0_a, u, gw0); gx15_0 = fmaf(W16_0_a, u, gx15_0);
      }
      if (gwp) gwp[2048] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W21_0_a * X9_0_a; float u = 0.f;
        u = fmaf(Y0_a, G86_0, u); gy0 = fmaf(q, G86_0, gy0);
        gw0 = fmaf(X9_0_a, u, gw0); gx9_0 = fmaf(W21_0_a, u, gx9_0);
      }
      { const float q = W21_0_a * X10_0_a; float u = 0.f;
        u = fmaf(Y0_a, G87_0, u); gy0 = fmaf(q, G87_0, gy0);
        gw0 = fmaf(X10_0_a, u, gw0); gx10_0 = fmaf(W21_0_a, u, gx10_0);
      }
      { const float q = W21_0_a * X11_0_a; float u = 0.f;
        u = fmaf(Y0_a, G88_0, u); gy0 = fmaf(q, G88_0, gy0);
        gw0 = fmaf(X11_0_a, u, gw0); gx11_0 = fmaf(W21_0_a, u, gx11_0);
      }
      { const float q = W21_0_a * X12_0_a; float u = 0.f;
        u = fmaf(Y0_a, G89_0, u); gy0 = fmaf(q, G89_0, gy0);
        gw0 = fmaf(X12_0_a, u, gw0); gx12_0 = fmaf(W21_0_a, u, gx12_0);
      }
      { const float q = W21_0_a * X13_0_a; float u = 0.f;
        u = fmaf(Y0_a, G90_0, u); gy0 = fmaf(q, G90_0, gy0);
        gw0 = fmaf(X13_0_a, u, gw0); gx13_0 = fmaf(W21_0_a, u, gx13_0);
      }
      { const float q = W21_0_a * X14_0_a; float u = 0.f;
        u = fmaf(Y0_a, G91_0, u); gy0 = fmaf(q, G91_0, gy0);
        gw0 = fmaf(X14_0_a, u, gw0); gx14_0 = fmaf(W21_0_a, u, gx14_0);
      }
      { const float q = W21_0_a * X15_0_a; float u = 0.f;
        u = fmaf(Y0_a, G92_0, u); gy0 = fmaf(q, G92_0, gy0);
        gw0 = fmaf(X15_0_a, u, gw0); gx15_0 = fmaf(W21_0_a, u, gx15_0);
      }
      if (gwp) gwp[2688] = gw0;
    }
    {
      float gw0 = 0.f;
      { const float q = W22_0_a * X9_0_a; float u = 0.f;
        u = fmaf(Y4_a, G93_0, u); gy4 = fmaf(q, G93_0, gy4);
        u = fmaf(Y5_a, G94_0, u); gy5 = fmaf(q, G94_0, gy5);
        u = fmaf(Y6_a, G95_0, u); gy6 = fmaf(q, G95_0, gy6);
        u = fmaf(Y7_a, G96_0, u); gy7 = fmaf(q, G96_0, gy7);
        u = fmaf(Y8_a, G97_0, u); gy8 = fmaf(q, G97_0, gy8);
        gw0 = fmaf(X9_0_a, u, gw0); gx9_0 = fmaf(W22_0_a, u, gx9_0);
      }
      { const float q = W22_0_a * X10_0_a; float u = 0.f;
        u = fmaf(Y4_a, G98_0, u); gy4 = fmaf(q, G98_0, gy4);
        u = fmaf(Y5_a, G99_0, u); gy5 = fmaf(q, G99_0, gy5);
        u = fmaf(Y7_a, G100_0, u); gy7 = fmaf(q, G100_0, gy7);
        gw0 = fmaf(X10_0_a, u, gw0); gx10_0 = fmaf(W22_0_a, u, gx10_0);
      }
      { const float q = W22_0_a * X11_0_a; float u = 0.f;
        u = fmaf(Y4_a, G101_0, u); gy4 = fmaf(q, G101_0, gy4);
        u = fmaf(Y5_a, G102_0, u); gy5 = fmaf(q, G102_0, gy5);
        u = fmaf(Y6_a, G103_0, u); gy6 = fmaf(q, G103_0, gy6);
        u = fmaf(Y7_a, G104_0, u); gy7 = fmaf(q, G104_0, gy7);
        u = fmaf(Y8_a, G105_0, u); gy8 = fmaf(q, G105_0, gy8);
        gw0 = fmaf(X11_0_a, u, gw0); gx11_0 = fmaf(W22_0_a, u, gx11_0);
      }
      { const float q = W22_0_a * X12_0_a; float u = 0.f;
        u = fmaf(Y4_a, G106_0, u); gy4 = fmaf(q, G106_0, gy4);
        u = fmaf(Y5_a, G107_0, u); gy5 = fmaf(q, G107_0, gy5);
        u = fmaf(Y6_a, G108_0, u); gy6 = fmaf(q, G108_0, gy6);
        u = fmaf(Y7_a, G109_0, u); gy7 = fmaf(q, G109_0, gy7);
        u = fmaf(Y8_a, G110_0, u); gy8 = fmaf(q, G110_0, gy8);
        gw0 = fmaf(X12_0_a, u, gw0); gx12_0 = fmaf(W22_0_a, u, gx12_0);
      }
      { const float q = W22_0_a * X13_0_a; float u = 0.f;
        u = fmaf(Y4_a, G111_0, u); gy4 = fmaf(q, G111_0, gy4);
        u = fmaf(Y5_a, G112_0, u); gy5 = fmaf(q, G112_0, gy5);
        u = fmaf(Y6_a, G113_0, u); gy6 = fmaf(q, G113_0, gy6);
        u = fmaf(Y7_a, G114_0, u); gy7 = fmaf(q, G114_0, gy7);
        u = fmaf(Y8_a, G115_0, u); gy8 = fmaf(q, G115_0, gy8);
        gw0 = fmaf(X13_0_a, u, gw0); gx13_0 = fmaf(W22_0_a, u, gx13_0);
      }
      { const float q = W22_0_a * X14_0_a; float u = 0.f;
        u = fmaf(Y5_a, G116_0, u); gy5 = fmaf(q, G116_0, gy5);
        u = fmaf(Y7_a, G117_0, u); gy7 = fmaf(q, G117_0, gy7);
        u = fmaf(Y8_a, G118_0, u); gy8 = fmaf(q, G118_0, gy8);
        gw0 = fmaf(X14_0_a, u, gw0); gx14_0 = fmaf(W22_0_a, u, gx14_0);
      }
      { const float q = W22_0_a * X15_0_a; float u = 0.f;
        u = fmaf(Y4_a, G119_0, u); gy4 = fmaf(q, G119_0, gy4);
        u = fmaf(Y5_a, G120_0, u); gy5 = fmaf(q, G120_0, gy5);
        u = fmaf(Y6_a, G121_0, u); gy6 = fmaf(q, G121_0, gy6);
        u = fmaf(Y7_a, G122_0, u); gy7 = fmaf(q, G122_0, gy7);
        u = fmaf(Y8_a, G123_0, u); gy8 = fmaf(q, G123_0, gy8);
        gw0 = fmaf(X15_0_a, u, gw0); gx15_0 = fmaf(W22_0_a, u, gx15_0);
      }
      if (gwp) gwp[2816] = gw0;
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
      atomicAdd(gxp + 1152, gx9_0);
      atomicAdd(gxp + 1280, gx10_0);
      atomicAdd(gxp + 1408, gx11_0);
      atomicAdd(gxp + 1536, gx12_0);
      atomicAdd(gxp + 1664, gx13_0);
      atomicAdd(gxp + 1792, gx14_0);
      atomicAdd(gxp + 1920, gx15_0);
    }
  }
  }
}

extern "C" int mm_tpw_l0123_fwd_n(long E, const int* rowptr, int nR, const int* eid, const int* send, const float* Y,
    long y_stride, const float* W, long w_stride, const float* X, long x_stride, float* out, long out_stride,
    hipStream_t stream) {
  MM_CHECK_ARG(nR >= 0, "bad sizes");
  MM_CHECK_ARG(y_stride >= 16 && w_stride >= 2944 && x_stride >= 2048 && out_stride >= 12672,
               "row strides smaller than the path table's widths");
  if (nR == 0) return MM_OK;
  const long waves = (long)nR * 2;
  // E < 0: unknown, shared where the receivers alone leave most of the chip idle
  // (a launch takes fewer than 2^32 threads)
  const bool shared = E < 0 ? waves <= 2048 : true && waves < (1L << 24) && E >= 18L * nR;
  dim3 grid((unsigned)(shared ? waves : (waves + 3) / 4)), block(256);
  hipLaunchKernelGGL(shared ? mm_tpw_l0123_fwd_shared_kernel : mm_tpw_l0123_fwd_kernel, grid, block, 0, stream, rowptr, nR, eid, send, Y, y_stride, W,
                     w_stride, X, x_stride, out, out_stride);
  return mm::launch_status("mm_tpw_l0123_fwd");
}

extern "C" int mm_tpw_l0123_fwd(const int* rowptr, int nR, const int* eid, const int* send, const float* Y,
    long y_stride, const float* W, long w_stride, const float* X, long x_stride,
    float* out, long out_stride, hipStream_t stream) {
  return mm_tpw_l0123_fwd_n(-1, rowptr, nR, eid, send, Y, y_stride, W, w_stride, X, x_stride, out, out_stride, stream);
}

extern "C" int mm_tpw_l0123_bwd_n(long E, const int* rowptr, int nR, const int* eid, const int* send, const float* Y,
    long y_stride, const float* W, long w_stride, const float* X, long x_stride, const float* gO, long g_stride,
    float* gW, long gw_stride, float* gYp, long gy_cb_stride, float* gX, long gx_stride, hipStream_t stream) {
  MM_CHECK_ARG(nR >= 0, "bad sizes");
  MM_CHECK_ARG(y_stride >= 16 && w_stride >= 2944 && x_stride >= 2048 && g_stride >= 12672,
               "row strides smaller than the path table's widths");
  MM_CHECK_ARG(!gW || gw_stride >= 2944, "gW row stride");
  MM_CHECK_ARG(!gX || gx_stride >= 2048, "gX row stride");
  if (nR == 0) return MM_OK;
  const long waves = (long)nR * 6;
  // E < 0: unknown, shared where the receivers alone leave most of the chip idle
  // (a launch takes fewer than 2^32 threads)
  const bool shared = E < 0 ? waves <= 2048 : waves <= 8192 && waves < (1L << 24) && E >= 18L * nR;
  dim3 grid((unsigned)(shared ? waves : (waves + 3) / 4)), block(256);
  hipLaunchKernelGGL(shared ? mm_tpw_l0123_bwd_shared_kernel : mm_tpw_l0123_bwd_kernel, grid, block, 0, stream, rowptr, nR, eid, send, Y, y_stride, W,
                     w_stride, X, x_stride, gO, g_stride, gW, gw_stride, gYp, gy_cb_stride, gX, gx_stride);
  return mm::launch_status("mm_tpw_l0123_bwd");
}

extern "C" int mm_tpw_l0123_bwd(const int* rowptr, int nR, const int* eid, const int* send, const float* Y,
    long y_stride, const float* W, long w_stride, const float* X, long x_stride,
    const float* gO, long g_stride, float* gW, long gw_stride, float* gYp, long gy_cb_stride, float* gX,
    long gx_stride, hipStream_t stream) {
  return mm_tpw_l0123_bwd_n(-1, rowptr, nR, eid, send, Y, y_stride, W, w_stride, X, x_stride, gO, g_stride, gW, gw_stride, gYp, gy_cb_stride, gX, gx_stride, stream);
}
