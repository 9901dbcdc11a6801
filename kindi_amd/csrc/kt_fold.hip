/* kt_fold.hip - the producers of a product's input, fused with its int8 quantization (k_rmsfold_qT, k_fold_fwht_qT,
   k_smfold_qT tcf.cu:370-426; their numbers are those of k_rmsfold kindi.cu:350-394 and ff_* tcf.cu:218-312).

   Few tokens (k_fold_q8; many: k_fold_many, below): one block of 512 threads per token row and HB block (NM = HB / 512), so
   a row's work is spread over C / HB blocks (the reference's grid): thread j holds columns c0 + j + 512 k in v[k], and every
   output of the chunk is made in the block. rmsfold's blocks each read the whole row (NF = C / 512 registers) for the
   norm, in the reference's order, as every block of the reference does:
     MODE 0 (rmsfold): xf = x + (r_0 + ... + r_{n-1}) (parts in order), s = 1 / sqrt((float)(S / C) + 1e-6) with S
                       the double sum of squares, xn = (xf s) w, v = sg xn;
     MODE 1 (fold):    v = sg x;
     MODE 2 (smfold):  v = sg[e] (SiLU(a) b) at the permuted source column of e;
   then the unnormalised Walsh-Hadamard transform of each HB-column block, the 1/sqrt(HB) scale (xo), and the int8 row
   per 128-column group with k_tc_q8's numbers (natural column order, XS/XA [M][C/128] as kt_quant_q8 writes them).

   Bit-exact with the reference:
   - S is summed in the reference's order: thread j over k in order; each 32-lane half of a wave by the xor butterfly
     16, 8, 4, 2, 1 (the reference's warp); the 16 half-wave sums by the same butterfly (its warp 0 with lanes 16 ..
     31 zero), which every thread evaluates from LDS. sqrt and the division are the correctly rounded fp32 ones, as the
     reference's IEEE sqrtf and division.
   - The transform's butterflies are the reference's pairs in the reference's stage order: stages 1 .. 32 between
     lanes of a wave; stages 64, 128, 256 (between the 8 waves) as one LDS exchange after which each thread runs the
     8-point transform of its column's 8 values (the same additions in the same order) and keeps its own output;
     stages 512 and up between the registers of one HB block. */
#include "kt_gemv.h"
#include "kt_fold.h"
#include "kt_launch.h"

/* one butterfly stage between lanes l and l ^ X: the lower lane keeps a + b, the upper a - b, as (-b) + a: negation
   is exact and the sum is the same rounded value. neg = the sign bit on lanes with bit X set. */
template <int X> __device__ __forceinline__ float kf_bfly(float v, unsigned neg){
  return __int_as_float(__float_as_int(v) ^ neg) + kf_xorf<X>(v);
}
/* 1 / sqrt(S / C + 1e-6) of a row: S from the 512 threads' sums in the reference's order (each 32-lane half by the xor
   butterfly, the 16 half-wave sums by the same one, evaluated by every thread) */
__device__ __forceinline__ float kf_norm(double acc, double* red, int j, int C){
  acc += kf_xord<16>(acc);
  acc += kf_xord<8>(acc);
  acc += kf_xord<4>(acc);
  acc += kf_xord<2>(acc);
  acc += kf_xord<1>(acc);
  if((j & 31) == 0) red[j >> 5] = acc;
  __syncthreads();
  double t[8];
#pragma unroll
  for(int i = 0; i < 8; ++i) t[i] = red[i] + red[i + 8];           /* offset 8 (offset 16 added zeros) */
#pragma unroll
  for(int i = 0; i < 4; ++i) t[i] = t[i] + t[i + 4];
  t[0] = t[0] + t[2];
  t[1] = t[1] + t[3];
  const double S = t[0] + t[1];
  const float ms = (float)(S / (double)C) + 1e-6f;
  return 1.0f / sqrtf(ms);                                         /* both correctly rounded */
}

template <int NM>
__device__ __forceinline__ void kf_fwht(float* v, float* sm, int j, int HB){
  const int l = j & 63;
#define KF_STAGE(X) { const unsigned ng = (l & X) ? 0x80000000u : 0u; \
    _Pragma("unroll") for(int k = 0; k < NM; ++k) v[k] = kf_bfly<X>(v[k], ng); }
  KF_STAGE(1) KF_STAGE(2) KF_STAGE(4) KF_STAGE(8) KF_STAGE(16) KF_STAGE(32)
#undef KF_STAGE
#pragma unroll
  for(int k = 0; k < NM; ++k) sm[k * 512 + j] = v[k];
  __syncthreads();
  /* stages 64, 128, 256 for this thread's column only: with A_t = the column's value in wave w ^ t,
     s1_t = stage 64 at wave w ^ t (t even), s2_t = stage 128 at w ^ t (t = 0, 4), then stage 256 at w; each is the
     reference's a + b or a - b of the same pair (the lower wave of a pair adds) */
  const int w = __builtin_amdgcn_readfirstlane(j >> 6);
#pragma unroll
  for(int k = 0; k < NM; ++k){
    float A[8];
#pragma unroll
    for(int t = 0; t < 8; ++t) A[t] = sm[k * 512 + l + 64 * (w ^ t)];
    float s1[8], s2[8];
#pragma unroll
    for(int t = 0; t < 8; t += 2) s1[t] = (w & 1) ? (A[t ^ 1] - A[t]) : (A[t] + A[t ^ 1]);
#pragma unroll
    for(int t = 0; t < 8; t += 4) s2[t] = (w & 2) ? (s1[t ^ 2] - s1[t]) : (s1[t] + s1[t ^ 2]);
    v[k] = (w & 4) ? (s2[4] - s2[0]) : (s2[0] + s2[4]);
  }
  const int hbe = HB >> 9;                                     /* registers a Hadamard block */
#pragma unroll
  for(int h = 1; h < 16; h <<= 1){
    if(h < hbe){
#pragma unroll
      for(int k = 0; k < NM; ++k)
        if(!(k & h) && k + h < NM){ const float a = v[k], b = v[k + h]; v[k] = a + b; v[k + h] = a - b; }
    }
  }
}

template <int MODE, int NM, int NF>
__global__ void __launch_bounds__(512) k_fold_q8(const KtFoldArgs a){
  __shared__ float sm[NM * 512];
  __shared__ double red[16];
  __shared__ float qm[NM * 8];
  __shared__ int qs[NM * 8], qs2[NM * 8];
  const int j = threadIdx.x, n = blockIdx.y, lane = j & 63, w = j >> 6, C = NM * 512, c0 = blockIdx.x * C;
  float v[NM];
  if(MODE == 0){
    const float* x = a.x + (long long)n * a.ldx;
    constexpr int CF = NF * 512;                                   /* the row */
    float xf[NF], wv[NM], sv[NM];
#pragma unroll
    for(int m = 0; m < NF; ++m) xf[m] = x[j + 512 * m];
#pragma unroll
    for(int k = 0; k < NM; ++k){ wv[k] = a.w[c0 + j + 512 * k]; sv[k] = a.sg[c0 + j + 512 * k]; }
    if(a.nparts > 0){
      const float* r = a.r + (long long)n * a.ldr;
      float rv[NF];
#pragma unroll
      for(int m = 0; m < NF; ++m) rv[m] = r[j + 512 * m];
      for(int p = 1; p < a.nparts; ++p){
#pragma unroll
        for(int m = 0; m < NF; ++m) rv[m] += r[(long long)p * CF + j + 512 * m];
      }
#pragma unroll
      for(int m = 0; m < NF; ++m) xf[m] = xf[m] + rv[m];
    }
    double acc = 0.0;
#pragma unroll
    for(int m = 0; m < NF; ++m){ const double d = (double)xf[m]; acc += d * d; }
    const float s = kf_norm(acc, red, j, CF);
    float* xw = a.xw ? a.xw + (long long)n * a.ldxw : nullptr;
    float* xn = a.xn ? a.xn + (long long)n * a.ldxn : nullptr;
    const int b0 = blockIdx.x * NM;                                /* the chunk's first register of the row */
#pragma unroll
    for(int k = 0; k < NM; ++k){
      const int e = c0 + j + 512 * k;
      float f = xf[k];
#pragma unroll
      for(int m = 0; m < NF; ++m) if(m != k && m == b0 + k) f = xf[m];
      const float nv = (f * s) * wv[k];
      if(xw && a.nparts > 0) xw[e] = f;
      if(xn) xn[e] = nv;
      v[k] = sv[k] * nv;
    }
  } else if(MODE == 1){
    const float* x = a.x + (long long)n * a.ldx;
#pragma unroll
    for(int k = 0; k < NM; ++k) v[k] = a.sg[c0 + j + 512 * k] * x[c0 + j + 512 * k];
  } else {
    const float* pa = a.x + (long long)n * a.ldx;
    const float* pb = a.r + (long long)n * a.ldr;
#pragma unroll
    for(int k = 0; k < NM; ++k){
      const int e = c0 + j + 512 * k;
      int src = e;
      if(a.rep > 1){
        const int h = e % a.hd, g = e / a.hd, rp = g % a.rep, kk = g / a.rep;
        src = h + a.hd * (kk + a.nk * rp);
      }
      const float xa = pa[src];
      const float m = (xa / (1.0f + expf(-xa))) * pb[src];
      v[k] = a.sg[e] * m;
    }
  }
  kf_fwht<NM>(v, sm, j, a.HB);
  const float sc = a.HB == 512 ? 0.044194173824159220878f : (a.HB == 1024 ? 0.03125f : 0.015625f);
  float* xo = a.xo ? a.xo + (long long)n * a.ldxo : nullptr;
#pragma unroll
  for(int k = 0; k < NM; ++k){
    v[k] = v[k] * sc;
    if(xo) xo[c0 + j + 512 * k] = v[k];
  }
  /* group 4 k + w / 2 = waves 2i, 2i + 1 of register k */
#pragma unroll
  for(int k = 0; k < NM; ++k){
    const float m = kf_wave_max(fabsf(v[k]));
    if(lane == 0) qm[k * 8 + w] = m;
  }
  __syncthreads();
  /* hp: rows 2n (the int8 row) and 2n + 1 (the residual r = v - q (amax / 127), one fma as the reference's compiler
     contracts it, at the fixed scale amax / 32258: q2 = clamp(rne(r (32258 / amax)), -127, 127); ff_q8 tcf.cu:150-205) */
  const long long n0 = a.hp ? 2 * n : n;
  int8_t* Q = a.Q + n0 * a.ldq;
  const int NG = a.C >> 7;
#pragma unroll
  for(int k = 0; k < NM; ++k){
    const float amax = fmaxf(qm[k * 8 + (w & ~1)], qm[k * 8 + (w | 1)]);
    const float id = amax != 0.0f ? 127.0f / amax : 0.0f;
    const int qi = __float2int_rn(v[k] * id);
    Q[c0 + j + 512 * k] = (int8_t)qi;
    const int sum = kf_wave_sum(qi);
    if(lane == 0) qs[k * 8 + w] = sum;
    if(a.hp){                                                    /* block-uniform */
      const float r = fmaf(-(float)qi, amax / 127.0f, v[k]);
      const int q2 = max(-127, min(127, __float2int_rn(r * (amax != 0.0f ? 32258.0f / amax : 0.0f))));
      Q[a.ldq + c0 + j + 512 * k] = (int8_t)q2;
      const int sum2 = kf_wave_sum(q2);
      if(lane == 0) qs2[k * 8 + w] = sum2;
    }
  }
  __syncthreads();
  if(lane == 0 && !(w & 1)){
#pragma unroll
    for(int k = 0; k < NM; ++k){
      const int g = (c0 >> 7) + 4 * k + (w >> 1);
      const float amax = fmaxf(qm[k * 8 + w], qm[k * 8 + w + 1]);
      a.XS[n0 * NG + g] = amax / 127.0f;
      a.XA[n0 * NG + g] = qs[k * 8 + w] + qs[k * 8 + w + 1];
      if(a.hp){
        a.XS[(n0 + 1) * NG + g] = amax / 32258.0f;
        a.XA[(n0 + 1) * NG + g] = qs2[k * 8 + w] + qs2[k * 8 + w + 1];
      }
    }
  }
}

/* ------------------------------------------------------------------ many tokens
   The same numbers with 8 consecutive columns a thread (512 a wave, up to 4096 a block): the transform's stages 1, 2, 4 are
   between a thread's registers, 8 .. 256 between lanes, 512 and up between the waves of an HB block (one LDS exchange), each
   the same pairs in the same stage order; a 128-column group is 16 lanes, so its maximum and sum take 4 lane steps for 8
   columns (6 for one in the kernel above), its divisions are made once for 8, and rows are read and written 16 bytes a lane
   where their addresses allow (vec). rmsfold: one block a row; the norm's sum is taken first in the reference's order
   (thread j over columns j + 512 m), the row kept in LDS.
   MI355X, 1000 tokens, against the kernel above on chunks of up to 8192 columns (rmsfold: the row): smfold of 12288 columns, HB
   4096, 45.1 -> 29.0 us, rmsfold of 4096 with one part and xw 21.3 -> 15.1, of 5120 at 33 / 256 tokens 10.2 / 11.3 -> 7.0 / 8.0.
   waves_per_eu holds the registers to three blocks a CU (80): rmsfold 57.8 against 66.5 us at 4096 tokens of 8192 columns (88 and
   two blocks without), smfold 51.3 against 56.5 at 2048 of 12288 (82 and two), 9.6 against 10.9 at 2048 of 1024 in HB 512. */
#define KF_VX 1                       /* x / r rows, sg and w in 16-byte loads */
#define KF_VO 2                       /* xw, xn, xo in 16-byte stores */
#define KF_VQ 4                       /* the int8 rows in 8-byte stores */
#define KF_ROW 8                      /* smfold: a block a row, its inputs taken into LDS before an output is written */
__device__ __forceinline__ void kf_ld8(float* v, const float* p, bool vec){
  if(vec){
    const float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else
#pragma unroll
    for(int i = 0; i < 8; ++i) v[i] = p[i];
}
/* a wave's 512 columns (lane l: 8 l .. + 7) to p, through t, 512 floats of LDS of the wave's own, so that a store's lanes are
   neighbours. Straight from the lanes a 16-byte store leaves every other 16 bytes of its lines to the next one: MI355X,
   rmsfold of 4096 columns with xw, xn and xo at 1000 / 4096 tokens 37.5 / 142 us that way, 18.6 / 70 so; smfold of 12288 with
   xo 50.4 / 212 against 32.9 / 148 (at two blocks a CU). kf_out: columns that t already holds */
__device__ __forceinline__ void kf_put8(float* t, const float* v, int l){
  *(float4*)(t + 8 * l) = make_float4(v[0], v[1], v[2], v[3]);
  *(float4*)(t + 8 * l + 4) = make_float4(v[4], v[5], v[6], v[7]);
}
__device__ __forceinline__ void kf_out(float* p, const float* t, int l, bool vec){
  if(vec){
#pragma unroll
    for(int i = 0; i < 2; ++i) *(float4*)(p + 256 * i + 4 * l) = *(const float4*)(t + 256 * i + 4 * l);
  } else
#pragma unroll
    for(int i = 0; i < 8; ++i) p[64 * i + l] = t[64 * i + l];
}
__device__ __forceinline__ void kf_st8(float* p, float* t, const float* v, int l, bool vec){
  kt_wave_sync();                                                  /* t's earlier columns are read */
  kf_put8(t, v, l);
  kt_wave_sync();
  kf_out(p, t, l, vec);
  kt_wave_sync();
}
__device__ __forceinline__ void kf_stq(int8_t* p, const int* q, bool vec){
  if(vec){
    uint2 o;
    o.x = (q[0] & 255) | (q[1] & 255) << 8 | (q[2] & 255) << 16 | (unsigned)q[3] << 24;
    o.y = (q[4] & 255) | (q[5] & 255) << 8 | (q[6] & 255) << 16 | (unsigned)q[7] << 24;
    *(uint2*)p = o;
  } else
#pragma unroll
    for(int i = 0; i < 8; ++i) p[i] = (int8_t)q[i];
}

template <int MODE>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(MODE == 1 ? 2 : 6))) k_fold_many(const KtFoldArgs a, int vec){
  extern __shared__ __attribute__((aligned(16))) float kf_lds[];    /* [8][2][64][4] exchange (2 KB a wave), then the row */
  __shared__ double red[16];
  float4* ex = (float4*)kf_lds;
  float* rowb = kf_lds + 4096;
  const int j = threadIdx.x, n = blockIdx.y, l = j & 63, C = a.C, nw = a.HB >> 9;    /* nw waves an HB block: 1, 2, 8 */
  const int w = __builtin_amdgcn_readfirstlane(j >> 6);
  const bool vx = vec & KF_VX, vo = vec & KF_VO, vq = vec & KF_VQ;
  float* tw = kf_lds + 512 * w;                                     /* this wave's part of the exchange */
  float s = 1.0f;
  if(MODE == 0){
    const float* x = a.x + (long long)n * a.ldx;
    const float* r = a.r + (long long)n * a.ldr;
    double acc = 0.0;
    for(int m0 = 0; m0 < C; m0 += 4096){                           /* 8 columns' loads together */
      float f[8];
#pragma unroll
      for(int m = 0; m < 8; ++m) f[m] = m0 + 512 * m < C ? x[m0 + 512 * m + j] : 0.0f;
      if(a.nparts > 0){
        float rv[8];
#pragma unroll
        for(int m = 0; m < 8; ++m) rv[m] = m0 + 512 * m < C ? r[m0 + 512 * m + j] : 0.0f;
        for(int p = 1; p < a.nparts; ++p)
#pragma unroll
          for(int m = 0; m < 8; ++m) if(m0 + 512 * m < C) rv[m] += r[(long long)p * C + m0 + 512 * m + j];
#pragma unroll
        for(int m = 0; m < 8; ++m) f[m] = f[m] + rv[m];
      }
#pragma unroll
      for(int m = 0; m < 8; ++m)
        if(m0 + 512 * m < C){                                      /* uniform */
          const double d = (double)f[m];
          acc += d * d;
          rowb[m0 + 512 * m + j] = f[m];
        }
    }
    s = kf_norm(acc, red, j, C);                                   /* its barrier covers the row too */
  }
  /* smfold's product for columns c .. c + 7; ld: loads to issue before its own, but behind single ones (registers) */
  auto silu = [&](int c, float* f, auto&& ld){
    const float* pa = a.x + (long long)n * a.ldx;
    const float* pb = a.r + (long long)n * a.ldr;
    float fb[8];
    if(a.rep > 1){
      auto src = [&](int e){ const int h = e % a.hd, g = e / a.hd; return h + a.hd * (g / a.rep + a.nk * (g % a.rep)); };
      if(a.hd % 8 == 0){                                           /* uniform: the 8 columns stay neighbours */
        const int sc = src(c);
        ld();
        kf_ld8(f, pa + sc, vx);
        kf_ld8(fb, pb + sc, vx);
      } else {
#pragma unroll
        for(int i = 0; i < 8; ++i){ const int sc = src(c + i); f[i] = pa[sc]; fb[i] = pb[sc]; }
        ld();
      }
    } else { ld(); kf_ld8(f, pa + c, vx); kf_ld8(fb, pb + c, vx); }
#pragma unroll
    for(int i = 0; i < 8; ++i) f[i] = (f[i] / (1.0f + expf(-f[i]))) * fb[i];
  };
  const bool whole = MODE == 0 || (MODE == 2 && (vec & KF_ROW));   /* uniform */
  if(MODE == 2 && whole){
    for(int c = 512 * w + 8 * l; c < C; c += 4096){
      float f[8];
      silu(c, f, []{});
      kf_put8(rowb + c - 8 * l, f, l);
    }
    __syncthreads();
  }
  for(int c0 = whole ? 0 : blockIdx.x * 4096; c0 < (whole ? C : (int)blockIdx.x * 4096 + 1); c0 += 4096){
    const int cb = c0 + 512 * w, c = cb + 8 * l;                   /* the wave's columns (uniform), the lane's */
    const bool on = c0 + 512 * w < C;                              /* wave-uniform */
    float v[8];
#pragma unroll
    for(int i = 0; i < 8; ++i) v[i] = 0.0f;
    if(on){
      if(MODE == 0 && a.xw && a.nparts > 0){                       /* before the loads below: fewer registers at once */
        kf_out(a.xw + (long long)n * a.ldxw + cb, rowb + cb, l, vo);
        kt_wave_sync();
      }
      float sg[8];
      auto ld_sg = [&]{ kf_ld8(sg, a.sg + c, vx); };
      if(MODE != 2 || whole) ld_sg();
      if(MODE == 0){
        float f[8], wv[8];
        kf_ld8(f, rowb + c, true);
        kf_ld8(wv, a.w + c, vx);
#pragma unroll
        for(int i = 0; i < 8; ++i) f[i] = (f[i] * s) * wv[i];
        if(a.xn) kf_st8(a.xn + (long long)n * a.ldxn + cb, tw, f, l, vo);
#pragma unroll
        for(int i = 0; i < 8; ++i) v[i] = sg[i] * f[i];
      } else if(MODE == 1){
        float f[8];
        kf_ld8(f, a.x + (long long)n * a.ldx + c, vx);
#pragma unroll
        for(int i = 0; i < 8; ++i) v[i] = sg[i] * f[i];
      } else {
        float f[8];
        if(whole) kf_ld8(f, rowb + c, true);
        else silu(c, f, ld_sg);
#pragma unroll
        for(int i = 0; i < 8; ++i) v[i] = sg[i] * f[i];
      }
#pragma unroll
      for(int h = 1; h < 8; h <<= 1)
#pragma unroll
        for(int i = 0; i < 8; ++i)
          if(!(i & h)){ const float p = v[i], q = v[i + h]; v[i] = p + q; v[i + h] = p - q; }
#define KF_STAGE(X) { const unsigned ng = (l & X) ? 0x80000000u : 0u; \
      _Pragma("unroll") for(int i = 0; i < 8; ++i) v[i] = kf_bfly<X>(v[i], ng); }
      KF_STAGE(1) KF_STAGE(2) KF_STAGE(4) KF_STAGE(8) KF_STAGE(16) KF_STAGE(32)
#undef KF_STAGE
    }
    if(nw > 1){                                                    /* uniform */
      ex[w * 128 + l] = make_float4(v[0], v[1], v[2], v[3]);
      ex[w * 128 + 64 + l] = make_float4(v[4], v[5], v[6], v[7]);
      __syncthreads();
      if(on)
#pragma unroll
        for(int hf = 0; hf < 2; ++hf){
          float A[8][4];                                           /* the column's values in waves w ^ t */
#pragma unroll
          for(int t = 0; t < 8; ++t)
            if(t < 2 || nw > 2){
              const float4 f = ex[((w ^ t) & 7) * 128 + 64 * hf + l];
              A[t][0] = f.x; A[t][1] = f.y; A[t][2] = f.z; A[t][3] = f.w;
            }
#pragma unroll
          for(int i = 0; i < 4; ++i){
            float s1[8], s2[8];
            s1[0] = (w & 1) ? (A[1][i] - A[0][i]) : (A[0][i] + A[1][i]);
            if(nw > 2){
#pragma unroll
              for(int t = 2; t < 8; t += 2) s1[t] = (w & 1) ? (A[t ^ 1][i] - A[t][i]) : (A[t][i] + A[t ^ 1][i]);
#pragma unroll
              for(int t = 0; t < 8; t += 4) s2[t] = (w & 2) ? (s1[t ^ 2] - s1[t]) : (s1[t] + s1[t ^ 2]);
              v[4 * hf + i] = (w & 4) ? (s2[4] - s2[0]) : (s2[0] + s2[4]);
            } else v[4 * hf + i] = s1[0];
          }
        }
      __syncthreads();                                             /* the next chunk writes the exchange again */
    }
    if(on){
      const float sc = a.HB == 512 ? 0.044194173824159220878f : (a.HB == 1024 ? 0.03125f : 0.015625f);
      float m = 0.0f;
#pragma unroll
      for(int i = 0; i < 8; ++i){
        v[i] = v[i] * sc;
        m = i == 0 ? fabsf(v[0]) : fmaxf(m, fabsf(v[i]));
      }
      m = fmaxf(m, kf_xorf<1>(m)); m = fmaxf(m, kf_xorf<2>(m)); m = fmaxf(m, kf_xorf<4>(m)); m = fmaxf(m, kf_xorf<8>(m));
      const float id = m != 0.0f ? 127.0f / m : 0.0f, xs = m / 127.0f;
      const long long n0 = a.hp ? 2 * (long long)n : n;
      const int NG = C >> 7, g = c >> 7;
      int q[8], sum = 0;
#pragma unroll
      for(int i = 0; i < 8; ++i){ q[i] = __float2int_rn(v[i] * id); sum += q[i]; }
      kf_stq(a.Q + n0 * a.ldq + c, q, vq);
      sum += kf_xor<1>(sum); sum += kf_xor<2>(sum); sum += kf_xor<4>(sum); sum += kf_xor<8>(sum);
      if((l & 15) == 0){ a.XS[n0 * NG + g] = xs; a.XA[n0 * NG + g] = sum; }
      if(a.hp){                                                    /* uniform: the residual's row */
        const float i2 = m != 0.0f ? 32258.0f / m : 0.0f;
        int q2[8], sum2 = 0;
#pragma unroll
        for(int i = 0; i < 8; ++i){
          const float r = fmaf(-(float)q[i], xs, v[i]);
          q2[i] = max(-127, min(127, __float2int_rn(r * i2)));
          sum2 += q2[i];
        }
        kf_stq(a.Q + (n0 + 1) * a.ldq + c, q2, vq);
        sum2 += kf_xor<1>(sum2); sum2 += kf_xor<2>(sum2); sum2 += kf_xor<4>(sum2); sum2 += kf_xor<8>(sum2);
        if((l & 15) == 0){ a.XS[(n0 + 1) * NG + g] = m / 32258.0f; a.XA[(n0 + 1) * NG + g] = sum2; }
      }
      if(a.xo) kf_st8(a.xo + (long long)n * a.ldxo + cb, tw, v, l, vo);
    }
  }
}

/* few tokens, an HB block a chunk: rmsfold (chunk, row), fold / smfold the chunk */
#define KF_EACH_ROW(X) X(0, 1, 1) X(0, 1, 2) X(0, 1, 3) X(0, 1, 4) X(0, 1, 5) X(0, 1, 6) X(0, 1, 7) X(0, 1, 8) X(0, 1, 9) \
  X(0, 1, 10) X(0, 1, 11) X(0, 1, 12) X(0, 1, 13) X(0, 1, 14) X(0, 1, 15) X(0, 1, 16) X(0, 2, 2) X(0, 2, 4) X(0, 2, 6) \
  X(0, 2, 8) X(0, 2, 10) X(0, 2, 12) X(0, 2, 14) X(0, 2, 16) X(0, 8, 8) X(0, 8, 16) \
  X(1, 1, 1) X(1, 2, 2) X(1, 8, 8) X(2, 1, 1) X(2, 2, 2) X(2, 8, 8)
#define KF_INST(MODE, NM, NF) template __global__ void k_fold_q8<MODE, NM, NF>(const KtFoldArgs);
KF_EACH_ROW(KF_INST)
#undef KF_INST
template __global__ void k_fold_many<0>(const KtFoldArgs, int);
template __global__ void k_fold_many<1>(const KtFoldArgs, int);
template __global__ void k_fold_many<2>(const KtFoldArgs, int);

#define KF_KEY(MODE, NM, NF) ((MODE) * 1024 + (NM) * 32 + (NF))
#define KF_FEW 32                     /* up to this many tokens, k_fold_q8 with one HB block a chunk */
/* ... and rows of up to KF_NARROW columns at any number of tokens, where k_fold_many would leave 6 or 7 of a block's 8 waves
   without columns of their own (MI355X, 64 / 4096 tokens, k_fold_many against k_fold_q8: rmsfold of 512 columns with one part
   4.3 / 19.6 -> 3.6 / 15.0 us, of 1024 in HB 1024 4.8 / 26.5 -> 4.2 / 21.7, smfold 3.6 / 13.7 -> 3.1 / 10.9 and 4.1 / 23.7 -> 3.8 /
   18.1). Not fold (512: 3.0 / 9.8 us on k_fold_q8, 2.9 / 5.5 on k_fold_many), nor smfold of two HB blocks (18.3 against 16.1) */
#define KF_NARROW 1024
#define KF_ROW_MAX 36352              /* columns of a row in LDS beside the exchange (160 KB a CU) */

/* host launcher (kt_api.hip validates the arguments) */
static bool kf_overlap(const float* p, int ldp, const float* q, int ldq, int M, int C){
  if(!p || !q) return false;
  const uintptr_t p0 = (uintptr_t)p, p1 = p0 + ((size_t)(M - 1) * ldp + C) * 4;
  const uintptr_t q0 = (uintptr_t)q, q1 = q0 + ((size_t)(M - 1) * ldq + C) * 4;
  return p0 < q1 && q0 < p1;
}
/* ... and rows that meet: [a | b | xo] rows of one buffer lie between one another without doing so */
static bool kf_rows_meet(const float* p, int ldp, const float* q, int ldq, int M, int C){
  if(!kf_overlap(p, ldp, q, ldq, M, C)) return false;
  const long long d = ((long long)(intptr_t)p - (long long)(intptr_t)q) / 4;        /* floats from q to p */
  for(int i = 0; i < M; ++i){                                       /* row i of p against the last row of q that starts before its end */
    const long long e = d + (long long)i * ldp;
    if(e + C <= 0) continue;
    const long long j = (e + C - 1) / ldq;
    if((j < M ? j : M - 1) * ldq + C > e) return true;
    if(ldp == ldq && j < M) return false;                           /* equal strides: the other rows lie the same way */
  }
  return false;
}

hipError_t kt_fold_launch(int mode, const KtFoldArgs& a, int M, hipStream_t s){
  /* rmsfold over chunks of a row: every chunk's block reads the whole row (x and the parts, for the norm) while it
     writes its own chunk of xw / xn / xo. When one of those outputs overlaps x or the parts, one block takes the row
     (each thread writes only the columns it has read), so no block can overwrite what another has still to read. */
  const int np = a.nparts > 0 ? a.nparts : 0;
  const bool alias = mode == 0 && (kf_overlap(a.xw, a.ldxw, a.x, a.ldx, M, a.C) || kf_overlap(a.xn, a.ldxn, a.x, a.ldx, M, a.C)
      || kf_overlap(a.xo, a.ldxo, a.x, a.ldx, M, a.C) || (np && (kf_overlap(a.xw, a.ldxw, a.r, a.ldr, M, np * a.C)
      || kf_overlap(a.xn, a.ldxn, a.r, a.ldr, M, np * a.C) || kf_overlap(a.xo, a.ldxo, a.r, a.ldr, M, np * a.C))));
  /* smfold's grouped-head order reads other chunks' columns (with one key group, nk 1, it is the plain order): where xo lies
     over an input, a block takes the row, its inputs in LDS before an output is written, at any number of tokens */
  const bool turned = mode == 2 && a.rep > 1 && a.nk > 1 && (kf_rows_meet(a.xo, a.ldxo, a.x, a.ldx, M, a.C)
                      || kf_rows_meet(a.xo, a.ldxo, a.r, a.ldr, M, a.C));
  if(turned && a.C > KF_ROW_MAX) return hipErrorInvalidValue;
  const bool narrow = a.C <= KF_NARROW && (mode == 0 || (mode == 2 && a.C == a.HB));
  if((M > KF_FEW || alias || turned) && !narrow){
    auto al = [](const void* p, int ld, int b){ return (uintptr_t)p % b == 0 && (long long)ld * (b == 8 ? 1 : 4) % b == 0; };
    int vec = 0;
    if(al(a.x, a.ldx, 16) && (!a.r || al(a.r, a.ldr, 16)) && al(a.sg, 0, 16) && (!a.w || al(a.w, 0, 16))) vec |= KF_VX;
    if((!a.xw || al(a.xw, a.ldxw, 16)) && (!a.xn || al(a.xn, a.ldxn, 16)) && (!a.xo || al(a.xo, a.ldxo, 16))) vec |= KF_VO;
    if(al(a.Q, a.ldq, 8)) vec |= KF_VQ;
    if(turned) vec |= KF_ROW;
    const bool row = mode == 0 || turned;
    const size_t lds = 16384 + (row ? (size_t)a.C * 4 : 0);
    const dim3 grid(row ? 1 : (a.C + 4095) / 4096, M);
    return kt_go(mode == 0 ? k_fold_many<0> : mode == 1 ? k_fold_many<1> : k_fold_many<2>, grid, dim3(512), lds, s, a, vec);
  }
  const int cw = narrow && (alias || (long long)M * (a.C / a.HB) > 512) ? a.C : a.HB;      /* past 2 blocks a CU, the row */
  const int nm = cw >> 9, nf = mode == 0 ? a.C >> 9 : nm;
  void (*k)(const KtFoldArgs) = nullptr;
  switch(KF_KEY(mode, nm, nf)){
#define KF_CASE(MODE, NM, NF) case KF_KEY(MODE, NM, NF): k = k_fold_q8<MODE, NM, NF>; break;
    KF_EACH_ROW(KF_CASE)
#undef KF_CASE
    default: return hipErrorInvalidValue;
  }
  return kt_go(k, dim3(a.C / cw, M), dim3(512), 0, s, a);
}
