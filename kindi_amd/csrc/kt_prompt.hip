/* kt_prompt.hip - the prefill product for few tokens (kt_tern_gemm where one tile of 32 tokens x 32 rows a wave leaves
   most of the GPU's SIMDs idle: the prompts of a chat turn).

   The numbers are k_tern_gemm_w's (kt_prefill.hip): Y[t][r] = sum_g fmaf((float)v(t, r, g), XS[t][g] * d[r][g], .) over
   the 128-column groups g in order (RS: fmaf(v, d, .), times XS[t][0] at the end), v the exact int32 of
   V_MFMA_I32_32X32X32_I8. The chain over g is serial by that definition, the values v are not: a block owns one tile of
   32 tokens x 32 weight rows and its NW = 4 or 8 waves take the groups in turn (wave w of round j: group NW j + w). A wave makes its
   group's values with the packed trits unpacked in registers and hands them over through LDS as floats (exact: |v| <=
   128 * 127); after one barrier a round every thread applies the round's NW groups, in order, to its own 16 / NW outputs.

   Every global read is a DMA to LDS (kt_dma.h), counted by hand: a wave's own stage of a round holds its group's
   activations (4 KB, 16-byte chunk c of row r at position c ^ ((r >> 1) & 7): no bank conflicts), packed trits (1 KB),
   row scales and token scales, and the values overwrite the activations once the matrix cores have read them. Three
   stages: the DMAs of round j + 2 go out after the barrier of round j, into the stage whose values every wave has
   finished with. (With the activations loaded straight into the lanes' operands, 16 bytes of 32 rows an instruction, the
   address unit bound it.) */
#include "kt_common.h"
#include "kt_dma.h"

typedef int kt_v4i __attribute__((ext_vector_type(4)));
typedef int kt_v16i __attribute__((ext_vector_type(16)));

#define KS_A 4096                     /* a stage's activations, then its values */
#define KS_B (KS_A + 1024)            /* packed trits end here */
#define KS_D (KS_B + 256)             /* row scales: 32 fp16 (a DMA writes 256 bytes) */
#define KS_STAGE (KS_D + 256)         /* token scales: 32 floats (256 bytes written) */
#define KS_NS 3

template <int NW, bool RS, bool DBG>
__global__ void __launch_bounds__(64 * NW) k_tern_gemm_ks(const uint32_t* __restrict__ codes,
    const uint16_t* __restrict__ scales, int R, int NG, const int8_t* __restrict__ XQ, int ldq,
    const float* __restrict__ XS, int M, float* __restrict__ Y, uint16_t* __restrict__ Y16, int ldy,
    int32_t* __restrict__ dbg, int gx, int gy){
  __shared__ __attribute__((aligned(16))) uint8_t lds[KS_NS][NW][KS_STAGE];
  constexpr int EPT = 16 / NW;                                     /* outputs a thread: 4 or 2 */
  constexpr int DMA = RS ? 6 : 7;                                  /* a wave's DMA instructions a round */
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, n = lane & 31, lr8 = lane >> 3, R8 = kt_r8(R);
  int bx, by;
  kt_xcd_tile(blockIdx.x, gx, gy, bx, by);
  const int r0 = bx * 32, n0 = by * 32;
  /* an offset past a buffer's range lands zeros (rows past the matrix, tokens past M: never stored) */
  const uint32_t OOB = 0x80000000u;
  const kt_v4i rx = kt_dma_rsrc(XQ, (uint32_t)M * (uint32_t)ldq);
  const kt_v4i rw = kt_dma_rsrc(codes, (uint32_t)R8 * (uint32_t)NG * 256u);
  const kt_v4i rh = kt_dma_rsrc(scales, (uint32_t)R8 * (uint32_t)NG * 16u);
  const kt_v4i rs = kt_dma_rsrc(XS, (uint32_t)M * (uint32_t)NG * 4u);
  const uint32_t lbase = kt_dma_lds(&lds[0][w][0]);
  /* activation DMA i: rows 8 i + lane / 8, source chunk (lane % 8) ^ ((row >> 1) & 7) */
  uint32_t xo[4];
#pragma unroll
  for(int i = 0; i < 4; ++i){
    const int tok = n0 + 8 * i + lr8;
    xo[i] = tok < M ? (uint32_t)tok * (uint32_t)ldq + (uint32_t)(((lane & 7) ^ (lr8 >> 1) ^ (4 * (i & 1))) * 16) : OOB;
  }
  /* packed trits: lane (h, n) takes half h of row n, which is its own operand */
  const int row = r0 + n;
  const uint32_t wo = (row >> 3) < R8 ? (uint32_t)((row >> 3) * NG * 16 + (row & 7)) * 16u : OOB;
  const int srg = (r0 >> 3) + (lane >> 2);
  const uint32_t ho = lane < 16 && srg < R8 ? (uint32_t)srg * (uint32_t)NG * 16u + (lane & 3) * 4 : OOB;
  const uint32_t so = lane < 32 && n0 + lane < M ? (uint32_t)(n0 + lane) * (uint32_t)NG * 4u : OOB;
  const int rounds = (NG + NW - 1) / NW;
  /* round j's group into stage q (past the last group it is read again: a wave's counts stay the same) */
  auto issue = [&](int j, int q){
    const int g = min(NW * j + w, NG - 1), nc = min(8, NG - (g & ~7));
    const uint32_t st = lbase + (uint32_t)(q * NW * KS_STAGE);
#pragma unroll
    for(int i = 0; i < 4; ++i) kt_dma16(rx, xo[i], g * 128, st + i * 1024);
    kt_dma16(rw, wo + (uint32_t)(h * (nc * 128)), (g >> 3) * 2048 + (g & 7) * 128, st + KS_A);
    kt_dma4(rh, ho, g * 16, st + KS_B);
    if(!RS) kt_dma4(rs, so, g * 4, st + KS_D);
  };
  const int tok0 = 8 * (EPT * w / 4) + 4 * h + EPT * w % 4;        /* this thread's outputs: tokens tok0 .. of row n */
  int aoff[4];
#pragma unroll
  for(int i = 0; i < 4; ++i) aoff[i] = n * 128 + (((4 * h + i) ^ ((n >> 1) & 7)) << 4);
  float acc[EPT];
#pragma unroll
  for(int e = 0; e < EPT; ++e) acc[e] = 0.0f;

  /* round j's values into stage q: this wave's DMAs of round j have landed when at most round j + 1's are in flight
     (loads retire in order) */
  auto make = [&](int j, int q){
    if(DBG || j + 1 >= rounds) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" :: "n"(DMA) : "memory");
    uint8_t* st = lds[q][w];
    const uint4 wq = *(const uint4*)(st + KS_A + lane * 16);
    kt_v4i A[4];
#pragma unroll
    for(int i = 0; i < 4; ++i) A[i] = *(const kt_v4i*)(st + aoff[i]);
    const uint32_t ww[4] = {wq.x, wq.y, wq.z, wq.w};
    kt_v16i c;
    /* MFMA i takes columns 16 i .. + 15 of both half units, for both operands */
#pragma unroll
    for(int i = 0; i < 4; ++i){
      kt_v4i b;
#pragma unroll
      for(int k = 0; k < 4; ++k)
        b[k] = (int)__builtin_amdgcn_perm(0x000100FFu, 0x000100FFu, (ww[i] >> (2 * k)) & 0x03030303u);
      c = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[i], b, i == 0 ? kt_v16i{} : c, 0, 0, 0);
    }
#pragma unroll
    for(int i = 0; i < 4; ++i)
      *(float4*)(st + (64 * i + lane) * 16) = make_float4((float)c[4 * i], (float)c[4 * i + 1], (float)c[4 * i + 2],
                                                          (float)c[4 * i + 3]);
    if(DBG){
      const int g = NW * j + w;
      if(g < NG && row < R)
#pragma unroll
        for(int e = 0; e < 16; ++e){
          const int tok = n0 + (e & 3) + 8 * (e >> 2) + 4 * h;
          if(tok < M) dbg[((long long)tok * R + row) * NG + g] = c[e];
        }
    }
  };
  /* round j from stage q: after the barrier its values are there and the stage of round j - 1 is free. Its groups are
     applied in order to this thread's outputs (tokens tok0 .. + EPT - 1 of the tile, row n) while the next round's values are made */
  auto round = [&](int j, int q){
    __syncthreads();
    float v[NW][EPT], s[NW][EPT];
    uint16_t hd[NW];
#pragma unroll
    for(int k = 0; k < NW; ++k){
      const uint8_t* sk = lds[q][k];
      const float* pv = (const float*)(sk + (64 * (EPT * w / 4) + lane) * 16 + (EPT * w % 4) * 4);
      const float* ps = (const float*)(sk + KS_D) + tok0;
#pragma unroll
      for(int e = 0; e < EPT; ++e){ v[k][e] = pv[e]; s[k][e] = RS ? 1.0f : ps[e]; }
      hd[k] = *(const uint16_t*)(sk + KS_B + 2 * n);
    }
    if(j > 0 && j + 2 < rounds) issue(j + 2, (q + 2) % KS_NS);
    if(j + 1 < rounds) make(j + 1, (q + 1) % KS_NS);
#pragma unroll
    for(int k = 0; k < NW; ++k)
      if(NW * j + k < NG){                                         /* uniform */
        const float d = kt_h2f(hd[k]);
#pragma unroll
        for(int e = 0; e < EPT; ++e) acc[e] = fmaf(v[k][e], RS ? d : s[k][e] * d, acc[e]);
      }
  };
#pragma unroll
  for(int q = 0; q < KS_NS; ++q) if(q < rounds) issue(q, q);
  make(0, 0);
  int j = 0;
  for(; j + KS_NS <= rounds; j += KS_NS)
#pragma unroll
    for(int q = 0; q < KS_NS; ++q) round(j + q, q);
#pragma unroll
  for(int q = 0; q < KS_NS - 1; ++q) if(j + q < rounds) round(j + q, q);
  const __amdgpu_buffer_rsrc_t rsx = __builtin_amdgcn_make_buffer_rsrc((void*)XS, (short)0, M * NG * 4, 0x00020000);
#pragma unroll
  for(int e = 0; e < EPT; ++e){
    const int t = n0 + tok0 + e;
    if(t < M && row < R){
      float y = acc[e];
      if(RS) y *= __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsx, (uint32_t)t * NG * 4, 0, 0));
      asm volatile("" : "+v"(y));                                  /* fp32, then fp16: two roundings */
      if(Y) Y[(long long)t * ldy + row] = y;
      if(Y16) Y16[(long long)t * ldy + row] = __half_as_ushort(__float2half_rn(y));
    }
  }
}

#define KT_KS(NW, RS, DBG) template __global__ void k_tern_gemm_ks<NW, RS, DBG>(const uint32_t*, const uint16_t*, int, int, \
    const int8_t*, int, const float*, int, float*, uint16_t*, int, int32_t*, int, int);
KT_KS(4, false, false) KT_KS(4, false, true) KT_KS(4, true, false) KT_KS(4, true, true)
KT_KS(8, false, false) KT_KS(8, false, true) KT_KS(8, true, false) KT_KS(8, true, true)
