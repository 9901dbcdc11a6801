/* kt_prefill.hip - the prefill product on packed trits (k_tc_mm2 tc_hip.cu:243-269, k_mm_g5q chunk.cu:858-918).

   Y[t][r] = sum_g fmaf((float)v(t, r, g), XS[t][g] * d[r][g], .) over the 128-column groups g in order, where
   v(t, r, g) = sum of t(r, c) q(t, c) over the group is an exact int32 from V_MFMA_I32_32X32X32_I8. RS (one activation
   scale a token): Y[t][r] = XS[t][0] sum_g fmaf(v, d[r][g], .), the order that takes one operation less an element.

   Block: 4 waves own 32 T tokens x 128 weight rows, wave w the tiles of rows 32 w .. + 31 (T = 1, 2). Every global read
   is a DMA to LDS (kt_dma.h), counted by hand, three stages of one group: the tokens' activations (shared by the waves;
   16-byte chunk c of row r at position c ^ ((r >> 1) & 7), no bank conflicts), each wave's packed trits (1 KB: lane
   (h, n) its own half-unit chunk), row scales and token scales. A wave unpacks its trits in registers (shift, mask,
   v_perm byte lookup), so no unpacked weight is ever stored, and the T tiles share the unpacking. MFMA i takes columns
   16 i .. 16 i + 15 of both half units (lane half h supplies half h), for both operands. With T = 2 the tiles alternate
   between two accumulator sets: each MFMA of a tile is followed by a quarter of the other tile's epilogue, held in that
   order by scheduling barriers, across the group's end too; the element scales XS d of both tiles come from one
   V_MFMA_F32_32X32X1 (an outer product: one rounding, as the multiply), so that the token scales are one LDS word a lane
   and not a broadcast of 16.

   What bounds it: a SIMD overlaps its matrix and vector instructions little (a register-only probe: 4 MFMAs
   69 ns, with 32 vector operations 92, with 64 128, with 128 203), so a tile's group costs 70 ns of MFMA and about 1 ns a
   vector operation: 32 of the epilogue, 44 / T of the unpacking; the LDS reads of the activations (4 KB a tile) come on
   top. Four tiles a wave take 11 operations of unpacking instead of 22, but two waves a SIMD and measured no better.
   MI355X, group scales, fp32 out, against the kernel before it (128 x 128 tiles, trits unpacked into LDS by the block):
   [17408 x 5120] at 128 / 256 / 1000 tokens 57.5 / 70 / 190 -> 32 / 47 / 134 us, [4096 x 12288] at 1000 124 -> 80,
   [12288 x 4096] 100 -> 77; per-row scales [12288 x 4096] at 512 / 2048 tokens 56 / 168 -> 46 / 138 us.

   MFMA 32x32x32 i8 register layouts on gfx950 (measured): A lane l holds row l % 32, k = 16 (l / 32) .. +15;
   B lane l holds column l % 32, the same k; D lane l register i holds column l % 32, row (i % 4) + 8 (i / 4) +
   4 (l / 32). V_MFMA_F32_32X32X1_2B: A lane l block l / 32, row l % 32; B the same columns; D registers 16 b .. of
   block b in the layout above. */
#include "kt_common.h"
#include "kt_dma.h"

typedef int kt_v4i __attribute__((ext_vector_type(4)));
typedef int kt_v16i __attribute__((ext_vector_type(16)));
typedef float kt_v32f __attribute__((ext_vector_type(32)));

#define PF_NW 4                       /* waves a block: 32 rows each */
#define PF_NS 3                       /* LDS stages */

template <int T, bool RS>
struct KtPf {
  static constexpr int A = 32 * T * 128, B = PF_NW * 1024, D = PF_NW * 256, S = RS ? 0 : PF_NW * 256;
  static constexpr int STAGE = A + B + D + S;                    /* activations, trits, row scales, token scales */
  static constexpr int DMA = T + 2 + (RS ? 0 : 1);               /* DMA instructions a wave a group */
};

template <int T, bool RS, bool DBG>
__global__ void __launch_bounds__(64 * PF_NW) __attribute__((amdgpu_waves_per_eu(2))) k_tern_gemm_w(const uint32_t* __restrict__ codes,
    const uint16_t* __restrict__ scales, int R, int NG, const int8_t* __restrict__ XQ, int ldq,
    const float* __restrict__ XS, int M, float* __restrict__ Y, uint16_t* __restrict__ Y16, int ldy,
    int32_t* __restrict__ dbg, int gx, int gy){
  typedef KtPf<T, RS> L;
  constexpr int NS = PF_NS;
  __shared__ __attribute__((aligned(16))) uint8_t lds[NS * L::STAGE];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, n = lane & 31, R8 = kt_r8(R);
  int bx, by;
  kt_xcd_tile(blockIdx.x, gx, gy, bx, by);
  const int r0 = bx * 32 * PF_NW + 32 * w, n0 = by * 32 * T;
  const uint32_t OOB = 0x80000000u;
  const kt_v4i rx = kt_dma_rsrc(XQ, (uint32_t)M * (uint32_t)ldq);
  const kt_v4i rw = kt_dma_rsrc(codes, (uint32_t)R8 * (uint32_t)NG * 256u);
  const kt_v4i rh = kt_dma_rsrc(scales, (uint32_t)R8 * (uint32_t)NG * 16u);
  const kt_v4i rs = kt_dma_rsrc(XS, (uint32_t)M * (uint32_t)NG * 4u);
  const uint32_t lbase = kt_dma_lds(lds);
  /* activation DMA k of this wave: rows 8 (w + 4 k) + lane / 8 of the token tile, source chunk (lane % 8) ^
     ((row >> 1) & 7) at chunk position lane % 8 */
  const int lr8 = lane >> 3;
  uint32_t xo[T];
#pragma unroll
  for(int k = 0; k < T; ++k){
    const int tok = n0 + 8 * (w + 4 * k) + lr8;
    xo[k] = tok < M ? (uint32_t)tok * (uint32_t)ldq + (uint32_t)(((lane & 7) ^ (lr8 >> 1) ^ (4 * (w & 1))) * 16) : OOB;
  }
  const int wrow = r0 + n, wrg = wrow >> 3;
  const uint32_t wo = wrg < R8 ? (uint32_t)(wrg * NG * 16 + (wrow & 7)) * 16u : OOB;
  const int srg = (r0 >> 3) + (lane >> 2);
  const uint32_t ho = lane < 16 && srg < R8 ? (uint32_t)srg * (uint32_t)NG * 16u + (lane & 3) * 4 : OOB;
  const int stok = n0 + 8 * T * w + lane;
  const uint32_t so = lane < 8 * T && stok < M ? (uint32_t)stok * (uint32_t)NG * 4u : OOB;

  auto issue = [&](int g, int q){
    const uint32_t st = lbase + (uint32_t)(q * L::STAGE);
#pragma unroll
    for(int k = 0; k < T; ++k) kt_dma16(rx, xo[k], g * 128, st + (w + 4 * k) * 1024);
    const int nc = min(8, NG - (g & ~7));
    kt_dma16(rw, wo + (uint32_t)(h * (nc * 128)), (g >> 3) * 2048 + (g & 7) * 128, st + L::A + w * 1024);
    kt_dma4(rh, ho, g * 16, st + L::A + L::B + w * 256);
    if(!RS) kt_dma4(rs, so, g * 4, st + L::A + L::B + L::D + w * 256);
  };
  int aoff[4];
#pragma unroll
  for(int i = 0; i < 4; ++i) aoff[i] = n * 128 + (((4 * h + i) ^ ((n >> 1) & 7)) << 4);
  const int boff = L::A + w * 1024 + lane * 16, doff = L::A + L::B + w * 256 + n * 2;
  /* the token scales: each wave staged 8 T tokens in 256 bytes. T = 2: token lane's; T = 1: tokens 4 h + e of each */
  const int soff = L::A + L::B + L::D + (T == 2 ? 256 * (lane >> 4) + 4 * (lane & 15) : 16 * h);
  float acc[T][16];
#pragma unroll
  for(int t = 0; t < T; ++t)
#pragma unroll
    for(int e = 0; e < 16; ++e) acc[t][e] = 0.0f;

  kt_v16i c[2] = {};
  kt_v32f s = {};
  float dp = 0.0f;
  auto put_dbg = [&](int t, const kt_v16i& v, int g){
    int t0 = n0 + 32 * t + 4 * h;
    asm volatile("" : "+v"(t0));                                  /* the addresses are made here, not kept over the loop */
    if(wrow < R)
#pragma unroll
      for(int e = 0; e < 16; ++e){
        const int tok = t0 + (e & 3) + 8 * (e >> 2);
        if(tok < M) dbg[((long long)tok * R + wrow) * NG + g] = v[e];
      }
  };
  auto group = [&](int g, int q){
    /* this wave's DMAs of group g have landed when at most the later groups' are in flight (loads retire in order);
       after the barrier every wave's have, and the stage of group g - 1 is no longer read */
    if(DBG || g + NS - 2 >= NG) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" :: "n"(L::DMA * (NS - 2)) : "memory");
    __syncthreads();
    if(g + NS - 1 < NG) issue(g + NS - 1, (q + NS - 1) % NS);
    const uint8_t* st = lds + q * L::STAGE;
    const uint4 wq = *(const uint4*)(st + boff);
    const uint16_t hd = *(const uint16_t*)(st + doff);
    float xv = 0.0f, xe[T == 1 && !RS ? 16 : 1];
    if(!RS && T > 1) xv = *(const float*)(st + soff);
    if(!RS && T == 1)
#pragma unroll
      for(int e = 0; e < 16; ++e) xe[e] = *(const float*)(st + soff + 256 * (e >> 2) + 4 * (e & 3));
    kt_v4i A[4], B[4];
#pragma unroll
    for(int i = 0; i < 4; ++i) A[i] = *(const kt_v4i*)(st + aoff[i]);
    const uint32_t ww[4] = {wq.x, wq.y, wq.z, wq.w};
#pragma unroll
    for(int i = 0; i < 4; ++i)
#pragma unroll
      for(int k = 0; k < 4; ++k)
        B[i][k] = (int)__builtin_amdgcn_perm(0x000100FFu, 0x000100FFu, (ww[i] >> (2 * k)) & 0x03030303u);
    const float d = kt_h2f(hd);
    if(T == 1){
#pragma unroll
      for(int i = 0; i < 4; ++i) c[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[i], B[i], i == 0 ? kt_v16i{} : c[0], 0, 0, 0);
#pragma unroll
      for(int e = 0; e < 16; ++e) acc[0][e] = fmaf((float)c[0][e], RS ? d : xe[e] * d, acc[0][e]);
      if(DBG) put_dbg(0, c[0], g);
      return;
    }
#pragma unroll
    for(int t = 0; t < T; ++t){
      const int cu = t & 1, tp = (t + T - 1) % T;
      const float m = t == 0 ? dp : d;
#pragma unroll
      for(int i = 0; i < 4; ++i){
        c[cu] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[i], B[i], i == 0 ? kt_v16i{} : c[cu], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if(t + 1 < T) A[i] = *(const kt_v4i*)(st + aoff[i] + (t + 1) * 4096);
#pragma unroll
        for(int e = 4 * i; e < 4 * i + 4; ++e)
          acc[tp][e] = fmaf((float)c[cu ^ 1][e], RS ? m : s[16 * (tp & 1) + e], acc[tp][e]);
        asm volatile("" : "+v"(acc[tp][4 * i]), "+v"(acc[tp][4 * i + 1]), "+v"(acc[tp][4 * i + 2]), "+v"(acc[tp][4 * i + 3]));
        __builtin_amdgcn_sched_barrier(0);
      }
      if(DBG && (t > 0 || g > 0)) put_dbg(tp, c[cu ^ 1], t == 0 ? g - 1 : g);
      if(!RS && t == 0){                                            /* the last group's second tile is done with s */
        s = __builtin_amdgcn_mfma_f32_32x32x1f32(xv, d, kt_v32f{}, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    dp = d;
  };
#pragma unroll
  for(int q = 0; q < NS - 1; ++q) if(q < NG) issue(q, q);
  int g = 0;
  for(; g + NS <= NG; g += NS)
#pragma unroll
    for(int q = 0; q < NS; ++q) group(g + q, q);
#pragma unroll
  for(int q = 0; q < NS - 1; ++q) if(g + q < NG) group(g + q, q);
  if(T > 1){                                                        /* the last group's last tile */
#pragma unroll
    for(int e = 0; e < 16; ++e) acc[T - 1][e] = fmaf((float)c[1][e], RS ? dp : s[16 + e], acc[T - 1][e]);
    if(DBG) put_dbg(T - 1, c[1], NG - 1);
  }
  const __amdgpu_buffer_rsrc_t rsx = __builtin_amdgcn_make_buffer_rsrc((void*)XS, (short)0, M * NG * 4, 0x00020000);
#pragma unroll
  for(int t = 0; t < T; ++t)
#pragma unroll
    for(int e = 0; e < 16; ++e){
      const int tok = n0 + 32 * t + (e & 3) + 8 * (e >> 2) + 4 * h;
      if(tok < M && wrow < R){
        float y = acc[t][e];
        if(RS) y *= __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsx, (uint32_t)tok * NG * 4, 0, 0));
        asm volatile("" : "+v"(y));                              /* fp32, then fp16: two roundings */
        if(Y) Y[(long long)tok * ldy + wrow] = y;
        if(Y16) Y16[(long long)tok * ldy + wrow] = __half_as_ushort(__float2half_rn(y));
      }
    }
}
#define KT_PF(T, RS, DBG) template __global__ void k_tern_gemm_w<T, RS, DBG>(const uint32_t*, const uint16_t*, int, int, \
    const int8_t*, int, const float*, int, float*, uint16_t*, int, int32_t*, int, int);
KT_PF(1, false, false) KT_PF(1, false, true) KT_PF(1, true, false) KT_PF(1, true, true)
KT_PF(2, false, false) KT_PF(2, false, true) KT_PF(2, true, false) KT_PF(2, true, true)
