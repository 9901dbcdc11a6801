/* kt_q8gemm.hip - the q8_0 product for many tokens on the matrix cores, dense or grouped (MoE prefill; lt_mm_*
   lightning.cu:958-1168, k_q8 dsv41_gpu.cu:131-296): kt_q8_gemv's numbers and tree, so its bits.

   A K slice (kt_kslices: one or two steps of 8 units of 32 columns) at a time: per k-lane c the chain
   fmaf((float)v, d_w * D[t][u], .) over the slice's units 8 s + c, the 8 chains by ((c0 + c1) + (c2 + c3)) + ((c4 + c5) +
   (c6 + c7)), the slice sums left to right. A unit's values v of 32 tokens x 32 rows are one V_MFMA_I32_32X32X32_I8; the
   products d_w D of a k-lane's two units one V_MFMA_F32_32X32X1_2B (block j = the slice's step j; one rounding, as the
   multiply).

   Block: 4 waves own 128 weight rows of one expert (or of the dense matrix), wave w the tiles of rows 32 w .. + 31, in
   passes of up to 64 entries (two tiles a wave) over the expert's list. A wave holds its slice's weights in registers (16
   units, 64 registers) for both tiles, and refills each unit for the next slice as soon as the last tile's matrix cores
   have read it, so the weight stream runs under the products: what is in flight a CU is registers (128 KB), not LDS.
   The slice of the activations and their scales, which every wave reads, reaches LDS by DMA (kt_dma.h): rows of 512
   bytes, 16-byte chunk i of row t at i ^ (t & 15); token scales [row][16], 4-float chunk i of row t at i ^ ((t >> 2) & 3).
   A unit past the matrix or the slice gets zero scales (its product is +0).

   Measured on MI355X (128 experts, 6 picks, even router, up [1856 x 2688] / down [2688 x 1856], against k_q8_mma): 96
   entries an expert 987 / 970 -> 386 / 373 us, 20: 271 / 264 -> 149 / 148, 12: 165 / 168 -> 146 / 146 (678 MB of weights: 4.6 TB/s).
   Nothing is refilled after a block's last slice: with the first slice read again there (KS + 1 slices for KS) 12 entries took
   156 / 167 us, 24: 178 / 176; from an empty buffer instead of behind a branch every length is 1 to 2% slower. At long
   lists (96 entries) counters give vector instructions 53% of the SIMDs' cycles and the matrix cores 17%, next to no overlap (a unit's
   results are taken at once), the rest waiting with 2 waves a SIMD (253 registers); without any global load they take 296 us. */
#include <type_traits>
#include "kt_common.h"
#include "kt_dma.h"

typedef int kt_v4i __attribute__((ext_vector_type(4)));
typedef int kt_v16i __attribute__((ext_vector_type(16)));
typedef float kt_v32f __attribute__((ext_vector_type(32)));

#define QG_T 64                       /* entries a pass */
/* X for the k-lanes c_ = 0 .. 7 as compile-time constants (the register arrays stay registers) */
#define KT_QG_1(N, X) { std::integral_constant<int, N> c_; X; }
#define KT_QG_C(X) KT_QG_1(0, X) KT_QG_1(1, X) KT_QG_1(2, X) KT_QG_1(3, X) KT_QG_1(4, X) KT_QG_1(5, X) KT_QG_1(6, X) KT_QG_1(7, X)
struct KtQg {
  uint8_t a[2][32 * 512];             /* two stages of one tile's slice */
  uint8_t x[2][32 * 64];
  float4 tot[4][2][4][64];            /* [wave][tile][register quad][lane]: the slice sums so far */
  uint32_t ro[QG_T], rd[QG_T];        /* byte offsets of the pass's rows and of their scales */
};

/* a k-lane's two units of the slice of ns steps from s0 (unit (j, c) = step s0 + j; this lane half h of row n: byte offset
   wf in a full step, wl in the last, of ncl units) and its row scale (lane half h: step s0 + h). A unit past the matrix or
   the slice reads a valid one of the row, with a zero scale. Always KT_QG_LOADS / 8 loads: the waits below count them */
#define KT_QG_LOADS 24
__device__ __forceinline__ void qg_ldw(const __amdgpu_buffer_rsrc_t rw, int c, int s0, int ns, int S, int ncl, int h,
                                       uint32_t wf, uint32_t wl, uint32_t db, kt_v4i& w0, kt_v4i& w1, uint16_t& d){
  const bool l0 = s0 >= S - 1, l1 = s0 + 1 >= S - 1, ok0 = !(l0 && c >= ncl), ok1 = ns > 1 && !(l1 && c >= ncl);   /* uniform */
  const uint32_t v0 = l0 ? wl : wf, v1 = l1 ? wl : wf, vd = (h ? ok1 : ok0) ? db : 0x80000000u;
  w0 = __builtin_bit_cast(kt_v4i, __builtin_amdgcn_raw_buffer_load_b128(rw, v0, ok0 ? s0 * 2048 + c * 128 : 0, 2));
  w1 = __builtin_bit_cast(kt_v4i, __builtin_amdgcn_raw_buffer_load_b128(rw, v1, ok1 ? s0 * 2048 + 2048 + c * 128 : 0, 2));
  d = __builtin_amdgcn_raw_buffer_load_b16(rw, vd, s0 * 128 + c * 16, 0);
}

template <bool GRP, bool DBG>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DBG ? 1 : 2))) k_q8_gemm(const KtGemvArgs a,
    const KtGroupedArgs ga, const int8_t* __restrict__ xq, const float* __restrict__ xd, int32_t* __restrict__ dbg, int KS, int P, int dv){
  __shared__ __attribute__((aligned(16))) KtQg L;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, n = lane & 31;
  const uint8_t* wbuf;
  float* yout;
  int R, NU, ldy, ldq, ldd, nrows, t_lo, t_hi, t_st, p0 = 0, bx;
  const int* xrow = nullptr;
  if(GRP){
    /* P blocks of one row tile (passes z, z + P, ..) on one XCD, so that its L2 serves the weights to all but the first. dv = P: 8
       ids apart, at one time. dv < 0 (minus the row tiles an XCD): the tiles' first passes before all others */
    const unsigned gx = (unsigned)(ga.R + 127) >> 7, q = blockIdx.x >> 3, dq = q / (unsigned)abs(dv), dr = q - dq * (unsigned)abs(dv);
    const int z = dv > 0 ? dr : dq;
    const unsigned tile = (dv > 0 ? dq : dr) * 8 + (blockIdx.x & 7);
    const int ie = tile / gx;
    bx = tile - ie * gx;
    const int nact = *ga.nact;
    if(ie >= nact) return;
    const int e = __builtin_amdgcn_readfirstlane(ga.act[ie]);
    wbuf = ga.wexp[e];
    R = ga.R; NU = ga.NU; ldy = ga.ldy; ldq = ga.ldq; ldd = ga.ldd; nrows = ga.nrows; xrow = ga.xrow; yout = ga.y;
    p0 = __builtin_amdgcn_readfirstlane(ga.off[e]); t_hi = __builtin_amdgcn_readfirstlane(ga.cnt[e]);
    t_lo = z * QG_T; t_st = P * QG_T;
    if(t_lo >= t_hi) return;
  } else {
    wbuf = (const uint8_t*)a.mat[0].codes;
    R = a.mat[0].R; NU = a.NU; ldy = a.mat[0].ldy; ldq = a.ldq; ldd = a.ldxs; nrows = a.M; yout = a.mat[0].y;
    bx = blockIdx.x; t_lo = blockIdx.y * QG_T; t_hi = min(a.M, t_lo + QG_T); t_st = QG_T;
  }
  const int R8 = kt_r8(R), S = kt_steps(NU), row = bx * 128 + 32 * w + n, rg = row >> 3;
  const uint32_t OOB = 0x80000000u;
  const kt_v4i rx = kt_dma_rsrc(xq, (uint32_t)nrows * (uint32_t)ldq);
  const kt_v4i rs = kt_dma_rsrc(xd, (uint32_t)nrows * (uint32_t)ldd * 4u);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)wbuf, (short)0, R8 * NU * 272, 0x00020000);
  const uint32_t la = kt_dma_lds(L.a), lx = kt_dma_lds(L.x);
  const int ao = n * 512 + ((h ^ (n & 15)) << 4), xo = n * 64 + ((2 * h) ^ ((n >> 2) & 3)) * 16;   /* this lane's operands */
  const uint32_t wb = rg < R8 ? (uint32_t)(rg * NU * 16 + (row & 7)) * 16u : OOB;
  const uint32_t db = rg < R8 ? (uint32_t)R8 * NU * 256u + (uint32_t)(rg * NU * 16 + (row & 7) * 2 + h * 128) : OOB;

  /* the slice's weights: unit (j, c) = step s0 + j, k-lane c; this lane half h of row n. A unit past the slice or the
     matrix reads the row's first one (not used). Row scales: lane half h holds step s0 + h's (zero past the end) */
  kt_v4i wq[2][8];
  uint16_t hq[8];
  const int ncl = NU - (S - 1) * KT_KL;                            /* units of the last step */
  const uint32_t wf = wb + (uint32_t)(h * 1024), wl = wb + (uint32_t)(h * ncl * 128);
  /* the tile of entries 32 tt .. of the pass: slice k's products added to tot; RF: the weights refilled for slice kn */
  auto tile = [&](bool rf, int st, int tt, int k, int s0, int ns, int sn, int nsn, int t0){
    const uint8_t* la_ = L.a[st];
    const uint8_t* lx_ = L.x[st];
    float pend[16], t01[16], t45[16];
    auto lane_c = [&](auto cc){
      constexpr int c = decltype(cc)::value;
      __builtin_amdgcn_sched_barrier(0);
      const kt_v4i A0 = *(const kt_v4i*)(la_ + (ao ^ (32 * c))), A1 = *(const kt_v4i*)(la_ + (ao ^ (32 * c)) + 256);
      const float x = *(const float*)(lx_ + (xo ^ (c & 4) * 4) + (c & 3) * 4);
      const kt_v32f s = __builtin_amdgcn_mfma_f32_32x32x1f32(x, kt_h2f(hq[c]), kt_v32f{}, 0, 0, 0);
      const kt_v16i v0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(A0, wq[0][c], kt_v16i{}, 0, 0, 0);
      const kt_v16i v1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(A1, wq[1][c], kt_v16i{}, 0, 0, 0);
      if(rf) qg_ldw(rw, c, sn, nsn, S, ncl, h, wf, wl, db, wq[0][c], wq[1][c], hq[c]);                                           /* uniform */
      __builtin_amdgcn_sched_barrier(0);
      if(DBG && row < R){
        int tb = t0 + 32 * tt + 4 * h;
        asm volatile("" : "+v"(tb));                               /* the addresses are made here, not kept */
#pragma unroll
        for(int e = 0; e < 16; ++e){
          const int t = tb + (e & 3) + 8 * (e >> 2);
          int32_t* o = dbg + ((long long)(p0 + t) * R + row) * NU + s0 * KT_KL + c;
          if(t < t_hi && s0 * KT_KL + c < NU) o[0] = v0[e];
          if(t < t_hi && ns == 2 && (s0 + 1) * KT_KL + c < NU) o[KT_KL] = v1[e];
        }
      }
      /* stage after stage over the 16 elements (each stage's results taken by an empty asm): independent instructions
         behind one another; the compiler's own order was each element's chain of five dependent ones in turn, and it
         sank the k-lanes' epilogues behind the last one's MFMAs and spilled */
      float f0[16], f1[16];
#define KT_QG_STAGE(X, V) _Pragma("unroll") for(int e = 0; e < 16; ++e) X; \
      _Pragma("unroll") for(int e = 0; e < 16; ++e) asm volatile("" : "+v"(V[e]))
      KT_QG_STAGE(f0[e] = (float)v0[e], f0);
      KT_QG_STAGE(f1[e] = (float)v1[e], f1);
      KT_QG_STAGE(f0[e] = fmaf(f0[e], s[e], 0.0f), f0);
      KT_QG_STAGE(f0[e] = fmaf(f1[e], s[16 + e], f0[e]), f0);
      if(!(c & 1)){ KT_QG_STAGE(pend[e] = f0[e], pend); }
      else if(c == 1){ KT_QG_STAGE(t01[e] = pend[e] + f0[e], t01); }
      else if(c == 3){ KT_QG_STAGE(pend[e] = pend[e] + f0[e], pend); KT_QG_STAGE(t01[e] = t01[e] + pend[e], t01); }
      else if(c == 5){ KT_QG_STAGE(t45[e] = pend[e] + f0[e], t45); }
      else {                                                       /* the slice sum */
        KT_QG_STAGE(pend[e] = pend[e] + f0[e], pend);
        KT_QG_STAGE(pend[e] = t45[e] + pend[e], pend);
        KT_QG_STAGE(t01[e] = t01[e] + pend[e], t01);
      }
#undef KT_QG_STAGE
    };
    KT_QG_C(lane_c(c_))
    __builtin_amdgcn_sched_barrier(0);
    /* the slices left to right: the sums so far wait in LDS (this lane's own words), the last slice's go out */
    float4* tq = &L.tot[w][tt][0][lane];
#pragma unroll
    for(int q = 0; q < 4; ++q){
      float4 f = make_float4(t01[4 * q], t01[4 * q + 1], t01[4 * q + 2], t01[4 * q + 3]);
      if(k > 0){                                                   /* uniform */
        const float4 o = tq[64 * q];
        f = make_float4(o.x + f.x, o.y + f.y, o.z + f.z, o.w + f.w);
      }
      if(k + 1 < KS) tq[64 * q] = f;                               /* uniform */
      else if(row < R){
        const int t = t0 + 32 * tt + 8 * q + 4 * h;
        float* o = yout + (long long)(p0 + t) * ldy + row;
        if(t < t_hi) o[0] = f.x;
        if(t + 1 < t_hi) o[ldy] = f.y;
        if(t + 2 < t_hi) o[2ll * ldy] = f.z;
        if(t + 3 < t_hi) o[3ll * ldy] = f.w;
      }
    }
  };
  KT_QG_C(qg_ldw(rw, c_, 0, S / KS, S, ncl, h, wf, wl, db, wq[0][c_], wq[1][c_], hq[c_]))
  /* tile tt of the pass, slice from s0: its activations and token scales into stage st */
  auto issue = [&](int st, int tt, int s0, int ns){
    /* activations: instruction i = rows 2 i, 2 i + 1; lane: row 2 i + lane / 32, chunk position lane % 32 */
#pragma unroll
    for(int q = 0; q < 4; ++q){
      const int i = w + 4 * q, r = 2 * i + h, ch = (lane & 16) | ((lane & 15) ^ (r & 15));
      const uint32_t off = (uint32_t)s0 * 256u + (uint32_t)ch * 16u, ro = L.ro[32 * tt + r];
      kt_dma16(rx, ro != OOB && off < (uint32_t)NU * 32u && ch < 16 * ns ? ro + off : OOB, 0, la + st * 16384 + i * 1024);
    }
    /* token scales: instruction i = rows 4 i .. + 3 */
#pragma unroll
    for(int q = 0; q < 2; ++q){
      const int i = w + 4 * q, r = 4 * i + (lane >> 4);
      const int uc = 4 * (((lane >> 2) & 3) ^ (i & 3)) + (lane & 3), u = s0 * KT_KL + uc;
      const uint32_t rd = L.rd[32 * tt + r];
      kt_dma4(rs, rd != OOB && u < NU && uc < 8 * ns ? rd + (uint32_t)u * 4u : OOB, 0, lx + st * 2048 + i * 256);
    }
  };
  for(int t0 = t_lo; t0 < t_hi; t0 += t_st){
    const int nt = min(QG_T, t_hi - t0), T = nt > 32 ? 2 : 1;
    if(tid < QG_T){
      const int p = p0 + t0 + tid;
      const bool ok = tid < nt;
      const int r = ok ? (xrow ? xrow[p] : p) : 0;
      L.ro[tid] = ok ? (uint32_t)r * (uint32_t)ldq : OOB;
      L.rd[tid] = ok ? (uint32_t)r * (uint32_t)ldd * 4u : OOB;
    }
    __syncthreads();
    issue(0, 0, 0, S / KS);
    int st = 0;
    bool refilled = false;                                         /* uniform */
    for(int k = 0; k < KS; ++k){
      const int s0 = k * S / KS, ns = (k + 1) * S / KS - s0;
      const int kn = k + 1 < KS ? k + 1 : 0, sn = kn * S / KS, nsn = (kn + 1) * S / KS - sn;
      for(int tt = 0; tt < T; ++tt){
        /* this wave's DMAs of the stage have landed; a refill's loads are newer and stay in flight. After the barrier
           every wave's have, and the other stage is no longer read */
        if(refilled && !DBG) asm volatile("s_waitcnt vmcnt(%0)" :: "n"(KT_QG_LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        refilled = tt + 1 == T;
        if(!refilled) issue(st ^ 1, tt + 1, s0, ns);
        else if(k + 1 < KS) issue(st ^ 1, 0, sn, nsn);
        tile(refilled && (k + 1 < KS || t0 + t_st < t_hi), st, tt, k, s0, ns, sn, nsn, t0);
        st ^= 1;
      }
    }
    __syncthreads();                                               /* the rows' table and the stages are rewritten */
  }
}

#define KT_QG(GRP, DBG) template __global__ void k_q8_gemm<GRP, DBG>(const KtGemvArgs, const KtGroupedArgs, const int8_t*, \
    const float*, int32_t*, int, int, int);
KT_QG(false, false) KT_QG(false, true) KT_QG(true, false) KT_QG(true, true)
