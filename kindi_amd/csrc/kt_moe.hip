/* kt_moe.hip - the MoE dispatch around the q8_0 expert products (lightning.cu:348-468 router / top-k,
   1318-1349 lt_moe_lists, 1352-1361 lt_moe_combine; grouped products lt_mm_* lightning.cu:958-1168).

     k_moe_topk     the router's top-k of each token (kt_topk.h): softmax over E logits (BASELINE) or Kindi's sigmoid +
                    bias scoring; the k largest, ties to the lower expert index, weights normalized over the chosen k.
     k_moe_sort     token-sorted lists: cnt / off per expert, xrow (entry -> token), where ((t, j) -> entry), and the
                    active experts in ascending order. Entries of one expert are in ascending flat index t k + j
                    (stable), so the lists are deterministic.
   (the grouped product itself, per active expert and its token list, is the decode product k_gemv_flat in its
   grouped mode, kt_gemv.h: the dense q8_0 product's lanes, arithmetic and summation tree; output row = entry)
     k_moe_route    k_moe_topk and k_moe_sort in one launch of one block, for up to 64 entries.
     k_moe_combine  x[t] += sum_j fmaf(gw[t k + j], yd[where[t k + j]], .) (+ ysh[t]); x and ysh rows ldx apart.
*/
#include "kt_common.h"
#include "kt_topk.h"


/* exclusive prefix sum over the wave's 64 lanes (6 lane shifts through ds_bpermute); *total = the sum */
__device__ __forceinline__ int kt_wave_excl_scan(int v, int lane, int* total){
  int inc = v;
#pragma unroll
  for(int d = 1; d < 64; d <<= 1){
    const int y = __builtin_amdgcn_ds_bpermute(((lane - d) & 63) << 2, inc);
    inc += lane >= d ? y : 0;
  }
  *total = __builtin_amdgcn_readlane(inc, 63);
  return inc - v;
}

__global__ void __launch_bounds__(64) k_moe_topk(const float* __restrict__ logits, int E, int k, const KtRouter rt,
                                                int* __restrict__ ids, float* __restrict__ gw){
  /* one wave per token; E <= 1024, k <= 16 */
  const int t = blockIdx.x;
  kt_topk_wave(logits + (long long)t * E, E, k, rt, ids + t * k, gw + t * k, threadIdx.x);
}

/* an exclusive scan of v over the block's 1024 threads (in-wave shuffle scan, then the 16 wave totals) */
__device__ __forceinline__ int kt_block_excl_scan(int v, int* wsum){
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int x = v;
#pragma unroll
  for(int d = 1; d < 64; d <<= 1){
    const int y = __shfl_up(x, d);
    if(lane >= d) x += y;
  }
  if(lane == 63) wsum[w] = x;
  __syncthreads();
  int pre = 0;
  for(int i = 0; i < w; ++i) pre += wsum[i];
  __syncthreads();
  return pre + x - v;
}

__device__ __forceinline__ void kt_moe_lists(const int* __restrict__ ids, int n, int E, int* __restrict__ cnt,
    int* __restrict__ off, int* __restrict__ xrow, int* __restrict__ where, int* __restrict__ act,
    int* __restrict__ nact, int k, int* __restrict__ wc){
  /* one block of 1024 threads; n = M k entries, E <= 1024; wc: 16 E ints of LDS. Counting with LDS atomics
     (order-free); offsets and the active list by block scans; placement in chunks of 1024 entries, one a thread: the
     lanes of a wave holding the same expert found by ten ballots over the expert's bits (the lane's rank among them
     in lane order), each wave's count per expert in wc, an exclusive scan of those over the 16 waves per expert; an
     entry's place = its expert's offset + the earlier waves' count + its rank, so an expert's entries keep
     ascending flat index (stable) */
  __shared__ int c[1024], o[1024], wsum[16];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  c[tid] = 0;
  __syncthreads();
  for(int i = tid; i < n; i += 1024) atomicAdd(&c[ids[i]], 1);
  __syncthreads();
  const int ce = tid < E ? c[tid] : 0;
  const int oe = kt_block_excl_scan(ce, wsum);
  const int ae = kt_block_excl_scan(ce > 0 ? 1 : 0, wsum);
  if(tid < E){
    o[tid] = oe;
    cnt[tid] = ce;
    off[tid] = oe;
    if(ce > 0) act[ae] = tid;
    if(tid == E - 1) *nact = ae + (ce > 0 ? 1 : 0);
  }
  for(int i0 = 0; i0 < n; i0 += 1024){
    for(int q = tid; q < 16 * E; q += 1024) wc[q] = 0;
    __syncthreads();
    const int i = i0 + tid;
    const bool valid = i < n;
    const int e = valid ? ids[i] : 0;
    unsigned long long eq = __ballot(valid);
#pragma unroll
    for(int b = 0; b < 10; ++b){
      const bool bit = (e >> b) & 1;
      const unsigned long long bal = __ballot(bit);
      eq &= bit ? bal : ~bal;
    }
    const int rk = __popcll(eq & ((1ull << lane) - 1ull));
    if(valid && rk == 0) wc[w * E + e] = __popcll(eq);
    __syncthreads();
    if(tid < E){
      int run = o[tid];
      for(int ww = 0; ww < 16; ++ww){ const int t = wc[ww * E + tid]; wc[ww * E + tid] = run; run += t; }
      o[tid] = run;                                              /* the next chunk continues here */
    }
    __syncthreads();
    if(valid){
      const int p = wc[w * E + e] + rk;
      xrow[p] = i / k;
      where[i] = p;
    }
    __syncthreads();                                             /* wc is cleared for the next chunk */
  }
}

extern "C" __global__ void __launch_bounds__(1024) k_moe_sort(const int* __restrict__ ids, int n, int E,
    int* __restrict__ cnt, int* __restrict__ off, int* __restrict__ xrow, int* __restrict__ where,
    int* __restrict__ act, int* __restrict__ nact, int k){
  extern __shared__ int kt_moe_wc[];                              /* 16 E */
  kt_moe_lists(ids, n, E, cnt, off, xrow, where, act, nact, k, kt_moe_wc);
}

/* the router and the lists in one launch (n = M k <= 64 entries, E <= 1024). The waves take the tokens in turn for the
   top-k (each token's is one wave's serial chain of k rounds, about 3 us: one wave doing them one after the other took
   23 us for 7 tokens of 128 experts, 6 picks; one token a wave 5.4 us); the picks meet in LDS, and wave 0 builds the lists
   while the others quantize x. Lists: lane p holds entry p's expert; the lanes holding the same one found by a ballot a
   bit of the expert index (an entry's rank among them in lane order, so an expert's entries keep ascending flat index,
   as kt_moe_sort), their count; lane l owns experts l per .. + per - 1 (per = ceil(E / 64)), offsets and the active list
   by prefix sums over lanes. The same outputs as k_moe_topk + k_moe_sort. */
#define KT_RT_WAVES 8
template <bool X>   /* x given */
__global__ void __launch_bounds__(64 * KT_RT_WAVES) k_moe_route(const float* __restrict__ logits, int M, int E, int k,
    const KtRouter rt, int* __restrict__ ids, float* __restrict__ gw, int* __restrict__ cnt, int* __restrict__ off,
    int* __restrict__ xrow, int* __restrict__ where, int* __restrict__ act, int* __restrict__ nact,
    const float* __restrict__ x, int ldx, int H, int8_t* __restrict__ Q, int ldq, float* __restrict__ D, int ldd){
  __shared__ int c[1024], o[1024], pick[64];
  const int lane = threadIdx.x & 63, n = M * k, W = blockDim.x >> 6;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for(int t = w; t < M; t += W){                                   /* wave-uniform */
    const int mine = kt_topk_wave(logits + (long long)t * E, E, k, rt, ids + t * k, gw + t * k, lane);
    if(lane < k) pick[t * k + lane] = mine;
  }
  for(int e = threadIdx.x; e < E; e += blockDim.x) c[e] = 0;
  /* the tokens' int8 rows, k_quant_q8's numbers (act 0): 16 blocks of 32 columns of one token at a time (512 columns), a
     32-lane half a block, so that a wave waits for memory once for 512 columns; by waves 1 .. while wave 0 builds the lists, the
     first ones' loads before the barrier. early: one or two tokens of many experts, where the top-k is the longer part (7 us
     at 512): the waves without a token, during the others' top-k. MI355X, 128 experts, 6 picks, x of 1024 / 2688 / 7168 columns:
     1 token 4.7 / 5.2 / 7.1 us, 7 tokens 7.9 / 14.9 / 30.9, 10 tokens 11.1 / 20.3 / 43.5 (token after token
     by all 7 waves, 112 blocks' work each time: 4.8 / 5.3 / 7.6, 12.6 / 16.0 / 31.5, 17.9 / 22.5 / 44.7; by three waves beside one that
     does every token's top-k: 5.6 / 5.7 / 8.6, 21.4 / 21.6 / 50.0, 29.2 / 29.5 / 70.7) */
  if(X){
    const int nb = H >> 5, nc = (nb + 15) >> 4, nq = M * nc, l = lane & 31, h = lane >> 5;
    const bool early = 4 * M <= W && E > 256;                      /* uniform */
    const int step = early ? W - M : W - 1;
    int i = early ? w - M : w - 1;
    const bool on = i >= 0 && i < nq;                              /* wave-uniform */
    float v[8];
    int qt = 0, qc = 0;                                            /* uniform: the token and the 512 columns v is of */
    auto ld = [&]{
      const float* xt = x + (long long)qt * ldx + qc * 512 + lane;
#pragma unroll
      for(int q = 0; q < 8; ++q) v[q] = 16 * qc + 2 * q + h < nb ? xt[64 * q] : 0.0f;
    };
    if(on){
      qt = i / nc;
      qc = i - qt * nc;
      ld();
    }
    if(!early) __syncthreads();
    if(on)
      for(; i < nq; i += step){
        float u[8];
#pragma unroll
        for(int q = 0; q < 8; ++q) u[q] = v[q];
        const int left = nb - 16 * qc - h;
        int8_t* Qt = Q + (long long)qt * ldq + qc * 512 + lane;
        float* Dt = D + (long long)qt * ldd + qc * 16 + h;
        for(qc += step; qc >= nc; qc -= nc) ++qt;
        if(i + step < nq) ld();
#pragma unroll
        for(int q = 0; q < 8; ++q){
          float a = fabsf(u[q]);
          a = fmaxf(a, kf_xorf<1>(a)); a = fmaxf(a, kf_xorf<2>(a)); a = fmaxf(a, kf_xorf<4>(a));
          a = fmaxf(a, kf_xorf<8>(a)); a = fmaxf(a, kf_xorf<16>(a));
          const float id = a != 0.0f ? 127.0f / a : 0.0f;
          if(2 * q < left){
            Qt[64 * q] = (int8_t)__float2int_rn(u[q] * id);
            if(l == 0) Dt[2 * q] = __half2float(__float2half_rn(a / 127.0f));
          }
        }
      }
    if(early) __syncthreads();
  } else __syncthreads();
  if(w > 0) return;
  const bool valid = lane < n;
  const int ep = valid ? pick[lane] : 0;
  unsigned long long eq = __ballot(valid);
#pragma unroll
  for(int b = 0; b < 10; ++b){
    const bool bit = (ep >> b) & 1;
    const unsigned long long bal = __ballot(bit);
    eq &= bit ? bal : ~bal;
  }
  const int rank = __popcll(eq & ((1ull << lane) - 1ull));
  if(valid && rank == 0) c[ep] = __popcll(eq);
  /* c[] and o[] by this wave only from here: a wave barrier suffices */
  auto sync = []{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  };
  sync();
  const int per = (E + 63) >> 6;
  int tot = 0, na = 0;
  for(int i = 0; i < per; ++i){
    const int e = lane * per + i, ce = e < E ? c[e] : 0;
    tot += ce;
    na += ce > 0 ? 1 : 0;
  }
  int tall, all;
  int base = kt_wave_excl_scan(tot, lane, &tall), abase = kt_wave_excl_scan(na, lane, &all);
  for(int i = 0; i < per; ++i){
    const int e = lane * per + i;
    if(e < E){
      const int ce = c[e];
      cnt[e] = ce;
      off[e] = base;
      o[e] = base;
      if(ce > 0) act[abase++] = e;
      base += ce;
    }
  }
  if(lane == 0) *nact = all;
  sync();
  if(valid){
    const int pos = o[ep] + rank;
    xrow[pos] = lane / k;
    where[lane] = pos;
  }
}

#define KT_RT(X) template __global__ void k_moe_route<X>(const float*, int, int, int, const KtRouter, int*, float*, int*, int*, \
    int*, int*, int*, int*, const float*, int, int, int8_t*, int, float*, int);
KT_RT(false) KT_RT(true)

extern "C" __global__ void __launch_bounds__(256) k_moe_combine(const float* __restrict__ yd, const float* __restrict__ ysh,
    const int* __restrict__ where, const float* __restrict__ gw, int k, int cols, float* __restrict__ x, int ldx){
  /* grid (column blocks of 256, tokens): one column of one token a thread, so its k loads are in flight together;
     the pairs of the token read once a block */
  __shared__ int wp[16];
  __shared__ float gp[16];
  const int t = blockIdx.y, i = blockIdx.x * 256 + threadIdx.x;
  if(threadIdx.x < k){ wp[threadIdx.x] = where[t * k + threadIdx.x]; gp[threadIdx.x] = gw[t * k + threadIdx.x]; }
  __syncthreads();
  if(i < cols){
    float s = 0.0f;
    for(int j = 0; j < k; ++j) s = fmaf(gp[j], yd[(long long)wp[j] * cols + i], s);
    x[(long long)t * ldx + i] += ysh ? s + ysh[(long long)t * ldx + i] : s;
  }
}
