// The decode GEMV on the matrix core (4 to 8 rows of x, with the tile loop 1 to 8, int8 weights): the products, prologues
// and epilogues of gemv.hip, whose launcher decides which form runs.
//
// The form of gemv.hip spends one FMA per weight and row of x and reads x from LDS for every few rows of W; past three
// rows of x that sets its time, not the weights' bytes. Here x is split into three bf16 pieces, hi + mid + lo = x exactly (8
// significant bits each, by truncation), int8 weights are exact in bf16, and a v_mfma_f32_16x16x32_bf16 multiplies 16
// output rows by 16 columns = (piece, row of x): every product is exact and is summed in fp32, where an fp32 FMA chain
// rounds each partial sum once (error against 64 bits 7e-8 to 1.6e-7 here, 1.1e-7 to 2.2e-7 there). Up to five rows of x
// fit one MFMA, eight take two. Weights come in as there (a wave load covers 4 rows x 256 contiguous bytes: fragment-order
// loads would touch another cache line with every lane), go through a 4 KB wave-private LDS tile (16-byte chunks
// XOR-swizzled by row: no bank conflicts) and become A fragments.
// Measured on MI355X (graph-replayed, weights past the L2, group scales; us at 4 / 5 / 8 rows of x): gate/up 7168 x 1024 with
// norm and SwiGLU 6.3 / 6.4 / 7.7 (the FMA form of gemv.hip 6.7 / 9.8 / 10.0, at 8-row tiles past 4 rows), 5120 x 1024 with
// the norm 5.7 / 5.9 / 7.9 (5.9 / 7.7 / 7.9), 1024 x 2048 accumulating 4.2 / 4.6 / 5.2 (4.4 / 5.1 / 5.2). At 3 rows the two
// were equal (gate/up 7.2 and 6.9), at one row the FMA form was faster (6.4 and 5.3); kernels for fewer than 4 rows exist
// only with the tile loop.
#include <type_traits>

#include "gemv_common.h"

namespace q35 {

constexpr int gemv_ct(int mp) { return (3 * mp + 15) / 16; }  // MFMA column tiles of 3 pieces x mp rows
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));

// four consecutive values' pieces, packed in pairs: [piece][pair]
__device__ __forceinline__ void split3(const f32x4& x, u32x2 (&o)[3]) {
  uint32_t h[4], m[4], l[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float v = __builtin_canonicalizef(x[e]);  // (a NaN keeps its quiet bit in the truncated piece)
    h[e] = __float_as_uint(v);
    const float hf = __uint_as_float(h[e] & 0xffff0000u);
    const float r = fabsf(hf) < __builtin_inff() ? v - hf : 0.f;  // exact; inf and NaN live in hi alone
    m[e] = __float_as_uint(r);
    l[e] = __float_as_uint(r - __uint_as_float(m[e] & 0xffff0000u));
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {  // the high halves of two words
    o[0][q] = __builtin_amdgcn_perm(h[2 * q + 1], h[2 * q], 0x07060302);
    o[1][q] = __builtin_amdgcn_perm(m[2 * q + 1], m[2 * q], 0x07060302);
    o[2][q] = __builtin_amdgcn_perm(l[2 * q + 1], l[2 * q], 0x07060302);
  }
}
// 8 int8 values as bf16 (exact)
__device__ __forceinline__ bf16x8 w8_bf16(uint32_t w0, uint32_t w1) {
  bf16x8 r;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint32_t w = e < 4 ? w0 : w1;
    r[e] = (__bf16)(float)((int32_t)(w << (24 - 8 * (e & 3))) >> 24);
  }
  return r;
}

// four values of x row m at column k, as pieces
template <int MP>
__device__ __forceinline__ void put_pieces(char* xs, int stride, int m, int k, const f32x4& v) {
  u32x2 pc[3];
  split3(v, pc);
#pragma unroll
  for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x2*>(xs + (p * MP + m) * stride + 2 * k) = pc[p];
}

// One K step (256 inputs): weights w (rows g + 4 r, bytes 16 j .. + 15) through the wave's tile, times the x pieces at
// xc (the step's first column), into acc (GS: the two groups' sums scaled by sc[row][group])
template <int CT, bool GS>
__device__ __forceinline__ void gemv_mfma_step(char* wt, const u32x4 (&w)[4], const f32x2u (&sc)[4], const char* xc,
                                               const uint32_t (&boff)[CT], f32x4 (&acc)[CT]) {
  const int lane = threadIdx.x & 63, kg = lane >> 4, j = lane & 15;
  asm volatile("" ::: "memory");  // (LDS operations of a wave complete in order)
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = kg + 4 * r;
    *reinterpret_cast<u32x4*>(wt + row * 256 + ((j ^ row) << 4)) = w[r];
  }
  asm volatile("" ::: "memory");
  u32x4 a[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) a[i] = *reinterpret_cast<const u32x4*>(wt + j * 256 + (((4 * i + kg) ^ j) << 4));
  f32x4 ga[CT];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const bf16x8 wf = w8_bf16(a[i][2 * h], a[i][2 * h + 1]);
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        const bf16x8 xf = *reinterpret_cast<const bf16x8*>(xc + boff[c] + 128 * i + 16 * h);
        if constexpr (GS) ga[c] = mfma16(wf, xf, (i & 1) == 0 && h == 0 ? zero4() : ga[c]);
        else acc[c] = mfma16(wf, xf, acc[c]);
      }
    }
    if constexpr (GS) {
      if (i & 1) {
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[c][r] += sc[r][i >> 1] * ga[c][r];
      }
    }
  }
}

// x's columns kb0 .. kb0 + Kb - 1 into LDS as pieces (row p * MP + m holds piece p of x row m, `stride` bytes apart:
// 16 rows at one column fall in distinct 16-byte slots), with the prologues of gemv_kernel: NORM stages
// (x + xadd)(1 + nw), leaves the sums of squares per wave in ssw and writes the sum to xout from block 0; GN the gated
// norm. The first chunk's operands are loaded before `issue` sends out the weights, so that the staging does not wait
// behind them.
template <int MP, bool NORM, bool GN, class Issue>
__device__ __forceinline__ void stage_pieces(char* xs, int stride, const float* __restrict__ x, int64_t ldx, int M, int K,
                                             int kb0, int Kb, const float* __restrict__ xadd,
                                             const float* __restrict__ nw, float eps, float* __restrict__ xout,
                                             const GemvAux& aux, float (*ssw)[MP], Issue&& issue) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kf = 4 * tid;
  constexpr int FV = NORM ? MP : 1;
  f32x4 fv[FV], fa[FV], fw = zero4();
#pragma unroll
  for (int m = 0; m < FV; ++m) {
    fv[m] = zero4();
    fa[m] = zero4();
  }
  if (NORM) {
    if (kf < K) {
      fw = *reinterpret_cast<const f32x4*>(nw + kf);
#pragma unroll
      for (int m = 0; m < FV; ++m) {
        if (MP < 8 || m < M) fv[m] = *reinterpret_cast<const f32x4*>(x + m * ldx + kf);
        if ((MP < 8 || m < M) && xadd) fa[m] = *reinterpret_cast<const f32x4*>(xadd + m * ldx + kf);
      }
    }
  } else if (!GN) {
    const int m0 = kf / Kb, k0 = kf - m0 * Kb;
    if (m0 < M && kf < MP * Kb) fv[0] = *reinterpret_cast<const f32x4*>(x + m0 * ldx + kb0 + k0);
  }
  constexpr int kGnPre = GN ? 2 : 1;
  f32x4 go[kGnPre], gz[kGnPre], gw[kGnPre];
  float gh[kGnPre];
  if constexpr (GN) {
#pragma unroll
    for (int q = 0; q < kGnPre; ++q) {
      go[q] = zero4(); gz[q] = zero4(); gw[q] = zero4(); gh[q] = 1.f;
      const int i = tid + q * (int)blockDim.x;
      const int m = (4 * i) / Kb, kk = kb0 + 4 * i - m * Kb;
      if (i < MP * Kb / 4 && m < M) {
        go[q] = *reinterpret_cast<const f32x4*>(x + m * ldx + kk);
        gz[q] = *reinterpret_cast<const f32x4*>(aux.z + m * aux.ldz + kk);
        gw[q] = *reinterpret_cast<const f32x4*>(nw + (kk & (kGemvHead - 1)));
        if (aux.hs) gh[q] = aux.hs[kk / kGemvHead];
      }
    }
  }
  issue();
  asm volatile("" ::: "memory");
  if (NORM) {
    float ss[MP];
#pragma unroll
    for (int m = 0; m < MP; ++m) ss[m] = 0.f;
    auto chunk = [&](int k, const f32x4& w, const f32x4 (&v)[FV], const f32x4 (&a)[FV]) {
#pragma unroll
      for (int m = 0; m < FV; ++m) {
        f32x4 t = v[m];
        if (xadd) {
#pragma unroll
          for (int e = 0; e < 4; ++e) t[e] += a[m][e];
        }
        if (xout && blockIdx.x == 0 && (MP < 8 || m < M)) *reinterpret_cast<f32x4*>(xout + m * ldx + k) = t;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          ss[m] += t[e] * t[e];
          t[e] *= 1.f + w[e];
        }
        put_pieces<MP>(xs, stride, m, k, t);
      }
    };
    // the first chunk outside the loop: inside it, the wait for its operands would merge with the loop's own loads into
    // a wait for everything, the weights included
    if (kf < K) chunk(kf, fw, fv, fa);
    for (int k = kf + 4 * (int)blockDim.x; k < K; k += 4 * (int)blockDim.x) {
      const f32x4 w = *reinterpret_cast<const f32x4*>(nw + k);
      f32x4 v[FV], a[FV];
#pragma unroll
      for (int m = 0; m < FV; ++m) {
        v[m] = a[m] = zero4();
        if (MP < 8 || m < M) v[m] = *reinterpret_cast<const f32x4*>(x + m * ldx + k);
        if ((MP < 8 || m < M) && xadd) a[m] = *reinterpret_cast<const f32x4*>(xadd + m * ldx + k);
      }
      chunk(k, w, v, a);
    }
#pragma unroll
    for (int m = 0; m < MP; ++m) {
      const float t = wave_sum_f(ss[m]);
      if (lane == 0) ssw[wave][m] = t;
    }
  } else if (GN) {
    // gated RMSNorm per head of 128 inputs, a head's 32 quads in one half wave (see gemv_kernel)
    auto quad = [&](int i, const f32x4& o, const f32x4& zz, const f32x4& w, float hsc) {
      const int m = (4 * i) / Kb, k = 4 * i - m * Kb;
      const float ss = half_sum_f(o[0] * o[0] + o[1] * o[1] + o[2] * o[2] + o[3] * o[3]);
      const float r = rsqrtf(ss * (1.f / kGemvHead) + eps);
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = w[e] * (o[e] * r) * gsilu(zz[e]) * hsc;
      put_pieces<MP>(xs, stride, m, k, v);
    };
#pragma unroll
    for (int q = 0; q < kGnPre; ++q) {  // (the first quads outside the loop, as above)
      const int i = tid + q * (int)blockDim.x;
      if (i < MP * Kb / 4) quad(i, go[q], gz[q], gw[q], gh[q]);
    }
    for (int i = tid + kGnPre * (int)blockDim.x; i < MP * Kb / 4; i += blockDim.x) {
      const int m = (4 * i) / Kb, kk = kb0 + 4 * i - m * Kb;
      f32x4 o = zero4(), zz = zero4(), w = zero4();
      float hsc = 1.f;
      if (m < M) {
        o = *reinterpret_cast<const f32x4*>(x + m * ldx + kk);
        zz = *reinterpret_cast<const f32x4*>(aux.z + m * aux.ldz + kk);
        w = *reinterpret_cast<const f32x4*>(nw + (kk & (kGemvHead - 1)));
        if (aux.hs) hsc = aux.hs[kk / kGemvHead];
      }
      quad(i, o, zz, w, hsc);
    }
  } else {
    auto put = [&](int i, const f32x4& v) {
      const int m = (4 * i) / Kb, k = 4 * i - m * Kb;
      put_pieces<MP>(xs, stride, m, k, v);
    };
    if (tid < MP * Kb / 4) put(tid, fv[0]);  // (the first quad outside the loop, as above)
    for (int i = tid + (int)blockDim.x; i < MP * Kb / 4; i += blockDim.x) {
      const int m = (4 * i) / Kb, k = 4 * i - m * Kb;
      put(i, m < M ? *reinterpret_cast<const f32x4*>(x + m * ldx + kb0 + k) : zero4());
    }
  }
}

template <int MP, int EPI, int U, bool NORM, bool GS, bool GN>
__global__ __launch_bounds__(512) void gemv_mfma_kernel(const float* __restrict__ x, int64_t ldx,
                                                        const int8_t* __restrict__ W,
                                                        const float* __restrict__ wscale, float* __restrict__ y,
                                                        int64_t ldy, int M, int N, int K,
                                                        const q35_push* __restrict__ pushes, int npush, int T,
                                                        const float* __restrict__ xadd, const float* __restrict__ nw,
                                                        float eps, float* __restrict__ xout, GemvAux aux) {
  Q35_ARGS_UPFRONT(x, ldx, W, wscale, y, ldy, M, N, K, pushes, npush, T, xadd, nw, eps, xout);
  static_assert(!(GN && NORM), "one prologue");
  constexpr int CT = gemv_ct(MP);
  extern __shared__ __attribute__((aligned(16))) char dyn[];  // the waves' weight tiles, then the pieces of x
  __shared__ float ssw[8][MP];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int NW = blockDim.x >> 6;
  const int kg = lane >> 4, j = lane & 15;
  const int n0 = blockIdx.x * 16;
  const int nsplit = gridDim.y;
  const int spb = (K / 256 + nsplit - 1) / nsplit;
  const int sb = (int)blockIdx.y * spb, se = min(K / 256, sb + spb);
  if (sb >= se) return;
  const int kb0 = sb * 256, Kb = (se - sb) * 256;
  const int stride = 2 * Kb + 16;
  char* const xs = dyn + NW * kWTile;
  char* const wt = dyn + wave * kWTile;
  const int8_t* wr[4];
  const float* sr[4];  // GS: scales of rows 4 kg + r (the accumulator's rows), 2 per K step
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    wr[r] = W + (size_t)min(n0 + kg + 4 * r, N - 1) * K + 16 * j;
    sr[r] = GS ? wscale + (size_t)min(n0 + 4 * kg + r, N - 1) * (K >> 7) : nullptr;
  }
  u32x4 wc[U][4];
  f32x2u wsc[U][4];
  auto issue = [&](int s0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int st = min(s0 + u * NW, se - 1);
#pragma unroll
      for (int r = 0; r < 4; ++r) wc[u][r] = *reinterpret_cast<const u32x4*>(wr[r] + st * 256);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (GS) wsc[u][r] = *reinterpret_cast<const f32x2u*>(sr[r] + 2 * st);
      }
    }
  };
  float cvw[kGemvConvMaxK], cvs[kGemvConvMaxK - 1], cvb = 0.f;
  int pn = 0x7fffffff;
  stage_pieces<MP, NORM, GN>(xs, stride, x, ldx, M, K, kb0, Kb, xadd, nw, eps, xout, aux, ssw, [&] {
    if (EPI == kEpiSwiglu) pn = push_neuron(pushes, npush);
    issue(sb + wave);
    if constexpr (EPI == kEpiConv) {  // the epilogue thread's taps, bias and conv state, loaded behind the weights
  #pragma unroll
      for (int i = 0; i < kGemvConvMaxK; ++i) cvw[i] = 0.f;
  #pragma unroll
      for (int i = 0; i < kGemvConvMaxK - 1; ++i) cvs[i] = 0.f;
      const int rr = tid / MP, m = tid - rr * MP, nn = n0 + rr;
      if (tid < 16 * MP && m < M && nn < aux.cc) {
  #pragma unroll
        for (int i = 0; i < kGemvConvMaxK; ++i)
          if (i < aux.ck) cvw[i] = aux.cw[(size_t)nn * aux.ck + i];
  #pragma unroll
        for (int i = 0; i < kGemvConvMaxK - 1; ++i)
          if (i < aux.ck - 1) cvs[i] = aux.cst[((size_t)m * (aux.ck - 1) + i) * aux.cc + nn];
        if (aux.cb) cvb = aux.cb[nn];
      }
    }
  });
  lds_barrier();  // (the weights stay in flight)
  f32x4 acc[CT];
  uint32_t boff[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    acc[c] = zero4();
    boff[c] = (uint32_t)(min(16 * c + j, 3 * MP - 1) * stride + 32 * kg);
  }
  for (int s0 = sb + wave; s0 < se; s0 += U * NW) {
    if (s0 != sb + wave) issue(s0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int st = s0 + u * NW;
      if (st >= se) break;
      gemv_mfma_step<CT, GS>(wt, wc[u], wsc[u], xs + (st - sb) * 512, boff, acc);
    }
  }
  // the wave's sums into its weight tile: [column][16 rows]
  asm volatile("" ::: "memory");
#pragma unroll
  for (int c = 0; c < CT; ++c) *reinterpret_cast<f32x4*>(wt + ((16 * c + j) * 16 + 4 * kg) * 4) = acc[c];
  __syncthreads();
  unsigned long long best_key = 0ull;
  // row rr of the tile, row m of x: the waves' sums per piece in wave order, then lo + mid, then hi
  auto rowsum = [&](int rr, int m) {
    float pv[3];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      float t[8];
#pragma unroll
      for (int w = 0; w < 8; ++w)
        t[w] = w < NW ? *reinterpret_cast<const float*>(dyn + w * kWTile + ((p * MP + m) * 16 + rr) * 4) : 0.f;
      pv[p] = ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
    }
    float v = pv[0] + (pv[1] + pv[2]);
    if (NORM) {
      float t[8];
#pragma unroll
      for (int w = 0; w < 8; ++w) t[w] = w < NW ? ssw[w][m] : 0.f;
      v *= rsqrtf((((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]))) / (float)K + eps);
    }
    return v;
  };
  if (EPI != kEpiSwiglu) {
    if (tid < 16 * MP) {
      const int rr = tid / MP, m = tid - rr * MP;
      const int nn = n0 + rr;
      if (m < M && nn < N) {
        float v = rowsum(rr, m);
        if (wscale && !GS) v *= wscale[nn];
        float* dst = y + m * ldy + nn;
        if (EPI == kEpiConv && nn < aux.cc) {
          // causal conv over the channel's last ck inputs (the conv state, then v) + SiLU; state <- [rows 1.. | v]
          float a = cvb;
#pragma unroll
          for (int i = 0; i < kGemvConvMaxK; ++i) {
            if (i >= aux.ck) break;
            a += cvw[i] * (i < aux.ck - 1 ? cvs[i] : v);
          }
          float* cs = aux.cst + (size_t)m * (aux.ck - 1) * aux.cc + nn;
#pragma unroll
          for (int i = 0; i < kGemvConvMaxK - 1; ++i) {
            if (i >= aux.ck - 1) break;
            cs[(size_t)i * aux.cc] = i + 1 < aux.ck - 1 ? cvs[i + 1] : v;
          }
          *dst = silu_f(a);
        } else if (EPI == kEpiAccumulate && nsplit > 1) {
          __hip_atomic_fetch_add(dst, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
          *dst = EPI == kEpiAccumulate ? *dst + v : v;
          if (EPI == kEpiStore && aux.amax) best_key = amax_key(v, nn);
        }
      }
    }
  } else if (const bool touched = pushes_touch(pn, n0 >> 1, (n0 >> 1) + 8); tid < 8 * MP) {
    // rows 2 q and 2 q + 1 of the tile are gate and up of neuron n0 / 2 + q
    const int qn = tid / MP, m = tid - qn * MP;
    const int ng = n0 + 2 * qn;
    const int neuron = ng >> 1;
    if (m < M && ng + 1 < N) {
      float gt = rowsum(2 * qn, m), up = rowsum(2 * qn + 1, m);
      if (wscale && !GS) { gt *= wscale[ng]; up *= wscale[ng + 1]; }
      float a = gsilu(gt) * up;
      const int row = min(m / T, 3);
      if (touched)
        for (int p = 0; p < npush; ++p) a = apply_push(pushes + p, neuron, row, a);
      y[m * ldy + neuron] = a;
      if (aux.cap) aux.cap[(int64_t)(m / T) * aux.ldcr + (int64_t)(m % T) * aux.ldc + neuron] = a;
    }
  }
  if constexpr (EPI == kEpiStore) {
    if (aux.amax) {  // the block's best key per row of x, then one device-scope atomic max per row (see gemv_kernel)
      __shared__ unsigned long long kbest[16 * MP];
      if (tid < 16 * MP) kbest[tid] = best_key;
      __syncthreads();
      if (tid < MP && tid < M) {
        unsigned long long k = 0ull;
        for (int rr = 0; rr < 16; ++rr) k = kbest[rr * MP + tid] > k ? kbest[rr * MP + tid] : k;
        if (k) __hip_atomic_fetch_max(aux.amax + tid, k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
}

// Products with many tiles (the LM head: 9496): a wave takes whole 16-row tiles (wave w of the grid tiles w, w + the
// number of waves, ...) over all of K, so nothing crosses waves and the loop has no barrier: the previous form's blocks
// crossed one per 16 rows. Rounds of four K steps (16 KB of weights per wave), each step's buffer refilled for the next
// round, of this tile or the next, as soon as its products are done. Two blocks of four waves per CU: 128 KB in flight.
// The pieces of a row are summed between the accumulator's columns with two lane exchanges. 151,936 x 1024 with group
// scales, the norm and the argmax, at 1 / 3 / 5 / 8 rows: 38.8 / 39.0 / 39.7 / 42.9 us (160 MB: 3.7-4.1 TB/s), the block tile
// loop of gemv.hip 34.5 / 44.4 / 79.4 / 80.5; without the argmax 35.2 / 35.3 / 35.7 / 39.6 and 31.5 / 40.5 / 77.8 / 78.0.
// Which of the two runs at 1 to 3 rows: gemv_tiles_on_mfma.
template <int MP, int EPI, bool NORM, bool GS>
__global__ __launch_bounds__(256, 2) void gemv_tiles_kernel(const float* __restrict__ x, int64_t ldx,
                                                            const int8_t* __restrict__ W,
                                                            const float* __restrict__ wscale, float* __restrict__ y,
                                                            int64_t ldy, int M, int N, int K,
                                                            const q35_push* __restrict__ pushes, int npush, int T,
                                                            const float* __restrict__ xadd,
                                                            const float* __restrict__ nw, float eps,
                                                            float* __restrict__ xout, GemvAux aux) {
  Q35_ARGS_UPFRONT(x, ldx, W, wscale, y, ldy, M, N, K, pushes, npush, T, xadd, nw, eps, xout);
  constexpr int CT = gemv_ct(MP), NW = 4;
  extern __shared__ __attribute__((aligned(16))) char dyn[];  // the waves' weight tiles, then the pieces of x
  __shared__ float ssw[NW][MP];
  __shared__ unsigned long long kbest[NW][16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = lane >> 4, j = lane & 15;
  const int stride = 2 * K + 16;
  char* const xs = dyn + NW * kWTile;
  char* const wt = dyn + wave * kWTile;
  const int ntiles = (N + 15) / 16, KS = K / 256, step = (int)gridDim.x * NW;
  int tile = (int)blockIdx.x * NW + wave;
  u32x4 wc[4][4];
  f32x2u wsc[4][4];
  const int8_t* wr[4];
  const float* sr[4];
  auto set_rows = [&](int t) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      wr[r] = W + (size_t)min(t * 16 + kg + 4 * r, N - 1) * K + 16 * j;
      sr[r] = GS ? wscale + (size_t)min(t * 16 + 4 * kg + r, N - 1) * (K >> 7) : nullptr;
    }
  };
  auto fetch = [&](int st, auto u_c) {
    constexpr int u = decltype(u_c)::value;
#pragma unroll
    for (int r = 0; r < 4; ++r) wc[u][r] = *reinterpret_cast<const u32x4*>(wr[r] + st * 256);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (GS) wsc[u][r] = *reinterpret_cast<const f32x2u*>(sr[r] + 2 * st);
    }
  };
  constexpr std::integral_constant<int, 0> c0;
  constexpr std::integral_constant<int, 1> c1;
  constexpr std::integral_constant<int, 2> c2;
  constexpr std::integral_constant<int, 3> c3;
  const bool any = tile < ntiles;
  auto first = [&] {
    if (any) {
      set_rows(tile);
      fetch(0, c0);
      fetch(min(1, KS - 1), c1);
      fetch(min(2, KS - 1), c2);
      fetch(min(3, KS - 1), c3);
    }
  };
  // (8 rows: the staging's rows of x beside the weights' registers would spill, so the weights go out after it)
  stage_pieces<MP, NORM, false>(xs, stride, x, ldx, M, K, 0, K, xadd, nw, eps, xout, aux, ssw, [&] {
    if constexpr (MP < 8) first();
  });
  if constexpr (MP == 8) first();
  lds_barrier();  // (the weights stay in flight)
  const int mc = j;  // the lane's row of x, where j < M
  float rsf = 1.f;
  if (NORM && mc < MP) {
    const float ss = (ssw[0][mc] + ssw[1][mc]) + (ssw[2][mc] + ssw[3][mc]);
    rsf = rsqrtf(ss / (float)K + eps);
  }
  uint32_t boff[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) boff[c] = (uint32_t)(min(16 * c + j, 3 * MP - 1) * stride + 32 * kg);
  unsigned long long best_key = 0ull;
  const bool vec = EPI != kEpiSwiglu && (ldy & 3) == 0 && ((uintptr_t)y & 15) == 0;
  f32x4 acc[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) acc[c] = zero4();
  int s0 = 0;
  while (tile < ntiles) {
    // the next round: of this tile, or the next tile's first
    const int cur = tile, sc0 = s0;
    const bool last = s0 + 4 >= KS;
    s0 = last ? 0 : s0 + 4;
    if (last) {
      tile += step;
      if (tile < ntiles) set_rows(tile);
    }
    const bool more = tile < ntiles;
    auto one = [&](auto u_c) {
      constexpr int u = decltype(u_c)::value;
      if (sc0 + u < KS) gemv_mfma_step<CT, GS>(wt, wc[u], wsc[u], xs + (sc0 + u) * 512, boff, acc);
      if (more) fetch(min(s0 + u, KS - 1), u_c);
    };
    one(c0);
    one(c1);
    one(c2);
    one(c3);
    if (!last) continue;
    // rows n .. n + 3 (n = 16 tile + 4 kg) of x row j: lo + mid, then hi
    const int n = cur * 16 + 4 * kg;
    f32x4 v;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (CT == 1) {
        const float mid = __shfl(acc[0][r], (lane & 48) + ((j + MP) & 15), 64);
        const float lo = __shfl(acc[0][r], (lane & 48) + ((j + 2 * MP) & 15), 64);
        v[r] = acc[0][r] + (mid + lo);
      } else {
        static_assert(CT == 1 || MP == 8, "piece columns: hi at j, mid at j + 8, lo at j of the second tile");
        const float mid = __shfl(acc[0][r], (lane & 48) + ((j + 8) & 15), 64);
        v[r] = acc[0][r] + (mid + acc[CT - 1][r]);
      }
      v[r] *= rsf;
      if (!GS) v[r] *= wscale ? wscale[min(n + r, N - 1)] : 1.f;
    }
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[c] = zero4();
    if (j >= M) continue;
    if constexpr (EPI == kEpiSwiglu) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        if (n + 2 * q + 1 >= N) break;
        const int neuron = (n >> 1) + q;
        float a = gsilu(v[2 * q]) * v[2 * q + 1];
        const int row = min(j / T, 3);
        for (int p = 0; p < npush; ++p) a = apply_push(pushes + p, neuron, row, a);  // (few products have both)
        y[j * ldy + neuron] = a;
        if (aux.cap) aux.cap[(int64_t)(j / T) * aux.ldcr + (int64_t)(j % T) * aux.ldc + neuron] = a;
      }
    } else {
      float* dst = y + j * ldy + n;
      if (vec && n + 4 <= N) {
        f32x4 o = v;
        if (EPI == kEpiAccumulate) {
          const f32x4 old = *reinterpret_cast<const f32x4*>(dst);
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = old[r] + v[r];
        }
        *reinterpret_cast<f32x4*>(dst) = o;
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < N) dst[r] = EPI == kEpiAccumulate ? dst[r] + v[r] : v[r];
      }
      if (EPI == kEpiStore && aux.amax) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const unsigned long long kk = n + r < N ? amax_key(v[r], n + r) : 0ull;
          best_key = kk > best_key ? kk : best_key;
        }
      }
    }
  }
  if constexpr (EPI == kEpiStore) {
    if (aux.amax) {  // the block's best key per row of x, then one device-scope atomic max per row (see gemv_kernel)
#pragma unroll
      for (int off = 16; off < 64; off <<= 1) {
        const unsigned long long o = __shfl_xor(best_key, off, 64);
        best_key = o > best_key ? o : best_key;
      }
      if (kg == 0) kbest[wave][j] = best_key;
      __syncthreads();
      if (tid < M) {
        unsigned long long k = 0ull;
        for (int w = 0; w < NW; ++w) k = kbest[w][tid] > k ? kbest[w][tid] : k;
        if (k) __hip_atomic_fetch_max(aux.amax + tid, k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
}

// the matrix-core form (int8 weights, one 16-row tile per block; 4 rows of x or more)
template <int EPI, int U, bool NORM, bool GS, bool GN>
void gemv_mfma_launch_u(const float* x, int64_t ldx, const int8_t* W, const float* wscale, float* y, int64_t ldy,
                        int64_t M, int64_t N, int64_t K, const q35_push* pushes, int npush, int64_t T, int nw,
                        int nsplit, const GemvArgs& na, hipStream_t st) {
  const int64_t spb = (K / 256 + nsplit - 1) / nsplit;
  const size_t lds = gemv_mfma_lds(nw, M, spb * 256);
  const dim3 grid((unsigned)((N + 15) / 16), (unsigned)nsplit), block(64 * nw);
#define Q35_GEMV_MFMA(MP)                                                                                          \
  hipLaunchKernelGGL((gemv_mfma_kernel<MP, EPI, U, NORM, GS, GN>), grid, block, lds, st, x, ldx, W, wscale, y, ldy, \
                     (int)M, (int)N, (int)K, pushes, npush, (int)T, na.xadd, na.nw, na.eps, na.xout, na.aux)
  switch (gemv_mfma_rows(M)) {
    case 4: Q35_GEMV_MFMA(4); break;
    case 5: Q35_GEMV_MFMA(5); break;
    default: Q35_GEMV_MFMA(8); break;
  }
#undef Q35_GEMV_MFMA
}

// the matrix-core form with a tile loop per wave (int8 weights, many tiles): two blocks per CU
template <int EPI, bool NORM, bool GS>
void gemv_tiles_launch(const float* x, int64_t ldx, const int8_t* W, const float* wscale, float* y, int64_t ldy,
                       int64_t M, int64_t N, int64_t K, const q35_push* pushes, int npush, int64_t T,
                       const GemvArgs& na, hipStream_t st) {
  const size_t lds = gemv_mfma_lds(4, M, K);
  const int64_t blocks = ((N + 15) / 16 + 3) / 4;
  const dim3 grid((unsigned)(blocks < kGemvTileBlocks ? blocks : kGemvTileBlocks)), block(256);
#define Q35_GEMV_TILES(MP)                                                                                         \
  hipLaunchKernelGGL((gemv_tiles_kernel<MP, EPI, NORM, GS>), grid, block, lds, st, x, ldx, W, wscale, y, ldy, (int)M, \
                     (int)N, (int)K, pushes, npush, (int)T, na.xadd, na.nw, na.eps, na.xout, na.aux)
  switch (gemv_mfma_rows(M)) {
    case 1: Q35_GEMV_TILES(1); break;
    case 2: Q35_GEMV_TILES(2); break;
    case 3: Q35_GEMV_TILES(3); break;
    case 4: Q35_GEMV_TILES(4); break;
    case 5: Q35_GEMV_TILES(5); break;
    default: Q35_GEMV_TILES(8); break;
  }
#undef Q35_GEMV_TILES
}

template <bool NORM, bool GN, bool GS, int EPI>
static int gemv_mfma_epi(const float* x, int64_t ldx, const int8_t* W, const float* wscale, float* y, int64_t ldy,
                         int64_t M, int64_t N, int64_t K, const q35_push* pushes, int npush, int64_t T, int nsplit,
                         const GemvArgs& na, hipStream_t st) {
  if constexpr (EPI != kEpiConv && !GN) {
    if (nsplit == 1 && (N + 15) / 16 > kGemvMaxBlocks) {
      gemv_tiles_launch<EPI, NORM, GS>(x, ldx, W, wscale, y, ldy, M, N, K, pushes, npush, T, na, st);
      return hipGetLastError() == hipSuccess ? Q35_OK : Q35_ELAUNCH;
    }
  }
  // 4 waves when a block has at most 4 K steps, else 8; a wave's steps in flight together up to 2
  const int64_t bsteps = (K / 256 + nsplit - 1) / nsplit;
  const int nw = bsteps <= 4 ? 4 : 8;
  if ((bsteps + nw - 1) / nw <= 1)
    gemv_mfma_launch_u<EPI, 1, NORM, GS, GN>(x, ldx, W, wscale, y, ldy, M, N, K, pushes, npush, T, nw, nsplit, na, st);
  else
    gemv_mfma_launch_u<EPI, 2, NORM, GS, GN>(x, ldx, W, wscale, y, ldy, M, N, K, pushes, npush, T, nw, nsplit, na, st);
  return hipGetLastError() == hipSuccess ? Q35_OK : Q35_ELAUNCH;
}

template <bool NORM, bool GN, bool GS>
static int gemv_mfma_gs(int epi, const float* x, int64_t ldx, const int8_t* W, const float* wscale, float* y,
                        int64_t ldy, int64_t M, int64_t N, int64_t K, const q35_push* pushes, int npush, int64_t T,
                        int nsplit, const GemvArgs& na, hipStream_t st) {
  if constexpr (NORM) {
    if (epi == kEpiConv)
      return gemv_mfma_epi<NORM, GN, GS, kEpiConv>(x, ldx, W, wscale, y, ldy, M, N, K, pushes, npush, T, nsplit, na, st);
  }
  if constexpr (!GN) {
    if (epi == kEpiSwiglu)
      return gemv_mfma_epi<NORM, GN, GS, kEpiSwiglu>(x, ldx, W, wscale, y, ldy, M, N, K, pushes, npush, T, nsplit, na,
                                                     st);
  }
  if (epi == kEpiAccumulate)
    return gemv_mfma_epi<NORM, GN, GS, kEpiAccumulate>(x, ldx, W, wscale, y, ldy, M, N, K, pushes, npush, T, nsplit, na,
                                                       st);
  return gemv_mfma_epi<NORM, GN, GS, kEpiStore>(x, ldx, W, wscale, y, ldy, M, N, K, pushes, npush, T, nsplit, na, st);
}

int gemv_mfma_run(bool norm, bool gn, bool gs, int epi, const float* x, int64_t ldx, const int8_t* W,
                  const float* wscale, float* y, int64_t ldy, int64_t M, int64_t N, int64_t K, const q35_push* pushes,
                  int npush, int64_t T, int nsplit, const GemvArgs& na, hipStream_t st) {
#define Q35_GEMV_RUN(NORM, GN, GS) \
  return gemv_mfma_gs<NORM, GN, GS>(epi, x, ldx, W, wscale, y, ldy, M, N, K, pushes, npush, T, nsplit, na, st)
  if (norm) {
    if (gs) Q35_GEMV_RUN(true, false, true);
    Q35_GEMV_RUN(true, false, false);
  }
  if (gn) {
    if (gs) Q35_GEMV_RUN(false, true, true);
    Q35_GEMV_RUN(false, true, false);
  }
  if (gs) Q35_GEMV_RUN(false, false, true);
  Q35_GEMV_RUN(false, false, false);
#undef Q35_GEMV_RUN
}

}  // namespace q35
