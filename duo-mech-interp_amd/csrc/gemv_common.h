// What the decode GEMV's two translation units share: gemv.hip (fp32 FMA) and gemv_mfma.hip (matrix core).
#pragma once
#include "q35_common.h"
#include "q35hip.h"

namespace q35 {

enum GemvEpi : int { kEpiStore = 0, kEpiAccumulate = 1, kEpiSwiglu = 2, kEpiConv = 3 };
constexpr int kEpiAccumulateFixed = 4;  // entry-point code: accumulate, every output summed in one fixed order
constexpr int kGemvConvMaxK = 8;  // conv taps supported by the conv epilogue
constexpr int kGemvHead = 128;    // head size of the gated-norm prologue
// Tiles of 16 output rows (8 for fp32 weights at more than 4 rows of x) past which blocks or waves loop over tiles, x staged
// once per block (the LM head: 9496); products with fewer take one tile per block (measured faster for them). Also the
// blocks of gemv.hip's loop: four of 4 waves per CU at 128 VGPRs.
constexpr int64_t kGemvMaxBlocks = 1024;
constexpr int64_t kGemvLds = 160 * 1024;  // LDS of a CU

// The matrix-core form: blocks of its tile loop (two per CU), bytes of a wave's weight tile (16 rows x one K step), the
// rows of x that it is compiled for, and the LDS of a block of nw waves that stages K columns of M rows (three bf16
// pieces each).
constexpr int64_t kGemvTileBlocks = 512;
constexpr int kWTile = 16 * 256;
constexpr int gemv_mfma_rows(int64_t M) { return M <= 5 ? (int)M : 8; }
constexpr size_t gemv_mfma_lds(int nw, int64_t M, int64_t K) {
  return (size_t)nw * kWTile + (size_t)3 * gemv_mfma_rows(M) * (2 * K + 16);
}

// Operands of the gated-norm prologue (GN) and of the conv epilogue (kEpiConv); unused by the other forms.
struct GemvAux {
  const float* z;    // GN: gate rows z[m * ldz + k]
  int64_t ldz;
  const float* hs;   // GN: per-head scale (may be NULL)
  const float* cw;   // conv: weights [cc][ck]
  const float* cb;   // conv: bias [cc] (may be NULL)
  float* cst;        // conv: state [M][ck - 1][cc]
  int cc, ck;        // conv: channels (outputs 0 .. cc - 1 are convolved), taps
  float* cap;        // SwiGLU: activation capture (may be NULL): row m, neuron n at
  int64_t ldc, ldcr; //   cap[(m / T) ldcr + (m % T) ldc + n]
  unsigned long long* amax;  // store: per-row argmax keys (may be NULL), see amax_key
};

// Argmax key of output n with value v: the order-preserving bits of v above the complement of n, so that the largest
// key is the largest value and, among equal values, the lowest index (as argmax_rows_kernel and torch.argmax). -0
// ranks as +0; NaN gets 0, the empty key, and never wins (the scan's strict comparisons). A real key is never 0.
__device__ __forceinline__ unsigned long long amax_key(float v, int n) {
  if (!(v == v)) return 0ull;
  if (v == 0.f) v = 0.f;
  uint32_t b = __float_as_uint(v);
  b = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
  return ((unsigned long long)b << 32) | (0xFFFFFFFFu - (uint32_t)n);
}

__device__ __forceinline__ float gsilu(float x) { return silu_f(x); }

// Whether any push record can touch neurons nlo .. nhi - 1 (a record for every neuron, or for one in the range): the
// model passes eight records per layer, unused ones matching no neuron, and an epilogue that walks them pays one memory
// round trip per record. Lane p of a wave takes record p (npush <= 64): push_neuron's load goes out ahead of the
// weights, pushes_touch votes on it in the epilogue.
__device__ __forceinline__ int push_neuron(const q35_push* ps, int npush) {
  const int p = threadIdx.x & 63;
  return p < npush ? ps[p].neuron : 0x7fffffff;
}
__device__ __forceinline__ bool pushes_touch(int pn, int nlo, int nhi) {
  return __any(pn < 0 || (pn >= nlo && pn < nhi));
}

// one push applied to activation a of neuron n (fields read straight from the record: no copy of the value array)
__device__ __forceinline__ float apply_push(const q35_push* ps, int n, int row, float a) {
  const int pn = ps->neuron;
  if (pn != n && pn >= 0) return a;
  const float v = ps->vals[row];
  return ps->mode ? a * v : a + v;
}

// sum over the 16 lanes of a DPP row (lanes 16 r .. 16 r + 15), result in every lane of the row
__device__ __forceinline__ float row16_sum_f(float v) { return add_xor<8>(add_xor4_quads(add_xor<2>(add_xor<1>(v)))); }

// sum over 32 lanes (lanes 0 .. 31 or 32 .. 63), and over the wave, in every lane
__device__ __forceinline__ float half_sum_f(float v) { return add_xor<16>(row16_sum_f(v)); }
__device__ __forceinline__ float wave_sum_f(float v) { return add_xor<32>(half_sum_f(v)); }

// the prologues' operands (GN: nw is the gated norm's weight) and the epilogues'
struct GemvArgs {
  const float* xadd;
  const float* nw;
  float eps;
  float* xout;
  GemvAux aux;
};

// The matrix-core form (int8 weights): gemv_mfma.hip. gs: group scales; norm / gn: the RMSNorm and gated-norm prologues
// (norm also runs the conv epilogue). nsplit > 1: split K over blocks (accumulate). Returns a q35 status.
int gemv_mfma_run(bool norm, bool gn, bool gs, int epi, const float* x, int64_t ldx, const int8_t* W,
                  const float* wscale, float* y, int64_t ldy, int64_t M, int64_t N, int64_t K, const q35_push* pushes,
                  int npush, int64_t T, int nsplit, const GemvArgs& na, hipStream_t st);

}  // namespace q35
