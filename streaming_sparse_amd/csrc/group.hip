// Clean-commit token grouping for gfx950: the order in which a committed
// chunk's 4608 tokens fill its 72 pages (RV/runtime.py:57-68 GroupingOps.group).
//
//   features  f = (k - mean k).bank / sqrt(128) scaled to unit RMS, plus
//             0.1 tanh(gate) times the unit-RMS centred softmax response of
//             v.group_v                                  (LE/all_sparse_model.py:16-23)
//   balanced  7 levels of splits (3,3,2,2,2 over the chunk, then 2,2 inside
//             each page): each group is centred, a direction starts at the
//             one-hot of its highest-variance feature, takes 4 power steps,
//             and the group is stably sorted by its projection
//                                                        (LE/response_hard.py:20-31)
//   pages     a page permutation (Config.page_order, RV/ops.py:25-28)
//   chunk 0   a stable re-sort by frame, so the anchor frame fills pages
//             0..23                                      (VR/runtime.py:358-363)
//
// Everything after the bf16 inputs is fp64, so the order does not hinge on
// float32 rounding.  The batch is layers x heads independent rows b; a row's
// features are 1.2 MB, so the passes over them in memory set the time of the
// first two levels, and the work of every level is laid out to need few:
//   project_kernel   grid (18 token blocks, B): raw key and value projections
//                    on the fp64 matrix pipe, with the block's share of every
//                    head-wide statistic (moments, softmax sums)
//   totals_kernel    grid (B): the statistics over the row, feature constants
//   features_kernel  grid (18, B): features, and the block's Gram matrix
//   direction_kernel grid (B): level 0's direction from the Gram matrix (the
//                    power step X^T (X d) is (X^T X) d: 32 x 32 per step
//                    instead of a pass over the rows)
//   keys_kernel, sort_kernel  grid (18, B), (B): level 0's projections, sort
//   level_kernel     grid (3 B), (9 B): levels 1 and 2 (groups of 1536 and
//                    512): Gram matrix, direction, projections and sort; rows
//                    are read where they lie, through the previous order
//   fused_levels_kernel  grid (B x 18): levels 3..6 inside each 256-row group
//   frames_kernel    grid (B): the first chunk's stable partition by frame
// 30 layers x 12 heads: 5.26 ms (a workgroup per row and seven passes over its
// rows per level, sums over rows through serial LDS walks, bitonic sorts in
// LDS) -> 1.92 ms: project 0.59, totals 0.01, features 0.24, level 0 0.24
// (direction 0.014, keys 0.11, sort 0.12), level 1 0.20, level 2 0.17, fused
// levels 0.49.  One layer x 12 heads: 862 -> 249 us.
#include "common.h"

#include <type_traits>

using namespace ssa;

namespace {

constexpr int kTokens = 4608;      // 3 frames x 1536
constexpr int kFrame = 1536;
constexpr int kR = 32;             // feature width
constexpr int kPages = 72;
constexpr double kScale = 0.08838834764831844055;   // 1 / sqrt(128)
constexpr int kBlkTok = 256;                        // tokens of a block
constexpr int kBlks = kTokens / kBlkTok;            // 18

typedef double f64x4 __attribute__((ext_vector_type(4)));

// D[16x16] += A[16x4] * B[4x16] in fp64.  Lane l: A row l % 16, k = l / 16;
// B col l % 16, same k; D col l % 16, rows l / 16 + 4 i for item i.
__device__ __forceinline__ f64x4 mfma64(double a, double b, f64x4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

struct GroupParams {
  const uint16_t* k;
  const uint16_t* v;
  long long layer_stride, tok_stride, head_stride;   // elements
  const float* bank;       // [B][32][128]
  const float* gv;         // [B][128][32]
  const float* gate;       // [B][32]
  const int32_t* page_dst; // [72] destination page of grouped page p, or null
  // x[0]: [B][4608][32] raw key projections, then the features.  x[1]: the
  // value projections; once the features are formed, per token block (8192
  // doubles) its Gram matrix at 0, level 0's sort keys at kKeysAt, and in
  // block 0 level 0's mean and direction at kVecAt.
  double* x[2];
  // ids[0] and ids[1]: [B][4608] orders; before them, the statistics of each
  // row (kStatInts ints of the whole array per row; doubles at 4-byte alignment)
  int32_t* ids[2];
  int32_t* order;          // [B][4608]
  int H, B;
};

__device__ __forceinline__ const uint16_t* row_ptr(const uint16_t* base, const GroupParams& p, int b, int t) {
  const int l = b / p.H, h = b % p.H;
  return base + (long long)l * p.layer_stride + (long long)t * p.tok_stride + (long long)h * p.head_stride;
}

constexpr int kBlkDoubles = kBlkTok * kR;           // one block's rows in x[0] or x[1]
constexpr int kGramDoubles = 3 * 256;               // tiles (0,0), (0,1), (1,1) of 16 x 16 features
constexpr int kKeysAt = 1024, kVecAt = 2048;
constexpr int kStatVals = 8;
constexpr int kStatInts = kBlks * kR * kStatVals * 2;
static_assert(kStatInts == 2 * kTokens, "a row's statistics fill its share of the order scratch");

struct alignas(4) Double4 { uint32_t w[2]; };       // a double at 4-byte alignment
__device__ __forceinline__ double get_double(const int32_t* p) {
  const Double4 d = *reinterpret_cast<const Double4*>(p);
  return __longlong_as_double((long long)(((unsigned long long)d.w[1] << 32) | d.w[0]));
}
__device__ __forceinline__ void put_double(int32_t* p, double v) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(v);
  *reinterpret_cast<Double4*>(p) = Double4{{(uint32_t)u, (uint32_t)(u >> 32)}};
}

// Statistics of one feature over a set of n tokens, raw key projections x
// and value projections v: mean and M2 = sum (x - mean)^2; with the softmax
// weights e = exp((x - mx) / sqrt(D)), mx = max x (the mean cancels): den =
// sum e, num = sum e v; and of the squared weights, W2 = sum e^2, their mean
// m2 of v and M = sum e^2 (v - m2)^2.  Sets merge without cancellation (every
// term of a merged sum of squares is non-negative), so that the response's
// sum of squares sum e^2 (v - mean_a)^2 = M + W2 (m2 - mean_a)^2 needs no
// pass of its own after mean_a = num / den is known.
struct Stat {
  double n, mean, M2, mx, den, num, W2, m2, M;
};

__device__ __forceinline__ double ratio(double a, double b) { return b > 0.0 ? a / b : 0.0; }

__device__ __forceinline__ Stat merge(const Stat& a, const Stat& b) {
  Stat o;
  o.n = a.n + b.n;
  const double d = b.mean - a.mean, wb = b.n / o.n;
  o.mean = fma(d, wb, a.mean);
  o.M2 = a.M2 + b.M2 + d * d * (a.n * wb);
  o.mx = fmax(a.mx, b.mx);
  const double fa = exp((a.mx - o.mx) * kScale), fb = exp((b.mx - o.mx) * kScale);
  o.den = a.den * fa + b.den * fb;
  o.num = a.num * fa + b.num * fb;
  const double wa2 = a.W2 * (fa * fa), wb2 = b.W2 * (fb * fb);
  o.W2 = wa2 + wb2;
  const double e = b.m2 - a.m2, w = ratio(wb2, o.W2);
  o.m2 = fma(e, w, a.m2);
  o.M = a.M * (fa * fa) + b.M * (fb * fb) + e * e * (wa2 * w);
  return o;
}

template <int O>
__device__ __forceinline__ Stat xor_stat(const Stat& s) {
  return Stat{s.n, xor_lane<O>(s.mean), xor_lane<O>(s.M2), xor_lane<O>(s.mx), xor_lane<O>(s.den),
              xor_lane<O>(s.num), xor_lane<O>(s.W2), xor_lane<O>(s.m2), xor_lane<O>(s.M)};
}

// raw[b][t][r] = k_t . bank_r and vp[b][t][r] = v_t . gv[:, r] in fp64 (exact
// products of bf16 and fp32 values) on v_mfma_f64_16x16x4: wave w takes
// features 16 (w % 2) .. + 15 of both projections for tokens 128 (w / 2) ..
// + 127 of the block, 16 at a time.  Lane (c = l % 16, g = l / 16) holds both
// weight matrices' feature c at dims 32 g .. 32 g + 31 in registers for the
// whole block and reads its share of a token row as 64 consecutive bytes (the
// k order of the product is free, so no LDS staging is needed).  Bound by the
// fp64 pipe: 27.2 GFLOP per 30-layer batch, 0.39 ms at the 70 TFLOP/s a loop
// of these products reaches, and the operands' conversions (to 0.51 ms) and
// the statistics (to 0.59 ms) share it; as fp64 vector FMAs with a conversion
// per operand the projections alone took 1.01 ms.
__global__ __launch_bounds__(256, 2) void project_kernel(GroupParams p) {
  __shared__ double sh[2][16][kStatVals];
  const int blk = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int f = wave & 1, half = wave >> 1, c = lane & 15, g = lane >> 4;
  double wk[32], wv[32];
  {
    const float* bk = p.bank + ((long long)b * kR + 16 * f + c) * kHeadDim + 32 * g;
    const float* gv = p.gv + (long long)b * kR * kHeadDim + (32 * g) * kR + 16 * f + c;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const f32x4 w = reinterpret_cast<const f32x4*>(bk)[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) wk[4 * i + e] = (double)w[e];
    }
#pragma unroll
    for (int s = 0; s < 32; ++s) wv[s] = (double)gv[s * kR];
  }
  const int t0 = blk * kBlkTok + 128 * half;
  u32x4 ka[4], va[4];
  auto load = [&](int i) {
    const uint16_t* kp = row_ptr(p.k, p, b, t0 + 16 * i + c) + 32 * g;
    const uint16_t* vp = row_ptr(p.v, p, b, t0 + 16 * i + c) + 32 * g;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      ka[j] = ldg16(kp + 8 * j);
      va[j] = ldg16(vp + 8 * j);
    }
  };
  load(0);
  Stat st{0.0, 0.0, 0.0, -INFINITY, 0.0, 0.0, 0.0, 0.0, 0.0};
  double s1 = 0.0, s2 = 0.0, shift = 0.0;
#pragma unroll 1
  for (int i = 0; i < 8; ++i) {
    f64x4 rk = {}, rv = {};
    u32x4 ck[4], cv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      ck[j] = ka[j];
      cv[j] = va[j];
    }
    if (i < 7) load(i + 1);
#pragma unroll
    for (int s = 0; s < 32; ++s) {
      const uint32_t a = ck[s >> 3][(s >> 1) & 3], v = cv[s >> 3][(s >> 1) & 3];
      rk = mfma64((double)(s & 1 ? bf16_hi(a) : bf16_lo(a)), wk[s], rk);
      rv = mfma64((double)(s & 1 ? bf16_hi(v) : bf16_lo(v)), wv[s], rv);
    }
    const long long e0 = ((long long)b * kTokens + t0 + 16 * i + g) * kR + 16 * f + c;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      p.x[0][e0 + 4 * j * kR] = rk[j];
      p.x[1][e0 + 4 * j * kR] = rv[j];
    }
    if (i == 0) shift = rk[0];
    const double mn = fmax(fmax(st.mx, fmax(rk[0], rk[1])), fmax(rk[2], rk[3]));
    const double fr = exp((st.mx - mn) * kScale), fr2 = fr * fr;
    st.mx = mn;
    st.den *= fr;
    st.num *= fr;
    st.W2 *= fr2;
    st.M *= fr2;
    // the squared weights' moments of the tile's 4 tokens about their own
    // weighted mean, then merged: two divisions per tile
    double e2[4], wt = 0.0, at = 0.0, mt = 0.0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const double d = rk[j] - shift;
      s1 += d;
      s2 = fma(d, d, s2);
      const double e = exp((rk[j] - mn) * kScale);
      st.den += e;
      st.num = fma(e, rv[j], st.num);
      e2[j] = e * e;
      wt += e2[j];
      at = fma(e2[j], rv[j], at);
    }
    const double vm = ratio(at, wt);
#pragma unroll
    for (int j = 0; j < 4; ++j) mt = fma(e2[j] * (rv[j] - vm), rv[j] - vm, mt);
    const double dm = vm - st.m2, wn = st.W2 + wt, w = ratio(wt, wn);
    st.m2 = fma(dm, w, st.m2);
    st.M += mt + dm * dm * (st.W2 * w);
    st.W2 = wn;
  }
  st.n = 32.0;
  st.mean = shift + s1 / 32.0;
  st.M2 = fmax(s2 - s1 * (s1 / 32.0), 0.0);
  st = merge(st, xor_stat<16>(st));
  st = merge(st, xor_stat<32>(st));
  if (half == 1 && g == 0) {
    double* d = sh[f][c];
    d[0] = st.mean; d[1] = st.M2; d[2] = st.mx; d[3] = st.den; d[4] = st.num; d[5] = st.W2; d[6] = st.m2; d[7] = st.M;
  }
  __syncthreads();
  if (half == 0 && g == 0) {
    const double* d = sh[f][c];
    st = merge(st, Stat{st.n, d[0], d[1], d[2], d[3], d[4], d[5], d[6], d[7]});
    int32_t* o = p.ids[0] + (long long)b * kStatInts + (blk * kR + 16 * f + c) * (2 * kStatVals);
    const double v[kStatVals] = {st.mean, st.M2, st.mx, st.den, st.num, st.W2, st.m2, st.M};
#pragma unroll
    for (int k = 0; k < kStatVals; ++k) put_double(o + 2 * k, v[k]);
  }
}

// The statistics of one row b over its 18 blocks, and the constants of each
// feature (kConsts doubles, over the row's statistics): mean, 1 / (sqrt(D)
// rms), max, mean_a, and 0.1 tanh(gate) n / (den rms2).  Thread: feature
// tid % 32, blocks tid / 32 + 8 i, then a tree over the 8 parts.
constexpr int kConsts = 5;
__global__ __launch_bounds__(256) void totals_kernel(GroupParams p) {
  __shared__ Stat sh[8][kR];
  __shared__ double sq[2][kR];
  const int b = blockIdx.x, tid = threadIdx.x, r = tid & 31, part = tid >> 5;
  int32_t* stats = p.ids[0] + (long long)b * kStatInts;
  auto block = [&](int blk) {
    const int32_t* o = stats + (blk * kR + r) * (2 * kStatVals);
    double v[kStatVals];
#pragma unroll
    for (int k = 0; k < kStatVals; ++k) v[k] = get_double(o + 2 * k);
    return Stat{(double)kBlkTok, v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]};
  };
  Stat st = merge(block(part), block(part + 8));
  if (part < kBlks - 16) st = merge(st, block(part + 16));
  for (int h = 4; h > 0; h >>= 1) {
    if (part >= h && part < 2 * h) sh[part][r] = st;
    __syncthreads();
    if (part < h) st = merge(st, sh[part + h][r]);
    __syncthreads();
  }
  const double mean_a = st.num / st.den;
  if (part == 0) {
    const double dm = st.m2 - mean_a, an = kTokens / st.den;
    sq[0][r] = st.M2 * (kScale * kScale);
    sq[1][r] = (an * an) * (st.M + st.W2 * dm * dm);
  }
  __syncthreads();
  if (part > 0) return;
  double q0 = 0.0, q1 = 0.0;
  for (int k = 0; k < kR; ++k) {
    q0 += sq[0][k];
    q1 += sq[1][k];
  }
  const double rms = fmax(sqrt(q0 / (kTokens * kR)), 1e-6), rms2 = fmax(sqrt(q1 / (kTokens * kR)), 1e-6);
  const double g = 0.1 * tanh((double)p.gate[b * kR + r]);
  int32_t* o = stats + r * (2 * kConsts);
  put_double(o + 0, st.mean);
  put_double(o + 2, kScale / rms);
  put_double(o + 4, st.mx);
  put_double(o + 6, mean_a);
  put_double(o + 8, g * kTokens / (st.den * rms2));
}

// Sums of a wave's Gram tiles and row sums into LDS, in the order of
// kGramDoubles then 32 sums.
struct Gram {
  f64x4 t[3] = {};
  double lo = 0.0, hi = 0.0;      // this lane's share of the sums of features c and c + 16
  // rows: lane (c, g) holds features c (xl) and c + 16 (xh) of row g of four
  __device__ __forceinline__ void add(double xl, double xh) {
    t[0] = mfma64(xl, xl, t[0]);
    t[1] = mfma64(xl, xh, t[1]);
    t[2] = mfma64(xh, xh, t[2]);
    lo += xl;
    hi += xh;
  }
  // over the four lane groups
  __device__ __forceinline__ void fold() {
    lo += xor_lane<16>(lo);
    lo += xor_lane<32>(lo);
    hi += xor_lane<16>(hi);
    hi += xor_lane<32>(hi);
  }
  template <bool ADD>
  __device__ __forceinline__ void store(double* d, int lane) const {
    const int c = lane & 15, g = lane >> 4;
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        double* e = d + 256 * k + (g + 4 * i) * 16 + c;
        *e = ADD ? *e + t[k][i] : t[k][i];
      }
    if (g == 0) {
      d[kGramDoubles + c] = ADD ? d[kGramDoubles + c] + lo : lo;
      d[kGramDoubles + 16 + c] = ADD ? d[kGramDoubles + 16 + c] + hi : hi;
    }
  }
};
constexpr int kGramAll = kGramDoubles + kR;

// Features of one token block: x = (raw - mean) / (sqrt(D) rms) + gate n /
// (den rms2) exp((raw - max) / sqrt(D)) (vp - mean_a), and the block's Gram
// matrix and sums over them.  Lane (c, g): features c and c + 16 of token g
// of four.  Bound by memory: both projections in, the features out, 1.27 GB
// per 30-layer batch.
__global__ __launch_bounds__(256) void features_kernel(GroupParams p) {
  __shared__ double red[2][kGramAll];
  const int blk = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c = lane & 15, g = lane >> 4;
  double k[2][kConsts];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int32_t* o = p.ids[0] + (long long)b * kStatInts + (c + 16 * i) * (2 * kConsts);
#pragma unroll
    for (int j = 0; j < kConsts; ++j) k[i][j] = get_double(o + 2 * j);
  }
  const long long at = ((long long)b * kTokens + blk * kBlkTok + 64 * wave + g) * kR + c;
  double* x = p.x[0] + at;
  const double* v = p.x[1] + at;
  Gram gram;
#pragma unroll 1
  for (int i0 = 0; i0 < 16; i0 += 4) {
    double xr[4][2], vr[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        xr[i][h] = x[(4 * (i0 + i)) * kR + 16 * h];
        vr[i][h] = v[(4 * (i0 + i)) * kR + 16 * h];
      }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      double f[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const double e = exp((xr[i][h] - k[h][2]) * kScale);
        f[h] = fma(k[h][4] * e, vr[i][h] - k[h][3], (xr[i][h] - k[h][0]) * k[h][1]);
        x[(4 * (i0 + i)) * kR + 16 * h] = f[h];
      }
      gram.add(f[0], f[1]);
    }
  }
  gram.fold();
  // waves 2 and 3 store, waves 0 and 1 add, then the two halves together; the
  // value projections are read by now, so their space takes the result
  if (wave >= 2) gram.store<false>(red[wave - 2], lane);
  __syncthreads();
  if (wave < 2) gram.store<true>(red[wave], lane);
  __syncthreads();
  double* o = p.x[1] + ((long long)b * kBlks + blk) * kBlkDoubles;
  for (int i = tid; i < kGramAll; i += 256) o[i] = red[0][i] + red[1][i];
}

// Direction of a group of n rows from its Gram matrix and sums about `shift`
// (mean = shift + sum / n): starts at the one-hot of the highest-variance
// feature (first of equals), takes 4 power steps on the centred Gram matrix,
// each normalised (norm clamped at 1e-8).  One wave; lane i % 32 holds row i.
// gram: kGramAll doubles in LDS; vec: 32 doubles of LDS for the direction.
__device__ __forceinline__ double power_direction(const double* gram, double n, double* vec, int lane) {
  const int i = lane & 31;
  double row[kR];
  const double si = gram[kGramDoubles + i] / n;
#pragma unroll
  for (int j = 0; j < kR; ++j) {
    const double v = i < 16 ? (j < 16 ? gram[i * 16 + j] : gram[256 + i * 16 + j - 16])
                            : (j < 16 ? gram[256 + j * 16 + i - 16] : gram[512 + (i - 16) * 16 + j - 16]);
    row[j] = fma(-si, gram[kGramDoubles + j], v);
  }
  double var = row[0];
#pragma unroll
  for (int j = 1; j < kR; ++j) var = j == i ? row[j] : var;
  int axis = i;
  auto better = [&](double ov, int oi) {
    if (ov > var || (ov == var && oi < axis)) {
      var = ov;
      axis = oi;
    }
  };
  better(xor_lane<16>(var), xor_lane<16>(axis));
  better(xor_lane<8>(var), xor_lane<8>(axis));
  better(xor_lane<4>(var), xor_lane<4>(axis));
  better(xor_lane<2>(var), xor_lane<2>(axis));
  better(xor_lane<1>(var), xor_lane<1>(axis));
  double d = i == axis ? 1.0 : 0.0;
#pragma unroll 1
  for (int it = 0; it < 4; ++it) {
    vec[i] = d;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    double y[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int j = 0; j < kR; ++j) y[j & 3] = fma(row[j], vec[j], y[j & 3]);
    d = (y[0] + y[1]) + (y[2] + y[3]);
    double q = d * d;
    q += xor_lane<16>(q);
    q += xor_lane<8>(q);
    q += xor_lane<4>(q);
    q += xor_lane<2>(q);
    q += xor_lane<1>(q);
    d /= fmax(sqrt(q), 1e-8);
    __builtin_amdgcn_wave_barrier();
  }
  return d;
}

// Level 0's mean and direction of one row b, from its blocks' Gram matrices
// (the features' mean over the row is zero up to rounding, so the sums need
// no shift).
__global__ __launch_bounds__(256) void direction_kernel(GroupParams p) {
  __shared__ double gram[kGramAll];
  __shared__ double vec[kR];
  const int b = blockIdx.x, tid = threadIdx.x;
  double* x1 = p.x[1] + (long long)b * kBlks * kBlkDoubles;
  for (int i = tid; i < kGramAll; i += 256) {
    double v[kBlks];
#pragma unroll
    for (int k = 0; k < kBlks; ++k) v[k] = x1[k * kBlkDoubles + i];
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < kBlks; ++k) s += v[k];
    gram[i] = s;
  }
  __syncthreads();
  if (tid >= 64) return;
  const double d = power_direction(gram, kTokens, vec, tid);
  if (tid < kR) {
    x1[kVecAt + tid] = gram[kGramDoubles + tid] / kTokens;
    x1[kVecAt + kR + tid] = d;
  }
}

// Ascending key of a double (-0.0 and +0.0 equal, as the sort compares them).
__device__ __forceinline__ unsigned long long order_key(double s) {
  if (s == 0.0) s = 0.0;
  const unsigned long long u = (unsigned long long)__double_as_longlong(s);
  return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}

// Sum over the 8 lanes of a lane group (lanes 8q..8q+7): quad permutations,
// then the half-row mirror (lane l ^ 7, which holds the sum of l ^ 4's quad).
template <int CTRL>
__device__ __forceinline__ double dpp(double x) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(x);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, 0xF, 0xF, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ double sum8(double x) {
  x += dpp<0xB1>(x);
  x += dpp<0x4E>(x);
  x += dpp<0x141>(x);
  return x;
}

// x of lane l plus x of lane l ^ O (O = 8, 16, 32); the swaps return both
// lanes of a pair.  With two values, the lanes whose bit O is clear get the
// sum of x over the pair, the others that of y.
template <int O>
__device__ __forceinline__ double add_xor(double x, double y) {
  static_assert(O == 16 || O == 32, "lane swaps");
  const unsigned long long u = (unsigned long long)__double_as_longlong(x);
  const unsigned long long v = (unsigned long long)__double_as_longlong(y);
  auto swap = [](uint32_t a, uint32_t b) {
    return O == 16 ? __builtin_amdgcn_permlane16_swap(a, b, false, false)
                   : __builtin_amdgcn_permlane32_swap(a, b, false, false);
  };
  const auto l = swap((uint32_t)u, (uint32_t)v), h = swap((uint32_t)(u >> 32), (uint32_t)(v >> 32));
  return __longlong_as_double((long long)(((unsigned long long)h[0] << 32) | l[0])) +
         __longlong_as_double((long long)(((unsigned long long)h[1] << 32) | l[1]));
}
template <int O>
__device__ __forceinline__ double add_xor(double x) {
  if constexpr (O == 8)
    return x + dpp<0x128>(x);
  else
    return add_xor<O>(x, x);
}

// Centred projections of 4 features of a row on the direction, summed over
// the 8 lanes that share the row.
__device__ __forceinline__ double project_row(const double* x, const double (&mean)[4], const double (&dir)[4]) {
  double pr = 0.0;
#pragma unroll
  for (int c = 0; c < 4; ++c) pr = fma(x[c] - mean[c], dir[c], pr);
  return sum8(pr);
}

// Level 0's sort keys of one token block.  Thread: features 4 q .. 4 q + 3
// (q = tid % 8) of rows tid / 8 + 32 i.  Bound by reading the features once.
__global__ __launch_bounds__(256) void keys_kernel(GroupParams p) {
  const int blk = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, q = tid & 7, rs = tid >> 3;
  double* x1 = p.x[1] + (long long)b * kBlks * kBlkDoubles;
  const double* x = p.x[0] + ((long long)b * kBlks + blk) * kBlkDoubles + 4 * q;
  double mean[4], dir[4], xr[8][4];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int c = 0; c < 4; ++c) xr[i][c] = x[(rs + 32 * i) * kR + c];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    mean[c] = x1[kVecAt + 4 * q + c];
    dir[c] = x1[kVecAt + kR + 4 * q + c];
  }
  auto* key = reinterpret_cast<unsigned long long*>(x1 + (long long)blk * kBlkDoubles + kKeysAt);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const double pr = project_row(xr[i], mean, dir);
    if (q == 0) key[rs + 32 * i] = order_key(pr);
  }
}

// v of lane l ^ O without the LDS crossbar: 4 is the half-row mirror (l ^ 7)
// of the reversed quads (l ^ 3).
template <int O>
__device__ __forceinline__ uint32_t xor_word(uint32_t v) {
  if constexpr (O == 4) {
    const int r = __builtin_amdgcn_update_dpp(0, (int)v, 0x1B, 0xF, 0xF, false);
    return (uint32_t)__builtin_amdgcn_update_dpp(0, r, 0x141, 0xF, 0xF, false);
  } else {
    return xor_lane<O>(v);
  }
}

template <int O>
__device__ __forceinline__ unsigned long long xor_key(unsigned long long v) {
  const uint32_t lo = xor_word<O>((uint32_t)v), hi = xor_word<O>((uint32_t)(v >> 32));
  return ((unsigned long long)hi << 32) | lo;
}

// Ascending bitonic sort of a wave's 512 (key, position) pairs, element 8
// lane + i in item i: distances 1, 2 and 4 inside the lane, 8 .. 256 by
// lane exchanges, no LDS.  Positions break ties, so the order is stable.
__device__ __forceinline__ void sort512(unsigned long long (&key)[8], uint32_t (&pos)[8], int lane) {
  auto inner = [&](auto dist, int k) {
    constexpr int J = decltype(dist)::value;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (i & J) continue;
      const bool asc = ((8 * lane + i) & k) == 0;
      const unsigned long long a = key[i], c = key[i | J];
      const uint32_t pa = pos[i], pc = pos[i | J];
      if ((a > c || (a == c && pa > pc)) == asc) {
        key[i] = c;
        key[i | J] = a;
        pos[i] = pc;
        pos[i | J] = pa;
      }
    }
  };
  auto outer = [&](auto lanes, int k) {
    constexpr int L = decltype(lanes)::value;
    const bool want_min = ((lane & L) == 0) == (((8 * lane) & k) == 0);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const unsigned long long a = key[i], c = xor_key<L>(a);
      const uint32_t pa = pos[i], pc = xor_word<L>(pa);
      if ((a > c || (a == c && pa > pc)) == want_min) {
        key[i] = c;
        pos[i] = pc;
      }
    }
  };
#pragma unroll 1
  for (int k = 2; k <= 512; k <<= 1) {
#pragma unroll 1
    for (int j = k >> 1; j >= 8; j >>= 1) {
      switch (j) {
        case 256: outer(std::integral_constant<int, 32>{}, k); break;
        case 128: outer(std::integral_constant<int, 16>{}, k); break;
        case 64: outer(std::integral_constant<int, 8>{}, k); break;
        case 32: outer(std::integral_constant<int, 4>{}, k); break;
        case 16: outer(std::integral_constant<int, 2>{}, k); break;
        default: outer(std::integral_constant<int, 1>{}, k); break;
      }
    }
    if (k >= 8) inner(std::integral_constant<int, 4>{}, k);
    if (k >= 4) inner(std::integral_constant<int, 2>{}, k);
    inner(std::integral_constant<int, 1>{}, k);
  }
}

// Ranks of the elements of RUNS sorted runs of 512 (keys in LDS, run w's
// positions all below run w + 1's) in the whole: each element's place in its
// own run plus, for each other run, the number of its keys that come first
// (ties: those of an earlier run).  out(rank, pos) takes each element.  Used
// by wave w for its own run.
template <int RUNS, typename Out>
__device__ __forceinline__ void rank_runs(const unsigned long long (*runs)[512], int w,
                                          const unsigned long long (&key)[8], const uint32_t (&pos)[8], int lane,
                                          Out out) {
  int rank[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) rank[i] = 8 * lane + i;
#pragma unroll 1
  for (int o = 0; o < RUNS; ++o) {
    if (o == w) continue;
    const unsigned long long* run = runs[o];
    // an earlier run counts its keys <= key, a later one those < key
    const bool ties = o < w;
    int at[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) at[i] = 0;
#pragma unroll 1
    for (int s = 256; s > 0; s >>= 1) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const unsigned long long x = run[at[i] + s - 1];
        if (x < key[i] || (ties && x == key[i])) at[i] += s;
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const unsigned long long x = run[at[i]];
      rank[i] += at[i] + (x < key[i] || (ties && x == key[i]) ? 1 : 0);
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) out(rank[i], pos[i]);
}

// Level 0's stable order of one row: 9 waves sort runs of 512 tokens in
// registers, then merge by rank.
__global__ __launch_bounds__(576) void sort_kernel(GroupParams p) {
  __shared__ unsigned long long runs[kTokens / 512][512];
  const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const double* x1 = p.x[1] + (long long)b * kBlks * kBlkDoubles;
  unsigned long long key[8];
  uint32_t pos[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int t = 512 * wave + 8 * lane + i;
    key[i] = reinterpret_cast<const unsigned long long*>(x1 + (long long)(t / kBlkTok) * kBlkDoubles +
                                                         kKeysAt)[t % kBlkTok];
    pos[i] = (uint32_t)t;
  }
  sort512(key, pos, lane);
#pragma unroll
  for (int i = 0; i < 8; ++i) runs[wave][8 * lane + i] = key[i];
  __syncthreads();
  int32_t* o = p.ids[1] + (long long)b * kTokens;
  rank_runs<kTokens / 512>(runs, wave, key, pos, lane, [&](int rank, uint32_t t) { o[rank] = (int32_t)t; });
}

// Levels 1 and 2: each workgroup orders one group of N rows of one b (the
// rows ids[src][group] of x[0], read where they lie).  One pass for the
// group's Gram matrix, about its middle row (near the mean along the previous
// level's direction, so the centring loses nothing), on the fp64 matrix pipe;
// one for the projections; a wave sorts each run of 512, the runs merge by
// rank.  Bound by those two passes over the rows.
template <int N, int THREADS>
__global__ __launch_bounds__(THREADS) void level_kernel(GroupParams p, int src) {
  constexpr int kWaves = THREADS / 64, kHalf = kWaves / 2, kGroups = kTokens / N;
  __shared__ union {
    double red[kHalf][kGramAll];
    unsigned long long runs[N / 512][512];
  } u;
  __shared__ unsigned short tok[N];
  __shared__ double vec[kR], mean_s[kR], dir_s[kR];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.x / kGroups, gi = blockIdx.x % kGroups;
  const double* x = p.x[0] + (long long)b * kTokens * kR;
  const long long row0 = (long long)b * kTokens + gi * N;
  for (int i = tid; i < N; i += THREADS) tok[i] = (unsigned short)p.ids[src][row0 + i];
  __syncthreads();
  {
    const int c = lane & 15, g = lane >> 4;
    const double* mid = x + (int)tok[N / 2] * kR;
    const double s0 = mid[c], s1 = mid[c + 16];
    Gram gram;
    constexpr int kRows = N / kWaves, kSteps = kRows / 4;     // a wave's rows, four per step
    static_assert(kSteps % 8 == 0, "eight steps at a time");
#pragma unroll 1
    for (int i0 = 0; i0 < kSteps; i0 += 8) {
      double xl[8], xh[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const double* xr = x + (int)tok[kRows * wave + 4 * (i0 + i) + g] * kR + c;
        xl[i] = xr[0];
        xh[i] = xr[16];
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) gram.add(xl[i] - s0, xh[i] - s1);
    }
    gram.fold();
    if (wave >= kHalf) gram.store<false>(u.red[wave - kHalf], lane);
    __syncthreads();
    if (wave < kHalf) gram.store<true>(u.red[wave], lane);
    __syncthreads();
    for (int i = tid; i < kGramAll; i += THREADS) {
      double v = u.red[0][i];
#pragma unroll
      for (int k = 1; k < kHalf; ++k) v += u.red[k][i];
      u.red[0][i] = v;
    }
    __syncthreads();
    if (wave == 0) {
      const double d = power_direction(u.red[0], N, vec, lane);
      if (lane < kR) {
        mean_s[lane] = mid[lane] + u.red[0][kGramDoubles + lane] / N;
        dir_s[lane] = d;
      }
    }
    __syncthreads();
  }
  const int q = tid & 7, rs = tid >> 3;
  double mean[4], dir[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    mean[c] = mean_s[4 * q + c];
    dir[c] = dir_s[4 * q + c];
  }
  unsigned long long* keys = &u.runs[0][0];
  constexpr int kSlots = THREADS / 8;      // rows at a time
  static_assert(N / kSlots % 4 == 0, "four rows per thread at a time");
#pragma unroll 1
  for (int i0 = 0; i0 < N / kSlots; i0 += 4) {
    double xr[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const double* xp = x + (int)tok[rs + kSlots * (i0 + i)] * kR + 4 * q;
#pragma unroll
      for (int c = 0; c < 4; ++c) xr[i][c] = xp[c];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const double pr = project_row(xr[i], mean, dir);
      if (q == 0) keys[rs + kSlots * (i0 + i)] = order_key(pr);
    }
  }
  __syncthreads();
  unsigned long long key[8];
  uint32_t pos[8];
  const bool sorts = wave < N / 512;
  if (sorts) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      pos[i] = (uint32_t)(512 * wave + 8 * lane + i);
      key[i] = keys[pos[i]];
    }
    sort512(key, pos, lane);
#pragma unroll
    for (int i = 0; i < 8; ++i) u.runs[wave][8 * lane + i] = key[i];
  }
  __syncthreads();
  if (!sorts) return;
  int32_t* o = p.ids[src ^ 1] + row0;
  rank_runs<N / 512>(u.runs, wave, key, pos, lane, [&](int rank, uint32_t i) { o[rank] = (int32_t)tok[i]; });
}

// Levels 3..6 of the balanced split in one workgroup per 256-row group (an
// 18th of the chunk, as level 2 leaves it): the group's fp64 rows and token
// ids stay in LDS; level l sorts every aligned block of n = 256 >> (l - 3)
// rows by the block's own projection, all blocks at once, and a permutation
// of row slots carries the order from level to level.  A level reads its rows
// from LDS once: wave w holds rows 32 w .. 32 w + 31 of the order in
// registers, lane (q = l % 8, rg = l / 8) features 4 q .. 4 q + 3 of rows 4 rg
// .. 4 rg + 3, and the power steps, sums over rows by lane exchanges and,
// where a block spans waves, one LDS round with one barrier each.  The sort
// runs one element per thread, by lane exchanges up to distance 32.  The last
// level writes the final order.  Bound by fp64 vector issue, two workgroups
// per CU: per 30-layer batch 0.49 ms, half of it power steps (with level 2 in
// here too, 512 rows and one workgroup per CU: 0.77 ms against 0.49 + 0.17; at
// the start 1.65 ms, with every pass from LDS and its sums through a 64-deep
// serial LDS walk).
constexpr int kFuse = 256;
constexpr int kFuseLevels = 4;
constexpr int kFuseThreads = 512;
constexpr int kFuseWaves = kFuseThreads / 64;
constexpr int kFusePad = kR + 2;   // doubles per LDS row

__global__ __launch_bounds__(kFuseThreads, 4) void fused_levels_kernel(GroupParams p, int src, int32_t* last_out) {
  __shared__ alignas(16) double xs[kFuse][kFusePad];   // 68 KB: rows in level 3's input order
  __shared__ unsigned short perm[2][kFuse];            // row slot at each position
  __shared__ unsigned short tok[kFuse];
  __shared__ alignas(16) double part[2][kFuseWaves][kR];       // per wave, one of two buffers in turn
  __shared__ unsigned long long key[kFuse];
  __shared__ unsigned short pos[kFuse];
  const int tid = threadIdx.x, lane = tid & 63, q = lane & 7, rg = lane >> 3;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.x / (kTokens / kFuse), gi = blockIdx.x % (kTokens / kFuse);
  const long long row0 = (long long)b * kTokens + (long long)gi * kFuse;
  if (tid < kFuse) {
    tok[tid] = (unsigned short)p.ids[src][row0 + tid];
    perm[0][tid] = (unsigned short)tid;
  }
  __syncthreads();
  {
    const double* x = p.x[0] + (long long)b * kTokens * kR;
    // 16 lanes per row, 16 bytes each
    const int c = tid & 15, r = tid >> 4;
    f32x4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = reinterpret_cast<const f32x4*>(x + (int)tok[r + 32 * i] * kR)[c];
#pragma unroll
    for (int i = 0; i < 8; ++i) reinterpret_cast<f32x4*>(&xs[r + 32 * i][0])[c] = v[i];
  }
  __syncthreads();
  int cur = 0, buf = 0;
#pragma unroll 1
  for (int lv = 0; lv < kFuseLevels; ++lv) {
    const int n = kFuse >> lv, nw = n / 32;       // block size, waves per block
    const int w0 = wave & ~(nw - 1);              // first wave of this wave's block
    // this lane's 4 rows x 4 features
    double x[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x4* xr = reinterpret_cast<const f32x4*>(&xs[perm[cur][32 * wave + 4 * rg + i]][4 * q]);
      union { f32x4 v[2]; double d[4]; } t;
      t.v[0] = xr[0];
      t.v[1] = xr[1];
#pragma unroll
      for (int c = 0; c < 4; ++c) x[i][c] = t.d[c];
    }
    // sum over the block's rows of a per-lane partial of its 4 features: the
    // wave's rows by lane exchanges that leave one feature per lane, then
    // through LDS over the block's waves and back to 4 features per lane
    auto sum_rows = [&](double (&a)[4]) {
      const double w = add_xor<8>(add_xor<16>(add_xor<32>(a[0], a[2]), add_xor<32>(a[1], a[3])));
      if (!(lane & 8)) part[buf][wave][4 * q + 2 * (lane >> 5) + ((lane >> 4) & 1)] = w;
      if (nw > 1) {
        __syncthreads();
      } else {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
      // row group rg takes the block's wave rg mod nw, then the row groups sum
      const double* pw = part[buf][w0 + (rg & (nw - 1))] + 4 * q;
#pragma unroll
      for (int c = 0; c < 4; ++c) a[c] = pw[c];
      if (nw >= 2) {
#pragma unroll
        for (int c = 0; c < 4; ++c) a[c] = add_xor<8>(a[c]);
      }
      if (nw >= 4) {
#pragma unroll
        for (int c = 0; c < 4; ++c) a[c] = add_xor<16>(a[c]);
      }
      if (nw == 8) {
#pragma unroll
        for (int c = 0; c < 4; ++c) a[c] = add_xor<32>(a[c]);
      }
      // the other buffer next: its readers are past the barrier above
      buf ^= 1;
    };
    double acc[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] = (x[0][c] + x[1][c]) + (x[2][c] + x[3][c]);
    sum_rows(acc);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const double mean = acc[c] * (1.0 / n);     // n is a power of two
      acc[c] = 0.0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[i][c] -= mean;
        acc[c] = fma(x[i][c], x[i][c], acc[c]);
      }
    }
    // highest-variance feature (first of equals) -> one-hot start direction
    sum_rows(acc);
    double var = acc[0];
    int axis = 4 * q;
#pragma unroll
    for (int c = 1; c < 4; ++c) {
      if (acc[c] > var) {
        var = acc[c];
        axis = 4 * q + c;
      }
    }
    auto better = [&](double ov, int oi) {
      if (ov > var || (ov == var && oi < axis)) {
        var = ov;
        axis = oi;
      }
    };
    better(xor_lane<1>(var), xor_lane<1>(axis));
    better(xor_lane<2>(var), xor_lane<2>(axis));
    better(xor_lane<4>(var), xor_lane<4>(axis));
    double dir[4], pr[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) dir[c] = 4 * q + c == axis ? 1.0 : 0.0;
    auto project = [&]() {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        double s = 0.0;
#pragma unroll
        for (int c = 0; c < 4; ++c) s = fma(x[i][c], dir[c], s);
        pr[i] = sum8(s);
      }
    };
#pragma unroll 1
    for (int it = 0; it < 4; ++it) {
      project();
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        acc[c] = 0.0;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[c] = fma(x[i][c], pr[i], acc[c]);
      }
      sum_rows(acc);
      // not normalised: the order of the projections does not depend on the
      // direction's length, which unit-RMS features keep within 4 powers of
      // 2^24 (the normalised form's clamp at 1e-8 is a length, too)
#pragma unroll
      for (int c = 0; c < 4; ++c) dir[c] = acc[c];
    }
    // projections -> sort keys (ascending score, ties -> current position)
    project();
    {
      // lane q < 4 writes row 4 rg + q
      const double s = q == 0 ? pr[0] : q == 1 ? pr[1] : q == 2 ? pr[2] : pr[3];
      if (q < 4) key[32 * wave + 4 * rg + q] = order_key(s);
    }
    __syncthreads();
    // bitonic sort of every aligned block of n, ascending (the direction bit
    // of the last stage is masked to the block): element tid of the first 256
    // threads
    unsigned long long k = ~0ull;
    uint32_t ps = (uint32_t)tid;
    if (tid < kFuse) k = key[tid];
    auto exchange = [&](int j, int kk, unsigned long long ok, uint32_t op) {
      const bool greater = k > ok || (k == ok && ps > op);
      const bool want_min = ((tid & j) == 0) == ((tid & kk & (n - 1)) == 0);
      if (greater == want_min) {
        k = ok;
        ps = op;
      }
    };
#pragma unroll 1
    for (int kk = 2; kk <= n; kk <<= 1) {
#pragma unroll 1
      for (int j = kk >> 1; j >= 64; j >>= 1) {
        __syncthreads();
        if (tid < kFuse) {
          key[tid] = k;
          pos[tid] = (unsigned short)ps;
        }
        __syncthreads();
        if (tid < kFuse) exchange(j, kk, key[tid ^ j], pos[tid ^ j]);
      }
      if (wave < kFuse / 64) {
        if (kk >= 64) exchange(32, kk, xor_key<32>(k), xor_word<32>(ps));
        if (kk >= 32) exchange(16, kk, xor_key<16>(k), xor_word<16>(ps));
        if (kk >= 16) exchange(8, kk, xor_key<8>(k), xor_word<8>(ps));
        if (kk >= 8) exchange(4, kk, xor_key<4>(k), xor_word<4>(ps));
        if (kk >= 4) exchange(2, kk, xor_key<2>(k), xor_word<2>(ps));
        exchange(1, kk, xor_key<1>(k), xor_word<1>(ps));
      }
    }
    if (tid < kFuse) perm[cur ^ 1][tid] = perm[cur][ps];
    cur ^= 1;
    __syncthreads();
  }
  // final order: position j is grouped page (gi * 256 + j) / 64, row j % 64
  if (tid < kFuse) {
    const int in_head = gi * kFuse + tid, page = in_head / 64;
    const int dpage = p.page_dst ? min(max(p.page_dst[page], 0), kPages - 1) : page;   // clamped: memory safety
    last_out[(long long)b * kTokens + dpage * 64 + in_head % 64] = tok[perm[cur][tid]];
  }
}

// Stable partition of each row's order by frame (token / 1536): the first
// chunk's anchor frame fills pages 0..23 (VR/runtime.py:358-363).
__global__ __launch_bounds__(256) void frames_kernel(const int32_t* in, int32_t* out) {
  __shared__ int wsum[4];
  const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int32_t* src = in + (long long)b * kTokens;
  int32_t* dst = out + (long long)b * kTokens;
  int cursor = 0;
  for (int f = 0; f < 3; ++f) {
    for (int c0 = 0; c0 < kTokens; c0 += 256) {
      const int val = src[c0 + tid];
      const bool on = val / kFrame == f;
      const unsigned long long bal = __ballot(on);
      if (lane == 0) wsum[w] = __popcll(bal);
      __syncthreads();
      int off = cursor;
      for (int u = 0; u < w; ++u) off += wsum[u];
      if (on) dst[off + __popcll(bal & ((1ull << lane) - 1ull))] = val;
      cursor += wsum[0] + wsum[1] + wsum[2] + wsum[3];
      __syncthreads();
    }
  }
}

}  // namespace

extern "C" {

int ssa_group_order(const void* k, const void* v, long long layer_stride, long long token_stride,
                    long long head_stride, const float* bank, const float* group_v, const float* gate,
                    const int32_t* page_dst, int first_chunk, int layers, int heads, double* scratch_x,
                    int32_t* scratch_ids, int32_t* order, hipStream_t stream) {
  if (layers <= 0 || heads <= 0 || !k || !v || !bank || !group_v || !gate || !scratch_x || !scratch_ids || !order ||
      layer_stride < 0 || token_stride < 0 || head_stride < 0)
    return (int)hipErrorInvalidValue;
  // rows are read 16 bytes at a time
  if ((((uintptr_t)k | (uintptr_t)v | (uintptr_t)bank | (uintptr_t)group_v) & 15) != 0 ||
      ((layer_stride | token_stride | head_stride) & 7) != 0)
    return (int)hipErrorInvalidValue;
  GroupParams p;
  p.k = (const uint16_t*)k;
  p.v = (const uint16_t*)v;
  p.layer_stride = layer_stride;
  p.tok_stride = token_stride;
  p.head_stride = head_stride;
  p.bank = bank;
  p.gv = group_v;
  p.gate = gate;
  p.page_dst = page_dst;
  p.H = heads;
  p.B = layers * heads;
  const long long rows = (long long)p.B * kTokens;
  p.x[0] = scratch_x;
  p.x[1] = scratch_x + rows * kR;
  p.ids[0] = scratch_ids;
  p.ids[1] = scratch_ids + rows;
  p.order = order;
  const dim3 blocks(kBlks, p.B), rows_grid(p.B), threads(256);
  hipLaunchKernelGGL(project_kernel, blocks, threads, 0, stream, p);
  hipLaunchKernelGGL(totals_kernel, rows_grid, threads, 0, stream, p);
  hipLaunchKernelGGL(features_kernel, blocks, threads, 0, stream, p);
  hipLaunchKernelGGL(direction_kernel, rows_grid, threads, 0, stream, p);
  hipLaunchKernelGGL(keys_kernel, blocks, threads, 0, stream, p);
  hipLaunchKernelGGL(sort_kernel, rows_grid, dim3(576), 0, stream, p);          // -> ids[1]
  hipLaunchKernelGGL((level_kernel<kTokens / 3, 512>), dim3(p.B * 3), dim3(512), 0, stream, p, 1);   // -> ids[0]
  hipLaunchKernelGGL((level_kernel<kTokens / 9, 256>), dim3(p.B * 9), threads, 0, stream, p, 0);      // -> ids[1]
  // levels 3..6 write the order (or the frame partition's input)
  int32_t* last_out = first_chunk ? p.ids[0] : order;
  hipLaunchKernelGGL(fused_levels_kernel, dim3(p.B * (kTokens / kFuse)), dim3(kFuseThreads), 0, stream, p, 1, last_out);
  if (first_chunk) hipLaunchKernelGGL(frames_kernel, dim3(p.B), threads, 0, stream, p.ids[0], order);
  return (int)hipGetLastError();
}

}  // extern "C"
