// Full_Pset swap correction for gfx950: page encodings, reader readout with
// FP64 mixture states, and the per-(remove, add) set-gain table with the
// apply step.
//
// Reference (VB = reproduction/vbench_current, VR = local_experiments/
// video_runtime_v1, LE = local_experiments):
//   encode  : f = per-part RMS-normalised [keys|mean|detail|stats] (712);
//             co = bf16(reader MLP(f)) [5,17], A = bf16(phi MLP(f)) [8,4],
//             meanB = mean.B, detailB = detail.(bf16(basis)^T B)
//             (VR/page.py:6-14, VR/runtime.py:89,160-164,
//              LE/e27_adaptive_query/core.py:4-11, coefficients.py:4-8)
//   rows    : per probe m of a query block and page p: lm = LSE_r z - LSE z,
//             rp/beta = co0 + sum_j tanh(u.A_j) co_{j+1} (VR/page.py:17-21),
//             approx = meanB + sum_a c_a detailB_a (VB/graph.py:199-201),
//             then the mixtures H (current selection), target (all exact)
//             and the background of non-candidate pages (VR/scores.py:62-68)
//   scores  : for 16 removes x 32 adds, the FP64 endpoint deltas of the
//             mixture after the swap and 2 E.delta - |delta|^2 averaged over
//             the 16 probes (VR/scores.py:69-91); pools and legality of
//             VB/quota_pool.py:3-46; argmax and the gain > 0 gate of
//             VR/scores.py:102-107; the LUT of VB/graph.py:210.
// The mixture background is kept uncentred (the translation by the
// mass-weighted mean cancels in every delta, VR/reader_reduce.py:55-56).
#include "common.h"

#include <mutex>
#include <type_traits>

using namespace ssa;

namespace {

constexpr int kMaxPages = 512;
constexpr int kAnchors = 24;
constexpr int kCurrent = 72;
constexpr int kFeatures = 712;
constexpr int kMaxHidden = 256;
constexpr int kEncRows = 16;        // pages (of any heads) per MLP workgroup
constexpr int kEncThreads = 512;
constexpr int kProjPages = 32;      // pages of one head per projection workgroup
constexpr int kCoefStride = 128;    // bf16 per page: co[85] | 0 x 11 | A[32]
constexpr int kCoefA = 96;
constexpr int kCand = 48;           // 16 removes + 32 adds
constexpr int kCandVals = 34;       // doubles per probe and candidate in the caller's scratch
constexpr int kCandStride = 26;     // doubles of a candidate: lm, beta (fp32), approx[16], rp[16] (fp32)
constexpr int kRowDoubles = 16 * kCand * kCandVals;   // a row's scratch: its 16 x 48 candidates, then its partials
constexpr int kPoolInts = 64;       // 48 candidate pages + 16 legal bit rows

// ------------------------------------------------------------- encoding ----

struct EncodeParams {
  const uint16_t *keys, *mean, *detail, *stats, *basis;
  int HP;
  const float *w1t, *b1, *w2r, *b2r, *w2p, *b2p;
  const double* B;
  uint16_t* coef;
  double *mean_b, *detail_b;
  int EP, heads, first, pages, hidden;
};

// Per-layer tensors of a batched encode (blockIdx.z = layer): the summary
// slab, the basis and the encodings of each layer; the weights are shared.
constexpr int kMaxLayers = 32;
struct EncodeLayers {
  const uint16_t *keys[kMaxLayers], *mean[kMaxLayers], *detail[kMaxLayers], *stats[kMaxLayers],
      *basis[kMaxLayers];
  uint16_t* coef[kMaxLayers];
  double *mean_b[kMaxLayers], *detail_b[kMaxLayers];
};
struct OneLayer {};

__device__ __forceinline__ float wave_sum(float v) {
  return wave_reduce(v, [](float a, float b) { return a + b; });
}

// D[16x16] += A[16x4] * B[4x16], fp32.  Lane l: A row l % 16, k = l / 16; B
// column l % 16, same k; D column l % 16, rows 4 (l / 16) + i for item i.
__device__ __forceinline__ f32x4 mfma16(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Four floats at 4-byte alignment.
struct alignas(4) Row4 { float v[4]; };
__device__ __forceinline__ Row4 row4(const float* p, int valid) {
  Row4 r;
  if (valid >= 4) {
    r = *reinterpret_cast<const Row4*>(p);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) r.v[i] = i < valid ? p[i] : 0.f;
  }
  return r;
}

constexpr int kFeatPad = 716, kHidPad = 260;     // floats per row: 16-byte aligned, rows on distinct banks
union EncSmem {
  struct {
    union {
      alignas(16) float f[kEncRows][kFeatPad];   // features
      alignas(16) float hid[kEncRows][kHidPad];  // hidden units, once the features are used
    } u;
    float l1[2][kEncRows][kHidPad];              // layer 1 sums of the two halves of the features
  } m;
  struct {
    double B[kHeadDim][16];
    double pb[8][16];                            // bf16(basis)^T B of the head
    uint16_t mean[kProjPages][kHeadDim + 8];
  } b;
};

// The encodings of pages of all heads: workgroups 2 t and 2 t + 1 run the
// reader and the phi MLP of pages 16 t .. 16 t + 15 of the flat (head, page)
// range, the workgroups after them meanB and detailB of 32 pages of one head.
// The MLPs are products of 16 pages by 16 units on the fp32 matrix pipe (fp32
// products and sums).  Layer 1: wave w takes hidden units 64 (w % 4) .. + 63
// over half w / 4 of the 712 features; lane (c = l % 16, g = l / 16) loads
// units 4 c .. 4 c + 3 of a feature's weight row (256 bytes per row and
// wave), well ahead, each item one product.  Products take 9.5 us of a
// workgroup's time (the fp32 matrix pipe is 37% busy on the 108 CUs that 72 x
// 12 pages fill), the latency of the steps around them the rest.  72 x 12
// pages, kernel trace of a correction call: 42 us (4 pages and both MLPs per
// workgroup as vector FMAs at one wave per SIMD, layer 2 as 256-long serial dot
// products, meanB after it) -> 29;  432 x 12 pages, captured, 136 -> 80.
template <class Layers>
__global__ __launch_bounds__(kEncThreads) void encode_kernel(EncodeParams p, Layers layers) {
  if constexpr (std::is_same_v<Layers, EncodeLayers>) {
    const int l = blockIdx.z;
    p.keys = layers.keys[l];
    p.mean = layers.mean[l];
    p.detail = layers.detail[l];
    p.stats = layers.stats[l];
    p.basis = layers.basis[l];
    p.coef = layers.coef[l];
    p.mean_b = layers.mean_b[l];
    p.detail_b = layers.detail_b[l];
  }
  __shared__ EncSmem smem;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int total = p.heads * p.pages;
  const int mlps = 2 * ((total + kEncRows - 1) / kEncRows);
  if ((int)blockIdx.x >= mlps) {
    auto& s = smem.b;
    const int chunks = (p.pages + kProjPages - 1) / kProjPages;
    const int h = (blockIdx.x - mlps) / chunks, g0 = ((blockIdx.x - mlps) % chunks) * kProjPages;
    const int npg = min(kProjPages, p.pages - g0);
    const long long page0 = (long long)h * p.HP + p.first + g0, enc0 = (long long)h * p.EP + p.first + g0;
    for (int i = tid; i < kHeadDim * 16; i += kEncThreads) s.B[i >> 4][i & 15] = p.B[i];
    for (int i = tid; i < npg * 16; i += kEncThreads)
      *reinterpret_cast<u32x4*>(&s.mean[i >> 4][8 * (i & 15)]) = ldg16(p.mean + (page0 + (i >> 4)) * kHeadDim + 8 * (i & 15));
    const int o = tid >> 2, part = tid & 3, e = tid & 15;
    uint16_t bs[32];
#pragma unroll
    for (int i = 0; i < 32; ++i) bs[i] = p.basis[((long long)h * kHeadDim + 4 * i + part) * 8 + (o >> 4)];
    __syncthreads();
    // four threads per element of pb, 32 of the 128 dims each
    double pb = 0.0;
#pragma unroll
    for (int i = 0; i < 32; ++i) pb = fma((double)bf16_to_f32(bs[i]), s.B[4 * i + part][o & 15], pb);
    pb += xor_lane<1>(pb);
    pb += xor_lane<2>(pb);
    if (part == 0) s.pb[o >> 4][o & 15] = pb;
    if ((tid >> 4) < npg) {
      double acc = 0.0;
#pragma unroll 16
      for (int d = 0; d < kHeadDim; ++d) acc = fma((double)bf16_to_f32(s.mean[tid >> 4][d]), s.B[d][e], acc);
      p.mean_b[(enc0 + (tid >> 4)) * 16 + e] = acc;
    }
    __syncthreads();
    for (int i = tid; i < npg * 48; i += kEncThreads) {
      const int pl = i / 48, a = (i / 16) % 3;
      double acc = 0.0;
#pragma unroll
      for (int k = 0; k < 8; ++k)
        acc += (double)bf16_to_f32(p.detail[(page0 + pl) * 24 + a * 8 + k]) * s.pb[k][i & 15];
      p.detail_b[((enc0 + pl) * 3 + a) * 16 + (i & 15)] = acc;
    }
    return;
  }
  auto& s = smem.m;
  const bool phi = blockIdx.x & 1;
  const int r0 = (blockIdx.x >> 1) * kEncRows;
  const int nrow = min(kEncRows, total - r0);

  // the first weight rows are requested before anything else
  const int H = p.hidden, c = lane & 15, g = lane >> 4;
  constexpr int kHalf = kFeatures / 2, kSteps = kHalf / 16;      // 356 = 22 x 16 + 4
  static_assert(kHalf == 16 * kSteps + 4, "one product after the full steps");
  constexpr int kAhead = 4;        // steps of weight rows in flight
  const int unit = 64 * (wave & 3) + 4 * c, half = wave >> 2;
  const int valid = H - unit;      // units past H load zero
  const float* w1 = p.w1t + (long long)(half * kHalf) * 2 * H + (phi ? H : 0) + min(unit, H - 1);
  Row4 wr[kAhead][4];
  auto load = [&](int st, Row4 (&r)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = row4(w1 + (long long)(16 * min(st, kSteps - 1) + 4 * g + i) * 2 * H, valid);
  };
#pragma unroll
  for (int st = 0; st < kAhead; ++st) load(st, wr[st]);
  const Row4 last = row4(w1 + (long long)(16 * kSteps + g) * 2 * H, valid);

  // features: wave w normalises rows 2 w and 2 w + 1 (rows past the last
  // re-read it; their outputs are not written)
  {
    u32x4 k4[2];
    uint32_t mw[2];
    float dv[2], sv[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = min(r0 + 2 * wave + i, total - 1);
      const long long pg = (long long)(r / p.pages) * p.HP + p.first + r % p.pages;
      k4[i] = ldg16(p.keys + pg * 512 + lane * 8);
      mw[i] = *reinterpret_cast<const uint32_t*>(p.mean + pg * 128 + lane * 2);
      dv[i] = lane < 24 ? bf16_to_f32(p.detail[pg * 24 + lane]) : 0.f;
      sv[i] = lane < 48 ? bf16_to_f32(p.stats[pg * 48 + lane]) : 0.f;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float kv[8];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        kv[2 * w] = bf16_lo(k4[i][w]);
        kv[2 * w + 1] = bf16_hi(k4[i][w]);
      }
      float ks = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) ks += kv[j] * kv[j];
      const float m0 = bf16_lo(mw[i]), m1 = bf16_hi(mw[i]);
      const float kd = sqrtf(wave_sum(ks) / 512.f) + 1e-4f;
      const float md = sqrtf(wave_sum(m0 * m0 + m1 * m1) / 128.f) + 1e-4f;
      const float dd = sqrtf(wave_sum(dv[i] * dv[i]) / 24.f) + 1e-4f;
      const float sd = sqrtf(wave_sum(sv[i] * sv[i]) / 48.f) + 1e-4f;
      float* f = s.u.f[2 * wave + i];
      *reinterpret_cast<f32x4*>(f + 8 * lane) = f32x4{kv[0] / kd, kv[1] / kd, kv[2] / kd, kv[3] / kd};
      *reinterpret_cast<f32x4*>(f + 8 * lane + 4) = f32x4{kv[4] / kd, kv[5] / kd, kv[6] / kd, kv[7] / kd};
      f[512 + 2 * lane] = m0 / md;
      f[512 + 2 * lane + 1] = m1 / md;
      if (lane < 24) f[640 + lane] = dv[i] / dd;
      if (lane < 48) f[664 + lane] = sv[i] / sd;
    }
  }
  __syncthreads();

  // layer 1: step s, item i of its four products: features 16 s + 4 g + i of
  // this half (the last step's one product: feature 352 + g)
  {
    if (64 * (wave & 3) < H) {
      const float* x = &s.u.f[c][half * kHalf];
      f32x4 acc[4] = {};
#pragma unroll 1
      for (int s0 = 0; s0 < kSteps; s0 += kAhead) {
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
          if (s0 + k < kSteps) {
            const f32x4 xv = *reinterpret_cast<const f32x4*>(x + 16 * (s0 + k) + 4 * g);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
              for (int t = 0; t < 4; ++t) acc[t] = mfma16(wr[k][i].v[t], xv[i], acc[t]);
            load(s0 + k + kAhead, wr[k]);
          }
        }
      }
      {
        const float xv = x[16 * kSteps + g];
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = mfma16(last.v[t], xv, acc[t]);
      }
      // acc[t] item i: page c, unit 64 (w % 4) + 4 (4 g + i) + t
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<f32x4*>(&s.l1[half][c][64 * (wave & 3) + 4 * (4 * g + i)]) =
            f32x4{acc[0][i], acc[1][i], acc[2][i], acc[3][i]};
    }
  }
  // layer 2: 85 reader or 32 phi outputs per page; wave w takes outputs 16 w
  // .. + 15 of all pages, hidden units 16 s + 4 g + i in product i of step s.
  // Its weights are requested here, ahead of the hidden units.
  const int outs = phi ? 32 : 85;
  const int o = 16 * wave + c;
  const float* w = (phi ? p.w2p : p.w2r) + (long long)min(o, outs - 1) * H;
  Row4 w2[16];
  if (16 * wave < outs) {
#pragma unroll
    for (int st = 0; st < 16; ++st) w2[st] = row4(w + 16 * st + 4 * g, H - 16 * st - 4 * g);
  }
  __syncthreads();
  for (int i = tid; i < kEncRows * kMaxHidden; i += kEncThreads) {
    const int r = i / kMaxHidden, j = i % kMaxHidden;
    float y = 0.f;
    if (j < H) {
      const float x = (s.l1[0][r][j] + s.l1[1][r][j]) + p.b1[(phi ? H : 0) + j];
      y = 0.5f * x * (1.0f + erff(x * 0.70710678118654752f));
    }
    s.u.hid[r][j] = y;
  }
  __syncthreads();
  if (16 * wave >= outs) return;
  f32x4 acc[4] = {};
#pragma unroll
  for (int st = 0; st < 16; ++st) {
    const f32x4 xv = *reinterpret_cast<const f32x4*>(&s.u.hid[c][16 * st + 4 * g]);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = mfma16(w2[st].v[i], xv[i], acc[i]);
  }
  if (c >= nrow) return;
  const int r = r0 + c;
  uint16_t* cf = p.coef + ((long long)(r / p.pages) * p.EP + p.first + r % p.pages) * kCoefStride;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int oo = 16 * wave + 4 * g + i;
    if (oo < outs) {
      const float y = ((acc[0][i] + acc[1][i]) + (acc[2][i] + acc[3][i])) + (phi ? p.b2p[oo] : p.b2r[oo]);
      cf[phi ? kCoefA + oo : oo] = to_bf16(y);
    } else if (!phi) {
      cf[oo] = 0;       // 85 .. 95: padding between co and A
    }
  }
}

// ----------------------------------------------------------------- pool ----

struct PsetParams {
  const uint16_t* q;
  long long q_head, q_block, q_row;
  int gathered;
  const uint16_t* rk;
  int HP;
  const uint16_t* coef;
  const double *mean_b, *detail_b;
  int EP;
  const float* wq;
  const float* risk;
  const float* lse;            // [H, T, 16] per-probe LSE over all reps (from the router)
  uint8_t* mask;
  int32_t* ids;
  const int32_t* own;
  const int32_t* heads;
  int HS;
  double* cand;
  int32_t* pool;
  double* gain;
  int32_t* info;
  double* scores;
  long long* stats;            // [3] executed swaps, corrected rows, non-finite legal scores
  int H, T, P, C;
};

__device__ __forceinline__ int own_page(const PsetParams& p, int h, int t) {
  // clamped into the window like the router's own page (memory safety)
  return min(max(p.own ? p.own[(long long)h * p.T + t] : p.P - p.T + t, 0), p.P - 1);
}

template <int O>
__device__ __forceinline__ unsigned long long xor_u64(unsigned long long v) {
  const uint32_t lo = xor_lane<O>((uint32_t)v), hi = xor_lane<O>((uint32_t)(v >> 32));
  return ((unsigned long long)hi << 32) | lo;
}

struct PoolSmem {
  uint8_t sel[kMaxPages];
  uint8_t isadd[kMaxPages];
  unsigned long long key[kMaxPages];
  int cnt[4];                  // movable history, movable current, unselected history, unselected current
  int spare[32];
};

// One workgroup per scoped (head, block): the stratified pools of
// VB/quota_pool.py:3-46 from one descending bitonic sort of 512 keys whose
// group field orders history removes > current removes > history adds >
// current adds; removes rank by ascending risk, adds by descending risk,
// ties -> lower page.  A 72-page window (the anchor frame is the chunk's
// first frame, every other page current: VB/quota_pool.py:21-33) has one
// remove group and one add group: up to 8 movable removes, then the anchor
// pages other than own; the unselected pages by descending risk, then the
// selected pages in page order; the movable removes x the first 16 add
// slots are legal.  One key per thread; 3 heads x 72 blocks, kernel trace:
// 9.5 us (two keys per thread, every step through LDS) -> 8.3 us.
__global__ __launch_bounds__(kMaxPages) void pset_pool_kernel(PsetParams p) {
  __shared__ PoolSmem s;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int hs = blockIdx.x / p.T, t = blockIdx.x % p.T;
  const int h = p.heads[hs];
  const int P = p.P;
  const long long rowoff = ((long long)h * p.T + t) * P;
  const int own = own_page(p, h, t);
  if (blockIdx.x == 0 && tid < 3) p.stats[tid] = tid == 1 ? (long long)p.HS * p.T : 0ll;
  const float risk = tid < P ? p.risk[rowoff + tid] : 0.f;
  const bool sel = tid < P ? p.mask[rowoff + tid] != 0 : true;
  s.sel[tid] = sel;
  s.isadd[tid] = 0;
  if (tid < 4) s.cnt[tid] = 0;
  __syncthreads();
  const bool first = P == kCurrent;
  const int pg = tid;
  unsigned long long key = 0ull;
  int group = 0;
  // a 72-page window counts every page in the history groups (4: removes,
  // 2: adds), so its removes and adds each form one contiguous run; its
  // adds range over all pages (an anchor page is selected in every mask
  // the router writes)
  if ((pg >= kAnchors || first) && pg < P) {
    const int cur = first ? 0 : pg >= P - kCurrent;
    const uint32_t ord = orderable(risk);
    uint32_t kv = 0;
    if (sel && pg != own && pg >= kAnchors) {
      group = cur ? 3 : 4;
      kv = ~ord;
    } else if (!sel) {
      group = cur ? 1 : 2;
      kv = ord;
    }
    if (group) key = ((unsigned long long)group << 60) | ((unsigned long long)kv << 20) | (unsigned long long)(1023 - pg);
  }
#pragma unroll
  for (int g = 1; g <= 4; ++g) {
    const int n = __popcll(__ballot(group == g));
    if (lane == 0 && n) atomicAdd(&s.cnt[4 - g], n);
  }
  // descending bitonic sort, one key per thread: partner distances up to 32
  // by lane exchanges, 64 to 256 through LDS
  auto exchange = [&](int j, int k, unsigned long long other) {
    const bool keep_max = ((tid & j) == 0) == ((tid & k) == 0);
    if ((other > key) == keep_max) key = other;
  };
#pragma unroll 1
  for (int k = 2; k <= kMaxPages; k <<= 1) {
#pragma unroll 1
    for (int j = k >> 1; j >= 64; j >>= 1) {
      s.key[tid] = key;
      __syncthreads();
      const unsigned long long other = s.key[tid ^ j];
      __syncthreads();
      exchange(j, k, other);
    }
    if (k >= 64) exchange(32, k, xor_u64<32>(key));
    if (k >= 32) exchange(16, k, xor_u64<16>(key));
    if (k >= 16) exchange(8, k, xor_u64<8>(key));
    if (k >= 8) exchange(4, k, xor_u64<4>(key));
    if (k >= 4) exchange(2, k, xor_u64<2>(key));
    exchange(1, k, xor_u64<1>(key));
  }
  s.key[tid] = key;
  __syncthreads();
  const int nmh = s.cnt[0], nmc = s.cnt[1], nuh = s.cnt[2], nuc = s.cnt[3];
  auto page_at = [&](int i) -> int { return 1023 - (int)(s.key[i] & 1023ull); };
  if (first) {
    // the selected pages in page order fill the add slots past the unselected ones
    if (wave == 0) {
      int cnt = 0;
      for (int base = 0; base < P; base += 64) {
        const int pg = base + lane;
        const bool on = pg < P && s.sel[pg];
        const unsigned long long bal = __ballot(on);
        const int r = cnt + __popcll(bal & ((1ull << lane) - 1ull));
        if (on && r < 32) s.spare[r] = pg;
        cnt += __popcll(bal);
      }
    }
    __syncthreads();
    if (tid < kCand) {
      const int sl = tid, used = min(nmh, 8);
      int page;
      if (sl < 16) {
        // the anchor pages other than own, in page order, stand in past the movable removes
        const int a = sl - used;
        page = sl < used ? page_at(sl) : a + (own < kAnchors && a >= own ? 1 : 0);
      } else {
        const int k = sl - 16;
        page = k < nuh ? page_at(nmh + k) : s.spare[k - nuh];
      }
      int32_t* po = p.pool + ((long long)hs * p.T + t) * kPoolInts;
      po[sl] = page;
      if (sl < 16) po[kCand + sl] = sl < used ? 0xffff : 0;
    }
    return;
  }
  // valid adds, then spare pages (neither selected nor a valid add), ascending
  if (tid < 32) {
    const int q = tid >> 4, k = tid & 15;
    const int n = q ? nuc : nuh;
    if (k < n) s.isadd[page_at(nmh + nmc + (q ? nuh : 0) + k)] = 1;
  }
  __syncthreads();
  if (wave == 0) {
    int cnt = 0;
    for (int base = 0; base < P; base += 64) {
      const int pg = base + lane;
      const bool fr = pg < P && !s.sel[pg] && !s.isadd[pg];
      const unsigned long long bal = __ballot(fr);
      const int r = cnt + __popcll(bal & ((1ull << lane) - 1ull));
      if (fr && r < 32) s.spare[r] = pg;
      cnt += __popcll(bal);
    }
    if (lane < 32 && lane >= cnt) s.spare[lane] = -1;
  }
  __syncthreads();
  if (tid < kCand) {
    const int sl = tid;
    int page;
    bool valid;
    if (sl < 16) {
      const int q = sl >> 3, k = sl & 7;
      valid = k < (q ? nmc : nmh);
      page = valid ? page_at((q ? nmh : 0) + k) : sl;          // anchor stands in (never legal)
    } else {
      const int q = (sl - 16) >> 4, k = (sl - 16) & 15;
      valid = k < (q ? nuc : nuh);
      page = valid ? page_at(nmh + nmc + (q ? nuh : 0) + k) : s.spare[sl - 16];   // spare (never legal)
      if (page < 0) {
        // no spare page left for this slot (the reference's pool would index
        // page P, past the window): an empty candidate -- zero mass (lm =
        // -inf), zero values -- that adds nothing to any sum, while every
        // page outside the pool stays in the background.  The rows kernel
        // writes no endpoint data for it (no page maps to the slot).
        double* c = p.cand + ((long long)hs * p.T + t) * kRowDoubles + sl * kCandStride;
        for (int m = 0; m < 16; ++m)
          for (int v = 0; v < kCandStride; ++v) c[(long long)m * kCand * kCandStride + v] = v == 0 ? -INFINITY : 0.0;
      }
    }
    int32_t* po = p.pool + ((long long)hs * p.T + t) * kPoolInts;
    po[sl] = page;
    if (sl < 16) {
      const int q = sl >> 3;
      const int na = q ? nuc : nuh;
      const uint32_t addbits = na >= 16 ? 0xffffu : ((1u << na) - 1u);
      po[kCand + sl] = valid ? (int32_t)(addbits << (16 * q)) : 0;
    }
  }
}

// ----------------------------------------------------------------- rows ----

constexpr int kSplit = 4;          // page ranges per (head, 4 blocks)
constexpr int kRowBlocks = 4;      // query blocks (64 probes) per workgroup
constexpr int kRowWaves = 8;
constexpr int kPartVals = 35;      // B[16], T[16], their masses sB and sT, max log mass
constexpr int kPartAt = 16 * kCand * kCandStride;     // [kSplit][kPartVals][16 probes], in a row's scratch
static_assert(kPartAt + kSplit * kPartVals * 16 <= kRowDoubles, "the partials fit behind the candidates");

struct RowsSmem {
  uint8_t sel[kRowBlocks][kMaxPages];
  int8_t slot[kRowBlocks][kMaxPages];       // remove slot (0..15) of a pool page, or -1
  int8_t aslot[kRowBlocks][kMaxPages];      // add slot (16..47), or -1: a 72-page pool may list a page in both
  float u[64][9];
  float L[64];
  alignas(16) uint8_t q[64 * 256];          // probe rows, chunk c of row r at chunk c ^ (r & 15)
  double part[4][kPartVals][64];
};

// 1 / x by the hardware reciprocal (1 ulp) and one Newton step.
__device__ __forceinline__ float recip(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return fmaf(fmaf(-x, r, 1.0f), r, r);
}

// tanh to within 1.6 ulp (just above the split, where the exponent's argument
// is rounded once), in the form of the Cephes library's tanhf: below 0.625 an
// odd polynomial, above it 1 - 2 / (e^2x + 1).  The coefficients are a weighted
// least-squares fit of (tanh x / x - 1) / x^2 of our own, 7e-9 relative.
__device__ __forceinline__ float tanh_f32(float x) {
  const float a = fabsf(x), t = x * x;
  const float pl = fmaf(fmaf(fmaf(fmaf(-0.005515433382242918f, t, 0.020469674840569496f), t, -0.05368810519576073f), t,
                             0.1333083212375641f), t, -0.3333325982093811f);
  const float e = __builtin_amdgcn_exp2f(a * (2.0f * kLog2e));
  const float big = fmaf(-2.0f, __builtin_amdgcn_rcpf(e + 1.0f), 1.0f);
  return a < 0.625f ? fmaf(pl * t, x, x) : copysignf(big, x);
}

// A wave-uniform read-only value through the scalar cache.
template <typename T>
using Const = const __attribute__((address_space(4))) T;
template <typename T>
__device__ __forceinline__ Const<T>* scalar(const T* p) {
  return (Const<T>*)(uintptr_t)p;
}

// One workgroup per (scoped head, 4 query blocks, page range): a lane holds
// one of the 64 probes and a wave walks the pages of its tiles one at a time,
// so everything that belongs to the page (meanB, detailB, the readout
// coefficients) is wave-uniform and comes through the scalar cache into
// scalar operands.  Per probe and page: the log mass lm = LSE_r z - LSE z,
// the readout (rp, beta) and the summary approximation; candidate pages write
// their endpoint data, the background pages (in no pool slot) enter the
// mixture sums B (the current selection's weights) and T (every page exact),
// which the scores kernel completes with the candidates.  Vector issue
// takes about two thirds of the time a CU holds a workgroup (~440 fp32 and
// fp64 instructions per page and 64 probes, the fp64 ones at half rate), and
// waves wait 47% of theirs, mostly for scalar loads (with the page data always
// in the scalar cache the kernel is 12% faster).  The scalar cache reads whole 4-byte words and drops the low
// bits of an address, so coefficients that start between two words (a view at
// an odd element; the encode kernel writes those too) take the instance
// without WORDS, which reads them one by one.  432 pages, 3 heads x 72 blocks, kernel trace: 94 us (32 probes
// per wave, page data broadcast from LDS, three accumulated mixtures, 369
// registers at one wave per SIMD) -> 54 us; the trace runs below the load
// clock.
template <bool WORDS>
__global__ __launch_bounds__(64 * kRowWaves, 2) void pset_rows_kernel(PsetParams p) {
  __shared__ RowsSmem s;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int NG = (p.T + kRowBlocks - 1) / kRowBlocks;
  const int sp = blockIdx.x % kSplit;
  const int hs = blockIdx.x / (kSplit * NG), t0 = (blockIdx.x / kSplit % NG) * kRowBlocks;
  const int h = __builtin_amdgcn_readfirstlane(p.heads[hs]);
  const int P = p.P;
  const int nrow = min(kRowBlocks, p.T - t0);

  // this range's page data towards the L2 (768 bytes per page): the scalar
  // loads of the page steps wait for each other, so none of them should be
  // the first to miss.  The requests are dropped once the setup is done.
  constexpr int kWaves = kSplit * kRowWaves, kWarm = (kMaxPages / kWaves + 7) / 8;
  const int share = sp * kRowWaves + wave;
  const int page0 = share * P / kWaves, page1 = (share + 1) * P / kWaves;
  u32x4 warm[kWarm][3];
#pragma unroll
  for (int i = 0; i < kWarm; ++i) {
    const int page = min(page0 + 8 * i + (lane >> 3), P - 1), c = lane & 7;
    const long long pe = (long long)h * p.EP + page;
    warm[i][0] = ldg16(p.coef + pe * kCoefStride + 16 * c);
    warm[i][1] = *reinterpret_cast<const u32x4*>(p.mean_b + pe * 16 + 2 * c);
    warm[i][2] = *reinterpret_cast<const u32x4*>(p.detail_b + pe * 48 + 6 * c);
  }
  // probe rows into LDS: row r = block r / 16, probe r % 16
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = (tid >> 4) + 32 * i, c = tid & 15;
    const int tb = min(t0 + (r >> 4), p.T - 1);
    const long long rr = p.gathered ? (r & 15) : probe_row(r & 15);
    const uint16_t* qq = p.q + (long long)h * p.q_head + (long long)tb * p.q_block + rr * p.q_row;
    *reinterpret_cast<u32x4*>(&s.q[r * 256 + ((c ^ (r & 15)) << 4)]) = ldg16(qq + 8 * c);
  }
  for (int i = tid; i < kRowBlocks * P; i += 64 * kRowWaves) {
    const int b = i / P, pg = i % P;
    const int tb = min(t0 + b, p.T - 1);
    s.sel[b][pg] = p.mask[((long long)h * p.T + tb) * P + pg] ? 1 : 0;
    s.slot[b][pg] = -1;
    s.aslot[b][pg] = -1;
  }
  __syncthreads();
  if (tid < kRowBlocks * kCand) {
    const int b = tid / kCand, sl = tid % kCand;
    const int tb = min(t0 + b, p.T - 1);
    const int page = p.pool[((long long)hs * p.T + tb) * kPoolInts + sl];
    if (page >= 0 && page < P) (sl < 16 ? s.slot : s.aslot)[b][page] = (int8_t)sl;
  }
  // reader query u = Wq . probe (fp32) and the probe LSE from the router
  {
    const int pr = tid >> 3, i = tid & 7;
    const f32x4* wr = reinterpret_cast<const f32x4*>(p.wq + i * 128);
    float acc = 0.f;
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      const u32x4 qv = *reinterpret_cast<const u32x4*>(&s.q[pr * 256 + ((c ^ (pr & 15)) << 4)]);
      const f32x4 w0 = wr[2 * c], w1 = wr[2 * c + 1];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        acc = fmaf(bf16_lo(qv[k]), w0[2 * k], acc);
        acc = fmaf(bf16_hi(qv[k]), w0[2 * k + 1], acc);
        acc = fmaf(bf16_lo(qv[2 + k]), w1[2 * k], acc);
        acc = fmaf(bf16_hi(qv[2 + k]), w1[2 * k + 1], acc);
      }
    }
    s.u[pr][i] = acc;
    if (i == 0) s.L[pr] = p.lse[((long long)h * p.T + min(t0 + (pr >> 4), p.T - 1)) * 16 + (pr & 15)];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kWarm; ++i) asm volatile("" ::"v"(warm[i][0]), "v"(warm[i][1]), "v"(warm[i][2]));
  const int blk = lane >> 4, m = lane & 15;
  float u[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) u[i] = s.u[lane][i];
  const double L = (double)s.L[lane];
  const uint16_t* rkh = p.rk + (long long)h * p.HP * 4 * kHeadDim;
  const float c2 = kLog2e / sqrtf((float)kHeadDim);    // logits in log2 units
  constexpr float kLn2 = 0.69314718055994531f;
  double* const row = p.cand + ((long long)hs * p.T + min(t0 + blk, p.T - 1)) * kRowDoubles;
  double* const mine = row + m * (kCand * kCandStride);
  const bool live = blk < nrow;

  double accT[16], accB[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) accT[e] = accB[e] = 0.0;
  double sT = 0.0, sB = 0.0, lmax = -INFINITY;

  // one page, its 4 rep logits of this lane's probe in z
  auto page_step = [&](int page, const float (&zr)[4]) {
    const long long pe = (long long)h * p.EP + page;
    const uint16_t* const cf = p.coef + pe * kCoefStride;
    Const<double>* mb = scalar(p.mean_b + pe * 16);
    Const<double>* db = scalar(p.detail_b + pe * 48);
    auto coef = [&](int i) {
      if constexpr (WORDS) {
        const uint32_t w = scalar(reinterpret_cast<const uint32_t*>(cf))[i >> 1];
        return i & 1 ? bf16_hi(w) : bf16_lo(w);
      } else {
        return bf16_to_f32(cf[i]);
      }
    };
    // rep softmax of the page (fp32), page log mass in fp64
    float z[4], w[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) z[r] = zr[r] * c2;
    const float zm = fmaxf(fmaxf(z[0], z[1]), fmaxf(z[2], z[3]));
    float sw = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      w[r] = __builtin_amdgcn_exp2f(z[r] - zm);
      sw += w[r];
    }
    const double lm = (double)((zm + __log2f(sw)) * kLn2) - L;
    const float isw = recip(sw);       // sw is in [1, 4]
    const double d0 = (w[0] + w[1] - w[2] - w[3]) * isw;
    const double d1 = (w[0] - w[1] + w[2] - w[3]) * isw;
    const double d2 = (w[0] - w[1] - w[2] + w[3]) * isw;
    // readout: F_j = tanh(u . A_j), val = co_0 + sum_j F_j co_{j+1}
    float F[4];
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      float acc = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) acc = fmaf(u[i], coef(kCoefA + 4 * i + jj), acc);
      F[jj] = tanh_f32(acc);
    }
    float val[17];
#pragma unroll
    for (int k = 0; k < 17; ++k) {
      float acc = 0.f;
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) acc = fmaf(F[jj], coef((jj + 1) * 17 + k), acc);
      val[k] = coef(k) + acc;
    }
    const double le = lm + (double)val[16];
    const bool sel = s.sel[blk][page];
    const int sl = s.slot[blk][page], sa = s.aslot[blk][page];
    const bool cand = sl >= 0 || sa >= 0;
    const double lg = sel ? le : lm;
    lmax = fmax(lmax, lg);
    // a candidate's share of the sums is the scores kernel's
    const double ex = cand ? 0.0 : (double)__builtin_amdgcn_exp2f((float)lg * kLog2e);
    const double et = cand ? 0.0 : (double)__builtin_amdgcn_exp2f((float)le * kLog2e);
    sB += ex;
    sT += et;
    double ap[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      ap[e] = mb[e] + (d0 * db[e] + d1 * db[16 + e] + d2 * db[32 + e]);
      const double v = ap[e] + (double)val[e];
      accB[e] += ex * (sel ? v : ap[e]);
      accT[e] += et * v;
    }
    if (__any(cand && live)) {
#pragma unroll 1
      for (int k = 0; k < 2; ++k) {
        const int at = k == 0 ? sl : sa;
        if (at < 0 || !live) continue;
        double* d = mine + at * kCandStride;
        union { double v[2]; u32x4 w; } t;
        t.v[0] = lm;
        t.w[2] = __float_as_uint(val[16]);
        t.w[3] = 0u;
        *reinterpret_cast<u32x4*>(d) = t.w;
#pragma unroll
        for (int e = 0; e < 16; e += 2) {
          t.v[0] = ap[e];
          t.v[1] = ap[e + 1];
          *reinterpret_cast<u32x4*>(d + 2 + e) = t.w;
        }
#pragma unroll
        for (int e = 0; e < 16; e += 4)
          *reinterpret_cast<f32x4*>(d + 18 + e / 2) = f32x4{val[e], val[e + 1], val[e + 2], val[e + 3]};
      }
    }
  };

  // the pages of this wave: an even share of the window, in tiles of 8 pages
  // from its first one
  const int pr = lane & 31, hh = lane >> 5;
  u32x4 fk[8];
  auto fetch = [&](int page) {
    const uint16_t* a = rkh + (long long)min(page * 4 + pr, P * 4 - 1) * kHeadDim + 64 * hh;
#pragma unroll
    for (int st = 0; st < 8; ++st) fk[st] = ldg16(a + 8 * st);
  };
  if (page0 < page1) fetch(page0);
#pragma unroll 1
  for (int tile = page0; tile < page1; tile += 8) {
    // the tile's reps against probes 0..31 and 32..63
    f32x16 sa = {}, sb = {};
#pragma unroll
    for (int st = 0; st < 8; ++st) {
      const int c = ((8 * hh + st) ^ (pr & 15)) << 4;
      sa = mfma32(fk[st], *reinterpret_cast<const u32x4*>(&s.q[pr * 256 + c]), sa);
      sb = mfma32(fk[st], *reinterpret_cast<const u32x4*>(&s.q[(32 + pr) * 256 + c]), sb);
    }
    if (tile + 8 < page1) fetch(tile + 8);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // items 4 j .. 4 j + 3 hold page 2 j in lanes 0..31, page 2 j + 1 in
      // lanes 32..63: the lane-half swap gives each page all 64 probes
      float z0[4], z1[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(sa[4 * j + r]), __float_as_uint(sb[4 * j + r]),
                                                        false, false);
        z0[r] = __uint_as_float(x[0]);
        z1[r] = __uint_as_float(x[1]);
      }
      const int page = tile + 2 * j;
      if (page < page1) page_step(page, z0);
      if (page + 1 < page1) page_step(page + 1, z1);
    }
  }
  // sums over the workgroup's waves, by halves
  auto vals = [&](auto f) {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      f(e, accB[e]);
      f(16 + e, accT[e]);
    }
    f(32, sB);
    f(33, sT);
  };
#pragma unroll
  for (int half = kRowWaves / 2; half > 0; half >>= 1) {
    if (wave >= half && wave < 2 * half) {
      double(*d)[64] = s.part[wave - half];
      vals([&](int v, double& x) { d[v][lane] = x; });
      d[34][lane] = lmax;
    }
    __syncthreads();
    if (wave < half) {
      double(*d)[64] = s.part[wave];
      vals([&](int v, double& x) { x += d[v][lane]; });
      lmax = fmax(lmax, d[34][lane]);
    }
    __syncthreads();
  }
  if (wave == 0 && live) {
    double* d = row + kPartAt + sp * (kPartVals * 16) + m;
    vals([&](int v, double& x) { d[16 * v] = x; });
    d[16 * 34] = lmax;
  }
}

// --------------------------------------------------------------- scores ----

constexpr int kPairs = 256;              // 16 removes x the 16 adds each may swap with
constexpr int kScoreWaves = 8, kScoreThreads = 64 * kScoreWaves;
struct ScoreSmem {
  union {
    alignas(16) double cand[kScoreWaves][kCand][kCandStride];   // per wave: one probe's candidate endpoints
    double acc[kScoreWaves][kPairs];                            // its sums over probes, once they are done
  } c;
  double V[kScoreWaves][16][kCand];                // endpoint vectors D(c - H) + e^(e-M) rp, [dim][candidate]
  double EV[kScoreWaves][kCand];                   // E . V of each candidate
  double S[kScoreWaves][kCand];                    // S_r (removes) / T_a (adds), shifted by the row max
  double ex[kScoreWaves][kCand][2];                // e^(lm+beta-M), e^(lm-M) of each candidate
  double wt[kScoreWaves][kCand][2];                // its weight in H and in the target
  double Hs[kScoreWaves][48];                      // H[16] | E[16] | ob[16] of the probe
  double part[kScoreWaves][36];                    // the probe's background sums over the splits
  uint32_t legal[16];
  uint8_t csel[kCand], cdup[kCand];      // candidate selected; an add page already listed as a remove
  int page[kMaxPages];                   // pool pages, then the compacted selection
  unsigned long long key[kMaxPages];     // LUT keys of the compacted selection
  float risk[kMaxPages];
  uint8_t sel[kMaxPages];
  double best[4];
  int besti[4], bad[4];
};

// One workgroup per scoped (head, block); wave w takes probes w and w + 8
// With every log mass shifted by the row max M, e^(-den) of a swap is
// 1/(S_r + T_a) where S_r = B + sum_{k!=r} e^(er_k-M) + e^(lr_r-M) and
// T_a = sum_{k!=a} e^(la_k-M) + e^(ea_a-M) (VR/scores.py:72-73), and each
// endpoint delta of VR/scores.py:81-88 factors into e^(-den) times a
// per-candidate vector, so delta(r,a) = (V_a - V_r) / (S_r + T_a); a pair's
// score then needs |V_a - V_r|^2 and the difference of the candidates' E . V.
// Of the 16 x 32 pairs only those inside a partition can be legal (remove r
// with adds 0..15 for r < 8, 16..31 otherwise; in a 72-page pool adds 0..15),
// so a lane scores 4 pairs per probe, its sums in registers.  Bound by the
// chain of dependent steps per probe, two probes per wave at two waves per
// SIMD.  3 heads x 72 blocks, kernel trace: 48 us (all 512 pairs, three fp64
// products per pair and dim, four probes per wave) -> 27 us; with its LDS reads
// in groups (a read behind a write or a lane's condition waited for itself) ->
// 25 us, the correction call 147.7 -> 145.5.
__global__ __launch_bounds__(kScoreThreads) void pset_scores_kernel(PsetParams p) {
  __shared__ ScoreSmem s;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int hs = blockIdx.x / p.T, t = blockIdx.x % p.T;
  const int h = p.heads[hs];
  const int P = p.P;
  const bool first = P == kCurrent;
  const long long rowbase = (long long)hs * p.T + t;
  const double* const row = p.cand + rowbase * kRowDoubles;
  const int32_t* po = p.pool + rowbase * kPoolInts;
  // A probe's candidates (48 x 26 doubles = 624 16-byte chunks) and split
  // partials are loaded one probe ahead: the loads of probe m + 8 are in
  // flight while probe m is scored.
  constexpr int kChunks = kCand * kCandStride / 2, kLoads = (kChunks + 63) / 64;
  u32x4 v[kLoads];
  double pv[kSplit];
  auto load_probe = [&](int m) {
    const u32x4* cd = reinterpret_cast<const u32x4*>(row + m * (kCand * kCandStride));
#pragma unroll
    for (int k = 0; k < kLoads; ++k) v[k] = cd[min(lane + 64 * k, kChunks - 1)];
#pragma unroll
    for (int k = 0; k < kSplit; ++k) pv[k] = row[kPartAt + (k * kPartVals + min(lane, kPartVals - 1)) * 16 + m];
  };
  load_probe(w);
  const int my_page = tid < kCand ? po[tid] : -1;
  if (tid < kCand) s.page[tid] = my_page;
  if (tid < 16) s.legal[tid] = (uint32_t)po[kCand + tid];
  for (int i = tid; i < P; i += kScoreThreads) {
    const long long r = ((long long)h * p.T + t) * P + i;
    s.risk[i] = p.risk[r];
    s.sel[i] = p.mask[r] ? 1 : 0;
  }
  __syncthreads();
  if (tid < kCand) {
    // a 72-page pool may list an add page among its removes: counted once
    bool dup = false;
    if (tid >= 16)
      for (int k = 0; k < 16; ++k) dup = dup || s.page[k] == my_page;
    s.cdup[tid] = dup;
    s.csel[tid] = my_page >= 0 && my_page < P && s.sel[my_page];
  }
  __syncthreads();
  auto wave_fence = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  // this lane's pairs: remove i, add j (slot 16 + j)
  auto pair_of = [&](int pr, int& i, int& j) {
    i = pr >> 4;
    j = (pr & 15) + (!first && i >= 8 ? 16 : 0);
  };
  auto rp_of = [](const double* c, int e) { return (double)reinterpret_cast<const float*>(c + 18)[e]; };
  double acc[kPairs / 64];
#pragma unroll
  for (int q = 0; q < kPairs / 64; ++q) acc[q] = 0.0;
#pragma unroll 1
  for (int m = w; m < 16; m += kScoreWaves) {
    // stage the probe's candidates and background sums, then request the next probe's
    {
      u32x4* dst = reinterpret_cast<u32x4*>(&s.c.cand[w][0][0]);
#pragma unroll
      for (int k = 0; k < kLoads; ++k)
        if (lane + 64 * k < kChunks) dst[lane + 64 * k] = v[k];
      double x = pv[0];
#pragma unroll
      for (int k = 1; k < kSplit; ++k) x = lane == 34 ? fmax(x, pv[k]) : x + pv[k];
      if (lane < kPartVals) s.part[w][lane] = x;
    }
    if (m + kScoreWaves < 16) load_probe(m + kScoreWaves);
    wave_fence();
    const double M = s.part[w][34], shift = exp(-M), B = s.part[w][32] * shift;
    const double* c = s.c.cand[w][min(lane, kCand - 1)];
    double EX = 0.0, LM = 0.0, D = 0.0;
    if (lane < kCand) {
      const double lmk = c[0], bk = (double)reinterpret_cast<const float*>(c + 1)[0];
      EX = exp(lmk + bk - M);
      LM = exp(lmk - M);
      D = fabs(bk) < 0.5 ? LM * expm1(fmin(fmax(bk, -0.5), 0.5)) : EX - LM;
      s.ex[w][lane][0] = EX;
      s.ex[w][lane][1] = LM;
      s.wt[w][lane][0] = s.cdup[lane] ? 0.0 : s.csel[lane] ? EX : LM;
      s.wt[w][lane][1] = s.cdup[lane] ? 0.0 : EX;
    }
    wave_fence();
    // H and the target: the background sums and the candidates (lane: dim
    // l % 16, candidates 12 (l / 16) .. + 11)
    {
      const int e = lane & 15, g = lane >> 4;
      double aH = 0.0, aT = 0.0, zH = 0.0, zT = 0.0;
#pragma unroll
      for (int k = 12 * g; k < 12 * g + 12; ++k) {
        const double* ck = s.c.cand[w][k];
        const double wh = s.wt[w][k][0], wx = s.wt[w][k][1], ap = ck[2 + e], full = ap + rp_of(ck, e);
        aH = fma(wh, s.csel[k] ? full : ap, aH);
        aT = fma(wx, full, aT);
        zH += wh;
        zT += wx;
      }
      aH += xor_lane<16>(aH);
      aT += xor_lane<16>(aT);
      zH += xor_lane<16>(zH);
      zT += xor_lane<16>(zT);
      aH += xor_lane<32>(aH);
      aT += xor_lane<32>(aT);
      zH += xor_lane<32>(zH);
      zT += xor_lane<32>(zT);
      const double bH = s.part[w][e], Hv = fma(bH, shift, aH) / (zH + B);
      if (g == 0) {
        s.Hs[w][e] = Hv;
        s.Hs[w][16 + e] = fma(s.part[w][16 + e], shift, aT) / (fma(s.part[w][33], shift, zT)) - Hv;
        s.Hs[w][32 + e] = bH / s.part[w][32];
      }
    }
    wave_fence();
    // per candidate: endpoint vector, its E . V and its share of the swap
    // denominator (leave-one-out sums over the other candidates of its group)
    if (lane < kCand) {
      double ev = 0.0, x[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        x[e] = D * (c[2 + e] - s.Hs[w][e]) + EX * rp_of(c, e);
        ev = fma(s.Hs[w][16 + e], x[e], ev);
      }
      // written once all is read: reads stay behind the writes before them
#pragma unroll
      for (int e = 0; e < 16; ++e) s.V[w][e][lane] = x[e];
      s.EV[w][lane] = ev;
      // every entry is read and the lane's own left out of the sum: a read
      // under a condition of the lane waits for itself
      const int g0 = lane < 16 ? 0 : 16, gn = lane < 16 ? 16 : 32, col = lane < 16 ? 0 : 1;
      double others[32];
#pragma unroll
      for (int k = 0; k < 32; ++k) others[k] = s.ex[w][min(g0 + k, kCand - 1)][col];
      double loo = 0.0;
#pragma unroll
      for (int k = 0; k < 32; ++k) loo += k < gn && g0 + k != lane ? others[k] : 0.0;
      s.S[w][lane] = lane < 16 ? B + loo + LM : loo + EX;
    }
    wave_fence();
    uint32_t badmask = 0u;
#pragma unroll
    for (int q = 0; q < kPairs / 64; ++q) {
      int i, j;
      pair_of(lane + 64 * q, i, j);
      const double den = s.S[w][i] + s.S[w][16 + j];
      const double inv = 1.0 / den;
      double dd = 0.0;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const double d = s.V[w][e][16 + j] - s.V[w][e][i];
        dd = fma(d, d, dd);
      }
      const double ed = (s.EV[w][16 + j] - s.EV[w][i]) * inv;
      dd *= inv * inv;
      // the reference's "bad" branch: max logs - den > 80, or a non-finite delta
      if (den < 1.8048513878454153e-35 || !(isfinite(inv) && isfinite(ed) && isfinite(dd))) badmask |= 1u << q;
      else acc[q] += 2.0 * ed - dd;
    }
    if (__any(badmask != 0u)) {
      // rare: the mixture after the swap rebuilt from the background and every
      // candidate (VR/scores.py:75-79), minus H
#pragma unroll
      for (int q = 0; q < kPairs / 64; ++q) {
        if (!((badmask >> q) & 1u)) continue;
        int i, j;
        pair_of(lane + 64 * q, i, j);
        const double den = s.S[w][i] + s.S[w][16 + j];
        double ed = 0.0, dd = 0.0;
#pragma unroll 1
        for (int e = 0; e < 16; ++e) {
          double nw = B * s.Hs[w][32 + e];
#pragma unroll 1
          for (int k = 0; k < kCand; ++k) {
            const double* ck = s.c.cand[w][k];
            const bool exact = k < 16 ? k != i : k == 16 + j;      // selected after the swap
            nw += exact ? s.ex[w][k][0] * (ck[2 + e] + rp_of(ck, e)) : s.ex[w][k][1] * ck[2 + e];
          }
          const double d = nw / den - s.Hs[w][e];
          ed += s.Hs[w][16 + e] * d;
          dd += d * d;
        }
        acc[q] += 2.0 * ed - dd;
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();      // the candidates' space takes the sums
#pragma unroll
  for (int q = 0; q < kPairs / 64; ++q) s.c.acc[w][lane + 64 * q] = acc[q];
  __syncthreads();
  // legality, argmax (ties -> lowest pair index), finiteness
  double best = -INFINITY;
  int besti = 0x7fffffff;
  int bad = 0;
  if (tid < kPairs) {
    int i, j;
    pair_of(tid, i, j);
    const int flat = 32 * i + j;
    double sc = 0.0;
#pragma unroll
    for (int k = 0; k < kScoreWaves; ++k) sc += s.c.acc[k][tid];
    sc /= 16.0;
    if (!((s.legal[i] >> j) & 1u)) sc = -1e30;
    if (!isfinite(sc)) bad += 1;
    else {
      best = sc;
      besti = flat;
    }
    if (p.scores) {
      p.scores[rowbase * 512 + flat] = sc;
      p.scores[rowbase * 512 + (flat ^ 16)] = -1e30;     // across partitions: never legal
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double ob = __shfl_xor(best, o);
    const int oi = __shfl_xor(besti, o);
    bad += __shfl_xor(bad, o);
    if (ob > best || (ob == best && oi < besti)) {
      best = ob;
      besti = oi;
    }
  }
  if (lane == 0 && w < kPairs / 64) {
    s.best[w] = best;
    s.besti[w] = besti;
    s.bad[w] = bad;
  }
  __syncthreads();
  best = s.best[0];
  besti = s.besti[0];
  bad = s.bad[0];
  for (int k = 1; k < kPairs / 64; ++k) {
    if (s.best[k] > best || (s.best[k] == best && s.besti[k] < besti)) {
      best = s.best[k];
      besti = s.besti[k];
    }
    bad += s.bad[k];
  }
  const bool exec = bad == 0 && best > 0.0;
  if (tid == 0) {
    p.gain[rowbase] = best;
    p.info[rowbase * 3 + 0] = exec ? 1 : 0;
    p.info[rowbase * 3 + 1] = besti;
    p.info[rowbase * 3 + 2] = bad;
    if (exec) atomicAdd((unsigned long long*)&p.stats[0], 1ull);
    if (bad) atomicAdd((unsigned long long*)&p.stats[2], (unsigned long long)bad);
  }
  if (!exec) return;
  const int rpg = s.page[besti >> 5], apg = s.page[16 + (besti & 31)];
  __syncthreads();
  if (tid == 0) {
    s.sel[rpg] = 0;
    s.sel[apg] = 1;
    const long long base = ((long long)h * p.T + t) * P;
    p.mask[base + rpg] = 0;
    p.mask[base + apg] = 1;
  }
  __syncthreads();
  // LUT of the new selection: own first, then the other selected pages by
  // descending risk, ties -> lower page (compact list, then rank within it)
  if (!p.ids) return;
  const int own = own_page(p, h, t);
  int32_t* ids = p.ids + ((long long)h * p.T + t) * p.C;
  if (w == 0) {
    int cnt = 0;
    for (int base = 0; base < P; base += 64) {
      const int pg = base + lane;
      const bool on = pg < P && s.sel[pg] && pg != own;
      const unsigned long long bal = __ballot(on);
      if (on) s.page[cnt + __popcll(bal & ((1ull << lane) - 1ull))] = pg;   // pool pages no longer needed
      cnt += __popcll(bal);
    }
    if (lane == 0) s.besti[0] = cnt;
  }
  __syncthreads();
  const int nsel = s.besti[0];
  // key (orderable risk, 1023 - page): a higher key ranks first, ties go to
  // the lower page; a page's slot is the count of listed keys above its own
  for (int i = tid; i < nsel; i += kScoreThreads) {
    const int x = s.page[i];
    s.key[i] = ((unsigned long long)orderable(s.risk[x]) << 32) | (uint32_t)(1023 - x);
  }
  __syncthreads();
  if (tid == 0) ids[0] = own;
  for (int i = tid; i < nsel; i += kScoreThreads) {
    const unsigned long long kx = s.key[i];
    int rank = 0;
    for (int k = 0; k < nsel; ++k) rank += s.key[k] > kx;
    if (1 + rank < p.C) ids[1 + rank] = s.page[i];
  }
  // a selection shorter than the table (quotas clamped to their partitions)
  // leaves -1 padding, as the router writes it
  for (int i = 1 + nsel + tid; i < p.C; i += kScoreThreads) ids[i] = -1;
}

// Both entry points: a non-null `layers` table runs `nlayers` layers in one
// launch (entry 0's tensors are also the single-layer arguments).
int encode_launch(const EncodeLayers* layers, int nlayers, const void* keys, const void* mean, const void* detail,
                  const void* stats, int head_pages, const void* basis, const float* w1t, const float* b1,
                  const float* w2_reader, const float* b2_reader, const float* w2_phi, const float* b2_phi,
                  const double* B, void* coef, double* mean_b, double* detail_b, int enc_pages, int heads,
                  int first_page, int pages, int hidden, hipStream_t stream) {
  if (heads <= 0 || pages <= 0 || first_page < 0 || first_page + pages > head_pages ||
      first_page + pages > enc_pages || hidden <= 0 || hidden > kMaxHidden)
    return (int)hipErrorInvalidValue;
  EncodeParams p;
  p.keys = (const uint16_t*)keys;
  p.mean = (const uint16_t*)mean;
  p.detail = (const uint16_t*)detail;
  p.stats = (const uint16_t*)stats;
  p.basis = (const uint16_t*)basis;
  p.HP = head_pages;
  p.w1t = w1t;
  p.b1 = b1;
  p.w2r = w2_reader;
  p.b2r = b2_reader;
  p.w2p = w2_phi;
  p.b2p = b2_phi;
  p.B = B;
  p.coef = (uint16_t*)coef;
  p.mean_b = mean_b;
  p.detail_b = detail_b;
  p.EP = enc_pages;
  p.first = first_page;
  p.pages = pages;
  p.hidden = hidden;
  p.heads = heads;
  const dim3 grid(2 * ((heads * pages + kEncRows - 1) / kEncRows) + heads * ((pages + kProjPages - 1) / kProjPages), 1,
                  nlayers);
  if (layers)
    hipLaunchKernelGGL((encode_kernel<EncodeLayers>), grid, dim3(kEncThreads), 0, stream, p, *layers);
  else
    hipLaunchKernelGGL((encode_kernel<OneLayer>), grid, dim3(kEncThreads), 0, stream, p, OneLayer{});
  return (int)hipGetLastError();
}

}  // namespace

extern "C" {

int ssa_encode(const void* keys, const void* mean, const void* detail, const void* stats, int head_pages,
               const void* basis, const float* w1t, const float* b1, const float* w2_reader, const float* b2_reader,
               const float* w2_phi, const float* b2_phi, const double* B, void* coef, double* mean_b,
               double* detail_b, int enc_pages, int heads, int first_page, int pages, int hidden,
               hipStream_t stream) {
  return encode_launch(nullptr, 1, keys, mean, detail, stats, head_pages, basis, w1t, b1, w2_reader, b2_reader,
                       w2_phi, b2_phi, B, coef, mean_b, detail_b, enc_pages, heads, first_page, pages, hidden, stream);
}

int ssa_encode_layers(int layers, const void* const* keys, const void* const* mean, const void* const* detail,
                      const void* const* stats, int head_pages, const void* const* basis, const float* w1t,
                      const float* b1, const float* w2_reader, const float* b2_reader, const float* w2_phi,
                      const float* b2_phi, const double* B, void* const* coef, double* const* mean_b,
                      double* const* detail_b, int enc_pages, int heads, int first_page, int pages, int hidden,
                      hipStream_t stream) {
  if (layers < 1 || layers > kMaxLayers || !keys || !mean || !detail || !stats || !basis || !coef || !mean_b ||
      !detail_b)
    return (int)hipErrorInvalidValue;
  EncodeLayers t;
  for (int l = 0; l < layers; ++l) {
    if (!keys[l] || !mean[l] || !detail[l] || !stats[l] || !basis[l] || !coef[l] || !mean_b[l] || !detail_b[l])
      return (int)hipErrorInvalidValue;
    t.keys[l] = (const uint16_t*)keys[l];
    t.mean[l] = (const uint16_t*)mean[l];
    t.detail[l] = (const uint16_t*)detail[l];
    t.stats[l] = (const uint16_t*)stats[l];
    t.basis[l] = (const uint16_t*)basis[l];
    t.coef[l] = (uint16_t*)coef[l];
    t.mean_b[l] = mean_b[l];
    t.detail_b[l] = detail_b[l];
  }
  return encode_launch(&t, layers, keys[0], mean[0], detail[0], stats[0], head_pages, basis[0], w1t, b1, w2_reader,
                       b2_reader, w2_phi, b2_phi, B, coef[0], mean_b[0], detail_b[0], enc_pages, heads, first_page,
                       pages, hidden, stream);
}

}  // extern "C"

namespace {

// The three launches of one Full_Pset correction, after argument checks.
int pset_launch(const void* q, long long q_head_stride, long long q_block_stride, long long q_row_stride,
                int gathered, const void* keys, int head_pages, const void* coef, const double* mean_b,
                const double* detail_b, int enc_pages, const float* wq, const float* risk, const float* probe_lse,
                uint8_t* mask, int32_t* ids, const int32_t* own, const int32_t* heads, int n_heads, double* cand,
                int32_t* pool, double* gain, int32_t* info, double* scores, long long* stats, int total_heads,
                int blocks, int pages, int count, hipStream_t stream) {
  // a 72-page window (the first chunk) or a window beyond the anchor frame
  // and the current chunk; any table size (an add slot past the spare pages
  // is an empty candidate)
  const bool first = pages == kCurrent;
  if (n_heads <= 0 || n_heads > total_heads || blocks <= 0 || pages > kMaxPages ||
      (!first && pages <= kAnchors + kCurrent) || head_pages < pages ||
      enc_pages < pages || count < (first ? kAnchors : 1) || count > pages ||
      heads == nullptr || probe_lse == nullptr || cand == nullptr || pool == nullptr || gain == nullptr ||
      info == nullptr || stats == nullptr)
    return (int)hipErrorInvalidValue;
  PsetParams p;
  p.q = (const uint16_t*)q;
  p.q_head = q_head_stride;
  p.q_block = q_block_stride;
  p.q_row = q_row_stride;
  p.gathered = gathered;
  p.rk = (const uint16_t*)keys;
  p.HP = head_pages;
  p.coef = (const uint16_t*)coef;
  p.mean_b = mean_b;
  p.detail_b = detail_b;
  p.EP = enc_pages;
  p.wq = wq;
  p.risk = risk;
  p.lse = probe_lse;
  p.mask = mask;
  p.ids = ids;
  p.own = own;
  p.heads = heads;
  p.HS = n_heads;
  p.cand = cand;
  p.pool = pool;
  p.gain = gain;
  p.info = info;
  p.scores = scores;
  p.stats = stats;
  p.H = total_heads;
  p.T = blocks;
  p.P = pages;
  p.C = count;
  const int groups = (blocks + kRowBlocks - 1) / kRowBlocks;
  hipLaunchKernelGGL(pset_pool_kernel, dim3(n_heads * blocks), dim3(kMaxPages), 0, stream, p);
  const dim3 rows_grid(n_heads * groups * kSplit), rows_block(64 * kRowWaves);
  if (((uintptr_t)coef & 3) == 0)
    hipLaunchKernelGGL(pset_rows_kernel<true>, rows_grid, rows_block, 0, stream, p);
  else
    hipLaunchKernelGGL(pset_rows_kernel<false>, rows_grid, rows_block, 0, stream, p);
  hipLaunchKernelGGL(pset_scores_kernel, dim3(n_heads * blocks), dim3(kScoreThreads), 0, stream, p);
  return (int)hipGetLastError();
}

// Scratch of the allocation-free entry point: for at most kScratchRows scoped
// (head, query block) rows, the candidate scratch [rows, kRowDoubles] fp64 (a
// row's candidates, then its partials), then the pools [rows,64] int32, each
// region at a fixed offset (45.18 MB in all).
// Every entry a call reads is written earlier in the same call (the pool
// kernel writes all 48 slots of each row, the rows kernel the candidates'
// endpoint data and every partial), so nothing in it must start at zero.
constexpr int kScratchRows = 216;   // 3 heads x 72 query blocks
constexpr size_t kCandRowBytes = (size_t)kRowDoubles * sizeof(double);
constexpr size_t kPoolRowBytes = (size_t)kPoolInts * sizeof(int32_t);
constexpr size_t kScratchPoolOff = kScratchRows * kCandRowBytes;
constexpr size_t kScratchBytes = kScratchPoolOff + kScratchRows * kPoolRowBytes;
static_assert(kCandRowBytes % 256 == 0, "regions stay 256-byte aligned");

}  // namespace

static __device__ __align__(256) uint8_t scratch[kScratchBytes];

namespace {

// Device address of `scratch` on each device, looked up once per device with
// that device current (the array's name in host code is only a stand-in).
constexpr int kMaxDevices = 64;
std::mutex scratch_mutex;
uint8_t* scratch_ptr[kMaxDevices] = {};

int device_scratch(uint8_t** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kMaxDevices) return (int)hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(scratch_mutex);
  if (scratch_ptr[dev] == nullptr) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    scratch_ptr[dev] = (uint8_t*)ptr;
  }
  *out = scratch_ptr[dev];
  return (int)hipSuccess;
}

}  // namespace

extern "C" {

int ssa_pset(const void* q, long long q_head_stride, long long q_block_stride, long long q_row_stride,
             int gathered, const void* keys, int head_pages, const void* coef, const double* mean_b,
             const double* detail_b, int enc_pages, const float* wq, const float* risk, const float* probe_lse,
             uint8_t* mask, int32_t* ids, const int32_t* own, const int32_t* heads, int n_heads, double* cand,
             double* rows, int32_t* pool, double* gain, int32_t* info, double* scores, long long* stats,
             int total_heads, int blocks, int pages, int count, hipStream_t stream) {
  (void)rows;
  return pset_launch(q, q_head_stride, q_block_stride, q_row_stride, gathered, keys, head_pages, coef, mean_b,
                     detail_b, enc_pages, wq, risk, probe_lse, mask, ids, own, heads, n_heads, cand, pool, gain, info,
                     scores, stats, total_heads, blocks, pages, count, stream);
}

int ssa_pset_noalloc(const void* q, long long q_head_stride, long long q_block_stride, long long q_row_stride,
                     int gathered, const void* keys, int head_pages, const void* coef, const double* mean_b,
                     const double* detail_b, int enc_pages, const float* wq, const float* risk,
                     const float* probe_lse, uint8_t* mask, int32_t* ids, const int32_t* own, const int32_t* heads,
                     int n_heads, double* gain, int32_t* info, double* scores, long long* stats, int total_heads,
                     int blocks, int pages, int count, hipStream_t stream) {
  if (n_heads <= 0 || blocks <= 0 || (long long)n_heads * blocks > kScratchRows) return (int)hipErrorInvalidValue;
  uint8_t* base = nullptr;
  const int e = device_scratch(&base);
  if (e != (int)hipSuccess) return e;
  return pset_launch(q, q_head_stride, q_block_stride, q_row_stride, gathered, keys, head_pages, coef, mean_b,
                     detail_b, enc_pages, wq, risk, probe_lse, mask, ids, own, heads, n_heads, (double*)base,
                     (int32_t*)(base + kScratchPoolOff), gain, info, scores, stats, total_heads, blocks, pages, count,
                     stream);
}

}  // extern "C"
