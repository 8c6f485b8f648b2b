// Kernels of the 3D convolutional Dij-column denoiser: BF16 MFMA convolutions
// (forward, data gradient, weight gradient) with FP32 accumulation, and the
// elementwise, pooling, loss, reduction and optimizer kernels of the network, behind
// the C ABI of include/hipdn.h. The reference has no learned component; these
// kernels serve the denoised Dij builder (pyradmc_amd/denoise.py).
//
// Layouts. Activations are BF16, position-major "nd" = [N][D][H][W][C] with C a
// multiple of 16; a tensor that feeds a weight gradient also has a channel-major copy
// "cm" = [C][N*D*H*W]. Weights: FP32 master [27][Cout][Cin] (tap = (kz*3+ky)*3+kx);
// BF16 forward copy wf = [27][Cout][Cin]; BF16 data-gradient copy wd = [27][Cin][Cout]
// with the taps flipped (tap -> 26 - tap), so the data gradient is a forward
// convolution of the output gradient.
//
// MFMA: v_mfma_f32_16x16x32_bf16 (gfx950). For D = A x B with A 16x32, B 32x16:
// lane l holds A[l % 16][8 (l / 16) + e], B[8 (l / 16) + e][l % 16] (e = 0..7), and
// D[4 (l / 16) + r][l % 16] (r = 0..3). Every operand is one aligned 16-byte load.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <limits>
#include <mutex>

#include "../../include/hipdn.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__device__ inline f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ inline bf16x8 load8(const __bf16* p) { return *reinterpret_cast<const bf16x8*>(p); }

__device__ inline bf16x8 zero8() {
  bf16x8 z;
#pragma unroll
  for (int e = 0; e < 8; ++e) z[e] = static_cast<__bf16>(0.0f);
  return z;
}

__device__ inline float act(float v, float slope) { return v >= 0.0f ? v : v * slope; }

// Where a convolution reads its input from (inference fuses the preceding element-wise
// step into the operand loads; the values are those the separate kernels would store):
// kSrcPlain x itself; kSrcUp the nearest 2x upsampling of x, which has half the output
// dims (k_up_fwd); kSrcAdd x + x2 rounded to bf16 per element (k_add); kSrcLow8 x whose
// channels beyond the first 8 are zero (the network's padded input), which the
// reduction then skips.
constexpr int kSrcPlain = 0, kSrcUp = 1, kSrcAdd = 2, kSrcLow8 = 3;

__device__ inline bf16x8 add8(bf16x8 a, bf16x8 b) {
  bf16x8 r;
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = static_cast<__bf16>(static_cast<float>(a[e]) + static_cast<float>(b[e]));
  return r;
}

// What a convolution does with its sums: y = act(bias + sum), rounded to bf16, into y_nd
// and (where given) the channel-major y_cm; with skip, y + skip rounded again (the values
// k_add would store) instead of y; with pred, only inp[p][0] + y[p][0] in float32 (the
// values k_loss would predict) and no y at all.
struct Epilogue {
  const float* bias;
  float slope;
  const __bf16* skip;
  __bf16* y_nd;
  __bf16* y_cm;
  float* pred;
  const __bf16* inp;
  int c_in;  // channels of inp
};

// Kinds of epilogue. All but k_conv_fwd_deep are built per kind, and the tiled kernels load what
// it needs (conv_other) before their k-steps, so that the loads run under the MFMAs; kEpiAny
// decides at run time (in k_conv_fwd that cost 1 to 5 %).
constexpr int kEpiPlain = 0, kEpiSkip = 1, kEpiPred = 2, kEpiAny = 3;

// What a lane's four sums of channels cb .. cb + 3 at position p are combined with.
template <int EPI>
__device__ inline uint2 conv_other(const Epilogue& E, int cb, long long p, int cout) {
  if ((EPI == kEpiSkip || EPI == kEpiAny) && E.skip) return *reinterpret_cast<const uint2*>(E.skip + p * cout + cb);
  if ((EPI == kEpiPred || EPI == kEpiAny) && E.pred && cb == 0) {
    unsigned short first;
    std::memcpy(&first, E.inp + p * E.c_in, 2);
    return make_uint2(first, 0u);
  }
  return make_uint2(0u, 0u);
}

// One lane's four sums: channels cb .. cb + 3 of position p.
template <int EPI>
__device__ inline void conv_store(const Epilogue& E, const f32x4& sum, uint2 other, int cb, long long p, int cout,
                                  long long P) {
  __bf16 out[4], with[4];
  std::memcpy(with, &other, 8);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float v = sum[r] + (E.bias ? E.bias[cb + r] : 0.0f);
    out[r] = static_cast<__bf16>(act(v, E.slope));
  }
  if (EPI == kEpiPred || (EPI == kEpiAny && E.pred)) {
    if (cb == 0) E.pred[p] = static_cast<float>(with[0]) + static_cast<float>(out[0]);
    return;
  }
  if (EPI == kEpiSkip || (EPI == kEpiAny && E.skip)) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      out[r] = static_cast<__bf16>(static_cast<float>(out[r]) + static_cast<float>(with[r]));
  }
  uint2 packed;
  std::memcpy(&packed, out, 8);
  *reinterpret_cast<uint2*>(E.y_nd + p * cout + cb) = packed;
  if (E.y_cm) {
#pragma unroll
    for (int r = 0; r < 4; ++r) E.y_cm[static_cast<long long>(cb + r) * P + p] = out[r];
  }
}

// ------------------------------------------------------------------ convolution
//
// y[p][co] = act(bias[co] + sum_{tap, ci} x[p + off(tap)][ci] wt[tap][co][ci]) with
// zero padding. One wave computes 16*TM output channels x 64 positions (4 blocks of
// 16); a workgroup of 4 waves covers 256 consecutive positions (P % 64 == 0). K = 27*cin runs in
// chunks of 32; each lane's 8 k values lie inside one tap since cin % 8 == 0.
template <int TM, int SRC, int EPI>
__global__ void __launch_bounds__(256) k_conv_fwd(const __bf16* __restrict__ x,
                                                  const __bf16* __restrict__ x2,
                                                  const __bf16* __restrict__ wt, Epilogue E, int n, int d, int h,
                                                  int w, int cin, int cout) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const long long P = static_cast<long long>(n) * d * h * w;
  const long long p0 = (static_cast<long long>(blockIdx.x) * 4 + wave) * 64;
  if (p0 >= P) return;  // whole wave past the end (P % 64 == 0); no barriers follow
  const int co0 = blockIdx.y * 16 * TM;
  const int col = lane & 15;
  const int kg = lane >> 4;

  int pn[4], pz[4], py[4], px[4];
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
    long long t = p0 + 16 * nb + col;
    px[nb] = static_cast<int>(t % w);
    t /= w;
    py[nb] = static_cast<int>(t % h);
    t /= h;
    pz[nb] = static_cast<int>(t % d);
    pn[nb] = static_cast<int>(t / d);
  }

  f32x4 acc[TM][4];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) acc[m][nb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  const int kc = SRC == kSrcLow8 ? 8 : cin;  // channels read per tap
  const int K = 27 * kc;
  for (int k0 = 0; k0 < K; k0 += 32) {
    const int k = k0 + 8 * kg;
    bf16x8 a[TM], b[4];
    if (k < K) {
      const int tap = k / kc;
      const int c = k - tap * kc;
      const int dz = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dx = tap % 3 - 1;
#pragma unroll
      for (int m = 0; m < TM; ++m)
        a[m] = load8(wt + (static_cast<long long>(tap) * cout + co0 + 16 * m + col) * cin + c);
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) {
        const int zz = pz[nb] + dz, yy = py[nb] + dy, xx = px[nb] + dx;
        if (zz >= 0 && zz < d && yy >= 0 && yy < h && xx >= 0 && xx < w) {
          if constexpr (SRC == kSrcUp) {
            const long long q =
                ((static_cast<long long>(pn[nb]) * (d >> 1) + (zz >> 1)) * (h >> 1) + (yy >> 1)) * (w >> 1) + (xx >> 1);
            b[nb] = load8(x + q * cin + c);
          } else {
            const long long q = ((static_cast<long long>(pn[nb]) * d + zz) * h + yy) * w + xx;
            b[nb] = load8(x + q * cin + c);
            if constexpr (SRC == kSrcAdd) b[nb] = add8(b[nb], load8(x2 + q * cin + c));
          }
        } else {
          b[nb] = zero8();
        }
      }
    } else {
#pragma unroll
      for (int m = 0; m < TM; ++m) a[m] = zero8();
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) b[nb] = zero8();
    }
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) acc[m][nb] = mfma16(a[m], b[nb], acc[m][nb]);
  }

#pragma unroll
  for (int m = 0; m < TM; ++m) {
    const int cb = co0 + 16 * m + 4 * kg;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
      const long long p = p0 + 16 * nb + col;
      conv_store<EPI>(E, acc[m][nb], conv_other<EPI>(E, cb, p, cout), cb, p, cout, P);
    }
  }
}

// The same convolution where 64-position waves are too few to fill the chip (the deep
// levels of a small batch). A wave's k-steps are a serial chain that waits for memory at
// every step, so a wave takes M x M tiles of 16 positions and 16 output channels (4 tm / M^2
// times as many waves as k_conv_fwd<tm> has) and loads its operands 8 (M = 1)
// or 4 k-steps ahead of their MFMAs. Bound by the instructions of a step's addresses with
// one wave per SIMD (37 us instead of 26 with the tap in vector registers), then by L2
// reads, which M = 2 halves. The k-steps keep k_conv_fwd's order: identical sums.
// (Splitting the k-steps over the waves of a workgroup took 22 and 28 us for the two below,
// but its sums round differently, which moved the weight gradients of a training step by
// 3 %.) Four 8^3 volumes of 128 -> 128 channels: 127 us as k_conv_fwd,
// 26 us so; four 16^3, 64 -> 64: 67 and 28 us.
template <int M, bool WIDE, int SRC>
__global__ void __launch_bounds__(256) k_conv_fwd_deep(const __bf16* __restrict__ x, const __bf16* __restrict__ x2,
                                                       const __bf16* __restrict__ wt, Epilogue E, int n, int d, int h,
                                                       int w, int cin, int cout) {
  constexpr int kDeep = M == 1 ? 8 : 4;
  const int lane = threadIdx.x & 63;
  const int col = lane & 15;
  const int kg = lane >> 4;
  const int P = n * d * h * w;  // P * cin and 27 * cin * cout fit an int (conv_fwd)
  const int co0 = blockIdx.y * 16 * M;
  const int p0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 16 * M;
  if (p0 >= P) return;  // P % 64 == 0: the other waves' positions are all inside

  // This lane's tap and first channel in the next k-step to load. Where the channels per tap
  // are a multiple of 32 all lanes of a step share a tap and what depends on it is scalar.
  const int kc = SRC == kSrcLow8 ? 8 : cin;  // channels read per tap
  const int steps = (27 * kc + 31) / 32;
  int tap = WIDE ? 0 : 8 * kg / kc;
  int c = WIDE ? 0 : 8 * kg - tap * kc;
  const int lane_c = WIDE ? 8 * kg : 0;

  int pn[M], pz[M], py[M], px[M], inside[M], at[M];  // inside: bit tap, the tap's voxel exists
#pragma unroll
  for (int i = 0; i < M; ++i) {
    const int p = p0 + 16 * i + col;
    int t = p;
    px[i] = t % w;
    t /= w;
    py[i] = t % h;
    t /= h;
    pz[i] = t % d;
    pn[i] = t / d;
    const int xs = (px[i] > 0) | 2 | (px[i] < w - 1) << 2;
    const int ys = (py[i] > 0) | 1 << 3 | (py[i] < h - 1) << 6;
    const int zs = (pz[i] > 0) | 1 << 9 | (pz[i] < d - 1) << 18;
    inside[i] = xs * ys * zs;  // no two of the products share a bit
    at[i] = p * cin + lane_c;
  }

  bf16x8 a[kDeep][M], b[kDeep][M];
  bool in[kDeep], ok[kDeep][M];
  // What lies past the last tap or outside the volume reads the tensor's first element,
  // always valid, and is replaced by zero where it is used: a replacement here would wait
  // for the load.
  auto load = [&](int j) {
    in[j] = tap < 27;
    const int tp = in[j] ? tap : 0;
    const int dz = tp / 9 - 1, dy = tp / 3 % 3 - 1, dx = tp % 3 - 1;
    const int from = in[j] ? tp * cout * cin + c : 0;
#pragma unroll
    for (int m = 0; m < M; ++m) a[j][m] = load8(wt + (from + ((co0 + 16 * m + col) * cin + lane_c)));
    const int shift = ((dz * h + dy) * w + dx) * cin + c;
#pragma unroll
    for (int i = 0; i < M; ++i) {
      ok[j][i] = in[j] && (inside[i] >> tp & 1);
      int q = at[i] + shift;
      if constexpr (SRC == kSrcUp)
        q = (((pn[i] * (d >> 1) + (pz[i] + dz >> 1)) * (h >> 1) + (py[i] + dy >> 1)) * (w >> 1) + (px[i] + dx >> 1)) * cin +
            lane_c + c;
      q = ok[j][i] ? q : 0;
      b[j][i] = load8(x + q);
      if constexpr (SRC == kSrcAdd) b[j][i] = add8(b[j][i], load8(x2 + q));
    }
    for (c += 32; c >= kc; c -= kc) ++tap;
  };
#pragma unroll
  for (int j = 0; j < kDeep; ++j) load(j);
  f32x4 acc[M][M];
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int i = 0; i < M; ++i) acc[m][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int s = 0; s < steps; s += kDeep) {
#pragma unroll
    for (int j = 0; j < kDeep; ++j) {
      if (s + j < steps) {
#pragma unroll
        for (int m = 0; m < M; ++m)
          if (!WIDE && !in[j]) a[j][m] = zero8();
#pragma unroll
        for (int i = 0; i < M; ++i) {
          if (!ok[j][i]) b[j][i] = zero8();
#pragma unroll
          for (int m = 0; m < M; ++m) acc[m][i] = mfma16(a[j][m], b[j][i], acc[m][i]);
        }
      }
      load(j);
    }
  }
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int i = 0; i < M; ++i) {
      const int cb = co0 + 16 * m + 4 * kg;
      const long long p = p0 + 16 * i + col;
      conv_store<kEpiAny>(E, acc[m][i], conv_other<kEpiAny>(E, cb, p, cout), cb, p, cout, P);
    }
}

// The same convolution for rows of KW = 32 voxels, or 64 (w == KW, h % (256 / KW) == 0,
// cout 16 x TM): a workgroup computes 256 / KW consecutive h-rows of one z-slice (256
// positions; each wave 64 of them) and first stages the input those rows read - 3 z x
// (rows + 2) h x (KW + 2) w positions with their one-voxel halo, zero outside the
// volume - in LDS (KW 32: 33, 65 or 130 KB for cin 16, 32 or 64; KW 64: 38 or 76 KB). Every tap's operand then comes
// from LDS instead of a gathered global load. The k-loop, MFMA operands and output are
// those of k_conv_fwd, so the two kernels give identical sums.
template <int TM, int CIN, int SRC, int EPI, int KW>
__global__ void __launch_bounds__(256) k_conv_fwd_tile(const __bf16* __restrict__ x,
                                                       const __bf16* __restrict__ x2,
                                                       const __bf16* __restrict__ wt, Epilogue E, int n, int d,
                                                       int h, int cout) {
  constexpr int kW = KW, kRows = 256 / KW, kTW = kW + 2, kTH = kRows + 2, kTZ = 3, kC8 = CIN / 8;
  __shared__ u32x4 tile[kTZ * kTH * kTW * kC8];
  const int rows = h / kRows;
  const int hb = static_cast<int>(blockIdx.x % rows);
  const long long t = blockIdx.x / rows;
  const int z = static_cast<int>(t % d);
  const int nn = static_cast<int>(t / d);
  const int h0 = kRows * hb;
  // The tile fill: each thread issues kFill loads before it stores any, so their
  // latencies overlap. A load whose position lies outside the volume (or past the tile)
  // reads the tensor's first element instead, always valid, and is replaced by zero.
  constexpr int kUnits = kTZ * kTH * kTW * kC8;
  constexpr int kFill = 8;
  for (int i0 = threadIdx.x; i0 < kUnits; i0 += 256 * kFill) {
    u32x4 v[kFill], v2[kFill];
    bool ok[kFill];
#pragma unroll
    for (int j = 0; j < kFill; ++j) {
      const int i = i0 + 256 * j;
      const int c8 = i % kC8;
      const int pos = i / kC8;
      const int xx = pos % kTW, yy = (pos / kTW) % kTH, zz = pos / (kTW * kTH);
      const int gz = z + zz - 1, gy = h0 + yy - 1, gx = xx - 1;
      ok[j] = i < kUnits && gz >= 0 && gz < d && gy >= 0 && gy < h && gx >= 0 && gx < kW;
      long long q;
      if constexpr (SRC == kSrcUp)
        q = ((static_cast<long long>(nn) * (d >> 1) + (gz >> 1)) * (h >> 1) + (gy >> 1)) * (kW >> 1) + (gx >> 1);
      else
        q = ((static_cast<long long>(nn) * d + gz) * h + gy) * kW + gx;
      q = ok[j] ? q : 0;
      v[j] = *reinterpret_cast<const u32x4*>(x + q * CIN + 8 * c8);
      if constexpr (SRC == kSrcAdd) v2[j] = *reinterpret_cast<const u32x4*>(x2 + q * CIN + 8 * c8);
    }
#pragma unroll
    for (int j = 0; j < kFill; ++j) {
      const int i = i0 + 256 * j;
      u32x4 val = v[j];
      if constexpr (SRC == kSrcAdd) {
        bf16x8 a8, b8;
        std::memcpy(&a8, &v[j], 16);
        std::memcpy(&b8, &v2[j], 16);
        a8 = add8(a8, b8);
        std::memcpy(&val, &a8, 16);
      }
      if (!ok[j]) val = u32x4{0u, 0u, 0u, 0u};
      if (i < kUnits) tile[i] = val;
    }
  }
  __syncthreads();

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int col = lane & 15;
  const int kg = lane >> 4;
  // Position block nb (16 positions) of this wave: row and first x within the rows.
  int blk_row[4], blk_x[4];
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
    blk_row[nb] = wave * (64 / kW) + (16 * nb) / kW;
    blk_x[nb] = (16 * nb) % kW;
  }
  const long long P = static_cast<long long>(n) * d * h * kW;
  const long long row0 = (static_cast<long long>(nn) * d + z) * h + h0;
  uint2 other[TM][4];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
      other[m][nb] = conv_other<EPI>(E, 16 * m + 4 * kg, (row0 + blk_row[nb]) * kW + blk_x[nb] + col, cout);
  f32x4 acc[TM][4];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) acc[m][nb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  constexpr int kKC = SRC == kSrcLow8 ? 8 : CIN;  // channels read per tap
  constexpr int K = 27 * kKC;
  // Weight fragments of k-step k0 (zero past K): global loads, issued one k-step ahead
  // of their MFMAs so that their latency overlaps the previous step's work.
  auto load_a = [&](int k0, bf16x8 (&a)[TM]) {
    const int k = k0 + 8 * kg;
    if (k < K) {
      const int tap = k / kKC;
      const int c = k - tap * kKC;
#pragma unroll
      for (int m = 0; m < TM; ++m)
        a[m] = load8(wt + (static_cast<long long>(tap) * cout + 16 * m + col) * CIN + c);
    } else {
#pragma unroll
      for (int m = 0; m < TM; ++m) a[m] = zero8();
    }
  };
  // Input fragments of k-step k0 from the LDS tile (zero past K).
  auto load_b = [&](int k0, bf16x8 (&b)[4]) {
    const int k = k0 + 8 * kg;
    if (k < K) {
      const int tap = k / kKC;
      const int c = k - tap * kKC;
      const int dz = tap / 9, dy = (tap / 3) % 3, dx = tap % 3;  // halo-shifted: 0..2
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) {
        const u32x4 v = tile[((dz * kTH + blk_row[nb] + dy) * kTW + dx + blk_x[nb] + col) * kC8 + c / 8];
        std::memcpy(&b[nb], &v, 16);
      }
    } else {
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) b[nb] = zero8();
    }
  };
  auto mfmas = [&](const bf16x8 (&a)[TM], const bf16x8 (&b)[4]) {
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) acc[m][nb] = mfma16(a[m], b[nb], acc[m][nb]);
  };
  // k-steps in order, two per trip: the next step's fragments load into the other
  // register set while this step's MFMAs run (ping-pong, no copies).
  bf16x8 a0[TM], a1[TM], b0[4], b1[4];
  load_a(0, a0);
  load_b(0, b0);
  for (int k0 = 0; k0 < K; k0 += 64) {
    load_a(k0 + 32, a1);
    load_b(k0 + 32, b1);
    mfmas(a0, b0);
    if (k0 + 32 >= K) break;
    load_a(k0 + 64, a0);
    load_b(k0 + 64, b0);
    mfmas(a1, b1);
  }

#pragma unroll
  for (int m = 0; m < TM; ++m) {
    const int cb = 16 * m + 4 * kg;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
      const long long p = (row0 + blk_row[nb]) * kW + blk_x[nb] + col;
      conv_store<EPI>(E, acc[m][nb], other[m][nb], cb, p, cout, P);
    }
  }
}

// Workgroups of k_conv_fwd_march to a CU that its registers are budgeted for: three of
// 16 -> 16 channels, else two; one less with the second input or skip that 16 channels
// prefetch.
template <int TM, int CIN, int SRC, int EPI>
constexpr int kMarchPerCu = (CIN * TM == 16 ? 3 : 2) - (CIN == 16 && (SRC == kSrcAdd || EPI == kEpiSkip) ? 1 : 0);

// The same convolution for rows of 64 voxels (w == 64, h % 4 == 0, cin 16 or 32, cout
// 16 x TM): the full-resolution layers, bound by the LDS reads of their input fragments
// (one 1 KiB fragment per MFMA and 16 output channels). A workgroup takes four h-rows and
// marches along z over zc slices with the three z-planes of a slice in an LDS ring: a
// plane is loaded once per workgroup (1.55 times in all, for the h and w halo) instead of
// once per slice it serves, and the next plane's loads run under this slice's MFMAs. The
// weight fragments of all k-steps stay in registers. 32-channel planes are kept as two
// halves of 16 channels, so that a fragment's lanes read 32-byte strides (64-byte strides
// conflict in the banks). The k-steps and their order are those of k_conv_fwd: identical
// sums. 32 windows of 96 x 64 x 64, us with a 3-plane tile per slice and now: 16 -> 16
// channels 445 and 260 (the copy rate's floor is 170), the 2-channel input 382 and 190,
// 32 -> 16 upsampled 870 and 400 (450 with the skip addition in its store).
template <int TM, int CIN, int SRC, int EPI>
__global__ void __launch_bounds__(256, (kMarchPerCu<TM, CIN, SRC, EPI>)) k_conv_fwd_march(
    const __bf16* __restrict__ x, const __bf16* __restrict__ x2, const __bf16* __restrict__ wt,
    Epilogue E, int n, int d, int h, int cout, int zc) {
  constexpr int kW = 64, kRows = 4, kTW = kW + 2, kTH = kRows + 2, kPos = kTH * kTW;
  constexpr int kKC = SRC == kSrcLow8 ? 8 : CIN;  // channels read per tap
  constexpr int kC8 = kKC / 8;
  constexpr int kPosUnits = kC8 >= 2 ? 2 : 1;      // 16-byte units of a position within a half
  constexpr int kHalf = kPos * kPosUnits;          // units of a half of a plane
  constexpr int kPlane = kPos * kC8;               // units of a plane
  constexpr int kPer = (kPlane + 255) / 256;
  constexpr int K = 27 * kKC, kSteps = (K + 31) / 32;
  __shared__ u32x4 ring[3 * kPlane];
  const int rows = h / kRows;
  const int zchunks = (d + zc - 1) / zc;
  const int hb = static_cast<int>(blockIdx.x % rows);
  const int t = static_cast<int>(blockIdx.x / rows);
  const int z0 = (t % zchunks) * zc;
  const int z1 = z0 + zc < d ? z0 + zc : d;
  const int nn = t / zchunks;
  const int h0 = kRows * hb;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int col = lane & 15;
  const int kg = lane >> 4;

  // This thread's units of a plane: place in the ring's slot, and in the tensor's plane
  // (the half-resolution one for an upsampled input); outside the rows nothing is loaded.
  u32x4 v[kPer], v2[kPer];
  auto load_plane = [&](int gz) {
    const bool zin = gz >= 0 && gz < d;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int i = static_cast<int>(threadIdx.x) + 256 * j;
      const int c8 = i % kC8, pos = i / kC8;
      const int gy = h0 + pos / kTW - 1, gx = pos % kTW - 1;
      const bool ok = zin && i < kPlane && gy >= 0 && gy < h && gx >= 0 && gx < kW;
      long long q;
      if constexpr (SRC == kSrcUp)
        q = ((static_cast<long long>(nn) * (d >> 1) + (gz >> 1)) * (h >> 1) + (gy >> 1)) * (kW >> 1) + (gx >> 1);
      else
        q = ((static_cast<long long>(nn) * d + gz) * h + gy) * kW + gx;
      // An element outside the volume reads the tensor's first one, always valid.
      q = ok ? q * CIN + 8 * c8 : 0;
      v[j] = *reinterpret_cast<const u32x4*>(x + q);
      if constexpr (SRC == kSrcAdd) v2[j] = *reinterpret_cast<const u32x4*>(x2 + q);
      if (!ok) {
        v[j] = u32x4{0u, 0u, 0u, 0u};
        if constexpr (SRC == kSrcAdd) v2[j] = u32x4{0u, 0u, 0u, 0u};
      }
    }
  };
  auto store_plane = [&](int slot) {
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int i = static_cast<int>(threadIdx.x) + 256 * j;
      const int c8 = i % kC8, pos = i / kC8;
      u32x4 val = v[j];
      if constexpr (SRC == kSrcAdd)
        val = __builtin_bit_cast(u32x4, add8(__builtin_bit_cast(bf16x8, v[j]), __builtin_bit_cast(bf16x8, v2[j])));
      if (i < kPlane) ring[slot * kPlane + (c8 / kPosUnits) * kHalf + pos * kPosUnits + c8 % kPosUnits] = val;
    }
  };

  // Weight fragments of every k-step (zero past K).
  bf16x8 a[kSteps][TM];
#pragma unroll
  for (int s = 0; s < kSteps; ++s) {
    const int k = 32 * s + 8 * kg;
    const bool in = k < K;
    const int tap = in ? k / kKC : 0, c = in ? k % kKC : 0;
#pragma unroll
    for (int m = 0; m < TM; ++m) {
      a[s][m] = load8(wt + (static_cast<long long>(tap) * cout + 16 * m + col) * CIN + c);
      if (!in) a[s][m] = zero8();
    }
  }
  // A lane's part of a fragment's place in the ring: its row and column, and its channels
  // where the four lane groups share a tap (their tap where they do not is added per step).
  const int lane_units = (wave * kTW + col) * kPosUnits +
                         (kC8 == 4 ? (kg >> 1) * kHalf + (kg & 1) : kC8 == 2 ? (kg & 1) : 0);

  load_plane(z0 - 1);
  store_plane(0);
  load_plane(z0);
  store_plane(1);
  load_plane(z0 + 1);
  int slot = 2;                              // of the plane in registers
  int pb[3] = {0, kPlane, 2 * kPlane};       // units of planes z - 1, z, z + 1
  const long long P = static_cast<long long>(n) * d * h * kW;
  for (int z = z0; z < z1; ++z) {
    store_plane(slot);
    __syncthreads();
    const long long row = ((static_cast<long long>(nn) * d + z) * h + h0 + wave) * kW;
    uint2 other[TM][4];
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int nb = 0; nb < 4; ++nb)
        other[m][nb] = conv_other<EPI>(E, 16 * m + 4 * kg, row + 16 * nb + col, cout);
    if (z + 1 < z1) load_plane(z + 2);
    // Fragments of k-step s (zero past K: a zero weight times an infinity is no zero). Taps
    // of the step's lane groups: kC8 groups share one.
    auto load_b = [&](int s, bf16x8 (&b)[4]) {
      constexpr int kTaps = 4 / kC8;  // taps of a step
      int at;
      if constexpr (kC8 == 4) {
        at = pb[s / 9] + ((s / 3 % 3) * kTW + s % 3) * kPosUnits;
      } else {
        at = 0;
#pragma unroll
        for (int g = kTaps - 1; g >= 0; --g) {
          const int tap = kTaps * s + g < 27 ? kTaps * s + g : 26;
          const int u = pb[tap / 9] + ((tap / 3 % 3) * kTW + tap % 3) * kPosUnits;
          at = kg / kC8 <= g ? u : at;
        }
      }
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) {
        const u32x4 f = ring[lane_units + at + 16 * nb * kPosUnits];
        std::memcpy(&b[nb], &f, 16);
        if (kTaps * (s + 1) > 27 && kTaps * s + kg / kC8 >= 27) b[nb] = zero8();
      }
    };
    f32x4 acc[TM][4];
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) acc[m][nb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    bf16x8 b[2][4];
    load_b(0, b[0]);
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      if (s + 1 < kSteps) load_b(s + 1, b[(s + 1) & 1]);
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) acc[m][nb] = mfma16(a[s][m], b[s & 1][nb], acc[m][nb]);
    }
#pragma unroll
    for (int m = 0; m < TM; ++m) {
      const int cb = 16 * m + 4 * kg;
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) {
        const long long p = row + 16 * nb + col;
        conv_store<EPI>(E, acc[m][nb], other[m][nb], cb, p, cout, P);
      }
    }
    __syncthreads();  // plane z - 1 is read no more: the next plane takes its slot
    const int first = pb[0];
    pb[0] = pb[1];
    pb[1] = pb[2];
    pb[2] = first;
    slot = slot == 2 ? 0 : slot + 1;
  }
}

// 8 channel-major elements x[c][row + x0 + dx .. + 7] of one W-row (w % 8 == 0,
// x0 % 8 == 0), zero outside [0, w): the tap's x shift as a funnel shift of aligned
// 16-byte loads.
__device__ inline bf16x8 load_row8(const __bf16* row, int x0, int w, int dx) {
  const u32x4 cur = *reinterpret_cast<const u32x4*>(row + x0);
  u32x4 out;
  if (dx == 0) {
    out = cur;
  } else if (dx > 0) {
    const u32x4 nxt = x0 + 8 < w ? *reinterpret_cast<const u32x4*>(row + x0 + 8) : u32x4{0, 0, 0, 0};
    out[0] = (cur[0] >> 16) | (cur[1] << 16);
    out[1] = (cur[1] >> 16) | (cur[2] << 16);
    out[2] = (cur[2] >> 16) | (cur[3] << 16);
    out[3] = (cur[3] >> 16) | (nxt[0] << 16);
  } else {
    const u32x4 prv = x0 > 0 ? *reinterpret_cast<const u32x4*>(row + x0 - 8) : u32x4{0, 0, 0, 0};
    out[0] = (cur[0] << 16) | (prv[3] >> 16);
    out[1] = (cur[1] << 16) | (cur[0] >> 16);
    out[2] = (cur[2] << 16) | (cur[1] >> 16);
    out[3] = (cur[3] << 16) | (cur[2] >> 16);
  }
  bf16x8 r;
  std::memcpy(&r, &out, 16);
  return r;
}

// A workgroup's weight-gradient block: the four waves' accumulators added in wave order,
// nine taps at a time through LDS, and written by the first wave.
// D[i = ci][j = co]: a lane holds ci = ci0 + 4 kg + r, co = co0 + col.
__device__ inline void store_wgrad(const f32x4 (&acc)[27], float4 (*sums)[9][64], float* out, int ci0, int co0,
                                   int cin, int cout) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
#pragma unroll
  for (int t0 = 0; t0 < 27; t0 += 9) {
    __syncthreads();
    if (wave > 0) {
#pragma unroll
      for (int t = 0; t < 9; ++t)
        sums[wave - 1][t][lane] = make_float4(acc[t0 + t][0], acc[t0 + t][1], acc[t0 + t][2], acc[t0 + t][3]);
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        float4 v = make_float4(acc[t0 + t][0], acc[t0 + t][1], acc[t0 + t][2], acc[t0 + t][3]);
#pragma unroll
        for (int w = 0; w < 3; ++w) {
          const float4 o = sums[w][t][lane];
          v.x += o.x;
          v.y += o.y;
          v.z += o.z;
          v.w += o.w;
        }
        *reinterpret_cast<float4*>(out + (static_cast<long long>(t0 + t) * cout + co0 + (lane & 15)) * cin + ci0 +
                                   4 * (lane >> 4)) = v;
      }
    }
  }
}

// Weight-gradient partials: part[s][tap][co][ci] = sum over split s's positions of
// dz[p][co] x[p + off(tap)][ci]. A workgroup owns one 16x16 (ci, co) block for all 27
// taps (108 accumulators a lane) and a contiguous range of positions, which its four waves
// take in chunks of 32; their sums add in wave order (store_wgrad). For rows that
// k_conv_wgrad_tile does not take.
__global__ void __launch_bounds__(256) k_conv_wgrad(const __bf16* __restrict__ x_cm,
                                                   const __bf16* __restrict__ dz_cm,
                                                   float* __restrict__ part, int n, int d, int h,
                                                   int w, int cin, int cout, long long per_split) {
  __shared__ float4 sums[3][9][64];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int col = lane & 15;
  const int kg = lane >> 4;
  const int ci0 = 16 * blockIdx.x;
  const int co0 = 16 * blockIdx.y;
  const int split = blockIdx.z;
  const long long P = static_cast<long long>(n) * d * h * w;
  const long long pbeg = static_cast<long long>(split) * per_split;
  const long long pend = pbeg + per_split < P ? pbeg + per_split : P;

  f32x4 acc[27];
#pragma unroll
  for (int t = 0; t < 27; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  const __bf16* xrow_c = x_cm + static_cast<long long>(ci0 + col) * P;
  const __bf16* dz_c = dz_cm + static_cast<long long>(co0 + col) * P;
  for (long long pb = pbeg + 32 * wave; pb < pend; pb += 128) {
    const long long p = pb + 8 * kg;  // this lane's 8 positions: one aligned W-row segment
    const bf16x8 b = load8(dz_c + p);
    long long t = p;
    const int x0 = static_cast<int>(t % w);
    t /= w;
    const int y = static_cast<int>(t % h);
    t /= h;
    const int z = static_cast<int>(t % d);
    const long long nn = t / d;
#pragma unroll
    for (int dzz = -1; dzz <= 1; ++dzz) {
#pragma unroll
      for (int dyy = -1; dyy <= 1; ++dyy) {
        const int zz = z + dzz, yy = y + dyy;
        const bool row_ok = zz >= 0 && zz < d && yy >= 0 && yy < h;
        const long long row_off = row_ok ? ((nn * d + zz) * h + yy) * w : 0;
#pragma unroll
        for (int dxx = -1; dxx <= 1; ++dxx) {
          const int tap = ((dzz + 1) * 3 + (dyy + 1)) * 3 + (dxx + 1);
          const bf16x8 a = row_ok ? load_row8(xrow_c + row_off, x0, w, dxx) : zero8();
          acc[tap] = mfma16(a, b, acc[tap]);
        }
      }
    }
  }
  store_wgrad(acc, sums, part + static_cast<long long>(split) * 27 * cout * cin, ci0, co0, cin, cout);
}

// The same partials for rows of W = 64, 32 or 16 voxels (w == W, h % (256 / W) == 0): a
// workgroup takes tiles of 256 positions (256 / W rows of one z-slice; each wave 64 of
// them) and stages the 16 input channels' rows of a tile - 3 z x (rows + 2) h, zero
// outside the volume - in LDS, so an element is loaded 4.5 times (W = 64) instead of 27,
// in runs of whole rows. The rows of one channel-major tensor lie the channel stride
// apart (2 MiB at 128^3 voxels), so gathering a tap's 16 channels straight from memory sent
// every load of a wave to one L2 channel. Rows are 8 elements longer than W: the zeros
// beyond both row ends, read by the +-1 shifts. The channel stride is an odd number of
// 16-byte units, so that 16 channels' reads spread over the banks. The next tile's loads
// are issued before this tile's products and stored to LDS after them.
// Four 64^3 volumes of 16 -> 16 channels: 172 us gathered, 57 us staged; 32^3, 64 -> 32:
// 158 and 50 us.
template <int W>
__global__ void __launch_bounds__(256, 2) k_conv_wgrad_tile(const __bf16* __restrict__ x_cm,
                                                         const __bf16* __restrict__ dz_cm,
                                                         float* __restrict__ part, int n, int d, int h, int cin,
                                                         int cout, int splits) {
  constexpr int kRows = 256 / W, kTH = kRows + 2, kStride = W + 8, kChannel = 3 * kTH * kStride + 8;
  constexpr int kUnits = 16 * 3 * kTH * (W / 8);  // 16-byte units of a tile
  constexpr int kPer = (kUnits + 255) / 256;
  static_assert(kChannel % 16 == 8, "the channel stride is an odd number of 16-byte units");
  constexpr int kSumBytes = 3 * 9 * 64 * static_cast<int>(sizeof(float4));
  constexpr int kBytes = 16 * kChannel * 2 > kSumBytes ? 16 * kChannel * 2 : kSumBytes;
  __shared__ __align__(16) unsigned char lds[kBytes];
  __bf16* tile = reinterpret_cast<__bf16*>(lds);
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int col = lane & 15;
  const int kg = lane >> 4;
  const int ci0 = 16 * blockIdx.x;
  const int co0 = 16 * blockIdx.y;
  const int split = blockIdx.z;
  const int rows = h / kRows;
  const long long P = static_cast<long long>(n) * d * h * W;
  const long long tiles = P / 256;
  const long long t_beg = tiles * split / splits, t_end = tiles * (split + 1) / splits;

  for (int i = threadIdx.x; i < kBytes / 16; i += 256)  // row ends (and all else) start as zeros
    reinterpret_cast<u32x4*>(lds)[i] = u32x4{0u, 0u, 0u, 0u};

  u32x4 next[kPer];
  bf16x8 dz_next[2];
  auto load_tile = [&](long long t) {
    const int hb = static_cast<int>(t % rows);
    const long long zt = t / rows;
    const int z = static_cast<int>(zt % d);
    const long long nn = zt / d;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int i = static_cast<int>(threadIdx.x) + 256 * j;
      const int x8 = i % (W / 8), row = (i / (W / 8)) % (3 * kTH), ch = i / (W / 8 * 3 * kTH);
      const int gz = z + row / kTH - 1, gy = hb * kRows + row % kTH - 1;
      const bool ok = i < kUnits && gz >= 0 && gz < d && gy >= 0 && gy < h;
      // An element outside the volume reads the tensor's first one, always valid.
      const long long at = ok ? static_cast<long long>(ci0 + ch) * P + ((nn * d + gz) * h + gy) * W + 8 * x8 : 0;
      const u32x4 v = *reinterpret_cast<const u32x4*>(x_cm + at);
      next[j] = ok ? v : u32x4{0u, 0u, 0u, 0u};
    }
    const __bf16* dz = dz_cm + static_cast<long long>(co0 + col) * P + t * 256 + 64 * wave + 8 * kg;
    dz_next[0] = load8(dz);
    dz_next[1] = load8(dz + 32);
  };
  auto store_tile = [&]() {
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int i = static_cast<int>(threadIdx.x) + 256 * j;
      const int x8 = i % (W / 8), row = (i / (W / 8)) % (3 * kTH), ch = i / (W / 8 * 3 * kTH);
      if (i < kUnits) *reinterpret_cast<u32x4*>(tile + ch * kChannel + row * kStride + 8 + 8 * x8) = next[j];
    }
  };

  f32x4 acc[27];
#pragma unroll
  for (int t = 0; t < 27; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  if (t_beg < t_end) load_tile(t_beg);
  for (long long t = t_beg; t < t_end; ++t) {
    __syncthreads();  // the previous tile's reads (or the clearing) are done
    store_tile();
    const bf16x8 dz[2] = {dz_next[0], dz_next[1]};
    __syncthreads();
    if (t + 1 < t_end) load_tile(t + 1);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int p = 64 * wave + 32 * c + 8 * kg;  // this lane's 8 positions of the tile
      const __bf16* base = tile + col * kChannel + (p / W) * kStride + 8 + p % W;
#pragma unroll
      for (int zy = 0; zy < 9; ++zy) {
        const __bf16* q = base + ((zy / 3) * kTH + zy % 3) * kStride;
        const u32x4 cur = *reinterpret_cast<const u32x4*>(q);
        const unsigned int before = *reinterpret_cast<const unsigned int*>(q - 2);
        const unsigned int after = *reinterpret_cast<const unsigned int*>(q + 8);
        u32x4 lo, hi;
        lo[0] = __builtin_amdgcn_alignbit(cur[0], before, 16);
        hi[3] = __builtin_amdgcn_alignbit(after, cur[3], 16);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          lo[k + 1] = __builtin_amdgcn_alignbit(cur[k + 1], cur[k], 16);
          hi[k] = lo[k + 1];
        }
        bf16x8 a;
        std::memcpy(&a, &lo, 16);
        acc[3 * zy] = mfma16(a, dz[c], acc[3 * zy]);
        std::memcpy(&a, &cur, 16);
        acc[3 * zy + 1] = mfma16(a, dz[c], acc[3 * zy + 1]);
        std::memcpy(&a, &hi, 16);
        acc[3 * zy + 2] = mfma16(a, dz[c], acc[3 * zy + 2]);
      }
    }
  }
  store_wgrad(acc, reinterpret_cast<float4(*)[9][64]>(lds), part + static_cast<long long>(split) * 27 * cout * cin,
              ci0, co0, cin, cout);
}

// out[i] = sum_s part[s][i] in a fixed order: wave g of the kWaves that share 64 outputs adds
// splits g, g + kWaves, ..., eight loads in flight, and the waves' sums add in wave order
// (launch_reduce has the choice of kWaves).
template <int kWaves>
__global__ void __launch_bounds__(64 * kWaves) k_reduce_splits(const float* __restrict__ part,
                                                               float* __restrict__ out, long long len, int splits) {
  __shared__ float sums[kWaves][64];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  for (long long i0 = static_cast<long long>(blockIdx.x) * 64; i0 < len; i0 += static_cast<long long>(gridDim.x) * 64) {
    const long long i = i0 + lane;
    float s = 0.0f;
    if (i < len) {
#pragma unroll 8
      for (int k = wave; k < splits; k += kWaves) s += part[static_cast<long long>(k) * len + i];
    }
    if constexpr (kWaves == 1) {
      if (i < len) out[i] = s;
    } else {
      sums[wave][lane] = s;
      __syncthreads();
      if (wave == 0 && i < len) {
        for (int g = 1; g < kWaves; ++g) s += sums[g][lane];
        out[i] = s;
      }
      __syncthreads();
    }
  }
}

// Per-channel sums of a channel-major tensor: part[s][c] over split s of the positions.
__global__ void __launch_bounds__(256) k_channel_sum(const __bf16* __restrict__ cm,
                                                     float* __restrict__ part, long long P,
                                                     long long per_split) {
  const int c = blockIdx.x;
  const int s = blockIdx.y;
  const long long beg = static_cast<long long>(s) * per_split;
  const long long end = beg + per_split < P ? beg + per_split : P;
  float acc = 0.0f;
  for (long long p = beg + threadIdx.x; p < end; p += blockDim.x)
    acc += static_cast<float>(cm[static_cast<long long>(c) * P + p]);
  __shared__ float red[256];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (static_cast<int>(threadIdx.x) < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[static_cast<long long>(s) * gridDim.x + c] = red[0];  // [split][C]
}

// ------------------------------------------------------------------- elementwise
//
// Thread = (position p, 8-channel group g): a wave has 64 consecutive positions of one
// group, so its channel-major writes are contiguous, and the next wave the same positions'
// next group, so a position's line is fetched once (with all positions of a group before
// the next group it came from memory once per group).
struct Place {
  long long p;
  int g;
};
__device__ inline Place place(long long i, int groups) {
  const long long wave = i >> 6;
  return {(wave / groups << 6) + (i & 63), static_cast<int>(wave % groups)};
}

__device__ inline void store_both(__bf16* nd, __bf16* cm, long long P, int C, long long p, int g,
                                  const float* v) {
  __bf16 o[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = static_cast<__bf16>(v[e]);
  bf16x8 packed;
  std::memcpy(&packed, o, 16);
  *reinterpret_cast<bf16x8*>(nd + p * C + 8 * g) = packed;
  if (cm) {
#pragma unroll
    for (int e = 0; e < 8; ++e) cm[static_cast<long long>(8 * g + e) * P + p] = o[e];
  }
}

// dz = dy * act'(y) (act'(y) = 1 for y > 0, slope otherwise), both layouts.
__global__ void k_act_bwd(const __bf16* __restrict__ y, const __bf16* __restrict__ dy,
                          __bf16* __restrict__ dz_nd, __bf16* __restrict__ dz_cm, long long P,
                          int C, float slope) {
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  const auto [p, g] = place(i, C / 8);
  if (p >= P) return;
  const bf16x8 yv = load8(y + p * C + 8 * g);
  const bf16x8 gv = load8(dy + p * C + 8 * g);
  float v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float gy = static_cast<float>(gv[e]);
    v[e] = static_cast<float>(yv[e]) > 0.0f ? gy : gy * slope;
  }
  store_both(dz_nd, dz_cm, P, C, p, g, v);
}

// y = a + b, both layouts.
__global__ void k_add(const __bf16* __restrict__ a, const __bf16* __restrict__ b,
                      __bf16* __restrict__ y_nd, __bf16* __restrict__ y_cm, long long P, int C) {
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  const auto [p, g] = place(i, C / 8);
  if (p >= P) return;
  const bf16x8 av = load8(a + p * C + 8 * g);
  const bf16x8 bv = load8(b + p * C + 8 * g);
  float v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = static_cast<float>(av[e]) + static_cast<float>(bv[e]);
  store_both(y_nd, y_cm, P, C, p, g, v);
}

// 2x2x2 average pooling: x [n][2d][2h][2w][C] -> y [n][d][h][w][C] (nd and cm).
__global__ void k_pool_fwd(const __bf16* __restrict__ x, __bf16* __restrict__ y_nd,
                           __bf16* __restrict__ y_cm, int n, int d, int h, int w, int C) {
  const long long P = static_cast<long long>(n) * d * h * w;
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  const auto [p, g] = place(i, C / 8);
  if (p >= P) return;
  long long t = p;
  const int xx = static_cast<int>(t % w);
  t /= w;
  const int yy = static_cast<int>(t % h);
  t /= h;
  const int zz = static_cast<int>(t % d);
  const long long nn = t / d;
  float v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int a = 0; a < 2; ++a)
    for (int b = 0; b < 2; ++b)
      for (int c = 0; c < 2; ++c) {
        const long long q = ((nn * 2 * d + 2 * zz + a) * 2 * h + 2 * yy + b) * 2 * w + 2 * xx + c;
        const bf16x8 s = load8(x + q * C + 8 * g);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += static_cast<float>(s[e]);
      }
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] *= 0.125f;
  store_both(y_nd, y_cm, P, C, p, g, v);
}

// Gradient of the pooling: dx[fine] = dy[coarse] / 8 (nd only). Dims are the fine
// ones (2d, 2h, 2w).
__global__ void k_pool_bwd(const __bf16* __restrict__ dy, __bf16* __restrict__ dx, int n, int d2,
                           int h2, int w2, int C) {
  const long long P = static_cast<long long>(n) * d2 * h2 * w2;
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  const auto [p, g] = place(i, C / 8);
  if (p >= P) return;
  long long t = p;
  const int xx = static_cast<int>(t % w2);
  t /= w2;
  const int yy = static_cast<int>(t % h2);
  t /= h2;
  const int zz = static_cast<int>(t % d2);
  const long long nn = t / d2;
  const long long q = ((nn * (d2 / 2) + zz / 2) * (h2 / 2) + yy / 2) * (w2 / 2) + xx / 2;
  const bf16x8 s = load8(dy + q * C + 8 * g);
  float v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = static_cast<float>(s[e]) * 0.125f;
  store_both(dx, nullptr, P, C, p, g, v);
}

// Nearest 2x upsampling: x [n][d][h][w][C] -> y [n][2d][2h][2w][C]. Dims are the fine
// ones.
__global__ void k_up_fwd(const __bf16* __restrict__ x, __bf16* __restrict__ y_nd,
                         __bf16* __restrict__ y_cm, int n, int d2, int h2, int w2, int C) {
  const long long P = static_cast<long long>(n) * d2 * h2 * w2;
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  const auto [p, g] = place(i, C / 8);
  if (p >= P) return;
  long long t = p;
  const int xx = static_cast<int>(t % w2);
  t /= w2;
  const int yy = static_cast<int>(t % h2);
  t /= h2;
  const int zz = static_cast<int>(t % d2);
  const long long nn = t / d2;
  const long long q = ((nn * (d2 / 2) + zz / 2) * (h2 / 2) + yy / 2) * (w2 / 2) + xx / 2;
  const bf16x8 s = load8(x + q * C + 8 * g);
  float v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = static_cast<float>(s[e]);
  store_both(y_nd, y_cm, P, C, p, g, v);
}

// Gradient of the upsampling: dx[coarse] = sum of dy over its 8 fine cells (nd only).
// Dims are the coarse ones.
__global__ void k_up_bwd(const __bf16* __restrict__ dy, __bf16* __restrict__ dx, int n, int d,
                         int h, int w, int C) {
  const long long P = static_cast<long long>(n) * d * h * w;
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  const auto [p, g] = place(i, C / 8);
  if (p >= P) return;
  long long t = p;
  const int xx = static_cast<int>(t % w);
  t /= w;
  const int yy = static_cast<int>(t % h);
  t /= h;
  const int zz = static_cast<int>(t % d);
  const long long nn = t / d;
  float v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int a = 0; a < 2; ++a)
    for (int b = 0; b < 2; ++b)
      for (int c = 0; c < 2; ++c) {
        const long long q = ((nn * 2 * d + 2 * zz + a) * 2 * h + 2 * yy + b) * 2 * w + 2 * xx + c;
        const bf16x8 s = load8(dy + q * C + 8 * g);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += static_cast<float>(s[e]);
      }
  store_both(dx, nullptr, P, C, p, g, v);
}

// Residual head and sigma-weighted squared error. pred = inp[p][0] + out[p][0];
// per-block partial of sum weight * (pred - target)^2; gradient with respect to out
// (channel 0; the other channels zero) = 2 weight (pred - target) * grad_scale, in
// both layouts. Also writes pred (float) when pred_out is not null.
__global__ void __launch_bounds__(256) k_loss(const __bf16* __restrict__ out,
                                              const __bf16* __restrict__ inp, int c_out, int c_in,
                                              const float* __restrict__ target,
                                              const float* __restrict__ weight,
                                              __bf16* __restrict__ dout_nd,
                                              __bf16* __restrict__ dout_cm,
                                              float* __restrict__ pred_out,
                                              float* __restrict__ partial, long long P,
                                              float grad_scale) {
  const long long p = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  float l = 0.0f;
  if (p < P) {
    const float pred = static_cast<float>(inp[p * c_in]) + static_cast<float>(out[p * c_out]);
    if (pred_out) pred_out[p] = pred;
    if (target) {
      const float diff = pred - target[p];
      const float wt = weight ? weight[p] : 1.0f;
      l = wt * diff * diff;
      if (dout_nd) {
        const __bf16 g = static_cast<__bf16>(2.0f * wt * diff * grad_scale);
        const __bf16 zero = static_cast<__bf16>(0.0f);
        for (int c = 0; c < c_out; ++c) {
          dout_nd[p * c_out + c] = c == 0 ? g : zero;
          if (dout_cm) dout_cm[static_cast<long long>(c) * P + p] = c == 0 ? g : zero;
        }
      }
    }
  }
  __shared__ float red[256];
  red[threadIdx.x] = l;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (static_cast<int>(threadIdx.x) < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0 && partial) partial[blockIdx.x] = red[0];
}

// FP32 master -> BF16 forward [27][cout][cin] and flipped, transposed data-gradient
// [27][cin][cout] copies.
__global__ void k_prepare_weights(const float* __restrict__ master, __bf16* __restrict__ wf,
                                  __bf16* __restrict__ wd, int cin, int cout) {
  const long long total = 27LL * cin * cout;
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const int ci = static_cast<int>(i % cin);
  const long long t = i / cin;
  const int co = static_cast<int>(t % cout);
  const int tap = static_cast<int>(t / cout);
  const __bf16 v = static_cast<__bf16>(master[i]);
  wf[i] = v;
  wd[(static_cast<long long>(26 - tap) * cin + ci) * cout + co] = v;
}

// Adam (Kingma and Ba 2015) with bias correction; zero gradients leave padding zero.
__global__ void k_adam(float* __restrict__ param, const float* __restrict__ grad,
                       float* __restrict__ m, float* __restrict__ v, long long len, float lr,
                       float beta1, float beta2, float eps, float corr1, float corr2,
                       float weight_decay) {
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= len) return;
  const float g = grad[i] + weight_decay * param[i];
  const float mi = beta1 * m[i] + (1.0f - beta1) * g;
  const float vi = beta2 * v[i] + (1.0f - beta2) * g * g;
  m[i] = mi;
  v[i] = vi;
  param[i] -= lr * (mi / corr1) / (sqrtf(vi / corr2) + eps);
}

unsigned int blocks_for(long long n, int threads) {
  return static_cast<unsigned int>((n + threads - 1) / threads);
}

// 256-thread workgroups of an elementwise kernel (place).
unsigned int place_blocks(long long P, int C) { return blocks_for((P + 63) / 64 * 64 * (C / 8), 256); }

hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

int launch_status() { return hipGetLastError() == hipSuccess ? HDN_OK : HDN_EHIP; }

bool shape_ok(int n, int d, int h, int w) { return n > 0 && d > 0 && h > 0 && w > 0; }

}  // namespace

namespace {

// Below kFillWaves 64-position waves a convolution runs as k_conv_fwd_deep, which reads more
// per MFMA; below kPairWaves its waves take one tile instead of 2 x 2. Measured at 12 x 8 x 8
// volumes of 128 -> 128 channels as k_conv_fwd, 2 x 2 tiles and single tiles: 576 waves 130,
// 135 and 213 us, 384 waves 130, 93 and 143 us, 192 waves 128, 48 and 73 us; 8^3 volumes:
// 128 waves 128, 48 and 50 us, 64 waves 128, 48 and 26 us.
constexpr long long kFillWaves = 512;
constexpr long long kPairWaves = 128;

// Slices of a marching workgroup: those for which the rounds that the workgroups take on the
// card, each as long as its slices and about two more for the first planes and the weights,
// are the shortest; where two are alike the longer (fewer planes loaded twice). A fixed
// length of six and up left small volumes on few CUs, and counts off a whole round left the
// last one nearly empty. 16 -> 16 channels over 1 x 8, 1 x 64, 2 x 96 and 16 x 96 slices of
// 64 x 64, us: a 3-plane tile per slice 7.8, 13.1, 29.4 and 225, marching with six slices or
// more 17.7, 18.5, 22.1 and 145, with this rule 7.8, 11.1, 20.3 and 134; 16 -> 32: 8.7, 18.7,
// 41.4 and 322; 25.6, 27.2, 33.3 and 256; 8.2, 17.2, 33.3 and 248.
constexpr int kCus = 256;

int march_slices(long long columns, int d, int per_cu) {
  const long long resident = static_cast<long long>(kCus) * per_cu;
  int best = 1;
  long long least = std::numeric_limits<long long>::max();
  for (int zc = 1; zc <= std::min(d, 128); ++zc) {
    const long long groups = columns * ((d + zc - 1) / zc);
    const long long cost = (groups + resident - 1) / resident * (zc + 2);
    if (cost <= least) {
      least = cost;
      best = zc;
    }
  }
  return best;
}

template <int TM, int CIN, int SRC, int EPI>
int launch_march(const __bf16* xb, const __bf16* x2b, const __bf16* wb, const Epilogue& E, int n, int d, int h,
                 int cout, hipStream_t stream) {
  const long long columns = static_cast<long long>(n) * (h / 4);
  // With 32 channels on either side, a tile per slice where a CU has fewer than three slices
  // (32 -> 16 over 24 slices 10.4 us and 11.7 marching, 16 -> 32 over 40 13.4 and 14.8, over 64
  // 18.7 and 17.2). 16 -> 32 of two added inputs hold one marching workgroup to a CU and are
  // faster so at any size (over 64 slices 21 and 31 us, over 32 x 96 763 and 917).
  constexpr bool kAlways = SRC == kSrcAdd && TM == 2;
  if constexpr (TM * CIN == 32) {
    if (kAlways || columns * d < 3 * kCus) {
      hipLaunchKernelGGL((k_conv_fwd_tile<TM, CIN, SRC, EPI, 64>), dim3(static_cast<unsigned int>(columns * d)),
                         dim3(256), 0, stream, xb, x2b, wb, E, n, d, h, cout);
      return launch_status();
    }
  }
  // The 2-channel input's planes and weights are half as large: four fit.
  const int zc = march_slices(columns, d, SRC == kSrcLow8 && TM * CIN == 16 ? 4 : kMarchPerCu<TM, CIN, SRC, EPI>);
  const dim3 blocks(static_cast<unsigned int>(columns * ((d + zc - 1) / zc)));
  if constexpr (!kAlways)
    hipLaunchKernelGGL((k_conv_fwd_march<TM, CIN, SRC, EPI>), blocks, dim3(256), 0, stream, xb, x2b, wb, E, n, d, h,
                       cout, zc);
  return launch_status();
}

template <int SRC, int EPI>
int conv_fwd(const __bf16* xb, const __bf16* x2b, const __bf16* wb, const Epilogue& E, int n, int d, int h, int w,
             int cin, int cout, hipStream_t stream) {
  if (w == 64 && h % 4 == 0 && (cin == 16 || cin == 32) && (cout == 16 || (cout == 32 && cin == 16))) {
    // Full-resolution layers.
    if (cin == 16 && cout == 32) return launch_march<2, 16, SRC, EPI>(xb, x2b, wb, E, n, d, h, cout, stream);
    if (cin == 16) return launch_march<1, 16, SRC, EPI>(xb, x2b, wb, E, n, d, h, cout, stream);
    return launch_march<1, 32, SRC, EPI>(xb, x2b, wb, E, n, d, h, cout, stream);
  }
  if (w == 32 && h % 8 == 0 && (cin == 16 || cin == 32 || cin == 64) && cout == 32) {
    // Half-resolution layers: the same staging, 8 rows of 32 per workgroup.
    const dim3 tiles(static_cast<unsigned int>(static_cast<long long>(n) * d * (h / 8)));
    if (cin == 16)
      hipLaunchKernelGGL((k_conv_fwd_tile<2, 16, SRC, EPI, 32>), tiles, dim3(256), 0, stream, xb, x2b, wb, E, n, d, h, cout);
    else if (cin == 32)
      hipLaunchKernelGGL((k_conv_fwd_tile<2, 32, SRC, EPI, 32>), tiles, dim3(256), 0, stream, xb, x2b, wb, E, n, d, h, cout);
    else
      hipLaunchKernelGGL((k_conv_fwd_tile<2, 64, SRC, EPI, 32>), tiles, dim3(256), 0, stream, xb, x2b, wb, E, n, d, h, cout);
    return launch_status();
  }
  const long long P = static_cast<long long>(n) * d * h * w;
  const int tm = cout % 64 == 0 ? 4 : (cout % 32 == 0 ? 2 : 1);
  const long long waves = P / 64 * (cout / (16 * tm));
  const long long most = std::numeric_limits<int>::max() / cin;
  if (waves < kFillWaves && P <= most && 27LL * cout <= most) {
    const int m = waves >= kPairWaves && cout % 32 == 0 ? 2 : 1;
    const dim3 deep(static_cast<unsigned int>((P / 16 / m + 3) / 4), static_cast<unsigned int>(cout / 16 / m));
    auto* kernel = &k_conv_fwd_deep<1, false, SRC>;
    if (SRC != kSrcLow8 && cin % 32 == 0)
      kernel = m == 2 ? &k_conv_fwd_deep<2, true, SRC> : &k_conv_fwd_deep<1, true, SRC>;
    else if (m == 2)
      kernel = &k_conv_fwd_deep<2, false, SRC>;
    hipLaunchKernelGGL(kernel, deep, dim3(256), 0, stream, xb, x2b, wb, E, n, d, h, w, cin, cout);
    return launch_status();
  }
  const dim3 grid(static_cast<unsigned int>((P + 255) / 256), static_cast<unsigned int>(cout / (16 * tm)));
  if (tm == 4)
    hipLaunchKernelGGL((k_conv_fwd<4, SRC, EPI>), grid, dim3(256), 0, stream, xb, x2b, wb, E, n, d, h, w, cin, cout);
  else if (tm == 2)
    hipLaunchKernelGGL((k_conv_fwd<2, SRC, EPI>), grid, dim3(256), 0, stream, xb, x2b, wb, E, n, d, h, w, cin, cout);
  else
    hipLaunchKernelGGL((k_conv_fwd<1, SRC, EPI>), grid, dim3(256), 0, stream, xb, x2b, wb, E, n, d, h, w, cin, cout);
  return launch_status();
}

// Weight-gradient partials of hdn_conv3d_wgrad_noalloc live here: a library-owned array
// each GPU holds from the code object's load until the process ends. In host code the
// name stands for a host-side shadow, not a device address: kernels get the address
// hipGetSymbolAddress returns for the current device.
__device__ __align__(256) float scratch[HDN_SCRATCH_FLOATS];

// Validates a weight-gradient call and returns the positions each split owns.
int wgrad_split(const void* x_cm, const void* dz_cm, int splits, int n, int d, int h, int w, int cin,
                int cout, long long* per_split_out) {
  if (!x_cm || !dz_cm || splits < 1 || !shape_ok(n, d, h, w)) return HDN_EINVAL;
  const long long P = static_cast<long long>(n) * d * h * w;
  if (w % 8 != 0 || P % 32 != 0 || cin % 16 != 0 || cout % 16 != 0 || cin < 16 || cout < 16)
    return HDN_EINVAL;
  long long per_split = (P + splits - 1) / splits;
  per_split = (per_split + 31) / 32 * 32;
  if (per_split * (splits - 1) >= P) return HDN_EINVAL;  // every split must own positions
  *per_split_out = per_split;
  return HDN_OK;
}

void launch_wgrad(const void* x_cm, const void* dz_cm, float* part, int splits, int n, int d, int h,
                  int w, int cin, int cout, long long per_split, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned int>(cin / 16), static_cast<unsigned int>(cout / 16),
                  static_cast<unsigned int>(splits));
  const __bf16* xb = static_cast<const __bf16*>(x_cm);
  const __bf16* db = static_cast<const __bf16*>(dz_cm);
  if (w == 64 && h % 4 == 0)
    hipLaunchKernelGGL(k_conv_wgrad_tile<64>, grid, dim3(256), 0, stream, xb, db, part, n, d, h, cin, cout, splits);
  else if (w == 32 && h % 8 == 0)
    hipLaunchKernelGGL(k_conv_wgrad_tile<32>, grid, dim3(256), 0, stream, xb, db, part, n, d, h, cin, cout, splits);
  else if (w == 16 && h % 16 == 0)
    hipLaunchKernelGGL(k_conv_wgrad_tile<16>, grid, dim3(256), 0, stream, xb, db, part, n, d, h, cin, cout, splits);
  else
    hipLaunchKernelGGL(k_conv_wgrad, grid, dim3(256), 0, stream, xb, db, part, n, d, h, w, cin, cout, per_split);
}

void launch_reduce(const float* part, float* out, long long len, int splits, hipStream_t stream) {
  const unsigned int blocks = static_cast<unsigned int>(std::min<long long>(blocks_for(len, 64), 65535));
  // Sixteen waves to 64 outputs where there are many splits to walk or too few outputs to fill
  // the CUs; else one, where sixteen would mostly wait for each other. us with 16 waves and
  // with one: 13 824 outputs of 768 splits 7.9 and 34.9, 55 296 of 256 9.8 and 14.1; 110 592 of
  // 96 11.7 and 8.0, 442 368 of 4 11.2 and 7.2, of 48 24.4 and 14.1.
  if (splits >= 256 || len < 16384)
    hipLaunchKernelGGL(k_reduce_splits<16>, dim3(blocks), dim3(64 * 16), 0, stream, part, out, len, splits);
  else
    hipLaunchKernelGGL(k_reduce_splits<1>, dim3(blocks), dim3(64), 0, stream, part, out, len, splits);
}

// Device address of `scratch` on each GPU, looked up once per device with that device
// current (each GPU holds its own copy of the array at its own address).
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
float* g_scratch_address[kMaxDevices] = {};

int scratch_for_current_device(void* stream, float** out) {
  int device = -1;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return HDN_EHIP;
  if (stream) {
    // The kernels run on the stream's device: it must be the current one, whose copy of
    // the array is the one looked up.
    int stream_device = -1;
    if (hipStreamGetDevice(as_stream(stream), &stream_device) != hipSuccess) return HDN_EHIP;
    if (stream_device != device) return HDN_EINVAL;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_address[device]) {
    void* address = nullptr;
    if (hipGetSymbolAddress(&address, HIP_SYMBOL(scratch)) != hipSuccess || !address) return HDN_EHIP;
    g_scratch_address[device] = static_cast<float*>(address);
  }
  *out = g_scratch_address[device];
  return HDN_OK;
}

}  // namespace

extern "C" {

int hdn_conv3d_fwd_fused(const void* x, const void* x2, int src, const void* wt, const float* bias, const void* skip,
                         const void* inp, int c_in, float* pred, void* y_nd, void* y_cm, int n, int d, int h, int w,
                         int cin, int cout, float slope, void* stream) {
  if (!x || !wt || !shape_ok(n, d, h, w)) return HDN_EINVAL;
  if (pred ? (!inp || c_in < 1 || skip || src != kSrcPlain) : !y_nd) return HDN_EINVAL;
  if (skip && src != kSrcPlain && src != kSrcUp) return HDN_EINVAL;
  const long long P = static_cast<long long>(n) * d * h * w;
  if (P % 64 != 0 || cin % 16 != 0 || cin < 16 || cout % 16 != 0 || cout < 16) return HDN_EINVAL;
  if (src == kSrcUp && (d % 2 || h % 2 || w % 2)) return HDN_EINVAL;
  if (src == kSrcAdd && !x2) return HDN_EINVAL;
  if (src != kSrcPlain && src != kSrcUp && src != kSrcAdd && src != kSrcLow8) return HDN_EINVAL;
  const __bf16* xb = static_cast<const __bf16*>(x);
  const __bf16* x2b = static_cast<const __bf16*>(x2);
  const __bf16* wb = static_cast<const __bf16*>(wt);
  const Epilogue E{bias,
                   slope,
                   static_cast<const __bf16*>(skip),
                   static_cast<__bf16*>(y_nd),
                   static_cast<__bf16*>(y_cm),
                   pred,
                   static_cast<const __bf16*>(inp),
                   c_in};
  const hipStream_t s = as_stream(stream);
  if (pred) return conv_fwd<kSrcPlain, kEpiPred>(xb, nullptr, wb, E, n, d, h, w, cin, cout, s);
  if (skip && src == kSrcUp) return conv_fwd<kSrcUp, kEpiSkip>(xb, nullptr, wb, E, n, d, h, w, cin, cout, s);
  if (skip) return conv_fwd<kSrcPlain, kEpiSkip>(xb, nullptr, wb, E, n, d, h, w, cin, cout, s);
  if (src == kSrcUp) return conv_fwd<kSrcUp, kEpiPlain>(xb, nullptr, wb, E, n, d, h, w, cin, cout, s);
  if (src == kSrcAdd) return conv_fwd<kSrcAdd, kEpiPlain>(xb, x2b, wb, E, n, d, h, w, cin, cout, s);
  if (src == kSrcLow8) return conv_fwd<kSrcLow8, kEpiPlain>(xb, nullptr, wb, E, n, d, h, w, cin, cout, s);
  return conv_fwd<kSrcPlain, kEpiPlain>(xb, nullptr, wb, E, n, d, h, w, cin, cout, s);
}

int hdn_conv3d_fwd_src(const void* x, const void* x2, int src, const void* wt, const float* bias, void* y_nd,
                       void* y_cm, int n, int d, int h, int w, int cin, int cout, float slope, void* stream) {
  return hdn_conv3d_fwd_fused(x, x2, src, wt, bias, nullptr, nullptr, 0, nullptr, y_nd, y_cm, n, d, h, w, cin, cout,
                              slope, stream);
}

int hdn_conv3d_fwd(const void* x, const void* wt, const float* bias, void* y_nd, void* y_cm, int n,
                   int d, int h, int w, int cin, int cout, float slope, void* stream) {
  return hdn_conv3d_fwd_src(x, nullptr, kSrcPlain, wt, bias, y_nd, y_cm, n, d, h, w, cin, cout, slope, stream);
}

int hdn_conv3d_wgrad(const void* x_cm, const void* dz_cm, float* part, int splits, int n, int d,
                     int h, int w, int cin, int cout, void* stream) {
  long long per_split = 0;
  const int rc = wgrad_split(x_cm, dz_cm, splits, n, d, h, w, cin, cout, &per_split);
  if (rc != HDN_OK || !part) return rc != HDN_OK ? rc : HDN_EINVAL;
  launch_wgrad(x_cm, dz_cm, part, splits, n, d, h, w, cin, cout, per_split, as_stream(stream));
  return launch_status();
}

int hdn_reduce_splits(const float* part, float* out, long long len, int splits, void* stream) {
  if (!part || !out || len < 1 || splits < 1) return HDN_EINVAL;
  launch_reduce(part, out, len, splits, as_stream(stream));
  return launch_status();
}

int hdn_conv3d_wgrad_noalloc(const void* x_cm, const void* dz_cm, float* grad, int splits, int n,
                             int d, int h, int w, int cin, int cout, void* stream) {
  long long per_split = 0;
  const int rc = wgrad_split(x_cm, dz_cm, splits, n, d, h, w, cin, cout, &per_split);
  if (rc != HDN_OK || !grad) return rc != HDN_OK ? rc : HDN_EINVAL;
  const long long len = 27LL * cout * cin;
  if (static_cast<long long>(splits) * len > HDN_SCRATCH_FLOATS) return HDN_ESIZE;
  float* part = nullptr;
  const int srv = scratch_for_current_device(stream, &part);
  if (srv != HDN_OK) return srv;
  // Every partial is written before it is read, so the array needs no clearing.
  const hipStream_t s = as_stream(stream);
  launch_wgrad(x_cm, dz_cm, part, splits, n, d, h, w, cin, cout, per_split, s);
  launch_reduce(part, grad, len, splits, s);
  return launch_status();
}

int hdn_channel_sum(const void* cm, float* part, long long P, int C, int splits, void* stream) {
  if (!cm || !part || P < 1 || C < 1 || splits < 1) return HDN_EINVAL;
  const long long per_split = (P + splits - 1) / splits;
  hipLaunchKernelGGL(k_channel_sum, dim3(static_cast<unsigned int>(C), static_cast<unsigned int>(splits)),
                     dim3(256), 0, as_stream(stream), static_cast<const __bf16*>(cm), part, P,
                     per_split);
  return launch_status();
}

int hdn_act_bwd(const void* y, const void* dy, void* dz_nd, void* dz_cm, long long P, int C,
                float slope, void* stream) {
  if (!y || !dy || !dz_nd || P < 1 || C % 8 != 0) return HDN_EINVAL;
  hipLaunchKernelGGL(k_act_bwd, dim3(place_blocks(P, C)), dim3(256), 0, as_stream(stream),
                     static_cast<const __bf16*>(y), static_cast<const __bf16*>(dy),
                     static_cast<__bf16*>(dz_nd), static_cast<__bf16*>(dz_cm), P, C, slope);
  return launch_status();
}

int hdn_add(const void* a, const void* b, void* y_nd, void* y_cm, long long P, int C, void* stream) {
  if (!a || !b || !y_nd || P < 1 || C % 8 != 0) return HDN_EINVAL;
  hipLaunchKernelGGL(k_add, dim3(place_blocks(P, C)), dim3(256), 0, as_stream(stream),
                     static_cast<const __bf16*>(a), static_cast<const __bf16*>(b),
                     static_cast<__bf16*>(y_nd), static_cast<__bf16*>(y_cm), P, C);
  return launch_status();
}

int hdn_pool_fwd(const void* x, void* y_nd, void* y_cm, int n, int d, int h, int w, int C,
                 void* stream) {
  if (!x || !y_nd || !shape_ok(n, d, h, w) || C % 8 != 0) return HDN_EINVAL;
  const long long P = static_cast<long long>(n) * d * h * w;
  hipLaunchKernelGGL(k_pool_fwd, dim3(place_blocks(P, C)), dim3(256), 0, as_stream(stream),
                     static_cast<const __bf16*>(x), static_cast<__bf16*>(y_nd),
                     static_cast<__bf16*>(y_cm), n, d, h, w, C);
  return launch_status();
}

int hdn_pool_bwd(const void* dy, void* dx, int n, int d2, int h2, int w2, int C, void* stream) {
  if (!dy || !dx || !shape_ok(n, d2, h2, w2) || C % 8 != 0 || d2 % 2 || h2 % 2 || w2 % 2)
    return HDN_EINVAL;
  const long long P = static_cast<long long>(n) * d2 * h2 * w2;
  hipLaunchKernelGGL(k_pool_bwd, dim3(place_blocks(P, C)), dim3(256), 0, as_stream(stream),
                     static_cast<const __bf16*>(dy), static_cast<__bf16*>(dx), n, d2, h2, w2, C);
  return launch_status();
}

int hdn_up_fwd(const void* x, void* y_nd, void* y_cm, int n, int d2, int h2, int w2, int C,
               void* stream) {
  if (!x || !y_nd || !shape_ok(n, d2, h2, w2) || C % 8 != 0 || d2 % 2 || h2 % 2 || w2 % 2)
    return HDN_EINVAL;
  const long long P = static_cast<long long>(n) * d2 * h2 * w2;
  hipLaunchKernelGGL(k_up_fwd, dim3(place_blocks(P, C)), dim3(256), 0, as_stream(stream),
                     static_cast<const __bf16*>(x), static_cast<__bf16*>(y_nd),
                     static_cast<__bf16*>(y_cm), n, d2, h2, w2, C);
  return launch_status();
}

int hdn_up_bwd(const void* dy, void* dx, int n, int d, int h, int w, int C, void* stream) {
  if (!dy || !dx || !shape_ok(n, d, h, w) || C % 8 != 0) return HDN_EINVAL;
  const long long P = static_cast<long long>(n) * d * h * w;
  hipLaunchKernelGGL(k_up_bwd, dim3(place_blocks(P, C)), dim3(256), 0, as_stream(stream),
                     static_cast<const __bf16*>(dy), static_cast<__bf16*>(dx), n, d, h, w, C);
  return launch_status();
}

int hdn_loss(const void* out, const void* inp, int c_out, int c_in, const float* target,
             const float* weight, void* dout_nd, void* dout_cm, float* pred, float* partial,
             long long P, float grad_scale, void* stream) {
  if (!out || !inp || P < 1 || c_out < 1 || c_in < 1) return HDN_EINVAL;
  if ((dout_nd || partial) && !target) return HDN_EINVAL;
  hipLaunchKernelGGL(k_loss, dim3(blocks_for(P, 256)), dim3(256), 0, as_stream(stream),
                     static_cast<const __bf16*>(out), static_cast<const __bf16*>(inp), c_out, c_in,
                     target, weight, static_cast<__bf16*>(dout_nd), static_cast<__bf16*>(dout_cm),
                     pred, partial, P, grad_scale);
  return launch_status();
}

int hdn_prepare_weights(const float* master, void* wf, void* wd, int cin, int cout, void* stream) {
  if (!master || !wf || !wd || cin < 1 || cout < 1) return HDN_EINVAL;
  hipLaunchKernelGGL(k_prepare_weights, dim3(blocks_for(27LL * cin * cout, 256)), dim3(256), 0,
                     as_stream(stream), master, static_cast<__bf16*>(wf), static_cast<__bf16*>(wd),
                     cin, cout);
  return launch_status();
}

int hdn_adam(float* param, const float* grad, float* m, float* v, long long len, float lr,
             float beta1, float beta2, float eps, int step, float weight_decay, void* stream) {
  if (!param || !grad || !m || !v || len < 1 || step < 1) return HDN_EINVAL;
  const float corr1 = 1.0f - std::pow(beta1, static_cast<float>(step));
  const float corr2 = 1.0f - std::pow(beta2, static_cast<float>(step));
  hipLaunchKernelGGL(k_adam, dim3(blocks_for(len, 256)), dim3(256), 0, as_stream(stream), param, grad,
                     m, v, len, lr, beta1, beta2, eps, corr1, corr2, weight_decay);
  return launch_status();
}

}  // extern "C"
