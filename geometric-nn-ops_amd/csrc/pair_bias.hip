// Pair-bias projection of attention with pair bias, for gfx950.
//
//   bias[b, h, u, v] = round( sum_c round(LN(z[b, u, v, :]))[c] * W[h, c] )
//   LN(x)[c] = (x[c] - mean) / sqrt(var + eps) * gamma[c]      (biased variance, no beta)
//
// which is _project_pair_bias of the reference (geometric_nn_ops_torch/triangle/_reference/
// attention_pair_bias.py:17-22: F.layer_norm without bias, rounded to z's dtype as
// F.layer_norm returns it, then F.linear with fp32 accumulation and the permute to
// [B, H, U, V]). One pass over the pair tensor z replaces the reference's LayerNorm
// output, linear output and permuted copy.
//
// Layout: a wave takes 32 consecutive pixels of the flattened [B, U, V] grid. Their rows are
// one contiguous range of z, read in memory order (whole lines per instruction; reading the
// fragments straight from memory takes 32 bytes of each of 32 lines per instruction, and the
// lines fall out of L1 before their other parts are used) and passed through a wave-private LDS
// tile into the MFMA's B fragment: two lanes per pixel, lane half g holding the 8-channel chunks
// 16 kk + 8 g (k = channel, column = pixel). Mean and variance are one exchange between the two
// lanes, and the projection is [32 heads][Zc] x [Zc][32 pixels] with the weights as A fragments
// (heads past H repeat the last one and are not stored; chunks past Zc are zero on both sides).
// The result has a pixel per lane, so each head's 32 values leave as one run. Bound by HBM
// (Zc * e bytes read per pixel against H * e written). Against eight-lane dot products on the
// vector ALU (H * Zc / 8 FMAs with an LDS read each and three shuffles per head and lane), which
// few heads still take (pair_bias_dot): 54 -> 18.4 us at 384 x 384 pixels, Zc = 128, H = 16, bf16.
//
// Also here: the gate and output projection of attention with pair bias (apb_gate_out_kernel,
// below), the part of the op after the attention itself.
#include <type_traits>

#include "gnn_common.hpp"
#include "gnn_internal.hpp"

namespace gnn {

namespace {

constexpr int PB_MAX_ZC = 256;
constexpr int PB_MAX_W = 8192;               // H * Zc <= 8192

// 8 consecutive elements: one vector load where the array is 16-byte aligned, else scalar loads
template <typename T>
__device__ __forceinline__ typename TypeOps<T>::V8 load8_any(const T* p, bool aligned) {
  if (aligned) return load8(p);
  typename TypeOps<T>::V8 v;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = p[e];
  return v;
}

// KS k-steps of 16 channels (Zc <= 16 * KS); waves per workgroup such that the LDS tiles of
// 32 padded rows each take at most 36 KB
template <typename T, int KS>
struct PairBiasCfg {
  static constexpr int PITCH = 16 * KS * (int)sizeof(T) + 16;  // bytes
  static constexpr int NW = PITCH * 32 <= 9 * 1024 ? 4 : PITCH * 32 <= 18 * 1024 ? 2 : 1;
  static constexpr int CHUNKS = KS * (int)sizeof(T) / 2;       // 16-byte chunks per lane
};

// fp32 products of channel pairs C0 .. C0 + N - 1, leaves of 4 or 8 pairs added as a binary tree (in order, so
// that few of its sums are live at a time)
template <int KS, int C0, int N>
__device__ __forceinline__ f32x16 pair_bias_sum(const f32x8 (&w)[KS], const f32x8 (&x)[KS]) {
  if constexpr (N > (KS > 4 ? 8 : 4)) {
    f32x16 s = pair_bias_sum<KS, C0, N / 2>(w, x);
    s += pair_bias_sum<KS, C0 + N / 2, N / 2>(w, x);
    return s;
  } else {
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
    for (int c = C0; c < C0 + N; ++c)
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(w[c / 8][c % 8], x[c / 8][c % 8], s, 0, 0, 0);
    return s;
  }
}

template <typename T, int KS>
__global__ __launch_bounds__((64 * PairBiasCfg<T, KS>::NW), (KS <= (sizeof(T) == 2 ? 8 : 4) ? 4 : 1)) void pair_bias_proj_kernel(const gnn_pair_bias_args a) {
  typedef typename TypeOps<T>::V8 V8;
  typedef PairBiasCfg<T, KS> Cfg;
  typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
  constexpr int PREC = sizeof(T) == 4 ? PREC_IEEE : PREC_NATIVE;
  __shared__ __align__(16) unsigned char tiles[Cfg::NW * 32 * Cfg::PITCH];
  const int Zc = (int)a.Zc, H = (int)a.H;
  const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5, wave = threadIdx.x >> 6;
  unsigned char* tile = tiles + wave * 32 * Cfg::PITCH;
  const int64_t npix = a.B * a.U * a.V;
  const int64_t p0 = ((int64_t)blockIdx.x * Cfg::NW + wave) * 32, p = p0 + l32;
  const bool ok = p < npix;

  // the 32 rows in memory order; rows past the last pixel repeat the last chunk
  const int cpr = Zc * (int)sizeof(T) / 16;  // 16-byte chunks per row
  const int64_t left = (npix - (p0 < npix ? p0 : npix - 1)) * cpr - 1;
  const u32x4_t* src = (const u32x4_t*)a.z + (p0 < npix ? p0 : npix - 1) * cpr;
  u32x4_t raw[Cfg::CHUNKS];
#pragma unroll
  for (int i = 0; i < Cfg::CHUNKS; ++i) {
    const int c = 64 * i + lane;
    raw[i] = src[c < left ? c : left];
  }
  // the first 32 heads' weights, requested before the rows are waited for
  const bool wal = ((uintptr_t)a.proj_w & 15) == 0;
  V8 w[KS];
  auto weights = [&](int h0) {
    const T* wrow = (const T*)a.proj_w + (int64_t)(h0 + l32 < H ? h0 + l32 : H - 1) * Zc + 8 * g;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) w[kk] = 16 * kk + 8 * g < Zc ? load8_any(wrow + 16 * kk, wal) : zero8<T>();
  };
  weights(0);
#pragma unroll
  for (int i = 0; i < Cfg::CHUNKS; ++i) {
    const int c = 64 * i + lane;
    const int r = Zc == 16 * KS ? c / (KS * (int)sizeof(T)) : c / cpr;
    if (r < 32) *reinterpret_cast<u32x4_t*>(tile + r * Cfg::PITCH + (c - r * cpr) * 16) = raw[i];
  }
  // Each pass over the row reads it from LDS again (the compiler would otherwise keep the
  // fp32 copies of all channels live and spill)
  auto chunk = [&](int kk) {
    return 16 * kk + 8 * g < Zc ? load8((const T*)(tile + l32 * Cfg::PITCH) + 16 * kk + 8 * g) : zero8<T>();
  };
  auto next_pass = [] {
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
  };
  next_pass();
  const float inv_zc = 1.0f / (float)Zc;
  float s = 0.f;
#pragma unroll
  for (int kk = 0; kk < KS; ++kk) {
    const f32x8 v = TypeOps<T>::to_f32(chunk(kk));
#pragma unroll
    for (int e = 0; e < 8; ++e) s += v[e];
  }
  const float mean = pair_sum(s) * inv_zc;
  next_pass();
  float q = 0.f;
#pragma unroll
  for (int kk = 0; kk < KS; ++kk) {
    const f32x8 v = TypeOps<T>::to_f32(chunk(kk));
    float t = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) t += (v[e] - mean) * (v[e] - mean);
    q += 16 * kk + 8 * g < Zc ? t : 0.f;
  }
  const float rstd = 1.0f / sqrtf(pair_sum(q) * inv_zc + a.eps);
  next_pass();
  // normalised, gamma-scaled and rounded to the input dtype (F.layer_norm's output)
  const T* gam = (const T*)a.ln_w;
  const bool gal = ((uintptr_t)gam & 15) == 0;
  V8 x[KS];
#pragma unroll
  for (int kk = 0; kk < KS; ++kk) {
    const int ch = 16 * kk + 8 * g;
    x[kk] = zero8<T>();
    if (ch < Zc) {
      f32x8 v = TypeOps<T>::to_f32(chunk(kk));
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (v[e] - mean) * rstd;
      if (gam) v *= TypeOps<T>::to_f32(load8_any(gam + ch, gal));
      x[kk] = TypeOps<T>::from_f32(v);
    }
  }

  const uint32_t V = (uint32_t)a.V, U = (uint32_t)a.U;
  const uint64_t r = (uint64_t)(ok ? p : 0) / V;
  const uint32_t v0 = (uint32_t)((uint64_t)(ok ? p : 0) - r * V);
  T* orow = (T*)a.out + (int64_t)(r / U) * a.out_stride[0] + (int64_t)(r % U) * a.out_stride[2] + v0;
  for (int h0 = 0; h0 < H; h0 += 32) {
    if (h0 > 0) weights(h0);
    f32x16 acc;
    if constexpr (sizeof(T) == 2) {
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) Mma<T, PREC>::step(acc, w[kk], x[kk]);
    } else {
      // sums over 8 channels (16 past 64), added as a tree: one sum over all 128 is 2.1e-7 off, the eight-lane
      // dot products were 1.1e-7 (Zc = 64: 1.5e-7 and 0.95e-7)
      acc = pair_bias_sum<KS, 0, 8 * KS>(w, x);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int h = h0 + 8 * (i / 4) + 4 * g + i % 4;
      if (ok && h < H) orow[h * a.out_stride[1]] = TypeOps<T>::from_f32(acc[i]);
    }
  }
}

// The same with dot products on the vector ALU, where heads are few: eight lanes per pixel (a wave
// holds 8 consecutive pixels), lane j loading the 8-channel chunks j, j + 8, ... of its row; LayerNorm
// sums over the 8 lanes with xor shuffles; the weights as fp32 in LDS; a head's 8 partial products meet
// through three shuffles and lane h % 8 stores it. Time grows with H, where the matrix unit forms 32
// heads whatever their number (in fp32 at 64 cycles per channel pair).
constexpr int PB_THREADS = 256;          // 4 waves
constexpr int PB_PIX = PB_THREADS / 8;   // pixels per workgroup and step
constexpr int PB_MAX_CHUNKS = PB_MAX_ZC / 64;

template <typename T>
__global__ __launch_bounds__(PB_THREADS) void pair_bias_dot_kernel(const gnn_pair_bias_args a) {
  __shared__ float ws[PB_MAX_W];
  __shared__ float gs[PB_MAX_CHUNKS * 64];
  const int Zc = (int)a.Zc, H = (int)a.H, V = (int)a.V, U = (int)a.U;
  const int tid = threadIdx.x;
  for (int i = tid; i < H * Zc; i += PB_THREADS) ws[i] = TypeOps<T>::to_f32(((const T*)a.proj_w)[i]);
  for (int i = tid; i < Zc; i += PB_THREADS)
    gs[i] = a.ln_w ? TypeOps<T>::to_f32(((const T*)a.ln_w)[i]) : 1.0f;
  __syncthreads();

  const int j = tid & 7;
  const int nch = Zc / 8;
  const int64_t npix = a.B * (int64_t)U * V;
  const float inv_zc = 1.0f / (float)Zc;
  for (int64_t p0 = (int64_t)blockIdx.x * PB_PIX; p0 < npix; p0 += (int64_t)gridDim.x * PB_PIX) {
    const int64_t p = p0 + (tid >> 3);
    const bool ok = p < npix;
    const T* row = (const T*)a.z + (ok ? p : 0) * Zc;
    f32x8 x[PB_MAX_CHUNKS];
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < PB_MAX_CHUNKS; ++c) {
      const int ch = j + 8 * c;
      if (ch < nch) {
        x[c] = TypeOps<T>::to_f32(load8(row + 8 * ch));
#pragma unroll
        for (int e = 0; e < 8; ++e) s += x[c][e];
      }
    }
    s += __shfl_xor(s, 1);
    s += __shfl_xor(s, 2);
    s += __shfl_xor(s, 4);
    const float mean = s * inv_zc;
    float q = 0.f;
#pragma unroll
    for (int c = 0; c < PB_MAX_CHUNKS; ++c) {
      if (j + 8 * c < nch) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float d = x[c][e] - mean;
          q += d * d;
        }
      }
    }
    q += __shfl_xor(q, 1);
    q += __shfl_xor(q, 2);
    q += __shfl_xor(q, 4);
    const float rstd = 1.0f / sqrtf(q * inv_zc + a.eps);
    // normalised, gamma-scaled and rounded to the input dtype (F.layer_norm's output)
#pragma unroll
    for (int c = 0; c < PB_MAX_CHUNKS; ++c) {
      const int ch = j + 8 * c;
      if (ch < nch) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          x[c][e] = TypeOps<T>::to_f32(TypeOps<T>::from_f32((x[c][e] - mean) * rstd * gs[8 * ch + e]));
      }
    }
    int64_t b = 0, u = 0, v = 0;
    if (ok) {
      v = p % V;
      const int64_t r = p / V;
      u = r % U;
      b = r / U;
    }
    T* orow = (T*)a.out + b * a.out_stride[0] + u * a.out_stride[2] + v;
    for (int h = 0; h < H; ++h) {
      const float* wh = ws + h * Zc;
      float acc = 0.f;
#pragma unroll
      for (int c = 0; c < PB_MAX_CHUNKS; ++c) {
        const int ch = j + 8 * c;
        if (ch < nch) {
#pragma unroll
          for (int e = 0; e < 8; ++e) acc = __builtin_fmaf(x[c][e], wh[8 * ch + e], acc);
        }
      }
      acc += __shfl_xor(acc, 1);
      acc += __shfl_xor(acc, 2);
      acc += __shfl_xor(acc, 4);
      if (ok && (h & 7) == j) orow[h * a.out_stride[1]] = TypeOps<T>::from_f32(acc);
    }
  }
}

template <typename T>
int launch_pb_dot(const gnn_pair_bias_args& a, hipStream_t stream) {
  const int64_t want = (a.B * a.U * a.V + PB_PIX - 1) / PB_PIX;
  const int64_t grid =
      std::min<int64_t>(want, 4 * (int64_t)persistent_grid((const void*)pair_bias_dot_kernel<T>, PB_THREADS, 0));
  hipLaunchKernelGGL(pair_bias_dot_kernel<T>, dim3((uint32_t)grid), dim3(PB_THREADS), 0, stream, a);
  return (int)hipGetLastError();
}

#ifndef GNN_PB_DOT  // 0 / 1: never / always the dot products
#define GNN_PB_DOT -1
#endif
// Whether heads are so few that the dot products are faster: their time grows with the heads, that of the
// matrix unit with the channels, and up to 16384 pixels (a wave of the matrix kernel for each half
// SIMD or less) the latter is its chain of loads, LDS passes and products. us, matrix unit / dot products:
//   pixels  Zc    fp32: H = 4      8          12         16      | bf16: H = 2      6          10
//   128^2   64    6.0 / 4.4   6.1 / 5.5   6.3 / 6.6               | 5.2 / 4.0   5.3 / 5.1   5.2 / 6.2
//           128   9.1 / 5.0   9.1 / 6.5   9.3 / 8.0   9.2 / 9.4   | 7.6 / 4.5   7.7 / 6.1   7.7 / 7.6
//           256   15.6 / 6.2  15.7 / 8.7  15.6 / 11.1 15.7 / 13.7 | 11.4 / 5.4  11.5 / 8.2  11.5 / 10.7
//   160^2   64    6.2 / 4.9   6.3 / 6.5                           | 5.2 / 4.4   5.3 / 6.0
//           128   11.6 / 6.1  11.6 / 8.7  11.8 / 11.2 11.8 / 13.7 | 7.7 / 5.1   7.7 / 7.5   7.7 / 10.0
//           256   16.2 / 8.7  16.2 / 13.2 16.5 / 17.8             | 11.8 / 6.6  11.9 / 11.0 11.9 / 15.6
//   256^2   64    7.9 / 8.4   8.0 / 11.3                          | 5.4 / 7.2
//           128   13.2 / 11.5 13.8 / 16.9                         | 7.9 / 8.6
//           256   38 / 21     39 / 28     40 / 36     40 / 44     | 13.1 / 12.3 13.5 / 20.4
//   384^2   64    17.8 / 16.9 18.3 / 22.9                         | 8.1 / 13.2
//           128   35 / 22     36 / 32     36 / 41     37 / 50     | 16.8 / 18.0
//           256   87 / 35     88 / 48     89 / 65     90 / 82     | 37 / 26     37 / 39
template <typename T, int KS>
bool pair_bias_dot(const gnn_pair_bias_args& a) {
  if (GNN_PB_DOT >= 0) return GNN_PB_DOT;
  const int64_t px = a.B * a.U * a.V;
  if (sizeof(T) == 4)
    return a.H <= (px <= 16384 ? std::min(2 * KS, 16) : px <= 32768 ? std::min(3 * KS / 2, 10) : 3 * KS / 4);
  return a.H <= (px <= 16384 ? std::min(3 * KS / 2, 10) : px <= 32768 ? std::min(KS / 2, 6) : KS > 8 ? 3 : 0);
}

template <typename T, int KS>
int launch_pb(const gnn_pair_bias_args& a, hipStream_t stream) {
  if (pair_bias_dot<T, KS>(a)) return launch_pb_dot<T>(a, stream);
  constexpr int pix = 32 * PairBiasCfg<T, KS>::NW;
  const int64_t grid = (a.B * a.U * a.V + pix - 1) / pix;
  if (grid >= ((int64_t)1 << 31)) return set_error(GNN_ERR_UNSUPPORTED, "pair_bias_proj: too many pixels");
  hipLaunchKernelGGL((pair_bias_proj_kernel<T, KS>), dim3((uint32_t)grid), dim3(2 * pix), 0, stream, a);
  return (int)hipGetLastError();
}
// the channel loops unroll over 64, 128 or 256 channels
template <typename T>
int launch_pb(const gnn_pair_bias_args& a, hipStream_t stream) {
  if (a.Zc <= 64) return launch_pb<T, 4>(a, stream);
  if (a.Zc <= 128) return launch_pb<T, 8>(a, stream);
  return launch_pb<T, 16>(a, stream);
}

// ---- gate and output projection ------------------------------------------------------
//   out = ( T(o) * T(sigmoid(T(s Wg^T + bg))) ) Wo^T + bo,
// each product's result rounded to T as the reference's F.linear / torch.sigmoid / multiply
// return it (attention_pair_bias.py:86-89). One workgroup (NW waves) per GT = 32 tokens:
// the tile's s rows and its o rows (the attention output, heads merged) are staged in LDS;
// gate pre-activations run on MFMA in passes of 32 NW channels (wave w: channels 32 w ..,
// A = Wg rows from global memory, fetched a chunk of k-steps ahead, B = s fragments from
// LDS), and each lane writes o * g over
// the o values it read, so the gated tile never leaves LDS; the output product then reads it
// as its B operand and its results leave through an LDS staging tile as 16-byte rows. No
// intermediate (g, o * g) reaches memory.
constexpr int GT = 32;       // tokens per workgroup

struct GateOutLds {
  size_t s, og, y, bias;
};
// goc: output channels per pass, 32 per wave
template <typename T>
__host__ __device__ inline GateOutLds gate_out_lds(int64_t Cs, int64_t D, int goc) {
  constexpr int pad = 16 / (int)sizeof(T);
  GateOutLds L;
  L.s = 0;
  L.og = L.s + (size_t)GT * (Cs + pad) * sizeof(T);
  L.y = L.og + (size_t)GT * (D + pad) * sizeof(T);
  L.bias = L.y + (size_t)GT * (goc + pad) * sizeof(T);
  return L;
}
// the biases follow as fp32 [D] and [Co]
__host__ __device__ inline size_t gate_out_lds_total(const GateOutLds& L, int64_t D, int64_t Co) {
  return L.bias + (size_t)(D + Co) * sizeof(float);
}

// acc += W[rows wrow.., k] * tile[token l32][k] over nk k-steps of 16 (nk a multiple of GK):
// the weight fragments (global memory, L2-resident) in chunks of GK k-steps, the next chunk
// requested before the current one's MFMAs so that the loads stay ahead of the products.
// Branches only around whole chunks, so a chunk's LDS reads and counter waits are straight
// code the compiler can schedule.
template <typename T, int PREC, int GK>
__device__ __forceinline__ void gate_out_gemm(f32x16& acc, const T* __restrict__ wrow, int nk, const T* tile, int ld,
                                              int l32, int g) {
  typedef typename TypeOps<T>::V8 V8;
  V8 wa[GK], wb[GK];
  auto load = [&](V8 (&w)[GK], int k0) {
#pragma unroll
    for (int j = 0; j < GK; ++j) w[j] = load8(wrow + 16 * (k0 + j));
  };
  auto mma = [&](const V8 (&w)[GK], int k0) {
#pragma unroll
    for (int j = 0; j < GK; ++j) Mma<T, PREC>::step(acc, w[j], load8(&tile[l32 * ld + 16 * (k0 + j) + 8 * g]));
  };
  load(wa, 0);
  for (int k0 = 0; k0 < nk; k0 += 2 * GK) {
    const bool second = k0 + GK < nk;  // uniform
    if (second) load(wb, k0 + GK);
    mma(wa, k0);
    if (second) {
      if (k0 + 2 * GK < nk) load(wa, k0 + 2 * GK);
      mma(wb, k0 + GK);
    }
  }
}
template <typename T, int PREC>
__device__ __forceinline__ void gate_out_gemm(f32x16& acc, const T* __restrict__ wrow, int nk, const T* tile, int ld,
                                              int l32, int g) {
  if (nk % 8 == 0) gate_out_gemm<T, PREC, 8>(acc, wrow, nk, tile, ld, l32, g);
  else gate_out_gemm<T, PREC, 2>(acc, wrow, nk, tile, ld, l32, g);  // widths are multiples of 32: nk is even
}

template <typename T, int PREC, int NW>
__global__ __launch_bounds__(64 * NW) void apb_gate_out_kernel(const gnn_apb_gate_out_args a) {
  typedef typename TypeOps<T>::V8 V8;
  typedef typename TypeOps<T>::V4 V4;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  constexpr int pad = 16 / (int)sizeof(T);
  constexpr int EPC = 16 / (int)sizeof(T);  // elements per 16-byte chunk
  constexpr int GO_THREADS = 64 * NW, GOC = 32 * NW;
  const int Cs = (int)a.Cs, D = (int)a.D, Co = (int)a.Co;
  const int SR = Cs + pad, OR = D + pad, YR = GOC + pad;
  const GateOutLds L = gate_out_lds<T>(Cs, D, GOC);
  T* ss = reinterpret_cast<T*>(smem_raw + L.s);
  T* og = reinterpret_cast<T*>(smem_raw + L.og);
  T* ys = reinterpret_cast<T*>(smem_raw + L.y);
  float* gb_s = reinterpret_cast<float*>(smem_raw + L.bias);
  float* ob_s = gb_s + D;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, g = lane >> 5;
  const int64_t t0 = (int64_t)blockIdx.x * GT;
  const int ntok = a.M - t0 < GT ? (int)(a.M - t0) : GT;

  // stage s [GT][Cs] and o [GT][D] (16-byte chunks, zeros past the last token), SB chunks
  // per thread loaded before any is stored, so their latencies overlap
  constexpr int SB = NW == 4 ? 8 : 2;
  typedef typename std::conditional<sizeof(T) == 2, V8, V4>::type Vc;  // 16 bytes of T
  auto stage = [&](const T* src, int64_t ld, int C, T* dst, int R) {
    const int cpr = C / EPC, n = GT * cpr;
    for (int base = 0; base < n; base += SB * GO_THREADS) {
      Vc v[SB];
#pragma unroll
      for (int i = 0; i < SB; ++i) {
        const int c = base + i * GO_THREADS + tid, r = c / cpr, k = (c - r * cpr) * EPC;
        v[i] = Vc{};
        if (c < n && r < ntok) {
          if constexpr (sizeof(T) == 2) v[i] = load8(src + (t0 + r) * ld + k);
          else v[i] = load4(src + (t0 + r) * ld + k);
        }
      }
#pragma unroll
      for (int i = 0; i < SB; ++i) {
        const int c = base + i * GO_THREADS + tid, r = c / cpr, k = (c - r * cpr) * EPC;
        if (c < n) {
          if constexpr (sizeof(T) == 2) store8(&dst[r * R + k], v[i]);
          else store4(&dst[r * R + k], v[i]);
        }
      }
    }
  };
  stage((const T*)a.s, a.s_ld, Cs, ss, SR);
  stage((const T*)a.o, a.o_ld, D, og, OR);
  for (int c = tid; c < D; c += GO_THREADS) gb_s[c] = a.g_b ? TypeOps<T>::to_f32(((const T*)a.g_b)[c]) : 0.f;
  for (int c = tid; c < Co; c += GO_THREADS) ob_s[c] = a.o_b ? TypeOps<T>::to_f32(((const T*)a.o_b)[c]) : 0.f;
  __syncthreads();

  // ---- gate: acc = [channel][token], channel = c0 + 32 wave + 8(r/4) + 4g + r%4, token l32
  for (int c0 = 0; c0 < D; c0 += GOC) {
    const int cw = c0 + 32 * wave;
    if (cw < D) {
      f32x16 acc;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = 0.f;
      gate_out_gemm<T, PREC>(acc, (const T*)a.g_w + (int64_t)(cw + l32) * Cs + 8 * g, Cs / 16, ss, SR, l32, g);
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        const int ch = cw + 8 * rg + 4 * g;
        const f32x4 b4 = *reinterpret_cast<const f32x4*>(&gb_s[ch]);
        f32x4 pre;
#pragma unroll
        for (int e = 0; e < 4; ++e) pre[e] = acc[4 * rg + e] + b4[e];
        // T(linear) -> T(sigmoid) -> T(o * g)
        const f32x4 pr = TypeOps<T>::to_f32(TypeOps<T>::from_f32(pre));
        f32x4 gv;
#pragma unroll
        for (int e = 0; e < 4; ++e) gv[e] = 1.0f / (1.0f + __expf(-pr[e]));
        const f32x4 gr = TypeOps<T>::to_f32(TypeOps<T>::from_f32(gv));
        T* op = &og[l32 * OR + ch];
        const f32x4 ov = TypeOps<T>::to_f32(load4(op));
        store4(op, TypeOps<T>::from_f32(ov * gr));
      }
    }
  }
  __syncthreads();

  // ---- output: acc = [out channel][token], passes of GOC channels staged through ys
  T* obase = (T*)a.out + t0 * a.out_ld;
  for (int c0 = 0; c0 < Co; c0 += GOC) {
    const int W = Co - c0 < GOC ? Co - c0 : GOC;
    const int cw = c0 + 32 * wave;
    if (32 * wave < W) {
      f32x16 acc;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = 0.f;
      gate_out_gemm<T, PREC>(acc, (const T*)a.o_w + (int64_t)(cw + l32) * D + 8 * g, D / 16, og, OR, l32, g);
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        const int ch = cw + 8 * rg + 4 * g;
        const f32x4 b4 = *reinterpret_cast<const f32x4*>(&ob_s[ch]);
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[4 * rg + e] + b4[e];
        store4(&ys[l32 * YR + 32 * wave + 8 * rg + 4 * g], TypeOps<T>::from_f32(v));
      }
    }
    __syncthreads();
    const int cpr = W / EPC;
    for (int c = tid; c < GT * cpr; c += GO_THREADS) {
      const int r = c / cpr, k = (c - r * cpr) * EPC;
      if (r < ntok) {
        if constexpr (sizeof(T) == 2)
          store8(obase + (int64_t)r * a.out_ld + c0 + k, load8(&ys[r * YR + k]));
        else
          store4(obase + (int64_t)r * a.out_ld + c0 + k, load4(&ys[r * YR + k]));
      }
    }
    if (c0 + GOC < Co) __syncthreads();  // the next pass rewrites ys
  }
}

template <typename T, int PREC, int NW>
int launch_gate_out(const gnn_apb_gate_out_args& a, hipStream_t stream, size_t smem) {
  const void* fn = (const void*)apb_gate_out_kernel<T, PREC, NW>;
  if (smem > 64 * 1024) (void)hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
  hipLaunchKernelGGL((apb_gate_out_kernel<T, PREC, NW>), dim3((uint32_t)((a.M + GT - 1) / GT)), dim3(64 * NW), smem,
                     stream, a);
  return (int)hipGetLastError();
}

constexpr size_t GO_MAX_LDS = 160 * 1024;

// Waves per workgroup. A call has one workgroup per 32 tokens, so few that most CUs stay idle
// and its time is one workgroup's chain of weight loads and MFMAs per pass of 32 channels a
// wave: widths above 128 take as many waves as the registers allow (16; 8 for fp32, whose
// fragments are twice as wide), so that D = 384 is one pass instead of three; narrower ones
// and widths whose tiles would not fit in LDS beside the wider output pass take 4.
// 384 tokens, c_s = D = 384, bf16: 25.6 -> 21.9 us.
template <typename T, int PREC>
int launch_gate_out(const gnn_apb_gate_out_args& a, hipStream_t stream) {
  constexpr int NW = sizeof(T) == 2 ? 16 : 8;
  const size_t wide = gate_out_lds_total(gate_out_lds<T>(a.Cs, a.D, 32 * NW), a.D, a.Co);
  if ((a.D > 128 || a.Co > 128) && wide <= GO_MAX_LDS) return launch_gate_out<T, PREC, NW>(a, stream, wide);
  const size_t smem = gate_out_lds_total(gate_out_lds<T>(a.Cs, a.D, 128), a.D, a.Co);
  if (smem > GO_MAX_LDS)
    return set_error(GNN_ERR_UNSUPPORTED, "apb_gate_out: c_s + attention width too large for the LDS tiles");
  return launch_gate_out<T, PREC, 4>(a, stream, smem);
}

}  // namespace

int apb_gate_out(const gnn_apb_gate_out_args& a, hipStream_t stream) {
  if (a.Cs % 32 != 0 || a.D % 32 != 0 || a.Co % 32 != 0)
    return set_error(GNN_ERR_UNSUPPORTED, "apb_gate_out: c_s, the attention width and c_out must be multiples of 32");
  if (a.M >= ((int64_t)1 << 31) * GT) return set_error(GNN_ERR_UNSUPPORTED, "apb_gate_out: too many tokens");
  switch (a.dtype) {
    case GNN_BF16: return launch_gate_out<bf16, PREC_NATIVE>(a, stream);
    case GNN_F16: return launch_gate_out<f16, PREC_NATIVE>(a, stream);
    case GNN_F32:
      return a.precision == GNN_PREC_BF16X3 ? launch_gate_out<float, PREC_BF16X3>(a, stream)
                                            : launch_gate_out<float, PREC_IEEE>(a, stream);
  }
  return set_error(GNN_ERR_ARG, "apb_gate_out: unknown dtype");
}

int pair_bias_proj(const gnn_pair_bias_args& a, hipStream_t stream) {
  if (a.Zc % 8 != 0 || a.Zc > PB_MAX_ZC)
    return set_error(GNN_ERR_UNSUPPORTED, "pair_bias_proj: c_z must be a multiple of 8 and at most 256");
  if (a.H * a.Zc > PB_MAX_W)
    return set_error(GNN_ERR_UNSUPPORTED, "pair_bias_proj: heads * c_z must be at most 8192");
  switch (a.dtype) {
    case GNN_BF16: return launch_pb<bf16>(a, stream);
    case GNN_F16: return launch_pb<f16>(a, stream);
    case GNN_F32: return launch_pb<float>(a, stream);
  }
  return set_error(GNN_ERR_ARG, "pair_bias_proj: unknown dtype");
}

}  // namespace gnn
