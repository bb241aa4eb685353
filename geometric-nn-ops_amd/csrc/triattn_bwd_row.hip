// Triangle attention backward for gfx950, row-resident variant of dq and dk / dv: 16-bit
// inputs, head dim 32, N_res <= BWD_ROW_MAX_N.
//
// Same mathematics as bwd_dq_kernel and bwd_dkdv_kernel (triattn_bwd.hip):
//   dP_ij = dO_i . v_j,  dS_ij = P_ij (dP_ij - Delta_i),  P_ij = exp(S_ij - lse_i),
//   dV_j = sum_i P_ij dO_i,  dK_j = sum_i dS_ij Q'_i,  dQ_i = scale * sum_j dS_ij k_j,
// the gradient of triangle_attention_torch (geometric_nn_ops_torch/triangle/_reference/
// triangle_attention.py:11-44) that the reference's Triton backward computes
// (geometric_nn_ops_torch/triangle/_kernels/triangle_attention.py:548-1087).
//
// What changes is the schedule, as in the forward's row kernel (triattn_row.hip): one
// workgroup of 8 waves per (b, s, h) row stages the operands the row's loops sweep ONCE in
// LDS and its waves then run their loops with no barrier (the tiled kernels re-stage a
// 64-row tile behind two barriers per step, exposing the load latency every step):
//   bwd_dq_row    K and V of the row (global_load_lds, chunks XOR-swizzled by (row / 4) % 4),
//                 the per-key mask term and a per-64-key-tile "no masked key" flag; the waves
//                 take 32-query blocks round robin and sweep every key tile. Also writes
//                 Delta = rowsum(dO * O) for bwd_dkdv_row and bwd_dbias.
//   bwd_dkdv_row  Q' = bf16(q * scale) (through registers: the product is rounded) and dO
//                 (global_load_lds) of the row, with its lse and Delta; the waves take
//                 32-key blocks round robin and sweep every query tile.
// These two serve N_res above BWD_FUSED_MAX_N; below it bwd_fused_row does the work of both.
// The pair-bias fragments of the next step are requested from global memory (L2: a bias
// plane is shared by every N_seq row) while the current one is computed. The reference's
// correction for rows whose keys are all masked (P of a masked key divided by N_res, which
// only changes such rows: elsewhere a masked key's P is exactly 0) joins the exponent, as
// P = exp2((S - lse) log2(e) - log2(N_res)) (see lost_lse_bound).
// Against the tiled kernels the results differ in their last bits: the exponent is one fma where
// |lse| is small (subtracts_first; bwd_dkdv_row always subtracts first), and the fused kernel
// adds dQ over the key blocks in an order that starts at the wave's own.
#include <type_traits>

#include "gnn_common.hpp"
#include "gnn_internal.hpp"

namespace gnn {

namespace {

constexpr float LOG2E_R = 1.4426950408889634f;
constexpr int RW = 8;             // waves per workgroup
constexpr int RNT = 64 * RW;      // threads per workgroup
constexpr int RT = 64;            // rows (keys or queries) per tile
constexpr int RROW = 64;          // bytes per staged row (32 x 16-bit)
constexpr int RTILE = RT * RROW;  // bytes per staged tile
constexpr int BWD_ROW_MAX_N = 1024;
constexpr int RMAX_TILES = BWD_ROW_MAX_N / RT;

// byte offset of (row r, 16-byte chunk c) of a staged [rows][32] tile, chunks XOR-swizzled
// by (r / 4) % 4 (the layout of bwd_dq_kernel / bwd_dkdv_kernel's tiles)
__device__ __forceinline__ int rswz(int r, int c) { return r * RROW + 16 * (c ^ ((r >> 2) & 3)); }

template <typename T>
__device__ __forceinline__ typename TypeOps<T>::V8 rrow8(const unsigned char* base, int r, int c) {
  return *reinterpret_cast<const typename TypeOps<T>::V8*>(base + rswz(r, c));
}

template <typename T>
__device__ __forceinline__ typename TypeOps<T>::V4 rtr4(const unsigned char* p) {
  typedef short v4i16 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) v4i16 lds_v4i16;
  const v4i16 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (lds_v4i16*)(__attribute__((address_space(3))) const unsigned char*)p);
  return __builtin_bit_cast(typename TypeOps<T>::V4, v);
}

// Transposed B fragment of a staged tile: k = rows row0 + 16 kk + 8 (e / 4) + 4 g + e % 4 (the
// 32x32 accumulator's row order), n = column lane % 32.
template <typename T>
__device__ __forceinline__ typename TypeOps<T>::V8 rtr_frag(const unsigned char* tile, int row0, int kk, int lane) {
  const int g = lane >> 5, r16 = lane & 15;
  const int col = 16 * ((lane >> 4) & 1) + 4 * (r16 & 3);
  typename TypeOps<T>::V8 f;
#pragma unroll
  for (int hh = 0; hh < 2; ++hh) {
    const int row = row0 + 16 * kk + 8 * hh + 4 * g + (r16 >> 2);
    const typename TypeOps<T>::V4 x = rtr4<T>(tile + rswz(row, col >> 3) + 2 * (col & 7));
#pragma unroll
    for (int e = 0; e < 4; ++e) f[4 * hh + e] = x[e];
  }
  return f;
}

template <typename T>
__device__ __forceinline__ typename TypeOps<T>::V8 racc_frag(const f32x16& a, int kk) {
  f32x8 x = {a[8 * kk + 0], a[8 * kk + 1], a[8 * kk + 2], a[8 * kk + 3],
             a[8 * kk + 4], a[8 * kk + 5], a[8 * kk + 6], a[8 * kk + 7]};
  return TypeOps<T>::from_f32(x);
}

template <typename T>
__device__ __forceinline__ void ridentity(typename TypeOps<T>::V8 (&idf)[2], int l32, int g) {
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int e = 0; e < 8; ++e) idf[t][e] = TypeOps<T>::from_f32(l32 == 16 * t + 8 * g + e ? 1.f : 0.f);
}

// Stage rows 0 .. ntiles * 64 - 1 of a [N][32] 16-bit operand (row stride rs elements) into
// a swizzled LDS image with global_load_lds_dwordx4: one instruction moves 16 rows (1 KB),
// lane l filling bytes 16 l .. 16 l + 15 = row l / 4, physical chunk l % 4, which holds
// logical chunk (l % 4) ^ ((l / 16) % 4). Rows past N repeat row N - 1 (finite values whose
// weights are zero).
template <typename T>
__device__ __forceinline__ void stage_rows_dma(unsigned char* dst, const T* src, int64_t rs, int N, int ntiles,
                                               int wave, int lane) {
  const int lrow = lane >> 2, ch = (lane & 3) ^ ((lane >> 4) & 3);
  for (int q = wave; q < ntiles * (RT / 16); q += RW) {
    const int r = min(16 * q + lrow, N - 1);
    __builtin_amdgcn_global_load_lds((const void*)(src + (int64_t)r * rs + 8 * ch),
                                     (__attribute__((address_space(3))) void*)(dst + q * 1024), 16, 0, 0);
  }
}

// Logical workgroup order of the row kernels: the two heads of a pair fastest (they share
// the 128-byte lines of the K / V / Q / dO rows at D = 32), then N_seq, so an XCD keeps the
// bias planes of few heads in its L2; odd H takes rows fastest.
__device__ __forceinline__ void row_coords(uint32_t w, int S, int H, int& b, int& s, int& h) {
  if (H % 2 == 0) {
    const uint32_t hi = w & 1u, rest = w >> 1;
    s = (int)(rest % (uint32_t)S);
    h = 2 * (int)((rest / (uint32_t)S) % (uint32_t)(H / 2)) + (int)hi;
  } else {
    s = (int)(w % (uint32_t)S);
    h = (int)((w / (uint32_t)S) % (uint32_t)H);
  }
  b = (int)(w / ((uint32_t)S * H));
}

// P = exp(S - lse) is exp2(fma(S, log2 e, -lse log2 e)), one fma per element, where the rounding of
// -lse log2 e does no harm: up to FAR_LSE it is at most 2^-16, which moves P by 1.1e-5 of itself, a
// twentieth of fp16's half ulp. It grows with |lse|; at the mask sentinel, or wherever the pair bias
// alone puts a query, S - lse is exact and the rounded product is off by whole powers of two (bf16:
// 0.5 at 1e7, 52 at 1e9). Queries there subtract lse from the logit first.
constexpr float FAR_LSE = 256.f;
__device__ __forceinline__ bool subtracts_first(const gnn_triattn_bwd_args& a, float lse) {
  return fabsf(lse) > FAR_LSE || (a.mask && lse <= 0.5f * a.mask_value);
}

// ------------------------------------------------------------------------------- dQ
struct DqRowHdr {
  float kterm[BWD_ROW_MAX_N];  // added to the scores of key j: 0, the mask sentinel, or -inf past N
  int plain[RMAX_TILES];       // tile t has no masked key and no key past N
  int dead;                    // no live key
};
constexpr int DQ_HDR = (int)((sizeof(DqRowHdr) + 255) / 256 * 256);

template <typename T, bool HAS_BIAS>
__global__ __launch_bounds__(RNT, 4) void bwd_dq_row_kernel(const gnn_triattn_bwd_args a) {
  typedef typename TypeOps<T>::V8 V8;
  extern __shared__ __align__(256) unsigned char smem_raw[];
  DqRowHdr& hdr = *reinterpret_cast<DqRowHdr*>(smem_raw);
  const int N = (int)a.N, H = (int)a.H, S = (int)a.S;
  const int ntiles = (N + RT - 1) / RT;
  unsigned char* ks = smem_raw + DQ_HDR;
  unsigned char* vs = ks + ntiles * RTILE;
  int b, s, h;
  row_coords(xcd_remap(blockIdx.x, gridDim.x), S, H, b, s, h);
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  const T* kp = (const T*)a.k + b * a.k_stride[0] + s * a.k_stride[1] + h * a.k_stride[3];
  const T* vp = (const T*)a.v + b * a.v_stride[0] + s * a.v_stride[1] + h * a.v_stride[3];
  stage_rows_dma<T>(ks, kp, a.k_stride[2], N, ntiles, wave, lane);
  stage_rows_dma<T>(vs, vp, a.v_stride[2], N, ntiles, wave, lane);
  if (wave == 0) {
    bool live = false;
    for (int t = 0; t < ntiles; ++t) {
      const int key = t * RT + lane;
      float kt = 0.f;
      if (key >= N)
        kt = -INFINITY;
      else if (a.mask && a.mask[b * a.mask_stride[0] + s * a.mask_stride[1] + (int64_t)key * a.mask_stride[2]] == 0)
        kt = a.mask_value;
      hdr.kterm[key] = kt;
      const bool plain = __ballot(kt != 0.f) == 0;
      if (lane == 0) hdr.plain[t] = plain;
      live |= __ballot(kt == 0.f) != 0;
    }
    if (lane == 0) hdr.dead = !live;
  }
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0): this wave's LDS DMA has landed
  __syncthreads();

  V8 idf[2];
  ridentity<T>(idf, l32, g);
  const int64_t lrow = (((int64_t)b * S + s) * H + h) * N;
  const int nqb = (N + 31) / 32;
  for (int qblk = wave; qblk < nqb; qblk += RW) {
    int Nq = N;  // opaque: keeps the tail compares of the bias loads inside the loop
    asm volatile("" : "+s"(Nq));
    const int qi = qblk * 32 + l32;
    const bool qok = qi < Nq;
    // this lane's query: Q' and dO as B operands (lane = query, 8 consecutive d)
    V8 qf[2], dof[2];
    float delta;
    {
      const T* qr = (const T*)a.q + b * a.q_stride[0] + s * a.q_stride[1] + h * a.q_stride[3] +
                    (int64_t)(qok ? qi : 0) * a.q_stride[2];
      const T* dr = (const T*)a.dout + b * a.do_stride[0] + s * a.do_stride[1] + h * a.do_stride[3] +
                    (int64_t)(qok ? qi : 0) * a.do_stride[2];
      const T* orow = (const T*)a.o + b * a.o_stride[0] + s * a.o_stride[1] + h * a.o_stride[3] +
                      (int64_t)(qok ? qi : 0) * a.o_stride[2];
      float part = 0.f;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const int d0 = 16 * kk + 8 * g;
        qf[kk] = qok ? TypeOps<T>::from_f32(TypeOps<T>::to_f32(load8(qr + d0)) * a.scale) : zero8<T>();
        dof[kk] = qok ? load8(dr + d0) : zero8<T>();
        const f32x8 x = TypeOps<T>::to_f32(qok ? load8(orow + d0) : zero8<T>());
        const f32x8 y = TypeOps<T>::to_f32(dof[kk]);
#pragma unroll
        for (int e = 0; e < 8; ++e) part = __builtin_fmaf(x[e], y[e], part);
      }
      // Delta = dO . O: the lane pair (g = 0, 1) holds the 32 columns between them
      delta = part + __shfl_xor(part, 32);
      if (qok && g == 0) a.delta[lrow + qi] = delta;
    }
    const float lse = qok ? a.lse[lrow + qi] : INFINITY;  // absent queries: p = 0
    // P = exp2(S log2 e - lse log2 e) takes one fma per element (lse is this lane's query's,
    // constant along the accumulator) unless a query of the wave has S - lse formed first.
    const bool first = hdr.dead || __any(qok && subtracts_first(a, lse));
    const float pl2 = hdr.dead || lse <= lost_lse_bound(a.mask, a.mask_value) ? -__log2f((float)N) : 0.f;
    const float nl2 = -lse * LOG2E_R;
    const T* brow = HAS_BIAS ? (const T*)a.bias + b * a.bias_stride[0] + h * a.bias_stride[1] +
                                   (int64_t)(qok ? qi : 0) * a.bias_stride[2]
                             : nullptr;
    // bias fragments of one 32-key step: keys 32 st + 16 t + 8 g + 0..7 of the lane's query
    V8 bb[2];
    auto load_bias = [&](int st) {
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) bb[t2] = load8_bias_tail<T>(brow, 32 * st + 16 * t2 + 8 * g, Nq);
    };
    if constexpr (HAS_BIAS) load_bias(0);
    f32x16 dq;
#pragma unroll
    for (int i = 0; i < 16; ++i) dq[i] = 0.f;

    // 32-key steps: S^T[key][q] = K Q'^T (+ bias) and dP^T[key][q] = V dO^T, rows = keys
    // 32 st + 8 (i / 4) + 4 g + i % 4, column = query
    const int nst = 2 * ntiles;
    for (int st = 0; st < nst; ++st) {
      const unsigned char* kt = ks + st * (RTILE / 2);
      const unsigned char* vt = vs + st * (RTILE / 2);
      const bool plain = hdr.plain[st >> 1] != 0;
      f32x16 sc, dp;
#pragma unroll
      for (int i = 0; i < 16; ++i) sc[i] = dp[i] = 0.f;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        Mma<T, PREC_NATIVE>::step(sc, rrow8<T>(kt, l32, 2 * kk + g), qf[kk]);
        Mma<T, PREC_NATIVE>::step(dp, rrow8<T>(vt, l32, 2 * kk + g), dof[kk]);
      }
      if constexpr (HAS_BIAS) {
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2) Mma<T, PREC_NATIVE>::step(sc, idf[t2], bb[t2]);
        if (st + 1 < nst) load_bias(st + 1);
      }
      f32x16 ds;
      if (plain && !first) {
#pragma unroll
        for (int i = 0; i < 16; ++i) ds[i] = fast_exp2(__builtin_fmaf(sc[i], LOG2E_R, nl2)) * (dp[i] - delta);
      } else if (!first) {
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          const f32x4 k4 = *reinterpret_cast<const f32x4*>(&hdr.kterm[32 * st + 8 * rg + 4 * g]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int i = 4 * rg + e;
            ds[i] = fast_exp2(__builtin_fmaf(sc[i] + k4[e], LOG2E_R, nl2)) * (dp[i] - delta);
          }
        }
      } else {
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          const f32x4 k4 = *reinterpret_cast<const f32x4*>(&hdr.kterm[32 * st + 8 * rg + 4 * g]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int i = 4 * rg + e;
            ds[i] = fast_exp2(__builtin_fmaf(sc[i] + k4[e] - lse, LOG2E_R, pl2)) * (dp[i] - delta);
          }
        }
      }
      // dQ += dS K: A = the dS^T accumulator (lane = query, k = keys), B = K read transposed
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
        Mma<T, PREC_NATIVE>::step(dq, racc_frag<T>(ds, kk), rtr_frag<T>(kt, 0, kk, lane));
    }
    // dq[m = query][n = d]: lane = d, rows = queries 32 qblk + 8 (i / 4) + 4 g + i % 4
    T* dqp = (T*)a.dq + b * a.dq_stride[0] + s * a.dq_stride[1] + h * a.dq_stride[3] + l32;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int qq = qblk * 32 + 8 * (i / 4) + 4 * g + (i % 4);
      if (qq < Nq) dqp[(int64_t)qq * a.dq_stride[2]] = TypeOps<T>::from_f32(dq[i] * a.scale);
    }
  }
}

// --------------------------------------------------------------------------- dK, dV
struct DkdvRowHdr {
  float lse[BWD_ROW_MAX_N];    // +inf for absent queries (p = 0)
  float ndelta[BWD_ROW_MAX_N];  // -Delta (0 for absent queries): the dP accumulators' start
  int row[RW];                  // per wave, of what it staged: 1 a live key, 2 a query past lost_lse_bound
};
constexpr int DKDV_HDR = (int)((sizeof(DkdvRowHdr) + 255) / 256 * 256);

template <typename T>
struct BiasRows {
  typename TypeOps<T>::V8 f[2];  // [t]: keys kbase + 16 t + 8 g + 0..7 of query row r0 + l32
};

template <typename T, bool HAS_BIAS>
__global__ __launch_bounds__(RNT, 4) void bwd_dkdv_row_kernel(const gnn_triattn_bwd_args a) {
  typedef typename TypeOps<T>::V8 V8;
  extern __shared__ __align__(256) unsigned char smem_raw[];
  DkdvRowHdr& hdr = *reinterpret_cast<DkdvRowHdr*>(smem_raw);
  const int N = (int)a.N, H = (int)a.H, S = (int)a.S;
  const int ntiles = (N + RT - 1) / RT;
  const int nrows = ntiles * RT;
  unsigned char* qs = smem_raw + DKDV_HDR;
  unsigned char* ds_ = qs + ntiles * RTILE;
  int b, s, h;
  row_coords(xcd_remap(blockIdx.x, gridDim.x), S, H, b, s, h);
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // dO by DMA; Q' = bf16(q * scale) through registers (rows past N are zero)
  const T* dop = (const T*)a.dout + b * a.do_stride[0] + s * a.do_stride[1] + h * a.do_stride[3];
  stage_rows_dma<T>(ds_, dop, a.do_stride[2], N, ntiles, wave, lane);
  {
    const T* qp = (const T*)a.q + b * a.q_stride[0] + s * a.q_stride[1] + h * a.q_stride[3];
    constexpr int U = 4;
    for (int base = 0; base < nrows * 4; base += RNT * U) {
      V8 x[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = base + u * RNT + tid, r = c >> 2;
        x[u] = (c < nrows * 4 && r < N) ? load8(qp + (int64_t)r * a.q_stride[2] + 8 * (c & 3)) : zero8<T>();
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = base + u * RNT + tid, r = c >> 2;
        if (c < nrows * 4)
          *reinterpret_cast<V8*>(qs + rswz(r, c & 3)) = TypeOps<T>::from_f32(TypeOps<T>::to_f32(x[u]) * a.scale);
      }
    }
    const int64_t lrow = (((int64_t)b * S + s) * H + h) * N;
    bool live = false, lost = false;
    for (int r = tid; r < nrows; r += RNT) {
      const float l = r < N ? a.lse[lrow + r] : INFINITY;
      hdr.lse[r] = l;
      hdr.ndelta[r] = r < N ? -a.delta[lrow + r] : 0.f;
      live |= r < N && (!a.mask || a.mask[b * a.mask_stride[0] + s * a.mask_stride[1] + r * a.mask_stride[2]] != 0);
      lost |= l <= lost_lse_bound(a.mask, a.mask_value);
    }
    const int row = (__any(live) ? 1 : 0) | (__any(lost) ? 2 : 0);
    if (lane == 0) hdr.row[wave] = row;
  }
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0): this wave's LDS DMA has landed
  __syncthreads();

  V8 idf[2];
  ridentity<T>(idf, l32, g);
  // both uniform over the workgroup. A row whose keys are all masked divides P by N_res in the exponent
  const bool dead = !__any(hdr.row[lane & (RW - 1)] & 1), lost = __any(hdr.row[lane & (RW - 1)] & 2);
  const float pl2 = dead ? -__log2f((float)N) : 0.f;
  if (lost && !dead) {  // a live row's queries past the bound: with dO and Delta divided, P^T dO and dS are
    const float inv_n = 1.0f / (float)N;
    for (int r = tid; r < N; r += RNT) {
      if (hdr.lse[r] > lost_lse_bound(a.mask, a.mask_value)) continue;
      hdr.ndelta[r] *= inv_n;
      for (int c = 0; c < 4; ++c) {
        V8* x = reinterpret_cast<V8*>(ds_ + rswz(r, c));
        *x = TypeOps<T>::from_f32(TypeOps<T>::to_f32(*x) * inv_n);
      }
    }
    __syncthreads();
  }
  const T* bias_plane = HAS_BIAS ? (const T*)a.bias + b * a.bias_stride[0] + h * a.bias_stride[1] : nullptr;
  const int nkb = (N + 31) / 32;
  const int nsub = 2 * ntiles;  // 32-query steps
  for (int kblk = wave; kblk < nkb; kblk += RW) {
    int Nk = N;  // opaque, as in the dq kernel
    asm volatile("" : "+s"(Nk));
    const int key = kblk * 32 + l32;
    const bool kok = key < Nk;
    // this lane's key: K and V as B operands (lane = key, 8 consecutive d)
    V8 kf[2], vf[2];
    {
      const T* kr = (const T*)a.k + b * a.k_stride[0] + s * a.k_stride[1] + h * a.k_stride[3] +
                    (int64_t)(kok ? key : 0) * a.k_stride[2];
      const T* vr = (const T*)a.v + b * a.v_stride[0] + s * a.v_stride[1] + h * a.v_stride[3] +
                    (int64_t)(kok ? key : 0) * a.v_stride[2];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        kf[kk] = kok ? load8(kr + 16 * kk + 8 * g) : zero8<T>();
        vf[kk] = kok ? load8(vr + 16 * kk + 8 * g) : zero8<T>();
      }
    }
    // key-side mask term: the sentinel for masked keys, -inf for keys past N (p = 0)
    float kbias = 0.f;
    if (!kok)
      kbias = -INFINITY;
    else if (a.mask && a.mask[b * a.mask_stride[0] + s * a.mask_stride[1] + (int64_t)key * a.mask_stride[2]] == 0)
      kbias = a.mask_value;
    // bias rows of the 32 queries of a step: A = bias[query][key] (lane = query, 8 keys)
    auto load_bias = [&](BiasRows<T>& br, int st) {
      const int qq = 32 * st + l32;
      const T* brow = bias_plane + (int64_t)(qq < Nk ? qq : 0) * a.bias_stride[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int k0 = kblk * 32 + 16 * t + 8 * g;
        br.f[t] = qq < Nk ? load8_bias_tail<T>(brow, k0, Nk) : zero8<T>();
      }
    };
    BiasRows<T> bb;
    if constexpr (HAS_BIAS) load_bias(bb, 0);
    f32x16 dk, dv;
#pragma unroll
    for (int i = 0; i < 16; ++i) dk[i] = dv[i] = 0.f;

    for (int st = 0; st < nsub; ++st) {
      const int r0 = 32 * st;
      // S[q][key] = Q' K^T (+ bias) and dP[q][key] - Delta_q = dO V^T - Delta (the accumulator
      // starts at -Delta): rows = queries r0 + 8 (i / 4) + 4 g + i % 4, column = key
      f32x16 sc, dp;
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        const f32x4 nd4 = *reinterpret_cast<const f32x4*>(&hdr.ndelta[r0 + 8 * rg + 4 * g]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          sc[4 * rg + e] = 0.f;
          dp[4 * rg + e] = nd4[e];
        }
      }
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        Mma<T, PREC_NATIVE>::step(sc, rrow8<T>(qs, r0 + l32, 2 * kk + g), kf[kk]);
        Mma<T, PREC_NATIVE>::step(dp, rrow8<T>(ds_, r0 + l32, 2 * kk + g), vf[kk]);
      }
      if constexpr (HAS_BIAS) {
#pragma unroll
        for (int t = 0; t < 2; ++t) Mma<T, PREC_NATIVE>::step(sc, bb.f[t], idf[t]);
        if (st + 1 < nsub) load_bias(bb, st + 1);
      }
      // P and dS for this lane's key and its 16 queries, 8 at a time (k-step kk of the
      // products): dV += P^T dO and dK += dS^T Q' with A = P / dS (lane = key, k = queries)
      // and B = the staged rows read transposed (k = queries, n = d)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        f32x8 pv, dv8;
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          const int rg = 2 * kk + hh;
          const f32x4 l4 = *reinterpret_cast<const f32x4*>(&hdr.lse[r0 + 8 * rg + 4 * g]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int i = 4 * rg + e;
            const float x = fast_exp2(__builtin_fmaf(sc[i] + kbias - l4[e], LOG2E_R, pl2));
            pv[4 * hh + e] = x;
            dv8[4 * hh + e] = x * dp[i];
          }
        }
        Mma<T, PREC_NATIVE>::step(dv, TypeOps<T>::from_f32(pv), rtr_frag<T>(ds_, r0, kk, lane));
        Mma<T, PREC_NATIVE>::step(dk, TypeOps<T>::from_f32(dv8), rtr_frag<T>(qs, r0, kk, lane));
      }
    }
    // dk / dv[m = key][n = d]: lane = d (l32), rows = keys 32 kblk + 8 (i / 4) + 4 g + i % 4
    T* dkp = (T*)a.dk + b * a.dk_stride[0] + s * a.dk_stride[1] + h * a.dk_stride[3] + l32;
    T* dvp = (T*)a.dv + b * a.dv_stride[0] + s * a.dv_stride[1] + h * a.dv_stride[3] + l32;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int kj = kblk * 32 + 8 * (i / 4) + 4 * g + (i % 4);
      if (kj < Nk) {
        dkp[(int64_t)kj * a.dk_stride[2]] = TypeOps<T>::from_f32(dk[i]);
        dvp[(int64_t)kj * a.dv_stride[2]] = TypeOps<T>::from_f32(dv[i]);
      }
    }
  }
}

// ------------------------------------------------------------------- dQ, dK and dV together
// Up to BWD_FUSED_MAX_N one workgroup takes a (b, s, h) row whole, so the logits and their exponents
// are formed once instead of once for dq and once for dk / dv: 10 products and 1 exponential per
// element pair of 32-blocks instead of 14 and 2 (QK^T, dO V^T and the bias count once).
//
// Q' = bf16(q * scale) and dO of the row sit in LDS (with -lse log2(e) and -Delta, which is formed
// here while o and dO pass through the staging registers), dQ accumulates in LDS in fp32, in the
// MFMA accumulator's own layout (16-byte reads and writes, the read being the product's initial
// accumulator). A wave owns KB blocks of 32 keys: K and V as B operands, K once more read transposed
// (the B operand of dQ += dS K), and the dK / dV accumulators, all in registers. Step t of wave w
// takes the queries of block (KB w + t) mod nb: the waves of a step update different dQ blocks, a
// barrier (which leaves the bias loads in flight) separates the steps, and so every sum has one fixed
// order. dS has its keys on the lanes, as dK's A operand needs it; dQ's A operand needs the queries
// there, so each 32 x 32 tile passes through a wave-private LDS tile and is read back transposed.
//
// KB = 2 (8 waves at N = 512, two workgroups of 4 at 256: two waves per SIMD, 256 registers) reads each
// Q' / dO fragment and updates dQ once for 64 keys; 256 < N <= 384, one workgroup per CU, takes KB = 1,
// whose 9 to 12 waves fill the SIMDs better than 5 or 6 (bf16, bias, H = 4, the call without the bias
// gradient: N = 320 121 against 142 us, 384 185 against 206; N = 128 41 against 33, 256 83 against 69).
// LDS bounds N: 264 bytes per query and 2 KB per wave.
// The same call on the two kernels: N = 256 104 -> 74 us, 384 247 -> 185, 512 537 -> 372. At N = 512 the
// vector ALU is busy 36% of the cycles (exponentials, conversions), the matrix unit 23% and LDS 33%; the
// rest is the chain of a tile (fragments, products, exponentials, the tile's way through LDS, dQ), which
// two waves per SIMD do not hide. Interleaved with the tile's C++ accesses (ordered by the compiler) and
// with the mask's branches inside the loop it took 453 us.
constexpr int BWD_FUSED_MAX_N = 512;

__host__ __device__ inline int fused_kb(int N) { return N > 256 && N <= 384 ? 1 : 2; }
__host__ __device__ inline int fused_waves(int N) {
  const int nb = (N + 31) / 32, kb = fused_kb(N);
  return (nb + kb - 1) / kb;
}
// LDS of a 32-query block: Q' and dO images, dQ in accumulator layout ([4][64 lanes] f32x4), then
// -lse log2(e) (lse itself where the row subtracts first; queries past N: p = 0) and -Delta
struct FusedBlock {
  unsigned char q[32 * RROW];
  unsigned char d[32 * RROW];
  f32x4 dq[4 * 64];
  float nl[32];
  float ndelta[32];
};
// then a 2 KB tile and a word of row flags for each wave
constexpr int FUSED_FLAGS = 64;
inline size_t fused_lds(int N) {
  return (size_t)((N + 31) / 32) * sizeof(FusedBlock) + fused_waves(N) * 2048 + FUSED_FLAGS;
}

// A 32 x 32 16-bit tile through LDS: write4 stores a lane's 16 values (row = lane % 32, columns
// 8 rg + 4 g .. + 3 in words 2 rg, 2 rg + 1) and read_tr reads both k-steps' transposed fragments,
// waiting for the data. In assembly, so that the compiler does not order its other LDS accesses
// (none of which touches the tile) around them; assembly blocks keep their order among themselves
// and a wave's LDS operations execute in order.
__device__ __forceinline__ void tile_write(const uint32_t (&o)[4], const uint64_t (&w)[4]) {
  asm volatile("ds_write_b64 %0, %4\n\tds_write_b64 %1, %5\n\tds_write_b64 %2, %6\n\tds_write_b64 %3, %7"
               :
               : "v"(o[0]), "v"(o[1]), "v"(o[2]), "v"(o[3]), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]));
}
template <typename V8>
__device__ __forceinline__ void tile_read_tr(uint32_t o0, uint32_t o1, V8 (&f)[2]) {
  typedef uint64_t u64x2_t __attribute__((ext_vector_type(2)));
  uint64_t r[4];
  asm volatile(
      "ds_read_b64_tr_b16 %0, %4\n\tds_read_b64_tr_b16 %1, %5\n\t"
      "ds_read_b64_tr_b16 %2, %4 offset:1024\n\tds_read_b64_tr_b16 %3, %5 offset:1024\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3])
      : "v"(o0), "v"(o1));
  f[0] = __builtin_bit_cast(V8, (u64x2_t{r[0], r[1]}));
  f[1] = __builtin_bit_cast(V8, (u64x2_t{r[2], r[3]}));
}

// Sum over the 4 lanes of a quad (every lane gets it)
__device__ __forceinline__ float quad_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, false));
}

template <typename T, bool HAS_BIAS, int KB>
__global__ __launch_bounds__(KB == 2 ? 512 : 768, KB == 2 ? 2 : 3) void bwd_fused_row_kernel(
    const gnn_triattn_bwd_args a) {
  typedef typename TypeOps<T>::V8 V8;
  typedef typename TypeOps<T>::V4 V4;
  extern __shared__ __align__(256) unsigned char smem_raw[];
  const int N = (int)a.N, H = (int)a.H, S = (int)a.S;
  const int nb = (N + 31) / 32, nrows = 32 * nb, nth = (int)blockDim.x;
  FusedBlock* blk = reinterpret_cast<FusedBlock*>(smem_raw);
  int b, s, h;
  row_coords(xcd_remap(blockIdx.x, gridDim.x), S, H, b, s, h);
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned char* tile = smem_raw + nb * sizeof(FusedBlock) + wave * 2048;  // this wave's dS tile [key][query]
  const int64_t lrow = (((int64_t)b * S + s) * H + h) * N;
  // per wave, of its keys and the queries that it stages: 1 a live key, 2 a query that subtracts first
  int* flags = reinterpret_cast<int*>(smem_raw + nb * sizeof(FusedBlock) + nth / 64 * 2048);

  // ---- this wave's keys: K and V as B operands (lane = key, 8 consecutive d), and the key-side
  // mask term (-inf for keys past N: p = 0)
  const int kb0 = KB * wave;
  V8 kf[KB][2], vf[KB][2];
  float kbias[KB];
  bool masked = false, live = false, first = false;
#pragma unroll
  for (int u = 0; u < KB; ++u) {
    const int key = 32 * (kb0 + u) + l32;
    const bool kok = key < N;
    const T* kr = (const T*)a.k + b * a.k_stride[0] + s * a.k_stride[1] + h * a.k_stride[3] +
                  (int64_t)(kok ? key : 0) * a.k_stride[2];
    const T* vr = (const T*)a.v + b * a.v_stride[0] + s * a.v_stride[1] + h * a.v_stride[3] +
                  (int64_t)(kok ? key : 0) * a.v_stride[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      kf[u][kk] = kok ? load8(kr + 16 * kk + 8 * g) : zero8<T>();
      vf[u][kk] = kok ? load8(vr + 16 * kk + 8 * g) : zero8<T>();
    }
    kbias[u] = 0.f;
    if (!kok)
      kbias[u] = -INFINITY;
    else if (a.mask && a.mask[b * a.mask_stride[0] + s * a.mask_stride[1] + (int64_t)key * a.mask_stride[2]] == 0)
      kbias[u] = a.mask_value;
    masked |= kbias[u] != 0.f;
    live |= kbias[u] == 0.f;
  }

  // ---- stage Q' and dO (rows past N are zero), form Delta, clear dQ
  {
    const T* qp = (const T*)a.q + b * a.q_stride[0] + s * a.q_stride[1] + h * a.q_stride[3];
    const T* dp = (const T*)a.dout + b * a.do_stride[0] + s * a.do_stride[1] + h * a.do_stride[3];
    const T* op = (const T*)a.o + b * a.o_stride[0] + s * a.o_stride[1] + h * a.o_stride[3];
    constexpr int U = 2;
    for (int base = 0; base < nrows * 4; base += nth * U) {
      V8 xq[U], xd[U], xo[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = base + u * nth + tid, r = c >> 2, d0 = 8 * (c & 3);
        const bool in = r < N;  // (N <= nrows, so chunks past the staged rows read nothing)
        xq[u] = in ? load8(qp + (int64_t)r * a.q_stride[2] + d0) : zero8<T>();
        xd[u] = in ? load8(dp + (int64_t)r * a.do_stride[2] + d0) : zero8<T>();
        xo[u] = in ? load8(op + (int64_t)r * a.o_stride[2] + d0) : zero8<T>();
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = base + u * nth + tid, r = c >> 2;
        const f32x8 x = TypeOps<T>::to_f32(xo[u]), y = TypeOps<T>::to_f32(xd[u]);
        float part = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) part = __builtin_fmaf(x[e], y[e], part);
        const float delta = quad_sum(part);
        if (c < nrows * 4) {
          FusedBlock& B = blk[r >> 5];
          *reinterpret_cast<V8*>(B.q + rswz(r & 31, c & 3)) =
              TypeOps<T>::from_f32(TypeOps<T>::to_f32(xq[u]) * a.scale);
          *reinterpret_cast<V8*>(B.d + rswz(r & 31, c & 3)) = xd[u];
          if ((c & 3) == 0) {
            B.ndelta[r & 31] = -delta;
            if (r < N) a.delta[lrow + r] = delta;
          }
        }
      }
    }
    for (int r = tid; r < nrows; r += nth) {
      const float l = r < N ? a.lse[lrow + r] : INFINITY;
      blk[r >> 5].nl[r & 31] = l;
      first |= r < N && subtracts_first(a, l);
    }
    const int f = (__any(live) ? 1 : 0) | (__any(first) ? 2 : 0);
    if (lane == 0) flags[wave] = f;
    for (int c = tid; c < nb * 256; c += nth) blk[c >> 8].dq[c & 255] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // per-lane byte offsets inside a block's images and the tile: row fragments (row l32, chunks
  // 2 kk + g), transposed reads (rows 16 kk + 8 hh + 4 g + .., see rtr_frag; kk adds 1024), tile rows
  const int o_row0 = rswz(l32, g), o_row1 = rswz(l32, 2 + g);
  const int r16 = lane & 15, tcol = 16 * ((lane >> 4) & 1) + 4 * (r16 & 3);
  const int o_tr0 = rswz(4 * g + (r16 >> 2), tcol >> 3) + 2 * (tcol & 7);
  const int o_tr1 = rswz(8 + 4 * g + (r16 >> 2), tcol >> 3) + 2 * (tcol & 7);
  const uint32_t t0 = lds_addr(tile);
  const uint32_t t_tr0 = t0 + o_tr0, t_tr1 = t0 + o_tr1;
  const uint32_t t_wr[4] = {t0 + rswz(l32, 0) + 8 * g, t0 + rswz(l32, 1) + 8 * g, t0 + rswz(l32, 2) + 8 * g,
                            t0 + rswz(l32, 3) + 8 * g};
  auto tr = [&](const unsigned char* img, int kk) -> V8 {  // rtr_frag(img, 0, kk, lane)
    const V4 x = rtr4<T>(img + o_tr0 + 1024 * kk), y = rtr4<T>(img + o_tr1 + 1024 * kk);
    return V8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
  };
  // K transposed (B operand of dQ: k = key in the accumulator's row order, n = d), through the tile
  V8 ktr[KB][2];
#pragma unroll
  for (int u = 0; u < KB; ++u) {
    *reinterpret_cast<V8*>(tile + o_row0) = kf[u][0];
    *reinterpret_cast<V8*>(tile + o_row1) = kf[u][1];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) ktr[u][kk] = tr(tile, kk);
    __builtin_amdgcn_wave_barrier();
  }
  V8 idf[2];
  ridentity<T>(idf, l32, g);
  // bias rows of a query block: A = bias[query][key] (lane = query, 8 keys); queries past N read
  // row N - 1 (their p is 0). The wave that holds the row's end zeroes the values of keys past N
  // (the identity product multiplies them with zeros: they may be NaN), chunks past N read chunk 0.
  const T* bias_plane = HAS_BIAS ? (const T*)a.bias + b * a.bias_stride[0] + h * a.bias_stride[1] : nullptr;
  const uint32_t bpitch = HAS_BIAS ? (uint32_t)a.bias_stride[2] : 0;
  const bool ktail = 32 * (kb0 + KB) > N;  // uniform; such a wave is a masked one
  V8 bb[KB][2];
  auto load_bias = [&](int u, int qb) {
    const uint32_t row = (uint32_t)min(32 * qb + l32, N - 1) * bpitch;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int k0 = 32 * (kb0 + u) + 16 * t + 8 * g;
      bb[u][t] = load8(bias_plane + (row + (k0 < N ? k0 : 0)));
    }
  };
  auto cut_bias = [&](int u) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int nv = N - (32 * (kb0 + u) + 16 * t + 8 * g);  // values of the chunk that are keys
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (e >= nv) bb[u][t][e] = TypeOps<T>::from_f32(0.f);
    }
  };
  if constexpr (HAS_BIAS) {
#pragma unroll
    for (int u = 0; u < KB; ++u) load_bias(u, kb0);
  }
  f32x16 dk[KB], dv[KB];
#pragma unroll
  for (int u = 0; u < KB; ++u)
#pragma unroll
    for (int i = 0; i < 16; ++i) dk[u][i] = dv[u][i] = 0.f;
  __syncthreads();
  // What the row's waves found together. Unless it subtracts first, lse and the key-side term join
  // the exponent in units of log2.
  const int found = flags[lane % (nth / 64)];
  const bool dead = !__any(found & 1);
  first = dead || __any(found & 2);
  const float nlog2 = -__log2f((float)N), qbound = lost_lse_bound(a.mask, a.mask_value);
  const float pl2 = dead ? nlog2 : 0.f;
  if (!first) {
    for (int r = tid; r < nrows; r += nth) blk[r >> 5].nl[r & 31] *= -LOG2E_R;
#pragma unroll
    for (int u = 0; u < KB; ++u) kbias[u] *= LOG2E_R;
    __syncthreads();
  }
  const int mode = first ? 2 : __any(masked) ? 1 : 0;  // uniform over the wave

  // MODE 0: no masked key in the wave's blocks and none past N. 1: the key-side term joins the
  // exponent. 2: the row subtracts lse from the logit first.
  auto sweep = [&](auto mode_) {
    constexpr int MODE = decltype(mode_)::value;
    int qb = kb0;
    for (int t = 0; t < nb; ++t) {
      FusedBlock& B = blk[qb];
      const int qn = qb + 1 == nb ? 0 : qb + 1;
      f32x16 dq;
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        const f32x4 v = B.dq[64 * rg + lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) dq[4 * rg + e] = v[e];
      }
#pragma unroll
      for (int u = 0; u < KB; ++u) {
        if (MODE > 0 && u > 0 && kb0 + u >= nb) continue;  // uniform; no key there
        // S[q][key] = Q' K^T (+ bias) and dP[q][key] - Delta_q = dO V^T - Delta (the accumulator
        // starts at -Delta): rows = queries 32 qb + 8 (i / 4) + 4 g + i % 4, column = key
        f32x16 sc, dp;
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          const f32x4 nd4 = *reinterpret_cast<const f32x4*>(&B.ndelta[8 * rg + 4 * g]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            sc[4 * rg + e] = 0.f;
            dp[4 * rg + e] = nd4[e];
          }
        }
        if constexpr (HAS_BIAS) {
          if (MODE > 0 && ktail) cut_bias(u);
#pragma unroll
          for (int t2 = 0; t2 < 2; ++t2) Mma<T, PREC_NATIVE>::step(sc, bb[u][t2], idf[t2]);
          load_bias(u, qn);
        }
        Mma<T, PREC_NATIVE>::step(sc, *reinterpret_cast<const V8*>(B.q + o_row0), kf[u][0]);
        Mma<T, PREC_NATIVE>::step(dp, *reinterpret_cast<const V8*>(B.d + o_row0), vf[u][0]);
        Mma<T, PREC_NATIVE>::step(sc, *reinterpret_cast<const V8*>(B.q + o_row1), kf[u][1]);
        Mma<T, PREC_NATIVE>::step(dp, *reinterpret_cast<const V8*>(B.d + o_row1), vf[u][1]);
        // P = exp2(S log2 e - lse log2 e [+ mask]), or with S - lse formed first (subtracts_first)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          const f32x4 l4 = *reinterpret_cast<const f32x4*>(&B.nl[8 * rg + 4 * g]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int i = 4 * rg + e;
            const float x = MODE == 0   ? __builtin_fmaf(sc[i], LOG2E_R, l4[e])
                            : MODE == 1 ? __builtin_fmaf(sc[i], LOG2E_R, l4[e] + kbias[u])
                                        : __builtin_fmaf(sc[i] + kbias[u] - l4[e], LOG2E_R,
                                                         l4[e] <= qbound ? nlog2 : pl2);
            sc[i] = fast_exp2(x);
            dp[i] *= sc[i];  // dS
          }
        }
        // dS through the tile (row = key), dV += P^T dO and dK += dS^T Q' meanwhile: A = P / dS
        // (lane = key, k = queries), B = the staged rows read transposed (k = queries, n = d)
        const V8 dsf[2] = {racc_frag<T>(dp, 0), racc_frag<T>(dp, 1)};
        typedef uint64_t u64x2_t __attribute__((ext_vector_type(2)));
        const u64x2_t d0 = __builtin_bit_cast(u64x2_t, dsf[0]), d1 = __builtin_bit_cast(u64x2_t, dsf[1]);
        const uint64_t dw[4] = {d0[0], d0[1], d1[0], d1[1]};
        tile_write(t_wr, dw);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          Mma<T, PREC_NATIVE>::step(dv[u], racc_frag<T>(sc, kk), tr(B.d, kk));
          Mma<T, PREC_NATIVE>::step(dk[u], dsf[kk], tr(B.q, kk));
        }
        // dQ += dS K: A = dS (lane = query, k = keys)
        V8 dst[2];
        tile_read_tr(t_tr0, t_tr1, dst);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) Mma<T, PREC_NATIVE>::step(dq, dst[kk], ktr[u][kk]);
      }
#pragma unroll
      for (int rg = 0; rg < 4; ++rg)
        B.dq[64 * rg + lane] = f32x4{dq[4 * rg], dq[4 * rg + 1], dq[4 * rg + 2], dq[4 * rg + 3]};
      qb = qn;
      // this wave's dQ block is written; after the barrier another wave takes it over
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
  };
  if (mode == 0)
    sweep(std::integral_constant<int, 0>{});
  else if (mode == 1)
    sweep(std::integral_constant<int, 1>{});
  else
    sweep(std::integral_constant<int, 2>{});

  // dk / dv[m = key][n = d]: lane = d (l32), rows = keys 32 block + 8 (i / 4) + 4 g + i % 4
  T* dkp = (T*)a.dk + b * a.dk_stride[0] + s * a.dk_stride[1] + h * a.dk_stride[3] + l32;
  T* dvp = (T*)a.dv + b * a.dv_stride[0] + s * a.dv_stride[1] + h * a.dv_stride[3] + l32;
#pragma unroll
  for (int u = 0; u < KB; ++u)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int kj = (kb0 + u) * 32 + 8 * (i / 4) + 4 * g + (i % 4);
      if (kj < N) {
        dkp[(int64_t)kj * a.dk_stride[2]] = TypeOps<T>::from_f32(dk[u][i]);
        dvp[(int64_t)kj * a.dv_stride[2]] = TypeOps<T>::from_f32(dv[u][i]);
      }
    }
  // dq[m = query][n = d]: the accumulator layout of each block
  T* dqg = (T*)a.dq + b * a.dq_stride[0] + s * a.dq_stride[1] + h * a.dq_stride[3] + l32;
  for (int c = wave; c < nb; c += nth / 64) {
#pragma unroll
    for (int rg = 0; rg < 4; ++rg) {
      const f32x4 v = blk[c].dq[64 * rg + lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int qq = 32 * c + 8 * rg + 4 * g + e;
        if (qq < N) dqg[(int64_t)qq * a.dq_stride[2]] = TypeOps<T>::from_f32(v[e] * a.scale);
      }
    }
  }
}

template <typename T, bool HAS_BIAS, int KB>
int launch_bwd_fused(const gnn_triattn_bwd_args& a, hipStream_t stream) {
  const void* fn = (const void*)bwd_fused_row_kernel<T, HAS_BIAS, KB>;
  const size_t smem = fused_lds((int)a.N);
  if (smem > 64 * 1024) (void)hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
  hipLaunchKernelGGL((bwd_fused_row_kernel<T, HAS_BIAS, KB>), dim3((uint32_t)(a.B * a.S * a.H)),
                     dim3(64 * fused_waves((int)a.N)), smem, stream, a);
  return (int)hipGetLastError();
}

template <typename T, bool HAS_BIAS>
int launch_bwd_row(const gnn_triattn_bwd_args& a, hipStream_t stream) {
  // (the fused kernel addresses the bias plane in unsigned 32 bits)
  if (a.N <= BWD_FUSED_MAX_N &&
      (!HAS_BIAS || (a.bias_stride[2] >= 0 && a.N * a.bias_stride[2] < ((int64_t)1 << 31))))
    return fused_kb((int)a.N) == 2 ? launch_bwd_fused<T, HAS_BIAS, 2>(a, stream)
                                   : launch_bwd_fused<T, HAS_BIAS, 1>(a, stream);
  const int64_t ntiles = (a.N + RT - 1) / RT;
  const dim3 grid((uint32_t)(a.B * a.S * a.H));
  const size_t smem_dq = DQ_HDR + 2 * (size_t)ntiles * RTILE;
  const size_t smem_dkdv = DKDV_HDR + 2 * (size_t)ntiles * RTILE;
  const void* fdq = (const void*)bwd_dq_row_kernel<T, HAS_BIAS>;
  const void* fdkdv = (const void*)bwd_dkdv_row_kernel<T, HAS_BIAS>;
  if (smem_dq > 64 * 1024) (void)hipFuncSetAttribute(fdq, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem_dq);
  if (smem_dkdv > 64 * 1024)
    (void)hipFuncSetAttribute(fdkdv, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem_dkdv);
  // dq first: it also writes Delta, which dk / dv reads
  hipLaunchKernelGGL((bwd_dq_row_kernel<T, HAS_BIAS>), grid, dim3(RNT), smem_dq, stream, a);
  hipLaunchKernelGGL((bwd_dkdv_row_kernel<T, HAS_BIAS>), grid, dim3(RNT), smem_dkdv, stream, a);
  return (int)hipGetLastError();
}

}  // namespace

bool triattn_bwd_row_applicable(const gnn_triattn_bwd_args& a) {
  return (a.dtype == GNN_BF16 || a.dtype == GNN_F16) && a.D == 32 && a.N >= 1 && a.N <= BWD_ROW_MAX_N &&
         a.B * a.S * a.H < ((int64_t)1 << 31);
}

int triattn_bwd_row_dq_dkdv(const gnn_triattn_bwd_args& a, hipStream_t stream) {
  if (a.dtype == GNN_BF16) return a.bias ? launch_bwd_row<bf16, true>(a, stream) : launch_bwd_row<bf16, false>(a, stream);
  return a.bias ? launch_bwd_row<f16, true>(a, stream) : launch_bwd_row<f16, false>(a, stream);
}

}  // namespace gnn
