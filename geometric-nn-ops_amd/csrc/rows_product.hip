// Products over the rows of two pixel-major tensors, C[o][i] = sum_m d[m][o] t[m][i]: the weight
// gradients of the linear layers of the multiplicative update (d the gradient of a layer's output,
// t its input, m the B N^2 pixels), and the ordered sum of partial results that they and the other
// backward kernels leave.
//
// The reference has no kernel for either: its gradients are autograd through F.linear
// (geometric_nn_ops_torch/triangle/_reference/trimul.py:85-97).
//
// rows_product_kernel. The output is small (4 c_hidden + c_z by c_z) and the contraction long (10^4
// to 10^6 rows), so the rows are cut into slices and a workgroup takes one 128 x 128 output block
// of one slice, leaving an fp32 partial; the slices of a block are added in a fixed order by
// reduce_parts_kernel. 4 waves of 64 x 64. Both operands are staged as they are stored, 128 columns
// of RS rows a stage, by global_load_lds (STAGES - 1 stages in flight, one barrier per stage), and the
// MFMA fragments are read down the columns: 16-bit types with ds_read_b64_tr_b16 (4 consecutive
// rows of a column per read, 16 rows per MFMA), fp32 as plain dwords (one row per lane half, 2 rows
// per 32x32x2 MFMA). Rows of LDS are 256 or 512 bytes, a multiple of the banks, so the rows that one
// read spans would collide: the source address of each lane permutes the row's 16-byte chunks
// (16-bit: 64-byte column blocks XOR row % 4; fp32: 128-byte halves XOR row % 2). The blocks of a
// slice follow each other on one XCD, whose L2 then serves t (and a 128-column block of d is read
// once); bound by HBM for 16-bit types and by the fp32 matrix rate for fp32.
// M = 384^2, [640 x 128] + [128 x 128], bf16: 66 us and 13 for the ordered sum, against 175 for the vendor's
// batched products on 64 slices and their sums; M = 201^2 fp32: 75 + 13 against 352 (an odd row count
// has no equal slices, and one vendor product of so few outputs leaves most CUs idle).
#include <algorithm>

#include "gnn_common.hpp"
#include "gnn_internal.hpp"

namespace gnn {

namespace {

constexpr int RP_NT = 256;     // 4 waves
constexpr int RP_BLK = 128;    // output block edge
// Workgroups per CU that the slice count aims at: two with 64 KB of stages each (bf16, M = 384^2,
// with launch: 77 us; one 81, three with 48 KB 83; five stages 77).
constexpr int RP_WGS = 2;
// Rows per slice at least: shorter ones cost more in partials than they save. fp32 goes down to 64 rows
// before it takes less than 32 slices, for shorter sums (1024 rows: 15.1 us with the ordered sum, at 128
// 16.1; 4096 rows stay at 128 with 22.6 us, at 64 24.3)
constexpr int RP_MIN_ROWS = 256, RP_MIN_ROWS_F32 = 64, RP_FULL_ROWS_F32 = 128;

template <typename T>
struct RowsProduct {
  static constexpr int STAGES = 4;
  static constexpr int RS = sizeof(T) == 2 ? 32 : 16;           // rows per stage
  static constexpr int ROWB = RP_BLK * (int)sizeof(T);          // bytes per LDS row
  static constexpr int OP_BYTES = RS * ROWB;                    // one operand's stage: 8 KB
  static constexpr int STAGE_BYTES = 2 * OP_BYTES;
  static constexpr int RPI = 1024 / ROWB;                       // rows per DMA instruction: 4 or 2
  static constexpr int Q = OP_BYTES / 1024 / 4;                 // DMA instructions per wave and operand: 2
  static constexpr int LDS = STAGES * STAGE_BYTES;
};

typedef __attribute__((address_space(3))) void lds_void_t;

template <int N_>
__device__ __forceinline__ void wait_vm_lgkm0() {
  static_assert(N_ >= 0 && N_ < 16, "vmcnt immediate");
  __builtin_amdgcn_s_waitcnt(0x070 | N_);  // vmcnt(N_) expcnt(7) lgkmcnt(0)
}

// The fragments of a 16-bit stage: two column blocks of each operand, two k-steps, each two
// transposed reads 8 rows apart (rows of 256 bytes). Waits for the data (see lds_addr).
template <typename V8>
__device__ __forceinline__ void read_stage16(const uint32_t (&ax)[2], const uint32_t (&ay)[2], V8 (&x)[2][2],
                                             V8 (&y)[2][2]) {
  static_assert(sizeof(V8) == 16, "8 16-bit values");
  uint64_t r[16];
  asm volatile(
      "ds_read_b64_tr_b16 %0, %16\n\tds_read_b64_tr_b16 %1, %16 offset:2048\n\t"
      "ds_read_b64_tr_b16 %2, %17\n\tds_read_b64_tr_b16 %3, %17 offset:2048\n\t"
      "ds_read_b64_tr_b16 %8, %18\n\tds_read_b64_tr_b16 %9, %18 offset:2048\n\t"
      "ds_read_b64_tr_b16 %10, %19\n\tds_read_b64_tr_b16 %11, %19 offset:2048\n\t"
      "ds_read_b64_tr_b16 %4, %16 offset:4096\n\tds_read_b64_tr_b16 %5, %16 offset:6144\n\t"
      "ds_read_b64_tr_b16 %6, %17 offset:4096\n\tds_read_b64_tr_b16 %7, %17 offset:6144\n\t"
      "ds_read_b64_tr_b16 %12, %18 offset:4096\n\tds_read_b64_tr_b16 %13, %18 offset:6144\n\t"
      "ds_read_b64_tr_b16 %14, %19 offset:4096\n\tds_read_b64_tr_b16 %15, %19 offset:6144\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5]), "=&v"(r[6]), "=&v"(r[7]),
        "=&v"(r[8]), "=&v"(r[9]), "=&v"(r[10]), "=&v"(r[11]), "=&v"(r[12]), "=&v"(r[13]), "=&v"(r[14]),
        "=&v"(r[15])
      : "v"(ax[0]), "v"(ax[1]), "v"(ay[0]), "v"(ay[1])
      : "memory");
  typedef uint64_t u64x2_t __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int kk = 0; kk < 2; ++kk)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      x[kk][b] = __builtin_bit_cast(V8, (u64x2_t{r[4 * kk + 2 * b], r[4 * kk + 2 * b + 1]}));
      y[kk][b] = __builtin_bit_cast(V8, (u64x2_t{r[8 + 4 * kk + 2 * b], r[8 + 4 * kk + 2 * b + 1]}));
    }
}

struct RowsProductGrid {
  int nb[GNN_ROWS_PRODUCT_MAX];  // output blocks of each product
  int total;                     // of all
  int64_t rps;                   // rows per slice
};

template <typename T>
__global__ __launch_bounds__(RP_NT, RP_WGS) void rows_product_kernel(const gnn_rows_product_args a, const RowsProductGrid G) {
  typedef RowsProduct<T> Cfg;
  __shared__ __align__(16) unsigned char smem[Cfg::LDS];
  const uint32_t w = xcd_remap(blockIdx.x, gridDim.x);
  int blk = (int)(w % (uint32_t)G.total), pi = 0;
  const int64_t slice = w / (uint32_t)G.total;
  while (blk >= G.nb[pi]) blk -= G.nb[pi++];
  const gnn_rows_product_item& P = a.p[pi];
  const int O = (int)P.O, I = (int)P.I;
  const int nbi = (I + RP_BLK - 1) / RP_BLK;
  const int o0 = blk / nbi * RP_BLK, i0 = blk % nbi * RP_BLK;
  const int64_t m0 = slice * G.rps, m1 = min(m0 + G.rps, a.rows);
  const int nkt = (int)((m1 - m0 + Cfg::RS - 1) / Cfg::RS);

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, g = lane >> 5;
  const int wm = wave >> 1, wn = wave & 1;

  // DMA: instruction q of a wave moves RPI rows of 128 columns; lane -> row lane / CPR, stored chunk
  // lane % CPR, which holds the row's chunk (lane % CPR) ^ swizzle(row). Columns past the operand's
  // repeat its last chunk and rows past the end the last row (in bounds; zeroed or never stored).
  constexpr int CPR = Cfg::ROWB / 16, EPC = 16 / (int)sizeof(T);
  const int drow = lane / CPR, dchunk = lane % CPR;
  auto swz = [](int row) { return sizeof(T) == 2 ? (row & 3) << 2 : (row & 1) << 3; };
  auto issue = [&](int kt) {
    unsigned char* st = smem + (kt % Cfg::STAGES) * Cfg::STAGE_BYTES;
#pragma unroll
    for (int q = 0; q < Cfg::Q; ++q) {
      const int ins = Cfg::Q * wave + q, r = Cfg::RPI * ins + drow;
      const int64_t m = min(m0 + (int64_t)kt * Cfg::RS + r, a.rows - 1);
      const int c = (dchunk ^ swz(r)) * EPC;
      __builtin_amdgcn_global_load_lds((const void*)((const T*)P.d + m * P.d_ld + min(o0 + c, O - EPC)),
                                       (lds_void_t*)(st + ins * 1024), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((const void*)((const T*)P.t + m * P.t_ld + min(i0 + c, I - EPC)),
                                       (lds_void_t*)(st + Cfg::OP_BYTES + ins * 1024), 16, 0, 0);
    }
  };

  // fp32: two sums, of the even and the odd row pairs, added at the end: slices of 128 rows are 1.47e-7
  // off, in one sum 2.04e-7 (the vendor's products and sums over 64 slices lay between: weight gradients
  // at N = 64, c_z = c_hidden = 128 4.0e-7, here 3.9e-7, with one sum 4.3e-7)
  f32x16 acc[2][2], odd[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[x][y][r] = odd[x][y][r] = 0.f;

#pragma unroll
  for (int st = 0; st < Cfg::STAGES - 1; ++st)
    if (st < nkt) issue(st);
  for (int kt = 0; kt < nkt; ++kt) {
    // this wave's DMA of stage kt has landed and its reads of stage kt - 1 have returned; after
    // the barrier every wave's part is in LDS and the buffer of stage kt - 1 is free
    const int ahead = min(Cfg::STAGES - 2, nkt - 1 - kt);
    if (ahead >= 2)
      wait_vm_lgkm0<4 * Cfg::Q>();
    else if (ahead == 1)
      wait_vm_lgkm0<2 * Cfg::Q>();
    else
      wait_vm_lgkm0<0>();
    asm volatile("s_barrier" ::: "memory");
    unsigned char* sx = smem + (kt % Cfg::STAGES) * Cfg::STAGE_BYTES;
    const int valid = (int)min<int64_t>(Cfg::RS, m1 - m0 - (int64_t)kt * Cfg::RS);
    if (valid < Cfg::RS) {  // uniform; the last stage of a slice: rows past its end are zeros
      typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
      for (int b = valid * Cfg::ROWB + 16 * tid; b < Cfg::OP_BYTES; b += 16 * RP_NT) {
        *reinterpret_cast<u32x4_t*>(sx + b) = u32x4_t{0u, 0u, 0u, 0u};
        *reinterpret_cast<u32x4_t*>(sx + Cfg::OP_BYTES + b) = u32x4_t{0u, 0u, 0u, 0u};
      }
      __syncthreads();
    }
    if (kt + Cfg::STAGES - 1 < nkt) issue(kt + Cfg::STAGES - 1);
    const unsigned char* sy = sx + Cfg::OP_BYTES;
    if constexpr (sizeof(T) == 2) {
      typedef typename TypeOps<T>::V8 V8;
      // column block b (32 columns), k-step kk: lane reads rows 16 kk + 4 g + q and 8 further
      // down, 4 columns, and receives 4 rows of its own column
      const int q = (lane & 15) >> 2;
      const int off = (4 * g + q) * Cfg::ROWB + 32 * ((lane >> 4) & 1) + 8 * (lane & 3);
      uint32_t ax[2], ay[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        ax[x] = lds_addr(sx + off + (((2 * wm + x) ^ q) << 6));
        ay[x] = lds_addr(sy + off + (((2 * wn + x) ^ q) << 6));
      }
      constexpr int KS = Cfg::RS / 16;
      V8 xf[KS][2], yf[KS][2];
      read_stage16(ax, ay, xf, yf);
#pragma unroll
      for (int kk = 0; kk < KS; ++kk)
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int y = 0; y < 2; ++y) Mma<T, PREC_NATIVE>::step(acc[x][y], xf[kk][x], yf[kk][y]);
    } else {
      // rows 2 kk + g: column 32 b + l32; the 128-byte block b of an odd row sits in the other half
      const int off = g * Cfg::ROWB + 4 * l32;
      auto col = [&](const unsigned char* s, int b, int kk) {
        return *reinterpret_cast<const float*>(s + off + 2 * kk * Cfg::ROWB + ((b ^ g) << 7));
      };
      constexpr int KS = Cfg::RS / 2;
      float xf[KS][2], yf[KS][2];
#pragma unroll
      for (int kk = 0; kk < KS; ++kk)
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          xf[kk][x] = col(sx, 2 * wm + x, kk);
          yf[kk][x] = col(sy, 2 * wn + x, kk);
        }
#pragma unroll
      for (int kk = 0; kk < KS; ++kk)
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int y = 0; y < 2; ++y) {
            f32x16& s = kk % 2 ? odd[x][y] : acc[x][y];
            s = __builtin_amdgcn_mfma_f32_32x32x2f32(xf[kk][x], yf[kk][y], s, 0, 0, 0);
          }
    }
  }

  // acc[x][y][r] = C[o0 + 64 wm + 32 x + 8 (r / 4) + 4 g + r % 4][i0 + 64 wn + 32 y + l32]
  float* out = P.partial + slice * (int64_t)O * I;
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      const int i = i0 + 64 * wn + 32 * y + l32;
      if constexpr (sizeof(T) == 4) acc[x][y] += odd[x][y];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int o = o0 + 64 * wm + 32 * x + 8 * (r / 4) + 4 * g + (r % 4);
        if (o < O && i < I) out[(int64_t)o * I + i] = acc[x][y][r];
      }
    }
}

RowsProductGrid rows_product_grid(const gnn_rows_product_args& a) {
  RowsProductGrid G{};
  for (int i = 0; i < a.count; ++i) {
    G.nb[i] = (int)(((a.p[i].O + RP_BLK - 1) / RP_BLK) * ((a.p[i].I + RP_BLK - 1) / RP_BLK));
    G.total += G.nb[i];
  }
  if (a.slice_rows > 0) {
    G.rps = a.slice_rows;
    return G;
  }
  const int64_t want = std::max<int64_t>(1, (int64_t)RP_WGS * compute_units() / G.total);
  const int64_t least = a.dtype == GNN_F32
                            ? std::max<int64_t>(RP_MIN_ROWS_F32, std::min<int64_t>(a.rows / 32, RP_FULL_ROWS_F32))
                            : RP_MIN_ROWS;
  const int64_t rows = std::max<int64_t>((a.rows + want - 1) / want, least);
  G.rps = (rows + 31) / 32 * 32;
  return G;
}

// ---- ordered sums of partial results ----------------------------------------------------
// dst[e] = sum over p of src[p stride + e] for every segment, in the segment's dtype and a fixed
// order. Segments of few parts (the weight gradients' slices) take a thread per element; those of
// many parts over few elements (per-workgroup column sums) take 8 elements a block, whose 32 thread
// groups add the parts p, p + 32, ... and meet in LDS in group order. 8 loads in flight per thread.
constexpr int RD_NT = 256;
constexpr int RD_E = 8, RD_G = RD_NT / RD_E;
constexpr int RD_FEW = 128;  // parts up to which a thread adds an element alone

__host__ __device__ inline int64_t reduce_blocks(const gnn_reduce_segment& s) {
  const int e = s.parts <= RD_FEW ? RD_NT : RD_E;
  return (s.n + e - 1) / e;
}

// Eight running sums, added pairwise at the end: 128 parts are 0.9e-7 off, in one sum 2.0e-7
__device__ __forceinline__ float sum_parts(const float* src, int64_t stride, int64_t p, int64_t parts, int step) {
  constexpr int UN = 8;
  float s[UN];
#pragma unroll
  for (int k = 0; k < UN; ++k) s[k] = 0.f;
  for (; p + (UN - 1) * step < parts; p += UN * step) {
#pragma unroll
    for (int k = 0; k < UN; ++k) s[k] += src[(p + k * step) * stride];
  }
#pragma unroll
  for (int k = 0; k < UN - 1; ++k)
    if (p + k * step < parts) s[k] += src[(p + k * step) * stride];
  return ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
}

__global__ __launch_bounds__(RD_NT) void reduce_parts_kernel(const gnn_reduce_args a) {
  __shared__ float red[RD_G][RD_E + 1];
  int64_t b = blockIdx.x;
  int si = 0;
  for (int64_t nb; b >= (nb = reduce_blocks(a.seg[si])); ++si) b -= nb;
  const gnn_reduce_segment& S = a.seg[si];
  float sum;
  int64_t i;
  if (S.parts <= RD_FEW) {  // uniform
    i = b * RD_NT + threadIdx.x;
    if (i >= S.n) return;
    sum = sum_parts(S.src + i, S.stride, 0, S.parts, 1);
  } else {
    const int e = threadIdx.x % RD_E, grp = threadIdx.x / RD_E;
    i = b * RD_E + e;
    red[grp][e] = i < S.n ? sum_parts(S.src + i, S.stride, grp, S.parts, RD_G) : 0.f;
    __syncthreads();
    if (grp != 0 || i >= S.n) return;
    float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < RD_G; ++k) part[k % 4] += red[k][e];
    sum = (part[0] + part[1]) + (part[2] + part[3]);
  }
  if (S.dtype == GNN_F32)
    ((float*)S.dst)[i] = sum;
  else if (S.dtype == GNN_BF16)
    ((bf16*)S.dst)[i] = (bf16)sum;
  else
    ((f16*)S.dst)[i] = (f16)sum;
}

}  // namespace

int64_t rows_product_slices(const gnn_rows_product_args& a) {
  const RowsProductGrid G = rows_product_grid(a);
  return (a.rows + G.rps - 1) / G.rps;
}

int rows_product(const gnn_rows_product_args& a, hipStream_t st) {
  const RowsProductGrid G = rows_product_grid(a);
  const int64_t nblk = (a.rows + G.rps - 1) / G.rps * G.total;
  if (nblk >= ((int64_t)1 << 31)) return set_error(GNN_ERR_UNSUPPORTED, "rows_product: grid too large");
  const dim3 grid((uint32_t)nblk), blk(RP_NT);
  switch (a.dtype) {
    case GNN_BF16: hipLaunchKernelGGL(rows_product_kernel<bf16>, grid, blk, 0, st, a, G); break;
    case GNN_F16: hipLaunchKernelGGL(rows_product_kernel<f16>, grid, blk, 0, st, a, G); break;
    default: hipLaunchKernelGGL(rows_product_kernel<float>, grid, blk, 0, st, a, G); break;
  }
  return (int)hipGetLastError();
}

int reduce_parts(const gnn_reduce_args& a, hipStream_t st) {
  int64_t nblk = 0;
  for (int i = 0; i < a.count; ++i) nblk += reduce_blocks(a.seg[i]);
  if (nblk >= ((int64_t)1 << 31)) return set_error(GNN_ERR_UNSUPPORTED, "reduce_parts: grid too large");
  hipLaunchKernelGGL(reduce_parts_kernel, dim3((uint32_t)nblk), dim3(RD_NT), 0, st, a);
  return (int)hipGetLastError();
}

}  // namespace gnn
