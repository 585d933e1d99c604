// NVFP4 GEMM for prefill chunks (more than 8 activation rows) on gfx950 matrix cores.
//
// Semantics: y[m][n] = global * sum_g e4m3(scale[n][g]) * sum_{j in g} e2m1(code[n][j]) * x[m][j], the prefill
// branch of matmul_nvfp4 (engine/src/kernels.cpp:116-137; the CPU decodes each weight row to FP32 and dots it
// with every input row, so the two differ only in FP32 rounding order).
//
// Design (MI355X; compute-bound once a chunk has hundreds of rows, bound by latency and filling the chip below):
//  - Operands as in the GEMV: weights in the prepared 16 x 128 tiles, dequantised exactly to f16 in registers;
//    activations in 8-row groups of the GEMV's operand (each row as f16 high and low parts, columns 2 r and
//    2 r + 1), so v_mfma_f32_16x16x32_f16 keeps ~22 bits of every activation and accumulates in FP32. BF16 rows come
//    in 16-row blocks of one part each (exact: their low parts are zero), half the matrix ops and operand bytes. With
//    XTG_GEMM_PARTS=1 (or GemvCall::parts = 1) a pair of groups feeds one matrix op with the 16 rows' high parts
//    only (f16 activations: rel-L2 ~2e-4 against FP32, the precision class of the reference's FP16 GPU prefill GEMM);
//    the default keeps both parts.
//  - A work-group of WN x KS waves owns WN RB row-blocks (16 WN RB output rows) and CB blocks of 16 operand columns.
//    Its KS slices of WN waves take a KS-th of the k-tiles each and are added in LDS at the end, in slice order.
//    Each k-tile (128 inputs) a slice stages its operand tile (4 KiB a block) in LDS by direct global-to-LDS loads,
//    double-buffered; each wave dequantises its RB weight tiles once, in registers, and runs them against all CB blocks:
//    4 RB CB matrix ops. Larger RB saves LDS reads, larger CB dequantisation, and both bytes loaded; smaller tiles and
//    more slices fill the chip when rows are few: gemm_cost chooses. In LDS the four chunks of an operand column are
//    rotated by half the column's index, so that the 16 lanes that read 16 columns at once touch every bank, while
//    each quad of lanes still loads 64 consecutive bytes.
//  - What bounds it, 16384 x 3072 at 512 rows (in the kernel 88 us, 103 GFLOP issued at 1.17 PFLOP/s; the register-staged
//    kernel before, 112 us): timing-only copies of a form that took 98 us took 62 us with the matrix ops alone (1.68
//    PFLOP/s; a large library f16 product reaches 1.4-1.57 here), 70 us with the LDS reads, 80 us with the
//    dequantisation too, and the loads made the rest.
//  - Tiles are dealt so that work-group i, which runs on XCD i mod 8, gets a contiguous run of tiles: the
//    work-groups of one XCD share weight tiles (consecutive m-tiles of one n-tile) in that XCD's L2.
#include <algorithm>
#include <cstdio>
#include <cstdlib>

#include "common.hpp"
#include "kernels.hpp"
#include "nvfp4.hpp"

namespace xtg::hip {

namespace {
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
}  // namespace

struct GemmArgs {
  const uint8_t* tiles[4];
  int nb[4];
  int n[4];
  float global[4];
  long long y_off[4];
  const float* col_scale[4];
  int tile_end[4];   // cumulative (n-tile x m-tile) counts per weight
  int nw, kt, m, groups, blocks, mtiles;   // groups of 8 rows, blocks of 16 operand columns
  int x16;           // PARTS = 1: the operand is stored in 16-row blocks of one part each (prep_x16)
  int vec;           // every output row starts on 16 bytes: float4 stores
  const char* op;    // group (or 16-row block) g's operand at op + g * op_stride; its row factors xop_bytes later
  size_t op_stride, xop_bytes;
  float* y;
};

template <int RB>
struct WTile {
  u32x4 c[RB];
  uint32_t s[RB];
};

// Row-blocks rb0 .. rb0 + RB - 1 of k-tile kt (a row-block past the last reloads the last one).
template <int RB>
__device__ inline WTile<RB> load_w(const uint8_t* tiles, int nb, int kt_count, int rb0, int kt, int lane) {
  WTile<RB> w;
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    const uint8_t* tile = tiles + (size_t(min(rb0 + r, nb - 1)) * size_t(kt_count) + size_t(kt)) * kTileBytes;
    w.c[r] = *reinterpret_cast<const u32x4*>(tile + 16 * lane);
    w.s[r] = uint32_t(*reinterpret_cast<const uint16_t*>(tile + 1024 + 2 * lane));
  }
  return w;
}

// This wave's share of k-tile kt's operand (its slice's CB column blocks) from global memory straight into LDS.
template <int CB, int WN>
__device__ __forceinline__ void load_x(uint4* buf, const char* const (&src)[CB * 4 / WN], int kt, int wn) {
#pragma unroll
  for (int i = 0; i < CB * 4 / WN; ++i)
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[i] + size_t(kt) * 4096),
                                     (__attribute__((address_space(3))) void*)(buf + size_t(wn + i * WN) * 64), 16, 0, 0);
}

// One k-tile's matrix ops from its LDS buffer.
template <int RB, int CB>
__device__ __forceinline__ void mma_ktile(const uint4* buf, const WTile<RB>& w, f32x4 (&acc)[RB][CB], int rd) {
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    f16x8 A[RB];
#pragma unroll
    for (int r = 0; r < RB; ++r) A[r] = dequant8(w.c[r][s], scale_pair(w.s[r], s >> 1));
#pragma unroll
    for (int c = 0; c < CB; ++c) {
      const f16x8 B = __builtin_bit_cast(f16x8, buf[size_t(c * 4 + s) * 64 + size_t(rd)]);
#pragma unroll
      for (int r = 0; r < RB; ++r) acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[r], B, acc[r][c], 0, 0, 0);
    }
  }
}

// Every load of this wave done (those into LDS too) and every LDS read of it.
__device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0070); }   // vmcnt(0) lgkmcnt(0)

// The wave's k-tiles k0 .. k1 - 1 in `iters` rounds of the work-group, two LDS buffers in turn: the next k-tile's
// operand (into LDS) and weights (into registers) are in flight during this one's math. The buffers are restrict
// parameters: the compiler then knows that the loads in flight do not touch the buffer being read, and puts no wait
// for them before its reads. A round begins with a barrier: its k-tile is complete (every wave has waited for its own
// share), and every wave is done reading the buffer that is loaded next. (Three and four buffers, with the weights
// through LDS too and the loads two or three rounds ahead, measured 0-15 % slower at nearly every size: fewer
// work-groups fit a CU.)
template <int RB, int CB, int WN>
__device__ __forceinline__ void gemm_loop(uint4* __restrict__ b0, uint4* __restrict__ b1,
                                          const char* const (&src)[CB * 4 / WN], const uint8_t* tiles, int nb, int KT,
                                          int rb0, int k0, int k1, int iters, f32x4 (&acc)[RB][CB], int wn, int lane,
                                          int rd) {
  uint4* const buf[2] = {b0, b1};
  const int last = max(min(k1, KT) - 1, 0);   // loads past the slice's end reload its last k-tile
  load_x<CB, WN>(b0, src, min(k0, last), wn);
  WTile<RB> w = load_w<RB>(tiles, nb, KT, rb0, min(k0, last), lane);
  for (int it = 0; it < iters; it += 2) {
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      if (it + p >= iters) break;
      wait_loads();
      __syncthreads();
      const int nx = min(k0 + it + p + 1, last);
      const WTile<RB> n = load_w<RB>(tiles, nb, KT, rb0, nx, lane);
      load_x<CB, WN>(buf[p ^ 1], src, nx, wn);
      __builtin_amdgcn_sched_barrier(0);   // the loads go out before the math
      if (k0 + it + p < k1) mma_ktile<RB, CB>(buf[p], w, acc, rd);
      w = n;
    }
  }
}

template <int RB, int CB, int WN, int KS, int PARTS, int OCC>
__global__ void __launch_bounds__(WN* KS * 64, OCC) gemm_kernel(const GemmArgs a) {
  extern __shared__ uint4 xs[];   // [buffer][slice][column block][step][lane]
  constexpr int kBuf = CB * 4 * 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % WN, ks = wave / WN;
  const int col = lane & 15, grp = lane >> 4;
  // the entry that lane slot `lane` of a staged (block, step) holds: column lc, chunk lg
  const int lc = lane >> 2, lg = ((lane & 3) - (lc >> 1)) & 3;
  const int rd = 4 * col + ((grp + (col >> 1)) & 3);   // and the slot of this lane's operand entry

  // which tile: work-group i runs on XCD i % 8; give each XCD a contiguous run of the tile order
  const int total = a.tile_end[a.nw - 1];
  const int per = total / 8;
  const int id = int(blockIdx.x);
  const int t = id < per * 8 ? (id % 8) * per + id / 8 : id;
  int wi = 0;
  while (wi < a.nw - 1 && t >= a.tile_end[wi]) ++wi;
  const int lt = t - (wi ? a.tile_end[wi - 1] : 0);
  const int ntile = lt / a.mtiles, mtile = lt % a.mtiles;
  const int rb0 = ntile * (WN * RB) + wn * RB;
  const int c0 = mtile * CB;
  const int nb = a.nb[wi], KT = a.kt;
  const uint8_t* tiles = a.tiles[wi];

  // this slice's k-tiles, and the most of any slice (the iterations every wave makes)
  const int k0 = KT * ks / KS, k1 = KT * (ks + 1) / KS, iters = (KT + KS - 1) / KS;

  // the wave's share of a k-tile's operand: entry (c, s) = wn + i WN of the slice's CB column blocks x 4 steps
  const char* src[CB * 4 / WN];
#pragma unroll
  for (int i = 0; i < CB * 4 / WN; ++i) {
    const int e = wn + i * WN, c = e >> 2, s = e & 3;
    if (PARTS == 1 && !a.x16)   // the high parts of a pair of groups
      src[i] = a.op + size_t(min(2 * (c0 + c) + (lc >> 3), a.groups - 1)) * a.op_stride +
               (size_t(s) * 64 + size_t(8 * (lc & 7) + lg)) * 16;
    else
      src[i] = a.op + size_t(min(c0 + c, a.blocks - 1)) * a.op_stride + (size_t(s) * 64 + size_t(4 * lc + lg)) * 16;
  }
  f32x4 acc[RB][CB];
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int c = 0; c < CB; ++c) acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};

  gemm_loop<RB, CB, WN>(xs + ks * kBuf, xs + (KS + ks) * kBuf, src, tiles, nb, KT, rb0, k0, k1, iters, acc, wn, lane, rd);

  // the slices' sums, in slice order, into slice 0's waves
  if constexpr (KS > 1) {
    f32x4* red = reinterpret_cast<f32x4*>(xs);
    wait_loads();   // the last round's prefetch has landed before the barrier below
#pragma unroll
    for (int s = 1; s < KS; ++s) {
      __syncthreads();
      if (ks == s) {
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
          for (int c = 0; c < CB; ++c) red[(size_t(wn) * RB * CB + size_t(r * CB + c)) * 64 + size_t(lane)] = acc[r][c];
      }
      __syncthreads();
      if (ks == 0) {
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
          for (int c = 0; c < CB; ++c) acc[r][c] += red[(size_t(wn) * RB * CB + size_t(r * CB + c)) * 64 + size_t(lane)];
      }
    }
    if (ks != 0) return;
  }

  // lane (grp, col) holds rows 4 grp .. 4 grp + 3 of its row-block for operand column col; PARTS = 2: columns 2 j
  // and 2 j + 1 (neighbour lanes) are row j's high and low parts; PARTS = 1: column col is row col of the pair
  const int n = a.n[wi];
  const float glob = a.global[wi];
  const float* cs = a.col_scale[wi];
#pragma unroll
  for (int c = 0; c < CB; ++c) {
    const int mrow = (c0 + c) * (PARTS == 1 ? 16 : 8) + (PARTS == 1 ? col : col >> 1);
    const bool row_ok = mrow < a.m;
    const int xrow = row_ok ? mrow : 0, per = a.x16 ? 16 : kMaxRows;   // rows per stored block
    const float xinv = reinterpret_cast<const float*>(a.op + size_t(xrow / per) * a.op_stride + a.xop_bytes)[xrow % per];
    const float f = glob * xinv;
    float* yp = a.y + a.y_off[wi] + (long long)mrow * n;
    constexpr int RS = PARTS == 1 || RB % 2 == 1 ? 1 : 2;   // two parts: the row's two lanes take a row-block each
#pragma unroll
    for (int r = 0; r < RB; r += RS) {
      f32x4 v = acc[r][c];
      int rb = rb0 + r;
      bool mine = row_ok;
      if constexpr (PARTS == 2) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += dpp<kDppXor1>(v[e]);
        if constexpr (RS == 2) {
          f32x4 u = acc[r + 1][c];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            u[e] += dpp<kDppXor1>(u[e]);
            v[e] = (col & 1) ? u[e] : v[e];
          }
          rb += col & 1;
        } else {
          mine = mine && (col & 1) == 0;
        }
      }
      const int n0 = rb * kTileRows + 4 * grp;
      if (mine && rb < nb) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] *= f;
        if (cs) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] *= n0 + e < n ? cs[n0 + e] : 0.f;
        }
        if (a.vec) {
          if (n0 < n) *reinterpret_cast<f32x4*>(yp + n0) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n0 + e < n) yp[n0 + e] = v[e];
        }
      }
    }
  }
}

// A launch shape, and the waves per SIMD that its registers allow.
struct GemmShape {
  int rb, cb, wn, ks, wps;
};
using GemmFn = void (*)(const GemmArgs);
#define XTG_GEMM_SHAPES(F)                                                                                   \
  F(4, 8, 4, 1, 2) F(4, 6, 4, 1, 2) F(4, 4, 4, 1, 3) F(4, 4, 4, 2, 3) F(3, 4, 4, 2, 4) F(2, 4, 4, 2, 5)         \
  F(4, 2, 4, 2, 4) F(2, 2, 4, 2, 7) F(1, 4, 4, 2, 8) F(1, 2, 4, 2, 8) F(1, 2, 4, 4, 8) F(1, 2, 2, 4, 8)
static const GemmShape kShapes[] = {
#define XTG_GEMM(R, C, W, K, O) {R, C, W, K, O},
    XTG_GEMM_SHAPES(XTG_GEMM)
#undef XTG_GEMM
};
static GemmFn gemm_fn(const GemmShape& g, int parts) {
#define XTG_GEMM(R, C, W, K, O)                        \
  if (g.rb == R && g.cb == C && g.wn == W && g.ks == K) \
    return parts == 1 ? gemm_kernel<R, C, W, K, 1, 2> : gemm_kernel<R, C, W, K, 2, 2>;
  XTG_GEMM_SHAPES(XTG_GEMM)
#undef XTG_GEMM
  return nullptr;
}

// The time of a launch in a shape, in us, from a model fitted to 62 sizes (9 to 2048 rows, 1040 to 8192 inputs, 1720
// to 16384 outputs, one and two parts) in 21 shapes: a CU's share of the work-groups runs in batches of what fits
// it; a batch's k-tile takes the work of its work-groups (matrix ops on the SIMD's queue and KiB loaded), which a CU
// with few waves overlaps less, or a round trip at least; adding up the K slices costs time too. Over 200 sizes (9 to
// 2048 rows of 10 products, FP32 and BF16) the shape with the least modelled time costs 2.4 % on average over the fastest
// one, 16 % at worst; with the rule before (by tile counts, and the kernel before) 3072 x 4096 took 27.7 us at 37 rows,
// 16384 x 3072 took 119.8 us at 512 rows and 2560 x 7168 in BF16 took 137.6 us at 1500 rows (whole calls), where now they
// take 12.8, 88.5 and 67.8 us.
static double gemm_cost(const GemvCall& c, const GemmShape& g, int blocks, int kt) {
  const int mt = (blocks + g.cb - 1) / g.cb, waves = g.wn * g.ks;
  long wgs = 0;
  for (int i = 0; i < c.nw; ++i) wgs += long((c.w[i]->nb + g.wn * g.rb - 1) / (g.wn * g.rb)) * mt;
  const int fit = std::max(1, std::min(160 / (8 * g.ks * g.cb), 4 * g.wps / waves));   // work-groups a CU holds
  const long per_cu = (wgs + 255) / 256;
  const double work = 0.0076 * g.rb * g.cb * waves + 0.0083 * (4.0 * g.ks * g.cb + 1.125 * g.rb * waves) + 0.0085 * waves;
  auto ktile = [&](long n) { return std::max(0.4, n * work) + 0.58 * 4.0 * work / waves; };
  const int rounds = (kt + g.ks - 1) / g.ks;
  double t = 0.1 * (g.ks - 1) * g.rb * g.cb + double(per_cu / fit) * rounds * ktile(fit);
  if (per_cu % fit) t += rounds * ktile(per_cu % fit);
  return t;
}

static std::string run_gemm(const GemvCall& c, const GemmShape& g, int parts, hipStream_t stream);

std::string launch_gemm(const GemvCall& c, hipStream_t stream) {
  XTG_CHECK(c.nw >= 1 && c.nw <= 4, "gemm: %d weights (1..4)", c.nw);
  XTG_CHECK(c.m >= 1, "gemm: %d rows", c.m);
  int parts = c.x16 ? 1 : c.parts;
  if (const char* env = c.x16 ? nullptr : std::getenv("XTG_GEMM_PARTS")) parts = std::atoi(env);
  XTG_CHECK(parts == 1 || parts == 2, "gemm: %d operand parts (1 or 2)", parts);
  const int groups = (c.m + kMaxRows - 1) / kMaxRows;
  const int blocks = parts == 1 ? (groups + 1) / 2 : groups;   // operand blocks of 16 columns
  const GemmShape* g = nullptr;
  // XTG_GEMM_SHAPE=RB,CB[,WN,KS] fixes the launch shape, for experiments
  if (const char* env = std::getenv("XTG_GEMM_SHAPE")) {
    int r = 0, cb = 0, wn = 0, ks = 0;
    const int n = std::sscanf(env, "%d,%d,%d,%d", &r, &cb, &wn, &ks);
    for (const GemmShape& s : kShapes)
      if (!g && n >= 2 && s.rb == r && s.cb == cb && (n < 4 || (s.wn == wn && s.ks == ks))) g = &s;
  }
  if (!g) {
    double best = 0;
    for (const GemmShape& s : kShapes) {
      const double t = gemm_cost(c, s, blocks, c.w[0]->kt);
      if (!g || t < best) {
        g = &s;
        best = t;
      }
    }
  }
  return run_gemm(c, *g, parts, stream);
}

static std::string run_gemm(const GemvCall& c, const GemmShape& g, int parts, hipStream_t stream) {
  const int kt = c.w[0]->kt;
  GemmArgs a{};
  a.groups = (c.m + kMaxRows - 1) / kMaxRows;
  a.blocks = parts == 1 ? (a.groups + 1) / 2 : a.groups;
  a.mtiles = (a.blocks + g.cb - 1) / g.cb;
  a.x16 = c.x16 ? 1 : 0;
  a.vec = reinterpret_cast<uintptr_t>(c.y) % 16 == 0;
  int end = 0;
  for (int i = 0; i < c.nw; ++i) {
    XTG_CHECK(c.w[i]->kt == kt, "gemm: input widths differ");
    a.tiles[i] = c.w[i]->tiles;
    a.nb[i] = c.w[i]->nb;
    a.n[i] = c.w[i]->n;
    a.global[i] = c.w[i]->global;
    a.y_off[i] = (long long)c.y_off[i];
    a.col_scale[i] = c.col_scale[i];
    if (c.w[i]->n % 4 != 0 || c.y_off[i] % 4 != 0) a.vec = 0;
    end += ((c.w[i]->nb + g.wn * g.rb - 1) / (g.wn * g.rb)) * a.mtiles;
    a.tile_end[i] = end;
  }
  for (int i = c.nw; i < 4; ++i) a.tile_end[i] = end;
  a.nw = c.nw;
  a.kt = kt;
  a.m = c.m;
  a.op = static_cast<const char*>(c.xop);
  a.op_stride = c.x16 ? op16_block_bytes(c.w[0]->k) : op_group_bytes(c.w[0]->k);
  a.xop_bytes = xop_bytes(c.w[0]->k);
  a.y = c.y;
  const dim3 grid{unsigned(end)}, block{unsigned(g.wn * g.ks * 64)};
  const GemmFn fn = gemm_fn(g, parts);
  const size_t lds = std::max<size_t>(size_t(2) * g.ks * g.cb * 4096, g.ks > 1 ? size_t(g.wn) * g.rb * g.cb * 1024 : 0);
  allow_lds(reinterpret_cast<const void*>(fn), lds);
  hipLaunchKernelGGL(fn, grid, block, lds, stream, a);
  HIP_CHECK(hipGetLastError());
  return strf(parts == 1 ? "gemm_kernel<%d, %d, %d, %d, f16>" : "gemm_kernel<%d, %d, %d, %d>", g.rb, g.cb, g.wn, g.ks);
}

}  // namespace xtg::hip
