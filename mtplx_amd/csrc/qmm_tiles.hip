// 4-bit affine quantized matmul past 64 rows (prompt chunks), gfx950.
//
//   y[m, n] = sum_k x[m, k] * (q[n, k] * s[n, k/gs] + b[n, k/gs])
//
// What bounds it: the matrix cores, once every weight is used by enough rows;
// in 64-row launches of qmm_rows_kernel each launch reads all weights again
// with a workgroup per 128 columns (136 for 17408) on 256 CUs. Here one launch
// covers all row tiles:
//  * a workgroup of 4 waves computes 64 rows x 128 columns, a wave 64 x 32 on
//    v_mfma_f32_32x32x16_bf16: per 64-k group 8 MFMAs (256 cycles) against 28
//    VALU instructions that unpack the weights and 32 that scale the group's
//    sums (240 cycles), which overlap between the two waves of a SIMD;
//  * x streams through an LDS double buffer quad by quad (256 k), weights
//    through a two-deep register ring from the tile-major packed layout 1, one
//    barrier per quad;
//  * the numerics are those of the other kernels: nibbles as the exact bf16
//    128 + q, each group's fp32 sum G scaled in fp32, and the bias term
//    sum_u (b_u - 128 s_u) * sum(x_u) in fp32: the group sums come from a pass
//    over x, split exactly into three bf16 (8 + 8 + 8 bits), and meet b and
//    -128 s, which are bf16 themselves, on the bf16 MFMA: all products exact,
//    accumulated in fp32, at half the cycles of the fp32 MFMA;
//  * workgroups of one column group follow each other on one XCD (workgroup b
//    runs on XCD b % 8), so the row tiles share its L2's weights;
//  * small grids are split by K (tiles_split), the parts' fp32 sums added in part
//    order by a second kernel.
// Measured: 512 rows, 17408 x 5120: 118-122 us (750-770 TFLOP/s; 272 in 64-row
// launches), 2048 rows: 453 us (806; 1080 then).
#include "qmv_args.hpp"

namespace mtp {

constexpr int kTiRows = 64;          // rows per workgroup
constexpr int kTiThreads = 256;
constexpr int kTiXBuf = kTiRows * 512;   // staged x of one quad
constexpr int kTiSBuf = kTiRows * 32;    // its group sums
constexpr int kTiLds = 2 * (kTiXBuf + kTiSBuf);

struct TilesParams {
  const uint16_t* x;
  const uint16_t* sums;    // [Q][M][16]: per half of a quad, its two groups' sums as (h, m, l, h, m, l, 0, 0)
  const uint32_t* w;
  uint16_t* y;
  int M, N, K, ldx, ldy;
  int row_tiles, groups;   // 64-row tiles; groups of four 32-column tiles
  float* part;             // [split][M][N] fp32 sums of the K parts (split > 1)
  int split;
};

// sums[q][m][8 half + ..]: each 64-k group's sum (fp32, added as the other
// kernels add it) as three bf16 that add up to it exactly.
__global__ __launch_bounds__(256) void tile_sums_kernel(const uint16_t* x, uint16_t* sums, int M, int Q, int ldx) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  const bf16x2_t one2 = __builtin_bit_cast(bf16x2_t, 0x3f803f80u);
  const int t = blockIdx.x * 256 + threadIdx.x;   // (m, q, half), half fastest
  if (t >= M * Q * 2) return;
  const int half = t & 1, q = (t >> 1) % Q, m = (t >> 1) / Q;
  const uint16_t* xr = x + (size_t)m * ldx + 256 * q + 128 * half;
  uint16_t o[8];
  o[6] = o[7] = 0;
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint4 c = *reinterpret_cast<const uint4*>(xr + 64 * g + 8 * j);
      s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, c.x), one2, s, false);
      s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, c.y), one2, s, false);
      s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, c.z), one2, s, false);
      s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, c.w), one2, s, false);
    }
    const uint16_t h = f2bf(s);
    const float r1 = s - bf2f(h);
    const uint16_t mm = f2bf(r1);
    o[3 * g] = h;
    o[3 * g + 1] = mm;
    o[3 * g + 2] = f2bf(r1 - bf2f(mm));
  }
  *reinterpret_cast<uint4*>(sums + ((size_t)q * M + m) * 16 + 8 * half) = *reinterpret_cast<const uint4*>(o);
}

struct TileQuad {
  uint4 w[4];
  uint4 sb;
};

__global__ __launch_bounds__(kTiThreads, 2) void qmm_tiles_kernel(TilesParams p) {
  extern __shared__ __align__(16) unsigned char lds[];   // x [2][64 rows][512 B], sums [2][64][32 B]
  const int i8 = blockIdx.x >> 3;
  const int rt = i8 % p.row_tiles;
  const int g = (i8 / p.row_tiles) * 8 + (blockIdx.x & 7);
  if (g >= p.groups) return;
  const int part = blockIdx.y;
  const int q0 = part * (p.K >> 8) / p.split;              // this part's first quad
  const int Q = (part + 1) * (p.K >> 8) / p.split - q0;    // and its quads (at least one)
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c32 = lane & 31, kq = lane >> 5;
  const int m0 = kTiRows * rt;
  const int M = p.M - m0 < kTiRows ? p.M - m0 : kTiRows;   // rows of this tile
  const int ct = 4 * g + wave;
  const bool has_tile = 32 * ct < p.N;
  const uint32_t* W = p.w + ((size_t)(has_tile ? ct : 0) * (p.K >> 8) + q0) * kPackQuadWords;
  const uint32_t* wl = W + lane * 4;
  const uint32_t* sl = W + 1024 + c32 * 4;
  const NibConsts nc = nib_consts();
  const uint32_t lds0 = lds_addr(lds);

  auto load_quad = [&](TileQuad& r, int q) {   // past the end: the last quad again, never used
    const size_t off = (size_t)(q < Q ? q : Q - 1) * kPackQuadWords;
#pragma unroll
    for (int u = 0; u < 4; ++u) r.w[u] = *reinterpret_cast<const uint4*>(wl + off + 256 * u);
    r.sb = *reinterpret_cast<const uint4*>(sl + off);
  };
  // x of quad q: wave instruction t holds rows 2 t, 2 t + 1 (16-byte piece kc of
  // row m at slot kc ^ (m & 15)); wave w takes t = w, w + 4, .., and waves 0 and 1
  // the sums of 32 rows each with one more.
  const uint16_t* xp[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int m = 2 * (wave + 4 * j) + (lane >> 5);
    xp[j] = p.x + (size_t)(m0 + (m < M ? m : M - 1)) * p.ldx + 256 * q0 + 8 * ((lane & 31) ^ (m & 15));
  }
  const int sm = 32 * (wave & 1) + (lane >> 1);   // waves 0 and 1: 32 rows each
  const uint16_t* sp = p.sums + ((size_t)q0 * p.M + m0 + (sm < M ? sm : M - 1)) * 16 + 8 * (lane & 1);
  auto stage = [&](int q) {
    if (q >= Q) return;   // uniform
    const uint32_t b = lds0 + (q & 1) * kTiXBuf;
#pragma unroll
    for (int j = 0; j < 8; ++j) dma16(xp[j] + 256 * q, b + 1024 * (wave + 4 * j));
    if (wave < 2) dma16(sp + (size_t)q * p.M * 16, lds0 + 2 * kTiXBuf + (q & 1) * kTiSBuf + 1024 * wave);
  };

  f32x16 acc[2];
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[0][r] = acc[1][r] = 0.f;

  auto compute = [&](const TileQuad& r, int b) {
    const unsigned char* xb = lds + b * kTiXBuf;
    const unsigned char* xs = lds + 2 * kTiXBuf + b * kTiSBuf;
    {
      // Bias: this half's two groups (u = 2 kq, 2 kq + 1) as 6 of the 8 k slots.
      const uint32_t sw = kq ? r.sb.y : r.sb.x, bw = kq ? r.sb.w : r.sb.z;
      const uint32_t nw = f2bf2(-128.f * __uint_as_float(sw << 16), -128.f * __uint_as_float(sw & 0xffff0000u));
      auto slots = [](uint32_t v) {   // (v0, v0, v0, v1, v1, v1, 0, 0)
        return __builtin_bit_cast(bf16x8, make_uint4(__builtin_amdgcn_perm(v, v, 0x01000100u), v,
                                                     __builtin_amdgcn_perm(v, v, 0x03020302u), 0u));
      };
      const bf16x8 bb = slots(bw), bs = slots(nw);
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(xs + (32 * rb + c32) * 32 + 16 * kq);
        acc[rb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, bs, acc[rb], 0, 0, 0);
        acc[rb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, bb, acc[rb], 0, 0, 0);
      }
    }
    const float sv[4] = {__uint_as_float(r.sb.x << 16), __uint_as_float(r.sb.x & 0xffff0000u),
                         __uint_as_float(r.sb.y << 16), __uint_as_float(r.sb.y & 0xffff0000u)};
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint32_t wv[4] = {r.w[u].x, r.w[u].y, r.w[u].z, r.w[u].w};
      f32x16 G[2];
#pragma unroll
      for (int r2 = 0; r2 < 16; ++r2) G[0][r2] = G[1][r2] = 0.f;
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) {
        const bf16x8 w = nibbles_to_bf16(wv[ii], nc);
        const int kc = 8 * u + 4 * kq + ii;
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
          const int m = 32 * rb + c32;
          const bf16x8 a = *reinterpret_cast<const bf16x8*>(xb + 512 * m + 16 * (kc ^ (m & 15)));
          G[rb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, w, G[rb], 0, 0, 0);
        }
      }
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int r2 = 0; r2 < 16; ++r2) acc[rb][r2] = fmaf(sv[u], G[rb][r2], acc[rb][r2]);
    }
  };

  TileQuad ring0, ring1;
  stage(0);
  asm volatile("" ::: "memory");
  load_quad(ring0, 0);
  load_quad(ring1, 1);
  // Quad q from ring slot cur and buffer q & 1. At the wait only the other ring
  // slot (5 loads) may be in flight; past the barrier every wave's x of quad q is in
  // LDS, and nobody reads the other buffer any more.
  auto step = [&](TileQuad& cur, int q) {
    asm volatile("" ::: "memory");   // (no load moves past the wait, which counts them)
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(5));
    lds_barrier();
    stage(q + 1);
    compute(cur, q & 1);
    asm volatile("" ::: "memory");
    load_quad(cur, q + 2);
  };
  // An odd last quad leaves the loop in its middle: with a path through the loop
  // that skips ring1, ring0's loads may be the newest that the compiler knows
  // of, and it waits for everything in flight (vmcnt(0), the DMAs just issued
  // among it) before it reads ring0.
  int q = 0;
  while (true) {
    step(ring0, q);
    if (q + 1 >= Q) break;
    step(ring1, q + 1);
    q += 2;
    if (q >= Q) break;
  }

  const int col = 32 * ct + c32;
  if (!has_tile || col >= p.N) return;
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int r2 = 0; r2 < 16; ++r2) {
      const int m = 32 * rb + 8 * (r2 >> 2) + 4 * kq + (r2 & 3);
      if (m >= M) continue;
      if (p.split > 1)
        p.part[((size_t)part * p.M + m0 + m) * p.N + col] = acc[rb][r2];
      else
        p.y[(size_t)(m0 + m) * p.ldy + col] = f2bf(acc[rb][r2]);
    }
}

// y = the K parts' sums, added in part order.
__global__ __launch_bounds__(256) void tile_parts_kernel(const float* part, uint16_t* y, long long n, int split) {
  for (long long i = blockIdx.x * 256ll + threadIdx.x; i < n; i += gridDim.x * 256ll) {
    float t = 0.f;
    for (int s = 0; s < split; ++s) t += part[s * n + i];
    y[i] = f2bf(t);
  }
}

}  // namespace mtp

using namespace mtp;

// K parts. A grid of fewer workgroups than CUs is split over them (128 rows,
// 5120 x 17408, 80 workgroups: 94.5 us whole, 44.4 in 3 parts; 65 rows, 1024 x
// 5120, 16 workgroups: 32.7, in 8 parts 16.0), two quads a part at least. One of
// one to two per CU takes the split with the least estimated time: a CU of the
// fullest XCD runs ceil(w s / CUs) parts of Q / s quads, 1.1 us each, and the
// parts cost a launch and a pass over their sums, 5 us and 8 bytes a sum at 5
// TB/s. Measured for one, two and three parts (K 1536 to 17408 of nine grids),
// it takes one within 2% of the best:
// 35 workgroups on an XCD's 32 CUs (448 rows, 5120 x 17408: 137, 125, 114 us; K
// 5120: 47.2, 48.1, 46.6), 40 (512 rows: 143, 129, 120; K 7168 62.8, 61.0, 59.3;
// K 5120 47.8, 48.7, 48.2), 48 (768 rows, 4096 x 17408: 150, 136, 146; K 7168
// 64.9, 65.1, 71.8), 60 (768 rows, 5120 x 17408: 160, 169, 174).
static int tiles_split(int M, int N, int K) {
  const long long blocks = (long long)cdiv(M, kTiRows) * cdiv(cdiv(N, 32), 4);
  const int cus = device_cus(), Q = K / 256;
  if (blocks >= 2 * cus) return 1;
  if (blocks >= cus) {
    const int w = cdiv(M, kTiRows) * cdiv(cdiv(cdiv(N, 32), 4), 8);   // workgroups on the fullest XCD
    auto us = [&](int s) {
      return 1.1 * Q * cdiv(8 * w * s, cus) / s + (s > 1 ? 5.0 + s * ((double)M * N) * 8.0 / 5e6 : 0.0);
    };
    const int s = us(2) < us(1) ? 2 : 1;
    return us(3) < us(s) ? 3 : s;   // (at most Q: below 3 quads the parts cost more than they can save)
  }
  long long s = cus / blocks;
  if (s > 8) s = 8;
  if (s > Q / 2) s = Q / 2;
  return s > 1 ? (int)s : 1;
}
static size_t tiles_sums_bytes(int M, int K) { return ((size_t)M * (K / 256) * 32 + 255) & ~(size_t)255; }

MTP_API size_t mtp_qmm_tiles_workspace_bytes(int M, int N, int K) {
  if (M < 1 || N < 1 || K < 256 || K % 256) return 0;
  const int s = tiles_split(M, N, K);
  return tiles_sums_bytes(M, K) + (s > 1 ? (size_t)s * M * N * 4 : 0);
}

MTP_API int mtp_qmm_affine4_tiles(const void* x, const void* w, void* y, int M, int N, int K, int group_size, void* ws,
                                  size_t ws_bytes, void* stream) {
  const char* who = "mtp_qmm_affine4_tiles";
  if (!x || !w || !y || M < 1 || N < 1 || K < 256 || K % 256 || ((uintptr_t)x & 15) || ((uintptr_t)w & 15)) {
    set_error("%s: need 16-byte aligned x and w, y, M, N >= 1, K a multiple of 256 (got M=%d N=%d K=%d)", who, M, N, K);
    return MTP_ERR_ARG;
  }
  if (group_size != 64 && group_size != 128) {   // (the pack holds a scale per 64-group for either)
    set_error("%s: group_size %d unsupported (64 or 128)", who, group_size);
    return MTP_ERR_UNSUPPORTED;
  }
  const size_t need = mtp_qmm_tiles_workspace_bytes(M, N, K);
  if (!ws || ws_bytes < need || ((uintptr_t)ws & 15)) {
    set_error("%s: a 16-byte aligned workspace of %zu B is needed, got %zu B", who, need, ws_bytes);
    return MTP_ERR_WORKSPACE;
  }
  TilesParams p = {};
  p.x = (const uint16_t*)x;
  p.sums = (const uint16_t*)ws;
  p.w = (const uint32_t*)w;
  p.y = (uint16_t*)y;
  p.M = M;
  p.N = N;
  p.K = K;
  p.ldx = K;
  p.ldy = N;
  p.row_tiles = cdiv(M, kTiRows);
  p.groups = cdiv(cdiv(N, 32), 4);
  p.split = tiles_split(M, N, K);
  p.part = reinterpret_cast<float*>(reinterpret_cast<unsigned char*>(ws) + tiles_sums_bytes(M, K));
  const long long blocks = 8ll * cdiv(p.groups, 8) * p.row_tiles;
  if (blocks > 0x7fffffffll || (long long)M * (K / 256) * 2 > 0x7fffff00ll) {
    set_error("%s: M=%d N=%d K=%d too large for one launch", who, M, N, K);
    return MTP_ERR_UNSUPPORTED;
  }
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(tile_sums_kernel, dim3(cdiv(M * (K / 256) * 2, 256)), dim3(256), 0, st, p.x, (uint16_t*)ws, M,
                     K / 256, K);
  (void)hipFuncSetAttribute((const void*)qmm_tiles_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kTiLds);
  hipLaunchKernelGGL(qmm_tiles_kernel, dim3((unsigned)blocks, p.split), dim3(kTiThreads), kTiLds, st, p);
  if (p.split > 1) {
    const long long n = (long long)M * N;
    const long long g = (n + 255) / 256;
    hipLaunchKernelGGL(tile_parts_kernel, dim3((unsigned)(g < 2048 ? g : 2048)), dim3(256), 0, st, p.part, p.y, n,
                       p.split);
  }
  return launch_check(who);
}
