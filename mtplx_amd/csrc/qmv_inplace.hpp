// Quantized matmul of a few rows over weights in the reference (MLX) layout,
// read in place: the routed experts of drop-in callers, and the formats that
// have no tile-major pack (8-bit, group 32).
//
//   y[m, n] = sum_k x[m, k] * (q[n, k] * s[n, k/gs] + b[n, k/gs])
//
// What bounds it: the weights are read once, so HBM does; a weight row is
// K * bits / 8 contiguous bytes, so lanes that each read their own row's
// 16-byte piece touch 32 or 64 cache lines per instruction and a quarter of
// each. Here 8 lanes read one row's whole 128-byte line, straight into LDS
// (no registers), and the MFMA operands come out of LDS:
//  * one wave streams "chunks" of 128 bytes (256 k of 4 bits, 128 k of 8) of 32
//    weight rows with the same k of x beside them into stages of its own. No
//    other wave reads a stage, so the stream needs no barrier; a stage's
//    operands go to registers and it is loaded again while they are computed
//    on. The waves of a workgroup split K by chunks (and the pair's matrices,
//    or two column groups, between them) and meet once per item (column tile
//    x row tile). One matrix has eight K parts whatever its rows: eight waves
//    with one each, or four with two (chunks of the one and of the other in
//    turn), and parts w and w + 4 are added before the four such sums are, in
//    order of w. So a row's output has the same bits whatever rows are beside
//    it (16 rows of 17408 x 5120, 8 bits, weights in the caches: 26.5 us; with
//    four parts in all, one per wave, 26.1, and other bits than the eight of
//    up to 4 rows). The experts have two parts;
//  * scales and biases of an item's columns come as whole rows, also straight
//    to LDS (up to 88 or 24 groups of a row at a time), an item ahead: fetched chunk
//    by chunk, every 4 bytes of them cost a cache line (8-bit, 32768 x 5120,
//    4 rows: 41.2 us against 36.1);
//  * 16-byte pieces of a line sit at slot piece ^ (row / 2 % 8), those of an x
//    row at slot piece ^ row (the loads are permuted, not the stores), so
//    operand reads of 16 rows spread over all 64 banks;
//  * v_mfma_f32_16x16x32_bf16 with A = x rows, B = weight columns. Within a
//    group, lane group g = l / 16 takes k [gs/4 * g, gs/4 * (g + 1)) in steps
//    of 8, so each lane's fields of a group are contiguous; x is read at the
//    same k. 4-bit fields become the exact bf16 128 + q (one AND-OR per pair),
//    8-bit fields the exact bf16 q; weights are never rounded;
//  * the group sums of x (the bias term) are one more MFMA per step with
//    B = 1: they come out in the layout of the products, in fp32;
//  * with at most 4 rows, x row m sits at A row 4m, so every lane finishes one
//    row's element per 16 columns; with more, row m sits at A row m.
// The items of one workgroup follow each other in the stream: the next item's
// first chunks are in flight while the last one's sums meet.
//
// Measured (MI355X, weights from HBM): 8-bit group 64, 17408 x 5120, 4 rows:
// 24 us (3.9 TB/s; 138 us with one lane per column on the VALU), 65536 x 5120:
// 66 us (5.4 TB/s). 256 experts of 2 x 1536 x 4096, 16 rows x 8 (59 of them
// with 1..4 rows): gate|up 90 us and down 48 us (4.4 and 4.2 TB/s) for those, 99
// and 55 with the others; 355 and 240 us before, each lane reading 16 bytes of
// its own row. A wave's own instructions bound it there: with one wave per SIMD, two,
// three or four stages all take 131 us (gate|up), with two waves 92.
#pragma once

#include "qmv_common.hpp"

#include <limits.h>

namespace mtp {

struct InplaceParams {
  const uint16_t* x;
  const uint8_t* w0;       // rows of K * bits / 8 bytes
  const uint8_t* w1;       // second matrix (fused SwiGLU pair), same shape
  const uint16_t* s0;
  const uint16_t* b0;
  const uint16_t* s1;
  const uint16_t* b1;
  uint16_t* y;
  float* yf;               // bf16-rounded fp32 output instead of y
  const float* xsums;      // chunk-sum table (mtp_chunk_sums), or null
  const uint32_t* rowmap;  // x row of output row i (null: i)
  const int32_t* expert_off;   // experts: rows of expert e are [off[e], off[e+1])
  const int32_t* active;       // [1 + E]: count, then the experts with rows; null: one matrix, M rows
  long long w_estride;     // bytes between experts' weights
  long long s_estride;     // scales between experts
  int M, N, K, ldx, ldy;
  int ntile;               // column tiles
};

constexpr int kInList = 128;    // experts listed in LDS at a time
template <int BITS, int GS, int R, bool DUAL, int NW, int KS, int ND>
struct InplaceShape {
  static constexpr int D = ND;                      // stages per wave
  static constexpr int KP = KS == 2 ? 2 : 8;        // K parts: chunk c of a scale segment is in part c % KP
  static constexpr int PW = KP / KS;                // parts per wave: its chunks take them in turn
  static_assert(KP % KS == 0 && PW <= 2, "one or two parts per wave");
  // Scale groups of one column staged at a time: a longer K takes its groups in
  // several segments. An LDS row is an odd number of 16-byte pieces, so 16
  // columns' reads fall in distinct banks. The experts' tiles of 16 rows stage
  // few groups and items, so that two workgroups (81 KB each) fit a CU, at
  // most 256 registers: their waves' own instructions bound them, and one wave
  // per SIMD leaves every wait open (256 experts of 1536 x 4096, 512 rows x 8:
  // 1366 us with 88 groups and one workgroup per CU, 1014 with 24 and two).
  static constexpr bool SMALL = R == 16 && ND == 1;
  static constexpr int GRP = SMALL ? 24 : 88;
  static constexpr int SROW = 2 * GRP;
  static constexpr int ITEMS = SMALL ? 16 : 32;     // items described in LDS at a time
  static constexpr int COLS = 32;                   // weight rows per wave
  static constexpr int CK = 1024 / BITS;            // k per chunk
  static constexpr int XB = CK * 2;                 // x bytes per row and chunk
  static constexpr int GPC = CK / GS;               // groups per chunk
  static constexpr int XR = R;                      // x rows staged (4 or 16)
  static constexpr int XI = XR * XB / 1024;         // x load instructions per chunk
  static constexpr int WI = COLS / 8;               // weight load instructions per chunk
  static constexpr int STAGE = COLS * 128 + XR * XB;
  static constexpr int SEG = GRP / GPC;         // chunks per scale segment
  static constexpr int TC = COLS * (NW / KS);         // weight rows per tile
  static constexpr int OC = DUAL ? TC / 2 : TC;       // output columns per tile
  static constexpr int SCAL = 2 * TC * SROW;       // one segment: scales [TC][row], then biases
  static constexpr int RED = 2 * NW * XR * COLS * 4;
  // What comes first in LDS: the experts listed, and the items described.
  struct Lists {
    int4 item[ITEMS];                // expert, column tile, first row, rows
    int rows[ITEMS][XR];             // x row of each staged row
    int e[kInList], r0[kInList], cum[kInList + 1];   // expert, its first row, row tiles before it
    int wcnt[NW], wtil[NW];          // per wave of the scan
  };
  static constexpr int LISTS = (sizeof(Lists) + 255) & ~255;
  static constexpr size_t lds() { return (size_t)LISTS + NW * D * STAGE + RED + 2 * SCAL; }
  static_assert(GRP % GPC == 0 && GRP % 8 == 0, "segments of whole chunks and 16-byte pieces");
  static_assert((GRP / 8) % 2 == 1, "odd rows");
  static_assert(XI >= 1, "a chunk of x is at least one load");
};

// GPC bf16 values in LDS, aligned to 2 * GPC bytes.
template <int GPC>
__device__ __forceinline__ void group_vals(const unsigned char* at, float (&o)[GPC]) {
  uint32_t v[GPC > 1 ? GPC / 2 : 1];
  if constexpr (GPC == 8) {
    const uint4 t = *reinterpret_cast<const uint4*>(at);
    v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
  } else if constexpr (GPC == 4) {
    const uint2 t = *reinterpret_cast<const uint2*>(at);
    v[0] = t.x; v[1] = t.y;
  } else if constexpr (GPC == 2) {
    v[0] = *reinterpret_cast<const uint32_t*>(at);
  } else {
    v[0] = *reinterpret_cast<const uint16_t*>(at);
  }
#pragma unroll
  for (int u = 0; u < GPC; ++u) o[u] = __uint_as_float((u & 1) ? (v[u >> 1] & 0xffff0000u) : (v[u >> 1] << 16));
}

// The work of one workgroup, number ``bid`` of the grid: all rows, or the rows
// of the experts with m_lo <= rows <= m_hi. Returns (to every thread) whether
// an expert has more rows than m_hi.
// VEC: scales straight to LDS, and x 16-byte aligned (else scales element by
// element, and x too where it is not aligned). XS: the bias term
// takes its group sums from the caller's chunk-sum table (p.xsums); those that
// take 128 s off the fields' 128 + q are the MFMA's as in the others.
template <int BITS, int GS, int R, bool DUAL, bool VEC, bool XS, int NW, int KS, int ND>
__device__ __forceinline__ bool inplace_body(const InplaceParams& p, unsigned char* const lds_base, int bid, int m_lo,
                                             int m_hi) {
  using S = InplaceShape<BITS, GS, R, DUAL, NW, KS, ND>;
  constexpr int COLS = S::COLS;
  static_assert(!DUAL || NW == 2 * KS, "the pair: half the waves on each matrix");
  constexpr int NT = NW * 64;
  constexpr int CT = COLS / 16;
  constexpr int RA = R == 4 ? 1 : 4;    // accumulators per 16 columns
  constexpr int SPG = GS / 32;          // MFMA steps per group
  constexpr int LPR = S::XB / 16;       // lanes per x row in a load
  constexpr int NL = S::WI + S::XI;     // loads per stage
  auto& L = *reinterpret_cast<typename S::Lists*>(lds_base);
  unsigned char* const smem = lds_base + S::LISTS;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kw = wave % KS, cg = wave / KS;   // K part; group of COLS weight rows (the pair: matrix)
  const int c16 = lane & 15, g = lane >> 4;
  const NibConsts nc = nib_consts();
  const int row_bytes = p.K * BITS / 8;
  const int Q = (p.K + S::CK - 1) / S::CK;
  const bool tail_k = (p.K % S::CK) != 0;
  const int sgroups = p.K / GS;
  const bool x_al = ((uintptr_t)p.x & 15) == 0;   // (rows are whole 64-byte steps apart)
  unsigned char* const stage0 = smem + (size_t)wave * S::D * S::STAGE;
  const uint32_t lds0 = lds_addr(stage0);
  float* const red = reinterpret_cast<float*>(smem + (size_t)NW * S::D * S::STAGE);
  unsigned char* const scal = smem + (size_t)NW * S::D * S::STAGE + S::RED;
  const uint32_t scal_lds = lds_addr(scal);
  const int nseg = (Q + S::SEG - 1) / S::SEG;
  // This wave's chunks of segment sg of an item: chunk SEG * sg + kw + KS * t.
  auto seg_chunks = [&](int sg) {
    const int n = Q - sg * S::SEG < S::SEG ? Q - sg * S::SEG : S::SEG;
    return n > kw ? (n - kw + KS - 1) / KS : 0;
  };

  // Lane constants of the loads: weights (row 8 i + lane / 8 of the tile, slot
  // lane % 8), x (row i * (64 / LPR) + lane / LPR, slot lane % LPR).
  const int w_piece = 16 * ((lane & 7) ^ (lane >> 4));   // (odd i: ^ 64)
  const int x_r = lane / LPR;
  const int x_slot = lane % LPR;

  // Scales: wave instruction i loads pieces 64 i .. + 63 of the buffer, piece
  // pc of row r (a column's scales, or its biases) at r * PR + pc.
  constexpr int PR = S::SROW / 16;
  constexpr int NI = 2 * S::TC * PR / 64;
  constexpr int NJ = (NI + NW - 1) / NW;
  static_assert(2 * S::TC * PR % 64 == 0, "whole wave instructions");
  int s_row[NJ], s_at[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int idx = 64 * (wave + NW * j) + lane;
    s_row[j] = idx / PR;
    s_at[j] = 8 * (idx - s_row[j] * PR);
  }

  // Operand addresses inside a stage. Weights: the lane's bytes of group u of
  // column 16 ct + c16 start at byte GB * u + GB/4 * g of the line, where GB =
  // GS * BITS / 8.
  constexpr int GB = GS * BITS / 8;
  auto w_addr = [&](int u, int o) {   // o: byte inside the lane's share
    const int byte = GB * u + (GB / 4) * g + o;
    return c16 * 128 + 16 * ((byte >> 4) ^ (c16 >> 1)) + (byte & 15);
  };
  const int a_row = R == 4 ? c16 >> 2 : c16;
  auto a_addr = [&](int u, int j) {   // x chunk of step j of group u
    const int ch = (GS / 8) * u + (GS / 32) * g + j;
    return COLS * 128 + a_row * S::XB + 16 * (ch ^ a_row);
  };

  // Base of experts [l0, l0 + kInList) of the active list, then their items.
  const int n_active = p.active ? p.active[0] : 1;
  int more = 0;   // an expert above m_hi
  for (int l0 = 0; l0 < n_active; l0 += kInList) {
    int n_list = 1;
    __syncthreads();
    if (p.active) {
      // The class's experts of this stretch in list order, with the running
      // count of their row tiles.
      const int l1 = n_active - l0 < kInList ? n_active - l0 : kInList;
      int nl = 0, nt = 0;
      for (int c0 = 0; c0 < l1; c0 += NT) {
        const int t = c0 + tid;
        int e = 0, r0 = 0, rows = 0;
        if (t < l1) {
          e = p.active[1 + l0 + t];
          r0 = p.expert_off[e];
          rows = p.expert_off[e + 1] - r0;
        }
        const bool in = t < l1 && rows >= m_lo && rows <= m_hi;
        const int above = __any(t < l1 && rows > m_hi) ? 1 << 16 : 0;
        const int tiles = in ? (rows + S::XR - 1) / S::XR : 0;
        const unsigned long long bal = __ballot(in);
        int inc = tiles;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
          const int v = __shfl_up(inc, off, 64);
          if (lane >= off) inc += v;
        }
        if (lane == 63) {
          L.wcnt[wave] = __popcll(bal) + above;
          L.wtil[wave] = inc;
        }
        __syncthreads();
        int at = nl, before = nt;
        for (int w = 0; w < NW; ++w) {
          const int c = L.wcnt[w] & 0xffff;
          if (w < wave) {
            at += c;
            before += L.wtil[w];
          }
          nl += c;
          nt += L.wtil[w];
          more |= L.wcnt[w] >> 16;
        }
        if (in) {
          const int i = at + __popcll(bal & ((1ull << lane) - 1ull));
          L.e[i] = e;
          L.r0[i] = r0;
          L.cum[i] = before + inc - tiles;
        }
        __syncthreads();
      }
      n_list = nl;
      if (tid == 0) L.cum[nl] = nt;
    } else if (tid == 0) {
      L.e[0] = 0;
      L.r0[0] = 0;
      L.cum[0] = 0;
      L.cum[1] = (p.M + S::XR - 1) / S::XR;
    }
    __syncthreads();
    const int n_items = L.cum[n_list] * p.ntile;

    // This workgroup's items bid, + gridDim.x, ..., S::ITEMS at a time.
    for (int i0 = bid; i0 < n_items; i0 += S::ITEMS * gridDim.x) {
      const int left = (n_items - i0 + (int)gridDim.x - 1) / (int)gridDim.x;
      const int ni = left < S::ITEMS ? left : S::ITEMS;
      __syncthreads();   // the last items' readers are done
      for (int j = tid; j < ni * S::XR; j += NT) {
        const int it = j / S::XR, r = j - it * S::XR;
        const int w = i0 + it * (int)gridDim.x;
        const int rt = w / p.ntile;   // row tile over all experts
        int lo = 0, hi = n_list;      // its expert: the last with cum <= rt
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (L.cum[mid] <= rt) lo = mid; else hi = mid;
        }
        const int e = L.e[lo];
        const int rows = p.active ? p.expert_off[e + 1] - L.r0[lo] : p.M;
        const int t0 = (rt - L.cum[lo]) * S::XR;
        const int n = rows - t0 < S::XR ? rows - t0 : S::XR;
        const int row = L.r0[lo] + t0 + (r < n ? r : n - 1);
        if (r == 0) L.item[it] = make_int4(e, w - rt * p.ntile, L.r0[lo] + t0, n);
        L.rows[it][r] = p.rowmap ? (int)p.rowmap[row] : row;
      }
      __syncthreads();

      // Prefetch iterator: item pf_it, segment pf_sg, chunk number pf_t of this
      // wave there.
      int pf_it = 0, pf_sg = 0, pf_t = 0, pf_n = 0;
      const uint8_t* w_base = nullptr;
      uint32_t w_off[S::WI];
      const uint16_t* x_ptr[S::XI];
      auto set_item = [&](int it) {
        const int e = __builtin_amdgcn_readfirstlane(L.item[it].x);
        const int tile = __builtin_amdgcn_readfirstlane(L.item[it].y);
        const int n0 = tile * S::OC + (DUAL ? 0 : cg * COLS);
        w_base = (DUAL && cg ? p.w1 : p.w0) + e * p.w_estride;
#pragma unroll
        for (int i = 0; i < S::WI; ++i) {
          const int col = n0 + 8 * i + (lane >> 3);
          w_off[i] = (uint32_t)((col < p.N ? col : p.N - 1) - tile * S::OC) * (uint32_t)row_bytes;
        }
        w_base += (long long)(tile * S::OC) * row_bytes;
#pragma unroll
        for (int i = 0; i < S::XI; ++i) {
          const int r = i * (64 / LPR) + x_r;
          x_ptr[i] = p.x + (size_t)L.rows[it][r] * p.ldx;
        }
      };
      // The scales and biases of segment sg of item it, into buffer (it * nseg
      // + sg) % 2, by the whole workgroup: 16-byte pieces straight to LDS (VEC;
      // a row's pieces past its last repeat it), else element by element.
      auto load_scales = [&](int it, int sg) {
        const int4 im = L.item[it];
        const int n0 = im.y * S::OC;
        const int g0 = sg * S::GRP;
        const int ng = sgroups - g0 < S::GRP ? sgroups - g0 : S::GRP;
        const int buf = ((it * nseg + sg) & 1) * S::SCAL;
        const size_t eo = (size_t)(im.x * p.s_estride) + g0;
        if constexpr (VEC) {
#pragma unroll
          for (int j = 0; j < NJ; ++j) {
            if (wave + NW * j < NI) {   // (the last round's waves may have none)
              const int c = s_row[j] % S::TC;
              const bool up = DUAL && c >= S::OC;
              const uint16_t* const src = s_row[j] >= S::TC ? (up ? p.b1 : p.b0) : (up ? p.s1 : p.s0);
              const int cc = DUAL ? c % S::OC : c, last = p.N - 1 - n0;
              const int at = s_at[j] < ng ? s_at[j] : ng - 8;
              dma16(src + (eo + (size_t)n0 * sgroups) + (size_t)(cc < last ? cc : last) * sgroups + at,
                    scal_lds + buf + 1024 * (wave + NW * j));
            }
          }
        } else {
          // (groups past K, of a last chunk that is not whole, as zero)
          const int np = S::GPC * Q - g0 < S::GRP ? S::GPC * Q - g0 : S::GRP;
          for (int t = tid; t < 2 * S::TC * np; t += NT) {
            const int row = t / np, u = t - row * np;
            const int c = row % S::TC;
            const int col = n0 + (DUAL ? c % S::OC : c);
            const bool up = DUAL && c >= S::OC;
            const uint16_t* const src = row >= S::TC ? (up ? p.b1 : p.b0) : (up ? p.s1 : p.s0);
            *reinterpret_cast<uint16_t*>(scal + buf + row * S::SROW + 2 * u) =
                u < ng ? src[eo + (size_t)(col < p.N ? col : p.N - 1) * sgroups + u] : (uint16_t)0;
          }
        }
      };
      // Moves the iterator to a chunk of this wave (or leaves it on its last).
      int last_sg = 0, last_t = 0;
      auto advance = [&]() {
        if (pf_t < pf_n) {
          last_sg = pf_sg;
          last_t = pf_t;
          return;
        }
        int it2 = pf_it, sg2 = pf_sg;
        while (true) {
          if (++sg2 == nseg) {
            sg2 = 0;
            if (++it2 == ni) {   // the end: stay
              pf_sg = last_sg;
              pf_t = last_t;
              return;
            }
          }
          if (seg_chunks(sg2) > 0) break;
        }
        pf_sg = last_sg = sg2;
        pf_t = last_t = 0;
        pf_n = seg_chunks(sg2);
        if (it2 != pf_it) {
          pf_it = it2;
          set_item(it2);
        }
      };
      // Loads of the iterator's chunk into the stage at LDS address st; the
      // iterator then moves on (past the end it loads its last chunk again,
      // which nobody reads).
      auto issue = [&](uint32_t st) {
        const int q = pf_sg * S::SEG + kw + KS * pf_t;
        int wb[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          wb[h] = 128 * q + (w_piece ^ (64 * h));
          if (tail_k && wb[h] >= row_bytes) wb[h] = row_bytes - 16;   // past K: a valid piece, times zero x
        }
#pragma unroll
        for (int i = 0; i < S::WI; ++i)
          dma16(w_base, w_off[i] + (uint32_t)wb[i & 1], st + 1024 * i);
#pragma unroll
        for (int i = 0; i < S::XI; ++i) {
          const int r = i * (64 / LPR) + x_r;
          int k = S::CK * q + 8 * (x_slot ^ (r & 15));
          if (tail_k && k >= p.K) k = 0;
          if (VEC || x_al) {
            dma16(x_ptr[i] + k, st + COLS * 128 + 1024 * i);
          } else {   // x at any element: the wave waits for it, and so for all loads before it
            uint32_t v[4];
#pragma unroll
            for (int h = 0; h < 4; ++h)
              v[h] = x_ptr[i][k + 2 * h] | (uint32_t)x_ptr[i][k + 2 * h + 1] << 16;
            *reinterpret_cast<uint4*>(stage0 + (st - lds0) + COLS * 128 + 1024 * i + 16 * lane) =
                make_uint4(v[0], v[1], v[2], v[3]);
          }
        }
        ++pf_t;
        advance();
      };

      // Sums of the wave's K parts.
      float acc[S::PW][CT][RA];
#pragma unroll
      for (int h = 0; h < S::PW; ++h)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int i = 0; i < RA; ++i) acc[h][ct][i] = 0.f;

      // Operands of one chunk in registers: the stage can be loaded again while
      // they are computed on.
      constexpr int WW = GS * BITS / 128;   // weight words per lane, group and 16 columns
      struct Ops {
        uint4 a[S::GPC][SPG];
        uint32_t w[S::GPC][CT][WW];
        float s[CT][S::GPC], b[CT][S::GPC];
      };
      // Chunk q (of segment sg) from stage st, its scales from buffer sc.
      auto fetch = [&](Ops& o, unsigned char* st, const unsigned char* sc, int sg, int q) {
        if (tail_k && q == Q - 1) {   // x past K: zero
          for (int t = lane; t < S::XR * LPR; t += 64) {
            const int r = t / LPR, slot = t % LPR;
            if (S::CK * q + 8 * (slot ^ (r & 15)) >= p.K)
              *reinterpret_cast<uint4*>(st + COLS * 128 + 16 * t) = make_uint4(0, 0, 0, 0);
          }
        }
#pragma unroll
        for (int u = 0; u < S::GPC; ++u) {
#pragma unroll
          for (int j = 0; j < SPG; ++j) o.a[u][j] = *reinterpret_cast<const uint4*>(st + a_addr(u, j));
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            if constexpr (WW == 1) {
              o.w[u][ct][0] = *reinterpret_cast<const uint32_t*>(st + 2048 * ct + w_addr(u, 0));
            } else if constexpr (WW == 2) {
              const uint2 v = *reinterpret_cast<const uint2*>(st + 2048 * ct + w_addr(u, 0));
              o.w[u][ct][0] = v.x;
              o.w[u][ct][1] = v.y;
            } else {
#pragma unroll
              for (int h = 0; h < WW; h += 4) {
                const uint4 v = *reinterpret_cast<const uint4*>(st + 2048 * ct + w_addr(u, 4 * h));
                o.w[u][ct][h] = v.x;
                o.w[u][ct][h + 1] = v.y;
                o.w[u][ct][h + 2] = v.z;
                o.w[u][ct][h + 3] = v.w;
              }
            }
          }
        }
        const int g0 = (q - sg * S::SEG) * S::GPC;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const unsigned char* const sp = sc + (COLS * cg + 16 * ct + c16) * S::SROW + 2 * g0;
          group_vals<S::GPC>(sp, o.s[ct]);
          group_vals<S::GPC>(sp + S::TC * S::SROW, o.b[ct]);
        }
      };
      auto compute = [&](const Ops& o, int q, float (&acc)[CT][RA]) {
        const bf16x8 ones = __builtin_bit_cast(bf16x8, make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u));
#pragma unroll
        for (int u = 0; u < S::GPC; ++u) {
          bf16x8 A[SPG];
          f32x4 X = {};
#pragma unroll
          for (int j = 0; j < SPG; ++j) {
            uint4 a = o.a[u][j];
            if constexpr (BITS == 4) {   // the k order of nibbles_to_bf16: (k0,k4) (k1,k5) (k2,k6) (k3,k7)
              uint4 t;
              t.x = __builtin_amdgcn_perm(a.z, a.x, 0x05040100u);
              t.y = __builtin_amdgcn_perm(a.z, a.x, 0x07060302u);
              t.z = __builtin_amdgcn_perm(a.w, a.y, 0x05040100u);
              t.w = __builtin_amdgcn_perm(a.w, a.y, 0x07060302u);
              a = t;
            }
            A[j] = __builtin_bit_cast(bf16x8, a);
            X = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[j], ones, X, 0, 0, 0);
          }
          float T[RA];
          if constexpr (XS) {
#pragma unroll
            for (int i = 0; i < RA; ++i) {
              const int m = R == 4 ? g : 4 * g + i;
              const int s0 = (S::CK * q + GS * u) >> 4;   // 16-value slices: 32 per 512 k, stride 8
              T[i] = 0.f;
#pragma unroll
              for (int s = 0; s < GS / 16; ++s) T[i] += m < p.M ? p.xsums[(size_t)(s0 + s) * 8 + m] : 0.f;
            }
          }
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            f32x4 G = {};
#pragma unroll
            for (int j = 0; j < SPG; ++j) {
              if constexpr (BITS == 4) {
                G = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[j], nibbles_to_bf16(o.w[u][ct][j], nc), G, 0, 0, 0);
              } else {
                uint32_t e[4];
#pragma unroll
                for (int h = 0; h < 2; ++h) {   // bytes -> exact bf16: the fp32 value's upper half
                  const uint32_t v = o.w[u][ct][2 * j + h];
                  const uint32_t f0 = __float_as_uint((float)(v & 0xff));
                  const uint32_t f1 = __float_as_uint((float)((v >> 8) & 0xff));
                  const uint32_t f2 = __float_as_uint((float)((v >> 16) & 0xff));
                  const uint32_t f3 = __float_as_uint((float)(v >> 24));
                  e[2 * h] = __builtin_amdgcn_perm(f1, f0, 0x07060302u);
                  e[2 * h + 1] = __builtin_amdgcn_perm(f3, f2, 0x07060302u);
                }
                G = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[j], __builtin_bit_cast(bf16x8, e), G, 0, 0, 0);
              }
            }
            // What the group's sum of x is multiplied by, beside the scale (XS: the table's sum by the bias).
            const float cf = BITS == 4 ? fmaf(-128.f, o.s[ct][u], XS ? 0.f : o.b[ct][u]) : o.b[ct][u];
#pragma unroll
            for (int i = 0; i < RA; ++i) {
              float& t = acc[ct][i];
              if constexpr (XS) t = fmaf(o.b[ct][u], T[i], t);
              t = fmaf(o.s[ct][u], G[i], fmaf(cf, X[i], t));
            }
          }
        }
      };

      // End of item it: the waves' sums meet in LDS (two areas in turn, so one
      // barrier per item suffices), added in wave order (eight parts: w and
      // w + 4 first), then stored.
      auto finish = [&](int it) {
        float* const rd = red + (size_t)(it & 1) * NW * S::XR * COLS;
        float* const mine = rd + (size_t)wave * S::XR * COLS;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int i = 0; i < RA; ++i) {
            const int m = R == 4 ? g : 4 * g + i;
            mine[m * COLS + 16 * ct + c16] = S::PW == 2 ? acc[0][ct][i] + acc[S::PW - 1][ct][i] : acc[0][ct][i];
#pragma unroll
            for (int h = 0; h < S::PW; ++h) acc[h][ct][i] = 0.f;
          }
        lds_barrier();
        const int4 im = L.item[it];
        for (int idx = tid; idx < S::XR * S::OC; idx += NT) {
          const int m = idx / S::OC, c = idx - m * S::OC;
          const int col = im.y * S::OC + c;
          if (m >= im.w || col >= p.N) continue;
          auto sum = [&](int cc) {   // column cc of the tile's weight rows
            auto part = [&](int w) { return rd[((cc / COLS * KS + w) * S::XR + m) * COLS + cc % COLS]; };
            float t = 0.f;
#pragma unroll
            for (int w = 0; w < (KS == 8 ? 4 : KS); ++w) t += KS == 8 ? part(w) + part(w + 4) : part(w);
            return t;
          };
          const float v = sum(c), up = DUAL ? sum(S::OC + c) : 0.f;
          const size_t o = (size_t)(im.z + m) * p.ldy + col;
          if (DUAL) {
            const float gs = round_bf(silu_f(round_bf(v)));
            p.y[o] = f2bf(gs * round_bf(up));
          } else if (p.yf) {
            p.yf[o] = round_bf(v);
          } else {
            p.y[o] = f2bf(v);
          }
        }
      };

      // The stream: segment by segment; every wave meets at each segment's end
      // (its scale buffer is free then, and the next segment's, loaded since
      // the one before, is complete: each wave has waited for all but its newest
      // stage), and at the item's last one the sums meet.
      load_scales(0, 0);
      if (nseg * ni > 1) load_scales(nseg > 1 ? 0 : 1, nseg > 1 ? 1 : 0);
      set_item(0);
      pf_n = seg_chunks(0);
      const bool any = pf_n > 0;   // (segment 0 is the longest or equal: a wave without chunks there has none)
      if (any) {
#pragma unroll
        for (int d = 0; d < S::D; ++d) issue(lds0 + d * S::STAGE);
        wait_vm<S::D * NL>();   // the scales
      } else {
        wait_vm<0>();
      }
      if constexpr (!VEC) __builtin_amdgcn_s_waitcnt(0);
      lds_barrier();
      int sel = 0;
      for (int it = 0; it < ni; ++it) {
        for (int sg = 0; sg < nseg; ++sg) {
          const unsigned char* const sc = scal + ((it * nseg + sg) & 1) * S::SCAL;
          const int n = any ? seg_chunks(sg) : 0;
          auto chunk = [&](int t, float (&acc)[CT][RA]) {
            wait_vm<(S::D - 1) * NL>();   // the other stages' loads may be in flight
            const int q = sg * S::SEG + kw + KS * t;
            Ops o;
            fetch(o, stage0 + sel * S::STAGE, sc, sg, q);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // its reads have returned: load it again
            issue(lds0 + sel * S::STAGE);
            compute(o, q, acc);
            sel = sel + 1 == S::D ? 0 : sel + 1;
          };
          for (int t = 0; t < n; t += S::PW) {
            chunk(t, acc[0]);
            if constexpr (S::PW == 2) {
              if (t + 1 < n) chunk(t + 1, acc[1]);
            }
          }
          // Its part of the next segment's scales: complete by the second chunk's
          // wait; with fewer chunks, waited for here.
          if (n > 0 && n < S::D) wait_vm<NL>();
          if (n == 0) wait_vm<0>();
          if (sg + 1 == nseg)
            finish(it);
          else
            lds_barrier();
          const int nx = it * nseg + sg + 2;   // the segment after next takes this one's buffer
          if (nx < ni * nseg) load_scales(nx / nseg, nx % nseg);
        }
      }
      wait_vm<0>();   // the stages are loaded again for the next items
    }
  }
  return more != 0;
}

// One matrix.
template <int BITS, int GS, int R, bool VEC, bool XS, int NW>
__global__ __launch_bounds__(NW * 64, 1) void qmv_inplace_kernel(InplaceParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  inplace_body<BITS, GS, R, false, VEC, XS, NW, NW, 2>(p, smem, blockIdx.x, 1, INT_MAX);
}

// Experts: those with at most 4 rows in tiles of 4, then, where there are such,
// the others in tiles of 16, all in one launch. A launch for each class costs
// the small calls, which wait for launches (4 rows x 8 of 256 experts through
// the three gathers of an unsorted block: 270-281 us, 258 with one launch each;
// 16 rows x 8 through the sorted block: 188 and 177; 512 rows x 8: 1045 and
// 1023). The second class is handed out from the last workgroup on: the first
// ones may hold an item more of the first. Two K parts and two column groups
// (the pair: its matrices) per workgroup: an item is twice as long as with four
// parts, and K = 1536 has 6 chunks (down 48 us against 59, gate|up 90 against 92).
template <int GS, bool DUAL, bool VEC>
struct InplaceExperts {
  using Few = InplaceShape<4, GS, 4, DUAL, 4, 2, 1>;
  using Many = InplaceShape<4, GS, 16, DUAL, 4, 2, 1>;
  static constexpr size_t lds() { return Few::lds() > Many::lds() ? Few::lds() : Many::lds(); }
  static_assert(Few::OC == Many::OC, "one column tile for both classes");
};
template <int GS, bool DUAL, bool VEC>
__global__ __launch_bounds__(256, 2) void qmv_inplace_experts(InplaceParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  if (inplace_body<4, GS, 4, DUAL, VEC, false, 4, 2, 1>(p, smem, blockIdx.x, 1, 4))
    inplace_body<4, GS, 16, DUAL, VEC, false, 4, 2, 1>(p, smem, gridDim.x - 1 - blockIdx.x, 5, INT_MAX);
}

// Launches it for bits 4/8 and groups 32/64/128 (experts: 4 bits, groups 64/128).
// ``dual``: the experts' fused SwiGLU pair (K % 256 == 0).
void inplace_launch(const InplaceParams& p, int bits, int gs, bool dual, hipStream_t st);

}  // namespace mtp
