// Launches of the in-place streaming matmul (qmv_inplace.hpp): the variant for
// a format and a row count, for one matrix or for the experts of a sort.
#include "qmv_inplace.hpp"

#include <climits>

namespace mtp {

template <int BITS, int GS, int R, bool DUAL, bool VEC, bool XS, int NW, int KS, int ND>
static void inplace_run(InplaceParams p, hipStream_t st) {
  using S = InplaceShape<BITS, GS, R, DUAL, NW, KS, ND>;
  auto k = qmv_inplace_kernel<BITS, GS, R, DUAL, VEC, XS, NW, KS, ND>;
  constexpr int lds = (int)S::lds();
  // Workgroups per CU by LDS, at most two.
  constexpr int per_cu = 160 * 1024 / (lds + S::FIXED) >= 2 ? 2 : 1;
  static_assert(lds + S::FIXED <= 160 * 1024, "a workgroup's LDS");
  (void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  p.ntile = cdiv(p.N, S::OC);
  int grid = per_cu * device_cus();
  if (!p.active) {
    const long long items = (long long)p.ntile * cdiv(p.M, R);
    if (items < grid) grid = (int)items;
  }
  hipLaunchKernelGGL(k, dim3(grid), dim3(NW * 64), lds, st, p);
}

// One matrix: 32 columns a workgroup, K split over all of its waves, in the
// same eight parts for any number of rows. Up to 4
// rows, 8 waves and two stages (17408 x 5120 of 8 bits 24.2 us, 5120 x 17408
// 23.9; two workgroups of 4 waves 23.8 and 27.1, with one stage 25.8 and
// 33.3); more rows, 4 waves, whose stages hold 16 rows of x (32768 x 5120, 16
// rows: 40.5 us, with one stage 48.8).
template <int BITS, int GS, bool VEC, bool XS>
static void inplace_dense(const InplaceParams& p, int max_rows, hipStream_t st) {
  if (max_rows <= 4)
    inplace_run<BITS, GS, 4, false, VEC, XS, 8, 8, 2>(p, st);
  else
    inplace_run<BITS, GS, 16, false, VEC, XS, 4, 4, 2>(p, st);
}

template <int BITS, int GS, bool DUAL, bool VEC>
static void inplace_rows(InplaceParams p, int max_rows, hipStream_t st) {
  if constexpr (!DUAL) {
    if (!p.active) {
      if constexpr (BITS == 4 && GS <= 64) {
        if (p.xsums) return inplace_dense<BITS, GS, VEC, true>(p, max_rows, st);   // the cross-row lane
      }
      return inplace_dense<BITS, GS, VEC, false>(p, max_rows, st);
    }
  }
  // Experts: those with at most 4 rows, then the others in tiles of 16. Two
  // K parts and two column groups (the pair: its matrices) per workgroup: an
  // item is twice as long as with four parts, and K = 1536 has 6 chunks (down
  // 48 us against 59, gate|up 90 against 92).
  if constexpr (BITS == 4 && GS >= 64) {
    p.m_lo = 1;
    p.m_hi = 4;
    inplace_run<BITS, GS, 4, DUAL, VEC, false, 4, 2, 1>(p, st);
    if (max_rows <= 4) return;
    p.m_lo = 5;
    p.m_hi = INT_MAX;
    inplace_run<BITS, GS, 16, DUAL, VEC, false, 4, 2, 1>(p, st);
  }
}

template <int BITS, int GS, bool DUAL>
static void inplace_vec(const InplaceParams& p, int max_rows, hipStream_t st) {
  // Scales straight to LDS in 16-byte pieces of eight groups where rows hold
  // whole pieces and the arrays are so aligned; else element by element. x may
  // start at any element too.
  auto aligned = [](const void* a) { return ((uintptr_t)a & 15) == 0; };
  const bool vec = (p.K / GS) % 8 == 0 && aligned(p.x) && aligned(p.s0) && aligned(p.b0) &&
                   (!DUAL || (aligned(p.s1) && aligned(p.b1)));
  if (vec) {
    inplace_rows<BITS, GS, DUAL, true>(p, max_rows, st);
  } else {
    inplace_rows<BITS, GS, DUAL, false>(p, max_rows, st);
  }
}

void inplace_launch(const InplaceParams& p, int bits, int gs, int max_rows, bool dual, hipStream_t st) {
  if (dual) {   // 4-bit, groups 64/128, K % 256 == 0, aligned scales (checked by the caller)
    if (gs == 64)
      inplace_vec<4, 64, true>(p, max_rows, st);
    else
      inplace_vec<4, 128, true>(p, max_rows, st);
  } else if (bits == 4) {
    if (gs == 32) inplace_vec<4, 32, false>(p, max_rows, st);
    else if (gs == 64) inplace_vec<4, 64, false>(p, max_rows, st);
    else inplace_vec<4, 128, false>(p, max_rows, st);
  } else {
    if (gs == 32) inplace_vec<8, 32, false>(p, max_rows, st);
    else if (gs == 64) inplace_vec<8, 64, false>(p, max_rows, st);
    else inplace_vec<8, 128, false>(p, max_rows, st);
  }
}

}  // namespace mtp
