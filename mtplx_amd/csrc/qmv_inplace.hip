// Launches of the in-place streaming matmul (qmv_inplace.hpp): the variant for
// a format and a row count, for one matrix or for the experts of a sort.
#include "qmv_inplace.hpp"

#include <limits.h>

namespace mtp {

// Launches kernel k, of ``threads`` threads and ``lds`` bytes of LDS: a
// workgroup per item, at most as many as the CUs hold (two each at most).
template <class Kernel>
static void inplace_run(Kernel k, const InplaceParams& p, int threads, int lds, long long items, hipStream_t st) {
  (void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  const long long most = (160 * 1024 / lds >= 2 ? 2ll : 1ll) * device_cus();
  hipLaunchKernelGGL(k, dim3((unsigned)(items < most ? items : most)), dim3(threads), lds, st, p);
}

// One matrix: 32 columns a workgroup, K split over all of its waves, in the
// same eight parts for any number of rows. Up to 4
// rows, 8 waves and two stages (17408 x 5120 of 8 bits 24.2 us, 5120 x 17408
// 23.9; two workgroups of 4 waves 23.8 and 27.1, with one stage 25.8 and
// 33.3); more rows, 4 waves, whose stages hold 16 rows of x (32768 x 5120, 16
// rows: 40.5 us, with one stage 48.8).
template <int BITS, int GS, int R, bool VEC, bool XS, int NW>
static void inplace_dense(InplaceParams p, hipStream_t st) {
  using S = InplaceShape<BITS, GS, R, false, NW, NW, 2>;
  static_assert(S::lds() <= 160 * 1024, "a workgroup's LDS");
  p.ntile = cdiv(p.N, S::OC);
  inplace_run(qmv_inplace_kernel<BITS, GS, R, VEC, XS, NW>, p, NW * 64, (int)S::lds(),
              (long long)p.ntile * cdiv(p.M, R), st);
}

template <int GS, bool DUAL, bool VEC>
static void inplace_experts(InplaceParams p, hipStream_t st) {
  using E = InplaceExperts<GS, DUAL, VEC>;
  static_assert(2 * E::lds() <= 160 * 1024, "two workgroups per CU");
  p.ntile = cdiv(p.N, E::Few::OC);
  inplace_run(qmv_inplace_experts<GS, DUAL, VEC>, p, 256, (int)E::lds(), LLONG_MAX, st);   // (the device knows how many items)
}

template <int BITS, int GS, bool DUAL, bool VEC>
static void inplace_rows(const InplaceParams& p, hipStream_t st) {
  if constexpr (BITS == 4 && GS >= 64) {
    if (p.active) return inplace_experts<GS, DUAL, VEC>(p, st);
  }
  if constexpr (!DUAL) {
    if constexpr (BITS == 4 && GS <= 64) {
      if (p.xsums)   // the cross-row lane
        return p.M <= 4 ? inplace_dense<BITS, GS, 4, VEC, true, 8>(p, st)
                        : inplace_dense<BITS, GS, 16, VEC, true, 4>(p, st);
    }
    return p.M <= 4 ? inplace_dense<BITS, GS, 4, VEC, false, 8>(p, st)
                    : inplace_dense<BITS, GS, 16, VEC, false, 4>(p, st);
  }
}

template <int BITS, int GS, bool DUAL>
static void inplace_vec(const InplaceParams& p, hipStream_t st) {
  // Scales straight to LDS in 16-byte pieces of eight groups where rows hold
  // whole pieces and the arrays are so aligned; else element by element. x may
  // start at any element too.
  auto aligned = [](const void* a) { return ((uintptr_t)a & 15) == 0; };
  const bool vec = (p.K / GS) % 8 == 0 && aligned(p.x) && aligned(p.s0) && aligned(p.b0) &&
                   (!DUAL || (aligned(p.s1) && aligned(p.b1)));
  if (vec) {
    inplace_rows<BITS, GS, DUAL, true>(p, st);
  } else {
    inplace_rows<BITS, GS, DUAL, false>(p, st);
  }
}

void inplace_launch(const InplaceParams& p, int bits, int gs, bool dual, hipStream_t st) {
  if (dual) {   // 4-bit, groups 64/128, K % 256 == 0, aligned scales (checked by the caller)
    if (gs == 64)
      inplace_vec<4, 64, true>(p, st);
    else
      inplace_vec<4, 128, true>(p, st);
  } else if (bits == 4) {
    if (gs == 32) inplace_vec<4, 32, false>(p, st);
    else if (gs == 64) inplace_vec<4, 64, false>(p, st);
    else inplace_vec<4, 128, false>(p, st);
  } else {
    if (gs == 32) inplace_vec<8, 32, false>(p, st);
    else if (gs == 64) inplace_vec<8, 64, false>(p, st);
    else inplace_vec<8, 128, false>(p, st);
  }
}

}  // namespace mtp
