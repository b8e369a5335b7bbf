// Discrete adjoint of the Biot time step (HIP, gfx950): FP32, FP64 or FP16 forward states,
// adjoint wavefields in the arithmetic type (float, double for FP64), FP64 gradient sums.
//
// One forward step n maps u^n (after the source of step n) to u^{n+1}:
//   velocity half step  D = delta(tau, p); D' = (1+a) D + c_V; c_V <- e (c_V + 2 a D)
//                       q' = W1 q - W2 sum D' - W3 D's;  v' = v + U1 sum D' - U2 (q' - q)
//   stress half step    E = delta(v', q'); E' = (1+a) E + c_T; c_T <- e (c_T + 2 a E)
//                       p' = p - P1 div_u' - P2 div_w';  tau' = tau + S1 .. + S2 .. + S3 div_w'
// (the folded C-PML carry, kernel.cu:188-196 algebraically).  Its transpose, applied backward, has
// two parts per half step:
//   local  : adjoints of the twelve post-PML derivatives from the adjoint state at the cell,
//            C-PML carry adjoints  lambda_E = (1+a) lambda_E' + 2 a e lambda_c,
//            lambda_c <- lambda_E' + e lambda_c, the cell-local field adjoints, and the FP64
//            sums of dJ/dK = lambda(output) x (forward term) for every coefficient K, with the
//            forward derivatives recomputed from the stored states;
//   gather : lambda_f(c) += sum_m w_m G(c - o_m), the transposed staggered differences,
//            written per cell so the result is deterministic (no atomics).
// A gather ends with the cell's new adjoint values, which are all that the next local part reads
// of them, so a backward step is two passes: the gather of step n+1's velocity half with the local
// part of step n's stress half (adj_stress), then the gather of that with the local part of step
// n's velocity half (adj_velocity).
// The derivative adjoints G between the passes: outside the absorbing slabs G is lambda_E', of
// which the stress half has 7 different ones and the velocity half 6, kept as full arrays; the
// derivatives along an axis whose slab the cell lies in are four records of G, laid out as the
// carries are.
// The passes are bound by their bytes: 137 values a cell and step (FP32: 548 B) and 160 B a slab
// membership, where four passes with twelve full arrays of G moved 175 and 96 B.  Per step, before and
// now: 128^3 FP32 343 and 320 us (about 4.1 TB/s), 192^3 1198 and 1000 us, 128^3 FP64 721 and 665, 90^3
// FP16M 236 and 107, 128^3 FP16T 687 and 320.
// With 16-bit storage everything runs in storage units (fields divided by their scales,
// coefficients as the kernels apply them); the host converts dJ/dK with the per-array factor.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "biot_adjoint.hpp"
#include "biot_packed.hpp"

namespace biot {
namespace {

using u32 = uint32_t;

template <typename T>
__device__ __forceinline__ T &at(void *base, u32 idx)
{
  return *reinterpret_cast<T *>(reinterpret_cast<char *>(base) + idx * (u32)sizeof(T));
}
template <typename T>
__device__ __forceinline__ const T &at(const void *base, u32 idx)
{
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + idx * (u32)sizeof(T));
}

// The twelve derivatives of a half step by axis and carry slot (kernel.cu:172-185, 188-216;
// 430-482): the field they difference, and whether forward (on the half-node profile) or backward
// (integer nodes).  Velocity half: x1 s1 y2 z2 | x2 y1 s2 z3 | x3 y3 z1 s3; stress half: uxx wx uyx
// uzx | uyy wy uxy uzy | uzz wz uxz uyz.
__device__ constexpr int der_field(bool vel, int ax, int m)
{
  constexpr int v[3][4] = {{6, 12, 9, 10}, {9, 7, 12, 11}, {10, 11, 8, 12}};
  constexpr int t[3][4] = {{0, 3, 1, 2}, {1, 4, 0, 2}, {2, 5, 0, 1}};
  return vel ? v[ax][m] : t[ax][m];
}
__device__ constexpr bool der_fwd(bool vel, int ax, int m)
{
  constexpr bool v[3][4] = {{true, true, false, false}, {false, true, true, false}, {false, false, true, true}};
  return vel ? v[ax][m] : m >= 2;
}
// the full array (AdjArgs gv / gt) that holds the derivative's G outside its slab.  Velocity half:
// the three S and the three Ds; stress half: uxx uyy uzz, div w, and the three shears xy xz yz.
__device__ constexpr int der_base(bool vel, int ax, int m)
{
  constexpr int v[3][4] = {{0, 3, 1, 2}, {0, 1, 4, 2}, {0, 1, 2, 5}};
  constexpr int t[3][4] = {{0, 3, 4, 5}, {1, 3, 4, 6}, {2, 3, 5, 6}};
  return vel ? v[ax][m] : t[ax][m];
}

// storage type S -> arithmetic type A (also the C-PML carry type)
template <typename S>
struct AdjT {
  using A = typename std::conditional<std::is_same<S, double>::value, double, float>::type;
  using C = typename std::conditional<std::is_same<S, float>::value, float, S>::type;  // forward carry
  using T = S;  // stored element of fields and coefficients
  static constexpr bool scaled = std::is_same<S, _Float16>::value;
  static constexpr bool res = false;
  static constexpr bool pk = false;
};
// FP16T / FP16C states: binary16 fields and coefficients, an int8 residual on the fields of MASK
// (FP16T tau and p, FP16C also v; value = h + r ulp(h)/256, as the forward kernels store it), float
// C-PML carries.  The mask is part of the type: tested at run time it put a branch around each of
// the 96 taps of a step (128^3 FP16T: 631 us a step, 292 without).
template <uint32_t MASK>
struct H16R {
  static constexpr uint32_t mask = MASK;
};
template <uint32_t MASK>
struct AdjT<H16R<MASK>> {
  using A = float;
  using C = float;
  using T = _Float16;
  static constexpr bool scaled = true;
  static constexpr bool res = true;
  static constexpr bool pk = false;
};
// FP16M states: binary16 fields; tau and p completed by the 4-bit residual of the cell's
// 4-byte record (value = h + r ulp(h)/16, as the forward kernels store it); float C-PML
// carries.  Its coefficients are read as FP16T stores them (binary16, packed per cell).
struct H16P {};
template <>
struct AdjT<H16P> {
  using A = float;
  using C = float;
  using T = _Float16;
  static constexpr bool scaled = true;
  static constexpr bool res = false;
  static constexpr bool pk = true;
};
// the residual unit ulp(h)/256 = 2^(e-33), e the biased exponent of h (subnormals e = 1)
__device__ __forceinline__ float res_unit(_Float16 h)
{
  const uint32_t u = __builtin_bit_cast(uint16_t, h);
  const int e = max((int)((u >> 10) & 31u), 1);
  return __builtin_bit_cast(float, (uint32_t)(e + 94) << 23);
}

struct CellIdx {
  int i, j, k;
  u32 c;
};

// the cell of thread t of block blk (AdjArgs: ADJ_BX consecutive cells of an x-y plane in ADJ_BZ
// planes); false outside the update box
template <class AT>
__device__ __forceinline__ bool cell_of(const AT &a, int h, u32 blk, u32 t, CellIdx &ci)
{
  const u32 tz = blk / (u32)a.gx, tx = blk - tz * (u32)a.gx;
  const u32 l = (u32)a.xy0 + tx * ADJ_BX + t % ADJ_BX;
  u32 q = __umulhi(l, a.nx_rcp);
  if (q * (u32)a.nx > l) --q;
  ci.j = (int)q;
  ci.i = (int)(l - q * (u32)a.nx);
  ci.k = h + (int)(tz * ADJ_BZ + t / ADJ_BX);
  ci.c = l + (u32)ci.k * (u32)a.sz;
  return ci.i >= h && ci.i < a.nx - h && ci.j >= h && ci.j < a.ny - h && ci.k < a.nz - h;
}

template <class AT>
__device__ __forceinline__ const void *fw_field(const AT &a, int q, int f)
{
  return a.slots + (uint64_t)q * a.sb + (uint64_t)f * a.fbytes;
}
template <class AT>
__device__ __forceinline__ const void *fw_carry(const AT &a, int q, int ax)
{
  return a.slots + (uint64_t)q * a.sb + a.coff[ax];
}
// the residuals of field f in state q (FP16T, FP16C)
template <class AT>
__device__ __forceinline__ const int8_t *fw_lo(const AT &a, int q, int f)
{
  return reinterpret_cast<const int8_t *>(a.slots + (uint64_t)q * a.sb + a.loff +
                                          (uint64_t)f * (uint64_t)a.nx * a.ny * a.nz);
}

// staggered difference of forward field f of state q at cell c, stride s (f and fwd fold to
// constants).  FP16M: the residual record of a point is addressed from the one record array, so the
// fields differenced there share its load.
template <typename S, int ORDER, class AT>
__device__ __forceinline__ typename AdjT<S>::A diff(const AT &a, int q, int f, u32 c, u32 s, bool fwd)
{
  using A = typename AdjT<S>::A;
  using T = typename AdjT<S>::T;
  const void *fp = fw_field(a, q, f);
  auto L = [&](u32 idx) {
    const T h = at<T>(fp, idx);
    if constexpr (AdjT<S>::res) {
      if ((S::mask >> f) & 1u) return (A)h + (A)fw_lo(a, q, f)[idx] * res_unit(h);
    }
    if constexpr (AdjT<S>::pk) {
      if ((PK_FIELDS >> f) & 1u)
        return (A)pk_join((float)h, pk_nib(at<u32>(a.slots + (uint64_t)q * a.sb + a.loff, idx), pk_slot(f)));
    }
    return (A)h;
  };
  if (fwd) {
    if constexpr (ORDER == 2) return L(c + s) - L(c);
    return A(9.0 / 8.0) * (L(c + s) - L(c)) + A(-1.0 / 24.0) * (L(c + 2 * s) - L(c - s));
  } else {
    if constexpr (ORDER == 2) return L(c) - L(c - s);
    return A(9.0 / 8.0) * (L(c) - L(c - s)) + A(-1.0 / 24.0) * (L(c + s) - L(c - 2 * s));
  }
}

template <int AX, class AT>
__device__ __forceinline__ u32 stride(const AT &a)
{
  return AX == 0 ? 1u : AX == 1 ? (u32)a.sy : (u32)a.sz;
}
// slab cell index on axis AX of the cell ci moved to position `pos` on that axis, or -1 outside
// the slabs
template <int AX, class AT>
__device__ __forceinline__ int slab_cell(const AT &a, const CellIdx &ci, int pos)
{
  const int nn = AX == 0 ? a.nx : (AX == 1 ? a.ny : a.nz);
  int p;
  if (pos < a.L[AX]) p = pos;
  else if (pos >= nn - a.R[AX]) p = a.L[AX] + pos - (nn - a.R[AX]);
  else return -1;
  const int w = a.L[AX] + a.R[AX];
  if (AX == 0) return p + w * (ci.j + a.ny * ci.k);
  if (AX == 1) return ci.i + a.nx * (p + w * ci.k);
  return ci.i + a.nx * (ci.j + a.ny * p);
}
// the record of four values of slab cell o of group g (0: velocity half, 1: stress half) in an
// array laid out as the carries are
template <typename E>
__device__ __forceinline__ void rec_load(E (&v)[4], const void *base, u32 g, u32 o, u32 sl)
{
  typedef E V4 __attribute__((ext_vector_type(4)));
  const V4 r = *reinterpret_cast<const V4 *>(reinterpret_cast<const char *>(base) + (g * sl + o) * (u32)(4 * sizeof(E)));
  v[0] = r.x, v[1] = r.y, v[2] = r.z, v[3] = r.w;
}
template <typename E>
__device__ __forceinline__ void rec_store(const E (&v)[4], void *base, u32 g, u32 o, u32 sl)
{
  typedef E V4 __attribute__((ext_vector_type(4)));
  V4 r;
  r.x = v[0], r.y = v[1], r.z = v[2], r.w = v[3];
  *reinterpret_cast<V4 *>(reinterpret_cast<char *>(base) + (g * sl + o) * (u32)(4 * sizeof(E))) = r;
}

// The transposed differences along axis AX of the four derivatives of a half step at cell ci:
// out[m] from G at the cells -h..h along the axis, each from the full array outside the axis's
// slabs and from the slab's record inside.  Away from the slabs (the whole stencil outside) there
// is nothing to choose.
template <typename A, int ORDER, bool VEL, int AX, class AT>
__device__ __forceinline__ void gather_axis(const AT &a, const CellIdx &ci, A (&out)[4])
{
  constexpr int h = ORDER / 2;
  const u32 s = stride<AX>(a);
  const int pos = AX == 0 ? ci.i : (AX == 1 ? ci.j : ci.k);
  const int nn = AX == 0 ? a.nx : (AX == 1 ? a.ny : a.nz);
  A v[4][2 * h + 1];
  auto base = [&](int m, int o) {
    return at<A>(VEL ? a.gv[der_base(true, AX, m)] : a.gt[der_base(false, AX, m)], ci.c + (u32)o * s);
  };
  if (pos - h < a.L[AX] || pos + h >= nn - a.R[AX]) {
#pragma unroll
    for (int o = -h; o <= h; ++o) {
      const int sc = slab_cell<AX>(a, ci, pos + o);
      A r[4];
      if (sc >= 0) {
        rec_load(r, a.gs[AX], VEL ? 0u : 1u, (u32)sc, (u32)a.slab[AX]);
      } else {
#pragma unroll
        for (int m = 0; m < 4; ++m) r[m] = base(m, o);
      }
#pragma unroll
      for (int m = 0; m < 4; ++m) v[m][o + h] = r[m];
    }
  } else {
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int o = -h; o <= h; ++o)
        if (der_fwd(VEL, AX, m) ? o < h : o > -h) v[m][o + h] = base(m, o);
  }
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    auto G = [&](int o) { return v[m][o + h]; };
    if constexpr (ORDER == 2) {
      out[m] = der_fwd(VEL, AX, m) ? G(-1) - G(0) : G(0) - G(1);
    } else {
      out[m] = der_fwd(VEL, AX, m) ? A(9.0 / 8.0) * (G(-1) - G(0)) + A(-1.0 / 24.0) * (G(-h) - G(1))
                                   : A(9.0 / 8.0) * (G(0) - G(1)) + A(-1.0 / 24.0) * (G(-1) - G(h));
    }
  }
}

// the N coefficients K[k0..k0+N) of cell c from the packed copy (storage units, times the
// per-array scale for 16-bit storage)
template <typename S, int N, class AT>
__device__ __forceinline__ void kblock(const AT &a, const void *base, u32 c, int k0,
                                       typename AdjT<S>::A (&out)[N])
{
  using A = typename AdjT<S>::A;
  using T = typename AdjT<S>::T;
  uint32_t d[packed::block_dwords<T, N>()];
  packed::load<T, N, true>(base, (uint64_t)a.nx * a.ny * a.nz, c, d);
#pragma unroll
  for (int e = 0; e < N; ++e) {
    if constexpr (AdjT<S>::scaled) out[e] = (A)packed::value<T>(d, e) * (A)a.ks[k0 + e];
    else out[e] = (A)packed::value<T>(d, e);
  }
}
// the N gradient sums of K[k0..k0+N) at cell c: float partial sums of the packed array p on
// FP32/FP16 handles, the FP64 sums themselves on FP64 handles
template <typename A, int N, class AT>
__device__ __forceinline__ void gload(const AT &a, const void *p, u32 c, int k0, double (&g)[N])
{
  if constexpr (std::is_same<A, double>::value) {
#pragma unroll
    for (int e = 0; e < N; ++e) g[e] = at<double>(a.gacc[k0 + e], c);
  } else {
    uint32_t d[packed::block_dwords<float, N>()];
    packed::load<float, N, false>(p, (uint64_t)a.nx * a.ny * a.nz, c, d);
#pragma unroll
    for (int e = 0; e < N; ++e) g[e] = (double)packed::value<float>(d, e);
  }
}
template <typename A, int N, class AT>
__device__ __forceinline__ void gstore(const AT &a, void *p, u32 c, int k0, const double (&g)[N])
{
  if constexpr (std::is_same<A, double>::value) {
#pragma unroll
    for (int e = 0; e < N; ++e) at<double>(a.gacc[k0 + e], c) = g[e];
  } else {
    uint32_t d[N];
#pragma unroll
    for (int e = 0; e < N; ++e) d[e] = __builtin_bit_cast(uint32_t, (float)g[e]);
    packed::store<float, N>(p, (uint64_t)a.nx * a.ny * a.nz, c, d);
  }
}

// contraction written out where the compiler has a choice, so that a gradient does not depend on
// how the passes are arranged
__device__ __forceinline__ float fmadd(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double fmadd(double a, double b, double c) { return fma(a, b, c); }
template <typename A>
__device__ __forceinline__ A product(A a, A b)
{
#pragma clang fp contract(off)
  return a * b;
}

// The four derivatives of one axis in the local part of a half step: the forward derivatives E
// (fields of state qf) and, in the axis's slab, its profile values, the forward carries (state qc)
// and the carry adjoints, a record each.  Both passes issue all of their loads before their first
// store: the compiler cannot prove the arrays distinct and never moves a load above a store, so
// this order keeps a cell's loads in flight together (one memory round trip instead of one per
// store).
template <typename S, int ORDER, bool VEL, int AX>
struct AxisLocal {
  using A = typename AdjT<S>::A;
  A E[4], e[2], aa[2], cf[4], lc[4], g[4];
  int sc;
  template <class AT>
  __device__ __forceinline__ void load(const AT &a, const CellIdx &ci, int qf, int qc)
  {
#pragma unroll
    for (int m = 0; m < 4; ++m)
      E[m] = diff<S, ORDER>(a, qf, der_field(VEL, AX, m), ci.c, stride<AX>(a), der_fwd(VEL, AX, m));
    const int pos = AX == 0 ? ci.i : (AX == 1 ? ci.j : ci.k);
    sc = slab_cell<AX>(a, ci, pos);
    if (sc >= 0) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {  // integer, half nodes
        e[b] = at<A>(a.prof[AX][2 * b], (u32)pos);
        aa[b] = at<A>(a.prof[AX][2 * b + 1], (u32)pos);
      }
      typename AdjT<S>::C c4[4];
      rec_load(c4, fw_carry(a, qc, AX), VEL ? 0u : 1u, (u32)sc, (u32)a.slab[AX]);
      rec_load(lc, a.lcarry[AX], VEL ? 0u : 1u, (u32)sc, (u32)a.slab[AX]);
#pragma unroll
      for (int m = 0; m < 4; ++m) cf[m] = (A)c4[m];
    }
  }
  // E becomes the post-PML forward derivatives, lc the updated carry adjoints, g the derivative
  // adjoints (in the slab) of lE, the adjoints of the post-PML derivatives
  __device__ __forceinline__ void apply(const A (&lE)[4])
  {
    if (sc < 0) return;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int b = der_fwd(VEL, AX, m) ? 1 : 0;
      const A one = A(1) + aa[b], two = A(2) * aa[b] * e[b];
      E[m] = fmadd(one, E[m], cf[m]);
      g[m] = fmadd(one, lE[m], product(two, lc[m]));
      lc[m] = fmadd(e[b], lc[m], lE[m]);
    }
  }
  template <class AT>
  __device__ __forceinline__ void store(const AT &a)
  {
    if (sc < 0) return;
    rec_store(g, a.gs[AX], VEL ? 0u : 1u, (u32)sc, (u32)a.slab[AX]);
    rec_store(lc, a.lcarry[AX], VEL ? 0u : 1u, (u32)sc, (u32)a.slab[AX]);
  }
};

// The adjoint sources of step it at cell c added to the adjoints l[m] of fields F0 + m, one rounding
// for the sample and one for the sum, as a kernel of its own adds them.
template <typename A, int F0, int N, class IT>
__device__ __forceinline__ void inject(const IT &j, u32 c, int it, A (&l)[N])
{
#pragma clang fp contract(off)
  if (!((j.has[c >> 5] >> (c & 31u)) & 1u)) return;
  int lo = 0, hi = j.ncells - 1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (j.cells[mid] < c) lo = mid + 1;
    else hi = mid;
  }
  for (u32 e = j.first[lo]; e < j.first[lo + 1]; ++e) {
    const int64_t r = j.ids[e];
#pragma unroll
    for (int m = 0; m < N; ++m) {
      const int ci = j.comp[F0 + m];
      if (ci < 0) continue;
      const float v = j.src[((int64_t)ci * j.nt + it) * j.nrec + r] * j.scale[F0 + m];
      l[m] = l[m] + (A)v;
    }
  }
}

// The loads of one axis at a time: left to itself the compiler issues a pass's hundred loads at
// once and keeps 200-218 registers for them, two waves a SIMD (FP64: one).  Ended phase by phase
// they take 127 and 165 (four and three waves), and the passes are faster: 192^3 FP32 996 -> 882 us a
// step, 128^3 FP64 689 -> 629.  (Capping the registers instead spills: 128^3 FP32 302 -> 602 us.)
__device__ __forceinline__ void phase() { __builtin_amdgcn_sched_barrier(0); }

// lambda(tau, p) += transposed differences of the velocity-half G of the step after; then the local
// part of the stress half of state q's step
template <typename S, int ORDER, class AT, class IT>
__device__ __forceinline__ void adj_stress(const AT &a, const IT &j, int q, int it, u32 blk, u32 t)
{
  using A = typename AdjT<S>::A;
  constexpr int h = ORDER / 2;
  CellIdx ci;
  if (!cell_of(a, h, blk, t, ci)) return;
  const u32 c = ci.c;
  A l[7];  // txx tyy tzz txy txz tyz p
#pragma unroll
  for (int f = 0; f < 7; ++f) l[f] = at<A>(a.lam[6 + f], c);
  A gx[4], gy[4], gz[4];  // x1 s1 y2 z2 | x2 y1 s2 z3 | x3 y3 z1 s3
  gather_axis<A, ORDER, true, 0>(a, ci, gx);
  phase();
  gather_axis<A, ORDER, true, 1>(a, ci, gy);
  phase();
  gather_axis<A, ORDER, true, 2>(a, ci, gz);
  l[0] += gx[0], l[1] += gy[1], l[2] += gz[2];
  l[3] += gy[0] + gx[2], l[4] += gz[0] + gx[3], l[5] += gz[1] + gy[3];
  l[6] += gx[1] + gy[2] + gz[3];
  inject<A, 6>(j, c, it, l);
  const A ltxx = l[0], ltyy = l[1], ltzz = l[2], ltxy = l[3], ltxz = l[4], ltyz = l[5], lp = l[6];
  phase();
  AxisLocal<S, ORDER, false, 0> X;  // uxx wx uyx uzx
  AxisLocal<S, ORDER, false, 1> Y;  // uyy wy uxy uzy
  AxisLocal<S, ORDER, false, 2> Z;  // uzz wz uxz uyz
  // velocities of state q+1 (after the velocity half step), carries of state q
  X.load(a, ci, q + 1, q);
  phase();
  Y.load(a, ci, q + 1, q);
  phase();
  Z.load(a, ci, q + 1, q);
  phase();
  A kt[8];  // K[14..21]: P1 P2 S1 S2 S3 Sxy Sxz Syz
  kblock<S, 8>(a, a.kt, c, K_P1, kt);
  double g[8];  // sums of K[14..21]
  gload<A, 8>(a, a.gpt, c, K_P1, g);
  const A P1 = kt[0], P2 = kt[1], S1 = kt[2], S2 = kt[3], S3 = kt[4];
  const A Sxy = kt[5], Sxz = kt[6], Syz = kt[7];
  const A lxx = S2 * ltxx + S1 * (ltyy + ltzz) - P1 * lp;
  const A lyy = S2 * ltyy + S1 * (ltxx + ltzz) - P1 * lp;
  const A lzz = S2 * ltzz + S1 * (ltxx + ltyy) - P1 * lp;
  const A lw = S3 * (ltxx + ltyy + ltzz) - P2 * lp;
  const A lxy = Sxy * ltxy, lxz = Sxz * ltxz, lyz = Syz * ltyz;
  X.apply({lxx, lw, lxy, lxz});
  Y.apply({lyy, lw, lxy, lyz});
  Z.apply({lzz, lw, lxz, lyz});
  // FP64 gradient sums: dJ/dK += lambda(output) x (forward term), kernel.cu:484-490
  const double divu = (double)X.E[0] + Y.E[0] + Z.E[0], divw = (double)X.E[1] + Y.E[1] + Z.E[1];
  g[0] += -(double)lp * divu;
  g[1] += -(double)lp * divw;
  g[2] += (double)ltxx * (Y.E[0] + Z.E[0]) + (double)ltyy * (X.E[0] + Z.E[0]) + (double)ltzz * (X.E[0] + Y.E[0]);
  g[3] += (double)ltxx * X.E[0] + (double)ltyy * Y.E[0] + (double)ltzz * Z.E[0];
  g[4] += ((double)ltxx + ltyy + ltzz) * divw;
  g[5] += (double)ltxy * (Y.E[2] + X.E[2]);
  g[6] += (double)ltxz * (Z.E[2] + X.E[3]);
  g[7] += (double)ltyz * (Z.E[3] + Y.E[3]);
  // stores
#pragma unroll
  for (int f = 0; f < 7; ++f) at<A>(a.lam[6 + f], c) = l[f];
  const A lE[7] = {lxx, lyy, lzz, lw, lxy, lxz, lyz};
#pragma unroll
  for (int d = 0; d < 7; ++d) at<A>(a.gt[d], c) = lE[d];
  X.store(a);
  Y.store(a);
  Z.store(a);
  gstore<A, 8>(a, a.gpt, c, K_P1, g);
}

// lambda(v', q') += transposed differences of the stress-half G; then the local part of the
// velocity half of state q's step
template <typename S, int ORDER, class AT, class IT>
__device__ __forceinline__ void adj_velocity(const AT &a, const IT &j, int q, int it, u32 blk, u32 t)
{
  using A = typename AdjT<S>::A;
  constexpr int h = ORDER / 2;
  CellIdx ci;
  if (!cell_of(a, h, blk, t, ci)) return;
  const u32 c = ci.c;
  constexpr int kU1[3] = {K_U1X, K_U1Y, K_U1Z}, kU2[3] = {K_U2X, K_U2Y, K_U2Z};
  constexpr int kW1[3] = {K_W1X, K_W1Y, K_W1Z}, kW2[3] = {K_W2X, K_W2Y, K_W2Z};
  constexpr int kW3[3] = {K_W3X, K_W3Y, K_W3Y};  // qz takes W3y (kernel.cu:220)
  A l[6], lv[3], lq[3];  // vx vy vz qx qy qz
#pragma unroll
  for (int m = 0; m < 6; ++m) l[m] = at<A>(a.lam[m], c);
  inject<A, 0>(j, c, it, l);
  A gx[4], gy[4], gz[4];  // uxx wx uyx uzx | uyy wy uxy uzy | uzz wz uxz uyz
  gather_axis<A, ORDER, false, 0>(a, ci, gx);
  phase();
  gather_axis<A, ORDER, false, 1>(a, ci, gy);
  phase();
  gather_axis<A, ORDER, false, 2>(a, ci, gz);
  lv[0] = l[0] + (gx[0] + gy[2] + gz[2]);
  lv[1] = l[1] + (gy[0] + gx[2] + gz[3]);
  lv[2] = l[2] + (gz[0] + gx[3] + gy[3]);
  lq[0] = l[3] + gx[1];
  lq[1] = l[4] + gy[1];
  lq[2] = l[5] + gz[1];
  phase();
  AxisLocal<S, ORDER, true, 0> X;  // x1 s1 y2 z2
  AxisLocal<S, ORDER, true, 1> Y;  // x2 y1 s2 z3
  AxisLocal<S, ORDER, true, 2> Z;  // x3 y3 z1 s3
  X.load(a, ci, q, q);
  phase();
  Y.load(a, ci, q, q);
  phase();
  Z.load(a, ci, q, q);
  phase();
  A kv[14];  // K[0..13]: U1 xyz, U2 xyz, W1 xyz, W2 xyz, W3x, W3y
  kblock<S, 14>(a, a.kv, c, 0, kv);
  double q0[3], q1[3];
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    q0[m] = (double)at<typename AdjT<S>::T>(fw_field(a, q, 3 + m), c);  // q carries no residual
    q1[m] = (double)at<typename AdjT<S>::T>(fw_field(a, q + 1, 3 + m), c);
  }
  double gv[14];  // sums of K[0..13]
  gload<A, 14>(a, a.gpv, c, 0, gv);
  // per component: lambda_qe = lambda_q' - U2 lambda_v'; lambda_S = U1 lambda_v' - W2 lambda_qe;
  // lambda_Ds = -W3 lambda_qe (qz takes W3y, kernel.cu:220)
  A lS[3], lDs[3], lqe[3], lqn[3];
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const A U1 = kv[kU1[m]], U2 = kv[kU2[m]], W1 = kv[kW1[m]], W2 = kv[kW2[m]], W3 = kv[kW3[m]];
    lqe[m] = lq[m] - U2 * lv[m];
    lS[m] = U1 * lv[m] - W2 * lqe[m];
    lDs[m] = -W3 * lqe[m];
    lqn[m] = U2 * lv[m] + W1 * lqe[m];  // lambda_q at step n (lambda_v is unchanged)
  }
  X.apply({lS[0], lDs[0], lS[1], lS[2]});
  Y.apply({lS[0], lS[1], lDs[1], lS[2]});
  Z.apply({lS[0], lS[1], lS[2], lDs[2]});
  // FP64 gradient sums with the forward terms of kernel.cu:218-225
  const double Ssum[3] = {(double)X.E[0] + Y.E[0] + Z.E[0], (double)X.E[2] + Y.E[1] + Z.E[1],
                          (double)X.E[3] + Y.E[3] + Z.E[2]};
  const double Ds[3] = {(double)X.E[1], (double)Y.E[2], (double)Z.E[3]};
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    gv[kU1[m]] += (double)lv[m] * Ssum[m];
    gv[kU2[m]] += -(double)lv[m] * (q1[m] - q0[m]);
    gv[kW1[m]] += (double)lqe[m] * q0[m];
    gv[kW2[m]] += -(double)lqe[m] * Ssum[m];
  }
  gv[K_W3X] += -(double)lqe[0] * Ds[0];
  gv[K_W3Y] += -(double)lqe[1] * Ds[1];  // qy's term, then qz's, into the one W3y sum
  gv[K_W3Y] += -(double)lqe[2] * Ds[2];
  // stores
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    at<A>(a.lam[m], c) = lv[m];
    at<A>(a.lam[3 + m], c) = lqn[m];
    at<A>(a.gv[m], c) = lS[m];
    at<A>(a.gv[3 + m], c) = lDs[m];
  }
  X.store(a);
  Y.store(a);
  Z.store(a);
  gstore<A, 14>(a, a.gpv, c, 0, gv);
}

// the float partial sums of a segment into the FP64 gradient sums, cleared for the next one
template <typename S, int ORDER, class AT>
__device__ __forceinline__ void adj_flush(const AT &a, u32 blk, u32 t)
{
  constexpr int h = ORDER / 2;
  CellIdx ci;
  if (!cell_of(a, h, blk, t, ci)) return;
  const u32 c = ci.c;
  const uint64_t n = (uint64_t)a.nx * a.ny * a.nz;
  uint32_t dv[14], dt[8];
  packed::load<float, 14, false>(a.gpv, n, c, dv);
  packed::load<float, 8, false>(a.gpt, n, c, dt);
  double tot[NKC];
#pragma unroll
  for (int k = 0; k < NKC; ++k) tot[k] = a.grad[k][c];
#pragma unroll
  for (int k = 0; k < NKC; ++k)
    a.grad[k][c] = tot[k] + (double)(k < 14 ? packed::value<float>(dv, k) : packed::value<float>(dt, k - 14));
  const uint32_t zero[14] = {};
  packed::store<float, 14>(a.gpv, n, c, zero);
  packed::store<float, 8>(a.gpt, n, c, zero);
}

// WHICH 0: the stress pass, 1: the velocity pass, 2: the flush
template <typename S, int ORDER, int WHICH, class AT, class IT>
__device__ __forceinline__ void adj_pass(const AT &a, const IT &j, int q, int it, u32 blk, u32 t)
{
  if constexpr (WHICH == 0) adj_stress<S, ORDER>(a, j, q, it, blk, t);
  else if constexpr (WHICH == 1) adj_velocity<S, ORDER>(a, j, q, it, blk, t);
  else adj_flush<S, ORDER>(a, blk, t);
}

// 256 cells a block, dealt out to the XCDs in runs of blocks as the forward kernels' tiles are
template <typename S, int ORDER, int WHICH>
__global__ void __launch_bounds__(ADJ_BX * ADJ_BZ) k_adj(const AdjArgs a, const InjectArgs j, int q, int it, int xg)
{
  const u32 blk = (u32)xcd_tile(blockIdx.x & 7, blockIdx.x >> 3, xg);
  if (blk < (u32)a.blocks) adj_pass<S, ORDER, WHICH>(a, j, q, it, blk, threadIdx.x);
}

// batched: argument tables read through the constant address space (uniform per block)
typedef __attribute__((address_space(4))) const AdjArgs CAdjArgs;
typedef __attribute__((address_space(4))) const int CInt;
typedef __attribute__((address_space(4))) const InjectArgs CInjectArgs;
typedef __attribute__((address_space(4))) const CopyEntry CCopyEntry;

__device__ __forceinline__ int shot_of_block(const AdjBatch &b, int blk)
{
  CInt *bs = (CInt *)b.block_start;
  int lo = 0, hi = b.nshots - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (bs[mid] <= blk) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

template <typename S, int ORDER, int WHICH>
__global__ void __launch_bounds__(ADJ_BX * ADJ_BZ) k_adj_batch(const AdjBatch b, int q, int it, int xg)
{
  const int blk = xcd_tile(blockIdx.x & 7, blockIdx.x >> 3, xg);
  if (blk >= b.total_blocks) return;
  const int s = shot_of_block(b, blk);
  const CAdjArgs &a = ((CAdjArgs *)b.shots)[s];
  const CInjectArgs &j = ((CInjectArgs *)b.inject)[s];
  adj_pass<S, ORDER, WHICH>(a, j, q, it, (u32)(blk - ((CInt *)b.block_start)[s]), threadIdx.x);
}

// J = 1/2 sum (d - obs)^2 in FP64, residual = d - obs
template <typename T>
__global__ void __launch_bounds__(256) k_misfit(const T *d, const float *obs, float *res, int64_t n, double *J)
{
  __shared__ double part[256];
  double acc = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const double r = (double)d[i] - (double)obs[i];
    if (res) res[i] = (float)r;
    acc += 0.5 * r * r;
  }
  part[threadIdx.x] = acc;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) part[threadIdx.x] += part[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(J, part[0]);
}

// ---- chain rule (the gather form of the host chain in biot_params.cpp) ----
__device__ __forceinline__ double harmonic4(double a, double b, double c, double d)
{
  if (a == 0 || b == 0 || c == 0 || d == 0) return 0.0;
  return 1.0 / (0.25 * (1 / a + 1 / b + 1 / c + 1 / d));
}

// One thread per window cell p sums what every coefficient that reads p's parameters passes
// back to it (the cells p and, one step down each axis the coefficient averages over, the cells
// below), so a cell's six gradients are written once, in a fixed order.  It runs once a gradient
// and is bound by its FP64 divisions: 0.33 ms at 128^3, where the single grid's chain took about
// 170 ms on one host thread, after a copy of all 22 FP64 gradient arrays (a 128^3, 100-step
// gradient: 253 -> 76 ms).  The scatter form (each coefficient adding to the cells it reads, ~30
// FP64 atomics a cell) summed in an order that changed from run to run.
struct VelGrad {
  double gA, gB, gc2;
};
// dJ/d(rho, rho_f, rho_f tphi averages) of axis m's velocity coefficients at cell c
__device__ __forceinline__ VelGrad vel_grad(const ChainArgs &a, int64_t c, int m, const int64_t (&step)[3])
{
  const double *rho = a.par[4], *rhof = a.par[5], *C1 = a.par[6], *tphi = a.par[7];
  bool c1zero = false, azero = false;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    c1zero |= 0.5 * (C1[c] + C1[c + step[d]]) == 0;
    azero |= 0.5 * (rho[c] + rho[c + step[d]]) == 0;
  }
  const double k1 = a.Cv * a.dt / a.Cp;  // velocity coefficient scale
  const int64_t c2i = c + step[m];
  const double A = 0.5 * (rho[c] + rho[c2i]), B = 0.5 * (rhof[c] + rhof[c2i]);
  const double c1 = 0.5 * (C1[c] + C1[c2i]);
  const double c2 = 0.5 * (tphi[c] * rhof[c] + tphi[c2i] * rhof[c2i]);
  const double D = (c2 - B * B / A) + 0.5 * a.dt * c1;
  auto gK = [&](int kk) { return a.grad[kk][c] * a.kfac[kk]; };
  VelGrad g{0, 0, 0};
  if (!c1zero) {
    const double gW1 = gK(K_W1X + m), gW2 = gK(K_W2X + m);
    // W3y multiplies the pressure term of both qy and qz, so its gradient holds both;
    // W3z is never read
    const double gW3 = m < 2 ? gK(K_W3X + m) : 0.0;
    const double D2 = D * D;
    const double dW1_dmp = a.dt * c1 / D2;
    const double dW3_dmp = -k1 * a.Hinv / D2;
    const double dW2_dmp = -k1 * a.Hinv * (B / A) / D2;
    const double gmp = gW1 * dW1_dmp + gW2 * dW2_dmp + gW3 * dW3_dmp;
    g.gA += gmp * B * B / (A * A) - gW2 * k1 * a.Hinv * B / (A * A * D);
    g.gB += gmp * (-2 * B / A) + gW2 * k1 * a.Hinv / (A * D);
    g.gc2 += gmp;
  }
  if (!azero) {
    const double gU1 = gK(K_U1X + m), gU2 = gK(K_U2X + m);
    g.gA += -gU1 * k1 * a.Hinv / (A * A) - gU2 * B / (A * A);
    g.gB += gU2 / A;
  }
  return g;
}

__global__ void __launch_bounds__(256) k_chain(const ChainArgs a)
{
  const int64_t wsy = a.wx, wsz = (int64_t)a.wx * a.wy;
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= wsz * a.wz) return;
  const int pos[3] = {(int)(p % a.wx), (int)((p / a.wx) % a.wy), (int)(p / wsz)};
  const int dims[3] = {a.wx, a.wy, a.wz};
  const int64_t step[3] = {1, wsy, wsz};
  // whether the cell dx, dy, dz steps below p has coefficients (the cells off the window's outer
  // planes do)
  auto holds = [&](int dx, int dy, int dz) {
    const int d[3] = {dx, dy, dz};
    bool ok = true;
#pragma unroll
    for (int m = 0; m < 3; ++m) ok = ok && pos[m] - d[m] >= 1 && pos[m] - d[m] < dims[m] - 1;
    return ok;
  };
  const double *mu = a.par[1], *alp = a.par[2], *M = a.par[3], *tphi = a.par[7];
  const double kk = a.dt * a.Cp / a.Cv;  // stress coefficient scale
  double g[6] = {0, 0, 0, 0, 0, 0};      // lambda mu alpha M rho rho_f
  if (holds(0, 0, 0)) {
    // stress side: K_P1 = C kk/dx, K_P2 = M kk/dx, K_S1 = lambda_c .., K_S2 = H .., K_S3 = C ..
    auto gK = [&](int k) { return a.grad[k][p] * a.kfac[k]; };
    const double al = alp[p], Mp = M[p];
    const double gC = (gK(K_P1) + gK(K_S3)) * kk * a.Hinv;
    const double glc = gK(K_S1) * kk * a.Hinv;
    const double gH = gK(K_S2) * kk * a.Hinv;
    const double gMd = gK(K_P2) * kk * a.Hinv;
    g[0] = glc + gH;
    g[1] = 2 * gH;
    g[2] = gC * Mp + (glc + gH) * 2 * al * Mp;
    g[3] = gMd + gC * al + (glc + gH) * al * al;
  }
  // shear: 4-cell harmonic means, d mu_bar / d mu_i = mu_bar^2 / (4 mu_i^2); p is a corner of
  // four quads in each coordinate plane
  constexpr int ax[3][2] = {{0, 1}, {0, 2}, {1, 2}};
  constexpr int kidx[3] = {K_SXY, K_SXZ, K_SYZ};
  const double mp = mu[p];
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const int64_t sa = step[ax[m][0]], sb = step[ax[m][1]];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      int d[3] = {0, 0, 0};
      d[ax[m][0]] = e & 1;
      d[ax[m][1]] = e >> 1;
      if (!holds(d[0], d[1], d[2])) continue;
      const int64_t c = p - (e & 1) * sa - (e >> 1) * sb;
      const double hm = harmonic4(mu[c], mu[c + sa], mu[c + sb], mu[c + sa + sb]);
      if (hm == 0) continue;
      g[1] += a.grad[kidx[m]][c] * a.kfac[kidx[m]] * kk * a.Hinv * hm * hm / (4 * mp * mp);
    }
  }
  // velocity side: p is the lower or the upper cell of each axis's averages
#pragma unroll
  for (int m = 0; m < 3; ++m)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      int d[3] = {0, 0, 0};
      d[m] = e;
      if (!holds(d[0], d[1], d[2])) continue;
      const VelGrad v = vel_grad(a, p - e * step[m], m, step);
      g[4] += 0.5 * v.gA;
      g[5] += 0.5 * v.gB + 0.5 * v.gc2 * tphi[p];
    }
  const int64_t o = (a.x0 + pos[0]) + (a.y0 + pos[1]) * a.msy + (a.z0 + pos[2]) * a.msz;
#pragma unroll
  for (int q = 0; q < 6; ++q) a.out[q][o] = a.add ? a.out[q][o] + g[q] : g[q];
}

// ---- batched state copies ----
__global__ void __launch_bounds__(256) k_copy_batch(const CopyEntry *tab)
{
  const CCopyEntry &e = ((CCopyEntry *)tab)[blockIdx.y];
  const uint64_t words = e.bytes >> 2;
  const uint32_t *src = (const uint32_t *)e.src;
  uint32_t *dst = (uint32_t *)e.dst;
  for (uint64_t w = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; w < words;
       w += (uint64_t)gridDim.x * blockDim.x)
    dst[w] = src[w];
  const uint32_t rem = (uint32_t)(e.bytes & 3);
  if (blockIdx.x == 0 && threadIdx.x < rem)
    ((uint8_t *)e.dst)[(words << 2) + threadIdx.x] = ((const uint8_t *)e.src)[(words << 2) + threadIdx.x];
}

struct SingleRun {
  const AdjArgs &a;
  const InjectArgs &j;
  int q, it;
  hipStream_t s;
  template <typename S, int O, int W>
  void pass()
  {
    const int xg = xcd_run(a.blocks, ADJ_BX * ADJ_BZ, (int64_t)a.blocks * ADJ_BX * ADJ_BZ);
    hipLaunchKernelGGL((k_adj<S, O, W>), dim3((unsigned)(8 * xcd_slots(a.blocks, xg))), dim3(ADJ_BX * ADJ_BZ), 0, s, a,
                       j, q, it, xg);
  }
};
struct BatchRun {
  const AdjBatch &b;
  int q, it;
  hipStream_t s;
  template <typename S, int O, int W>
  void pass()
  {
    const int xg = xcd_run(b.total_blocks, ADJ_BX * ADJ_BZ, (int64_t)b.total_blocks * ADJ_BX * ADJ_BZ);
    hipLaunchKernelGGL((k_adj_batch<S, O, W>), dim3((unsigned)(8 * xcd_slots(b.total_blocks, xg))), dim3(ADJ_BX * ADJ_BZ), 0, s, b,
                       q, it, xg);
  }
};

template <typename S, int O, class F>
hipError_t run_passes(F f, bool flush)
{
  if (flush) {
    f.template pass<S, O, 2>();
  } else {
    f.template pass<S, O, 0>();
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    f.template pass<S, O, 1>();
  }
  return hipGetLastError();
}
// the passes for the storage type of prec
template <class F>
hipError_t passes(int prec, int order, F f, bool flush)
{
  if (order != 2 && order != 4) return hipErrorInvalidValue;
  if (prec == PREC_FP32) return order == 2 ? run_passes<float, 2>(f, flush) : run_passes<float, 4>(f, flush);
  if (prec == PREC_FP64) return order == 2 ? run_passes<double, 2>(f, flush) : run_passes<double, 4>(f, flush);
  if (prec == PREC_FP16) return order == 2 ? run_passes<_Float16, 2>(f, flush) : run_passes<_Float16, 4>(f, flush);
  if (prec == PREC_FP16T)
    return order == 2 ? run_passes<H16R<COMP_FIELDS_T>, 2>(f, flush) : run_passes<H16R<COMP_FIELDS_T>, 4>(f, flush);
  if (prec == PREC_FP16C)
    return order == 2 ? run_passes<H16R<COMP_FIELDS_C>, 2>(f, flush) : run_passes<H16R<COMP_FIELDS_C>, 4>(f, flush);
  if (prec == PREC_FP16M) return order == 2 ? run_passes<H16P, 2>(f, flush) : run_passes<H16P, 4>(f, flush);
  return hipErrorInvalidValue;
}
}  // namespace

hipError_t launch_adjoint_step(int prec, int order, const AdjArgs &a, const InjectArgs &j, int q, int it, hipStream_t s)
{
  if (a.blocks == 0) return hipSuccess;
  return passes(prec, order, SingleRun{a, j, q, it, s}, false);
}

hipError_t launch_adjoint_flush(int prec, int order, const AdjArgs &a, hipStream_t s)
{
  if (a.blocks == 0 || prec == PREC_FP64) return hipSuccess;
  return passes(prec, order, SingleRun{a, InjectArgs{}, 0, 0, s}, true);
}

hipError_t launch_adjoint_flush_batch(int prec, int order, const AdjBatch &b, hipStream_t s)
{
  if (b.total_blocks <= 0 || prec == PREC_FP64) return hipSuccess;
  return passes(prec, order, BatchRun{b, 0, 0, s}, true);
}

hipError_t launch_adjoint_step_batch(int prec, int order, const AdjBatch &b, int q, int it, hipStream_t s)
{
  if (b.total_blocks <= 0) return hipSuccess;
  return passes(prec, order, BatchRun{b, q, it, s}, false);
}

hipError_t launch_misfit(const void *d, bool d_double, const float *obs, float *res, int64_t n,
                         double *J, hipStream_t s)
{
  if (n <= 0) return hipSuccess;
  const unsigned blocks = (unsigned)std::min<int64_t>((n + 255) / 256, 4096);
  if (d_double)
    hipLaunchKernelGGL(k_misfit<double>, dim3(blocks), dim3(256), 0, s, (const double *)d, obs, res, n, J);
  else
    hipLaunchKernelGGL(k_misfit<float>, dim3(blocks), dim3(256), 0, s, (const float *)d, obs, res, n, J);
  return hipGetLastError();
}

hipError_t launch_chain(const ChainArgs &c, hipStream_t s)
{
  const int64_t nw = (int64_t)c.wx * c.wy * c.wz;
  if (nw <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_chain, dim3((unsigned)((nw + 255) / 256)), dim3(256), 0, s, c);
  return hipGetLastError();
}

hipError_t launch_copy_batch(const CopyEntry *tab, int n, hipStream_t s)
{
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_copy_batch, dim3(1024, (unsigned)n), dim3(256), 0, s, tab);
  return hipGetLastError();
}

}  // namespace biot
