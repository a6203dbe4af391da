// Apply of dt*nu K + sigma M on structured meshes from two factors per element
// (ApplyDesc::ef), on the FP64 matrix units (gfx950).  First box elements:
//
// The operator is that of hc_apply.hip (EquationSystem::Mult,
// src/equation_systems/equation_system.cpp:200-204, on the system of
// FormLinearSystem, equation_system.cpp:132-190).  On a box element with
// J = diag(h) its integrals separate, and the p + 1 point rule integrates
// them exactly, so they are written with the exact 1-D matrices:
//   Mc  closed mass matrix (p + 1 Gauss-Lobatto points),
//   W   open mass matrix: diagonal, the Gauss-Legendre weights, because the
//       Lagrange basis on the p Gauss points is orthogonal,
//   Dg  the derivative of a closed 1-D function at the open points, which is
//       exact because it has degree p - 1.
// The curl of an ND field is then three differences (Dg along one axis), its
// mass matrix one contraction and two weights, and its transpose the same
// differences again:
//   c_x = D_y u_z - D_z u_y,  c_y = D_z u_x - D_x u_z,  c_z = D_x u_y - D_y u_x
//   f_a = dt nu ck_a Mc_a W W c_a,   ck_a = h_a^2 / |det J|
//   y_x = sigma mk_0 W Mc_y Mc_z u_x + D_z^T f_y - D_y^T f_z   (and cyclic)
// with no quadrature-point values: at order 3 about 220 multiply-adds of 4-wide
// contractions per 16 lanes and element layer against 600 for interpolation to
// the quadrature points and back.
//
// One 16-lane block of a wave holds the 4 x 4 (x, y) points of an element
// (orders 2 and 3; 2 x 2 elements at order 1, block-diagonal matrices), the z
// points are in registers.  A contraction along x or y of one plane is one
// v_mfma_f64_4x4x4_4b (four independent 4 x 4 products, one per 16-lane
// block); along z it is register arithmetic with compile-time tables.  Lane
// layouts (fast lane index f = lane % 4, slow s = lane / 16, block
// (lane / 4) % 4): "N" f = x, s = y; "T" f = y, s = x.  The instruction takes
// A[f][s], B[s][f] and returns D[s][f], so a value used as B is contracted
// along its slow axis and keeps its layout, used as A it is contracted along
// its slow axis and comes back transposed; no lane exchange is needed except
// for u_z and f_z (a product with the identity).
//
// A workgroup owns a column of tiles: ns elements (cx by cy) marched along z.
// The top plane of a layer is carried to the next one in registers; the face
// values of x and y neighbours meet in LDS (one barrier per layer, two
// buffers).  Elements on the lower x, y and z faces of a tile are computed by
// both tiles, so every output DOF is summed by one workgroup in a fixed order:
// one launch, no partial sums in memory, and the same bits for every tile
// shape.
//
// Trilinear elements (HEX; ApplyDesc::ef with vertices) march the same way, but
// their integrals do not separate: u is interpolated to the (p + 1)^3 points by
// matrix products along y and x and register arithmetic along z, the lane keeps
// its (x, y) point, takes the Jacobian there from the corners of the lower and
// upper vertex plane (the upper is carried to the next layer), applies mass and
// curl factors (adj(J^T J) sigma w / |det J| and J^T J dt nu w / |det J|) and the
// transposed stages follow.  Against 12 (p + 1)^3 stored factors per element
// read by the tile kernel of hc_apply_qp.hip this reads 24 bytes a vertex and 16
// an element.  About 680 FP64 vector instructions and 86 matrix products a layer
// at order 3 (480 and 62 at order 2) keep 244 registers, so two waves per SIMD
// and tiles of at most 32 elements, of whose work 1.5 x 1.1 is duplicated.  At
// 33x26x19 order 2 a SIMD issues vector instructions and products for 12 of 24 us;
// the rest is latency with two waves.  Measured, stored factors -> here: 48^3
// order 3 223 -> 157 us, 48^3 order 2 118 -> 106 us, 33x26x19 order 2 30 -> 24 us,
// 64^3 order 1 80 -> 38 us, 16^3 order 1 12 -> 7.4 us.  Error against extended precision over
// 40 meshes of 6x5x4 to 44x34x20: 9.1e-16 -> 7.2e-16 in the mean (the stored
// factors take the Jacobian from sums of coordinates, here from differences).
//
// The mass term alone (BOX_MASS: 10 matrix products a layer instead of 39 at
// order 2) and the product added to y (BOX_ADD) save the A-V block operator the
// curl of its mass product and its closing pass: 31x37x29 order 2 59 -> 47 us.
//
// Measured on boxes at 48^3 order 3 (9.08 M DOFs): 194 us per FP64 apply with the
// LDS-staged tile kernel and its face assembly, 69 us here (FP32 vectors: 114
// and 60 us).  Memory traffic is 160 MB (147 MB algorithmic, 30 us at the copy
// rate).  By the counters a layer takes 55 products (16 cycles each on a SIMD) and
// 248 other vector instructions (4 cycles; 150 of them FP64), which do not
// overlap: 14 + 16 us of the 65.  The rest is latency -- chains of dependent
// products, 152 scalar instructions and one barrier a layer, four waves per SIMD
// that 128 registers allow; the waves wait for 42 % of their cycles.  Of the work
// 1.31 x 1.08 is duplicated elements of tile and chunk faces.
#include "hc_basis.hpp"
#include "hc_kernels.hpp"

#include <algorithm>

namespace hc
{

namespace
{

// a b + c; NEG: bit 0 negates a (operand modifier of the FP64 form)
template <int NEG = 0>
__device__ inline double
mm(double a, double b, double c)
{
  return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, NEG);
}

} // namespace

// Global memory through a buffer resource at a wave-uniform base, with a 32-bit
// byte offset per lane: no vector arithmetic per access, and the hardware's
// range check takes the place of lane masks -- a lane whose offset is OOB loads
// zero and stores nothing.  Offsets are relative to the first row of a tile in
// the lowest plane of a layer (box_fits: p + 1 planes stay below 2^32 bytes; a
// mesh beyond that keeps the quadrature-point factors).
constexpr uint32_t OOB = 0xFFFFFFFFu;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

template <typename T>
__device__ inline __amdgpu_buffer_rsrc_t
rsrc(const T * p)
{
  return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, (int)(OOB - 1), 0x00027000);
}
template <typename T>
__device__ inline T
ldb(const T * base, uint32_t off, uint32_t sof = 0)
{
  if constexpr (sizeof(T) == 8)
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(rsrc(base), (int)off, (int)sof, 0));
  else
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(rsrc(base), (int)off, (int)sof, 0));
}
template <typename T>
__device__ inline void
stb(T * base, uint32_t off, T v, uint32_t sof = 0)
{
  if constexpr (sizeof(T) == 8)
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), rsrc(base), (int)off, (int)sof, 0);
  else
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), rsrc(base), (int)off, (int)sof, 0);
}

// LDS of the apply in doubles: 4 face arrays of 2 buffers and P planes, and the
// PEC values
template <int P, int NS>
constexpr int
box_lds()
{
  return 8 * P * (NS * (P == 1 ? 8 : 4) + 1) + (3 * P + 2) * 16 * NS;
}

// What a lane (f, s) of a block keeps of the 1-D matrices, by f * 4 + s.  (As
// selects over the entries this took 300 to 500 instructions of every launch.)
// Entry [f][s] of a matrix is its A operand, [s][f] its B operand; at order 1,
// where a block is 2 x 2 elements, the matrices are block-diagonal.
template <int N>
struct LaneTab
{
  double v[16][N];
};
template <int P>
constexpr LaneTab<6>
make_box_lanes()
{
  LaneTab<6> t{};
  const basis::BoxTab<P> b = basis::box_tab<P>();
  for (int f = 0; f < 4; f++)
    for (int s = 0; s < 4; s++)
    {
      const int pf = P == 1 ? f % 2 : f, ps = P == 1 ? s % 2 : s;
      double * v = t.v[f * 4 + s];
      if (pf > P || ps > P)
        continue;
      if (P > 1 || f / 2 == s / 2)
      {
        v[0] = b.M[pf][ps];
        v[1] = pf < P ? b.D[pf < P ? pf : 0][ps] : 0.0;
        v[2] = ps < P ? b.D[ps < P ? ps : 0][pf] : 0.0;
      }
      v[3] = pf < P ? b.w[pf < P ? pf : 0] : 0.0;
      v[4] = ps < P ? b.w[ps < P ? ps : 0] : 0.0;
    }
  return t;
}
// interpolation to the quadrature points (open, closed, derivative of closed),
// [f][s] and [s][f]; the lane's point (f, s) and its weight.  The lanes without
// a point of their own (order 2) take the last one's with weight zero: their
// determinant is then that of a quadrature point too, which is not zero where an
// edge of the element is collapsed (a corner's is, and 0 / 0 would spread from
// there through the matrix products).
template <int P>
constexpr LaneTab<10>
make_hex_lanes()
{
  LaneTab<10> t{};
  const basis::Tab<double> b = basis::tab<P, double>();
  for (int f = 0; f < 4; f++)
    for (int s = 0; s < 4; s++)
    {
      const int pf = P == 1 ? f % 2 : f, ps = P == 1 ? s % 2 : s;
      double * v = t.v[f * 4 + s];
      v[6] = b.qp[pf < P ? pf : P];
      v[7] = b.qp[ps < P ? ps : P];
      if (pf > P || ps > P)
        continue;
      if (P > 1 || f / 2 == s / 2)
      {
        v[0] = ps < P ? b.Bo[pf * P + (ps < P ? ps : 0)] : 0.0;
        v[1] = b.Bc[pf * (P + 1) + ps];
        v[2] = b.Gc[pf * (P + 1) + ps];
        v[3] = pf < P ? b.Bo[ps * P + (pf < P ? pf : 0)] : 0.0;
        v[4] = b.Bc[ps * (P + 1) + pf];
        v[5] = b.Gc[ps * (P + 1) + pf];
      }
      v[8] = b.qw[pf] * b.qw[ps];
    }
  return t;
}
template <int P>
__device__ constexpr LaneTab<6> box_lanes = make_box_lanes<P>();
template <int P>
__device__ constexpr LaneTab<10> hex_lanes = make_hex_lanes<P>();

// The corners (x, y) of an element on one vertex plane as they enter the
// trilinear map at reference point (a, b): the point, relative to corner (0, 0),
// and the two in-plane derivatives.  (Differences of coordinates are taken
// first throughout, so that the relative error does not grow with 1 / h.)
struct PlaneGeom
{
  double p[3], dx[3], dy[3];
};
__device__ inline PlaneGeom
plane_geom(const double * v, double a, double b)
{
#pragma clang fp contract(off)
  PlaneGeom g;
#pragma unroll
  for (int r = 0; r < 3; r++)
  {
    const double v00 = v[r], v10 = v[3 + r], v01 = v[6 + r], v11 = v[9 + r];
    const double e0 = v10 - v00, e1 = v11 - v01; // along x at y = 0, 1
    g.dx[r] = __builtin_fma(b, e1 - e0, e0);
    const double f0 = v01 - v00, f1 = v11 - v10; // along y at x = 0, 1
    g.dy[r] = __builtin_fma(a, f1 - f0, f0);
    g.p[r] = __builtin_fma(b, g.dy[r], a * e0);
  }
  return g;
}

// dt nu and sigma of a lane's element in the N and the T layout
struct Coef
{
  double nuN, sgN, nuT, sgT;
};

// The right-hand sides [r_begin, r_end) of tile `tile` of one instance.
template <int P, typename T, int NS, bool TABLE, int KIND, bool HEX>
__device__ __forceinline__ void
box_body(const ApplyDesc & ad, int tile, int r_begin, int r_end, double * lds)
{
#pragma clang fp contract(off)
  constexpr basis::BoxTab<P> tb = basis::box_tab<P>();
  constexpr int EJ = (P == 1) ? 2 : 1; // elements per axis in a 16-lane block
  constexpr int FS = 4 * EJ;           // face values per block, plane and array
  constexpr uint32_t SZ = sizeof(T);
  const Geom & g = ad.g;
  const int bcx = ad.bt.cx, bcy = ad.bt.cy;
  const int tx = tile % ad.bt.ntx;
  tile /= ad.bt.ntx;
  const int ty = tile % ad.bt.nty, tz = tile / ad.bt.nty;

  // face values; entry NS * FS is the zero that lanes without a neighbour add
  constexpr int FZ = NS * FS;
  using Face = double[P][FZ + 1];
  Face * const sX = (Face *)lds, * const sY = sX + 2, * const sZR = sX + 4, * const sZC = sX + 6;
  if (threadIdx.x < 2 * P)
  {
    const int b = threadIdx.x / P, k = threadIdx.x % P;
    sX[b][k][FZ] = sY[b][k][FZ] = sZR[b][k][FZ] = sZC[b][k][FZ] = 0.0;
  }

  const int lane = threadIdx.x & 63;
  const int lf = lane & 3, ls = lane >> 4;
  const int slot = (threadIdx.x >> 6) * 4 + ((lane >> 2) & 3);
  const int sx = slot % bcx, sy = slot / bcx;
  const int nx = g.n[0], ny = g.n[1], nz = g.n[2];
  const int xs = tx * (bcx * EJ - 1), ys = ty * (bcy * EJ - 1); // first computed element
  const int z0 = tz * ad.bt.zc, z1 = min(nz, z0 + ad.bt.zc);
  const int zs = z0 - (z0 > 0 ? 1 : 0);
  const bool sact = sy < bcy;
  const int pec = g.pec;

  // element and local point of this lane on each axis: index f / s of the lane
  const int ef = (P == 1) ? (lf >> 1) : 0, pf = (P == 1) ? (lf & 1) : lf;
  const int es = (P == 1) ? (ls >> 1) : 0, ps = (P == 1) ? (ls & 1) : ls;
  // N layout: x from f, y from s.  T layout: x from s, y from f.
  const int exN = xs + sx * EJ + ef, eyN = ys + sy * EJ + es;
  const int exT = xs + sx * EJ + es, eyT = ys + sy * EJ + ef;
  const bool vN = sact && exN < nx && eyN < ny, vT = sact && exT < nx && eyT < ny;
  auto face = [&](int axis, int gi, int n) {
    return (gi == 0 && ((pec >> (2 * axis)) & 1)) || (gi == n * P && ((pec >> (2 * axis + 1)) & 1));
  };
  const bool essx = face(1, eyN * P + ps, ny), essy = face(0, exN * P + pf, nx), essz = essx || essy;
  const bool essyL = HEX ? essy : face(0, exT * P + ps, nx); // lanes as they load u_y
  // lanes that read a DOF of the component, and those that write it
  const bool ldx = vN && pf < P && ps <= P, ldz = vN && pf <= P && ps <= P;
  const bool ldy = HEX ? vN && pf <= P && ps < P : vT && pf < P && ps <= P;
  const bool outN = vN && (exN > xs || tx == 0) && (eyN > ys || ty == 0);
  const bool topx = pf == P && exN == nx - 1, topy = ps == P && eyN == ny - 1;
  const bool ownx = outN && pf < P && (ps < P || topy);
  const bool owny = outN && ps < P && (pf < P || topx);
  const bool ownz = outN && (pf < P || topx) && (ps < P || topy);
  // some lane of the wave holds a PEC DOF of an x or y face; their values are
  // kept in LDS from load to store (own lane, component y transposed): planes
  // 1 .. p-1 of x and y and p planes of z of the layer, and the lowest plane of
  // x and y of the layer (by parity of z: the one above is known a layer early)
  const bool wave_ess = __any((vN && essz) || (vT && essyL)) != 0;
  using PecRow = double[16 * NS];
  PecRow * const sE = (PecRow *)(sX + 8);
  constexpr int EX = 0, EY = P - 1, EZ = 2 * P - 2, EX0 = 3 * P - 2, EY0 = 3 * P;
  const int eN = threadIdx.x, eT = HEX ? eN : (int)((threadIdx.x & ~51) | (lf << 4) | ls);
  // byte offsets inside a plane of each component, from the tile's first row
  const uint32_t cx0 = (uint32_t)g.cd[0][0], cy0 = (uint32_t)g.cd[1][0], cz0 = (uint32_t)g.cd[2][0];
  const uint32_t lxN = (sx * EJ + ef) * P + pf, lyN = (sy * EJ + es) * P + ps;
  const uint32_t oxN = (lyN * cx0 + lxN) * SZ, oyN = (lyN * cy0 + lxN) * SZ, ozN = (lyN * cz0 + lxN) * SZ;
  const uint32_t oyL = HEX ? oyN : (((sy * EJ + ef) * P + pf) * cy0 + (sx * EJ + es) * P + ps) * SZ;
  const uint32_t ilx = ldx ? oxN : OOB, ily = ldy ? oyL : OOB, ilz = ldz ? ozN : OOB; // loads
  // entries of a plane of each component
  const int64_t plx = g.cd[0][0] * g.cd[0][1], ply = g.cd[1][0] * g.cd[1][1], plz = g.cd[2][0] * g.cd[2][1];
  const uint32_t spx = (uint32_t)plx * SZ, spy = (uint32_t)ply * SZ, spz = (uint32_t)plz * SZ; // plane bytes
  const int64_t orgx = g.off[0] + (int64_t)ys * P * cx0 + xs * P;
  const int64_t orgy = g.off[1] + (int64_t)ys * P * cy0 + xs * P;
  const int64_t orgz = g.off[2] + (int64_t)ys * P * cz0 + xs * P;

  // face exchange: where this lane writes its upper faces and where it finds
  // the values of the element to the left (x - 1), below (y - 1) and diagonal
  const int wR = (slot * EJ + es) * 4 + lf; // row s = P, by x
  const int wC = (slot * EJ + ef) * 4 + ls; // column f = P, by y
  const bool hasL = pf == 0 && exN > xs, hasB = ps == 0 && eyN > ys;
  const int slL = (P == 1 && ef == 1) ? slot : slot - 1, slB = (P == 1 && es == 1) ? slot : slot - bcx;
  const int eL = (P == 1) ? 1 - ef : 0, eB = (P == 1) ? 1 - es : 0;
  const int rL = hasL ? (slL * EJ + eL) * 4 + ls : FZ;
  const int rB = hasB ? (slB * EJ + eB) * 4 + lf : FZ;
  // diagonal: row P of the element below the left one, at its x point P
  const int slD = (P == 1 && es == 1) ? slL : slL - bcx;
  const int rD = (hasL && hasB) ? (slD * EJ + eB) * 4 + ((P == 1) ? 2 * eL + 1 : P) : FZ;

  // matrix operands: lane (f, s) holds entry [f][s] as A and [s][f] as B
  const int lane16 = lf * 4 + ls;
  double opM = 0, opD = 0, opDt = 0, wf = 0, wsl = 0;
  if constexpr (!HEX)
  {
    const double * lo = box_lanes<P>.v[lane16];
    opM = lo[0];
    opD = lo[1]; // [open f][closed s]
    opDt = lo[2]; // [open s][closed f]
    wf = lo[3];
    wsl = lo[4];
  }
  const double opI = (lf == ls) ? 1.0 : 0.0;
  // lane weights of the element factors (mass x, y, z; curl x, y, z): the
  // weights of x and y are equal per axis up to the axis constants
  const double msc = ad.mscale, csc = ad.cscale;
  const double mk0 = ad.ef.mk[0] * msc, mk1 = ad.ef.mk[1] * msc, mk2 = ad.ef.mk[2] * msc;
  const double ck0 = ad.ef.ck[0] * csc, ck1 = ad.ef.ck[1] * csc, ck2 = -(ad.ef.ck[2] * csc);
  const double wfs = wf * wsl;
  // trilinear elements: interpolation to the quadrature points and its
  // transpose (operand entries [f][s] and [s][f]), the lane's point
  constexpr basis::Tab<double> qt = basis::tab<P, double>();
  double fBo = 0, fBc = 0, fGc = 0, bBo = 0, bBc = 0, bGc = 0, qa = 0, qb = 0, wxy = 0;
  if constexpr (HEX)
  {
    const double * lo = hex_lanes<P>.v[lane16];
    fBo = lo[0];
    fBc = lo[1];
    fGc = lo[2];
    bBo = lo[3];
    bBc = lo[4];
    bGc = lo[5];
    qa = lo[6];
    qb = lo[7];
    wxy = lo[8];
  }
  // vertices: the element's corner (0, 0) on a vertex plane, from the tile's first
  const double * vert = HEX ? ad.ef.vert + 3 * ((int64_t)ys * (nx + 1) + xs) : nullptr;
  const int64_t vpl = 3 * (int64_t)(nx + 1) * (ny + 1);
  const uint32_t ov = vN ? ((uint32_t)(sy * EJ + es) * (nx + 1) + sx * EJ + ef) * 24 : OOB;
  const uint32_t ov1 = vN ? ov + (uint32_t)(nx + 1) * 24 : OOB;
  auto load_corners = [&](int z, double (&v)[15]) { // and corner (0, 0) of the plane below
    const double * b = vert + z * vpl;
#pragma unroll
    for (int r = 0; r < 3; r++)
    {
      v[r] = ldb(b, ov, r * 8);
      v[3 + r] = ldb(b, ov, 24 + r * 8);
      v[6 + r] = ldb(b, ov1, r * 8);
      v[9 + r] = ldb(b, ov1, 24 + r * 8);
      v[12 + r] = ldb(z > 0 ? b - vpl : b, ov, r * 8);
    }
  };

  const T * qc = (const T *)ad.ef.qc + 2 * ((int64_t)ys * nx + xs);
  const uint32_t oeN = vN ? ((uint32_t)(sy * EJ + es) * nx + sx * EJ + ef) * 2 * SZ : OOB;
  const uint32_t oeT = vT ? ((uint32_t)(sy * EJ + ef) * nx + sx * EJ + es) * 2 * SZ : OOB;
  const int64_t epl = 2 * (int64_t)nx * ny;

  for (int rhs = r_begin; rhs < r_end; rhs++)
  {
    if (ad.done && gmem(ad.done)[(int64_t)rhs * ad.done_stride] != ad.gate)
      continue;
    const int64_t rof = (int64_t)rhs * g.off[3];
    const T * xv = (const T *)ad.x + rof;
    // offsets (entries) of the current layer's lowest plane of each component
    int64_t bx = orgx + (int64_t)zs * P * plx, by = orgy + (int64_t)zs * P * ply, bz = orgz + (int64_t)zs * P * plz;

    double ux[P + 1], uy[P + 1]; // this layer (uy in T layout)
    T nux[P], nuy[P], nuz[P];    // next layer, as loaded
    T nq[P == 1 ? 4 : 2];
    auto load_layer = [&](int64_t ax, int64_t ay, int64_t az, int z) {
#pragma unroll
      for (int k = 0; k < P; k++)
      {
        nux[k] = ldb(xv + ax, ilx, (k + 1) * spx);
        nuy[k] = ldb(xv + ay, ily, (k + 1) * spy);
        nuz[k] = ldb(xv + az, ilz, k * spz);
      }
      const T * q = qc + z * epl;
      nq[0] = ldb(q, oeN);
      nq[1] = ldb(q + 1, oeN);
      if constexpr (P == 1 && !HEX)
      {
        nq[2] = ldb(q, oeT);
        nq[3] = ldb(q + 1, oeT);
      }
    };
    {
      const bool zf = zs == 0 && (pec & 16);
      const T vx = ldb(xv + bx, ilx), vy = ldb(xv + by, ily);
      load_layer(bx, by, bz, zs);
      ux[0] = (zf || essx) ? 0.0 : (double)vx;
      uy[0] = (zf || essyL) ? 0.0 : (double)vy;
      sE[EX0 + (zs & 1)][eN] = (double)vx;
      sE[EY0 + (zs & 1)][eT] = (double)vy;
      // stores that store nothing: in the loop the loads of the next layer are
      // followed by 3 p stores, and the wait for them may count on that only
      // if every way into the loop has them
#pragma unroll
      for (int k = 0; k < 3 * P; k++)
        stb((T *)ad.y + rof, OOB, T(0), k);
    }
    PlaneGeom g0{}; // lower vertex plane of the layer
    double nv[15] = {};
    if constexpr (HEX)
    {
      load_corners(zs, nv);
      g0 = plane_geom(nv, qa, qb);
      load_corners(zs + 1, nv);
    }
    double carx = 0.0, cary = 0.0;
    int buf = 0;
    for (int z = zs; z < z1; z++)
    {
      double uz[P];
      const bool ztop = z == nz - 1 && (pec & 32); // PEC top plane: u_x, u_y read as zero
#pragma unroll
      for (int k = 0; k < P; k++)
      {
        ux[k + 1] = (double)nux[k];
        uy[k + 1] = (double)nuy[k];
        uz[k] = (double)nuz[k];
      }
      // PEC DOFs act as zero; their values go to LDS
      const bool stash = wave_ess || (z == 0 && (pec & 16));
      if (stash)
      {
#pragma unroll
        for (int k = 0; k < P; k++)
        {
          sE[EZ + k][eN] = uz[k];
          uz[k] = essz ? 0.0 : uz[k];
          if (k < P - 1)
          {
            sE[EX + k][eN] = ux[k + 1];
            sE[EY + k][eT] = uy[k + 1];
          }
          else
          {
            sE[EX0 + ((z + 1) & 1)][eN] = ux[P];
            sE[EY0 + ((z + 1) & 1)][eT] = uy[P];
          }
          ux[k + 1] = essx ? 0.0 : ux[k + 1];
          uy[k + 1] = essyL ? 0.0 : uy[k + 1];
        }
      }
      ux[P] = ztop ? 0.0 : ux[P];
      uy[P] = ztop ? 0.0 : uy[P];
      Coef cf;
      cf.nuN = (double)nq[0];
      cf.sgN = (double)nq[1];
      cf.nuT = (P == 1 && !HEX) ? (double)nq[P == 1 ? 2 : 0] : cf.nuN;
      cf.sgT = (P == 1 && !HEX) ? (double)nq[P == 1 ? 3 : 1] : cf.sgN;
      if (!HEX && z + 1 < z1)
        load_layer(bx + P * plx, by + P * ply, bz + P * plz, z + 1);
      // upper vertex plane of the layer, and the difference along z at the lane's point
      PlaneGeom g1;
      double jz[3];
      auto upper_plane = [&]() {
        g1 = plane_geom(nv, qa, qb);
#pragma unroll
        for (int r = 0; r < 3; r++)
          jz[r] = (nv[r] - nv[12 + r]) + (g1.p[r] - g0.p[r]);
      };
      if constexpr (HEX && P == 1)
        upper_plane();

      // the element products y = A_e u of the layer (first: with the loads of the
      // next one in the trilinear form; lanes without `use` have no element)
      double yx[P + 1], yy[P + 1], yz[P];
      auto products = [&](const double (&ux)[P + 1], const double (&uy)[P + 1], const double (&uz_)[P], const Coef & c, bool use,
                          auto first) {
      constexpr bool FIRST = decltype(first)::value;
      const double nuN = c.nuN, sgN = c.sgN, nuT = c.nuT, sgT = c.sgT;
      double uz[P];
#pragma unroll
      for (int k = 0; k < P; k++)
        uz[k] = uz_[k];
      if constexpr (HEX)
      {
        auto phase = []() { __builtin_amdgcn_sched_barrier(0); };
        constexpr int Q = P + 1;
        // x, y interpolation (y first: N -> T -> N): values and x, y derivatives
        double ux0[P + 1], uxy[P + 1], uy0[P + 1], uyx[P + 1], uz0[P], uzx[P], uzy[P];
#pragma unroll
        for (int k = 0; k <= P; k++)
        {
          const double a = mm(ux[k], fBc, 0.0), b = mm(ux[k], fGc, 0.0), c = mm(uy[k], fBo, 0.0);
          ux0[k] = mm(a, fBo, 0.0);
          uxy[k] = mm(b, fBo, 0.0);
          uy0[k] = mm(c, fBc, 0.0);
          uyx[k] = mm(c, fGc, 0.0);
        }
#pragma unroll
        for (int k = 0; k < P; k++)
        {
          const double a = mm(uz[k], fBc, 0.0), b = mm(uz[k], fGc, 0.0);
          uz0[k] = mm(a, fBc, 0.0);
          uzx[k] = mm(a, fGc, 0.0);
          uzy[k] = mm(b, fBc, 0.0);
        }
        phase();
        if constexpr (P > 1)
          upper_plane();
        const double sm0 = wxy * (sgN * msc), sc0 = wxy * (nuN * csc);
        // sums over the quadrature points along z of the transposed stage:
        // (value, y derivative) of x, (value, x derivative) of y, (value, x, y) of z
        double sx0[P + 1] = {}, sxy[P + 1] = {}, sy0[P + 1] = {}, syx[P + 1] = {}, sz0[P] = {}, szx[P] = {}, szy[P] = {};
#pragma unroll
        for (int q = 0; q < Q; q++)
        {
          double w0 = 0.0, w1 = 0.0, w2 = 0.0, c0 = 0.0, c1 = 0.0, c2 = 0.0;
#pragma unroll
          for (int k = 0; k <= P; k++)
          {
            const double Bc = qt.Bc[q * (P + 1) + k], Gc = qt.Gc[q * (P + 1) + k];
            w0 = __builtin_fma(Bc, ux0[k], w0);
            w1 = __builtin_fma(Bc, uy0[k], w1);
            c0 = __builtin_fma(-Gc, uy0[k], c0); // - d/dz u_y
            c1 = __builtin_fma(Gc, ux0[k], c1);  // + d/dz u_x
            c2 = __builtin_fma(Bc, uyx[k], c2);  // + d/dx u_y
            c2 = __builtin_fma(-Bc, uxy[k], c2); // - d/dy u_x
          }
#pragma unroll
          for (int k = 0; k < P; k++)
          {
            const double Bo = qt.Bo[q * P + k];
            w2 = __builtin_fma(Bo, uz0[k], w2);
            c0 = __builtin_fma(Bo, uzy[k], c0);  // + d/dy u_z
            c1 = __builtin_fma(-Bo, uzx[k], c1); // - d/dx u_z
          }
          // J = (d/dx, d/dy, d/dz) of the map; mass adj(J^T J) / |det|, curl J^T J / |det|
          double jx[3], jy[3];
#pragma unroll
          for (int r = 0; r < 3; r++)
          {
            jx[r] = __builtin_fma(qt.qp[q], g1.dx[r] - g0.dx[r], g0.dx[r]);
            jy[r] = __builtin_fma(qt.qp[q], g1.dy[r] - g0.dy[r], g0.dy[r]);
          }
          auto dot = [](const double * u, const double * v) {
            return __builtin_fma(u[0], v[0], __builtin_fma(u[1], v[1], u[2] * v[2]));
          };
          const double G00 = dot(jx, jx), G01 = dot(jx, jy), G02 = dot(jx, jz);
          const double G11 = dot(jy, jy), G12 = dot(jy, jz), G22 = dot(jz, jz);
          const double cr[3] = {__builtin_fma(jy[1], jz[2], -(jy[2] * jz[1])), __builtin_fma(jy[2], jz[0], -(jy[0] * jz[2])),
                                __builtin_fma(jy[0], jz[1], -(jy[1] * jz[0]))};
          const double det = __builtin_fabs(dot(jx, cr));
          const double rd = qt.qw[q] / (use ? det : 1.0); // (lanes without a point carry zeros)
          const double sm = sm0 * rd, sc = sc0 * rd;
          const double A00 = __builtin_fma(G11, G22, -(G12 * G12)), A01 = __builtin_fma(G02, G12, -(G01 * G22));
          const double A02 = __builtin_fma(G01, G12, -(G02 * G11)), A11 = __builtin_fma(G00, G22, -(G02 * G02));
          const double A12 = __builtin_fma(G01, G02, -(G00 * G12)), A22 = __builtin_fma(G00, G11, -(G01 * G01));
          auto row = [](double a, double b, double c, double u, double v, double w) {
            return __builtin_fma(a, u, __builtin_fma(b, v, c * w));
          };
          // (the diagonal term, the largest, is added last)
          const double m0 = sm * row(A00, A01, A02, w0, w1, w2), m1 = sm * row(A11, A01, A12, w1, w0, w2);
          const double m2 = sm * row(A22, A02, A12, w2, w0, w1);
          const double k0 = sc * row(G00, G01, G02, c0, c1, c2), k1 = sc * row(G11, G01, G12, c1, c0, c2);
          const double k2 = sc * row(G22, G02, G12, c2, c0, c1);
#pragma unroll
          for (int k = 0; k <= P; k++)
          {
            const double Bc = qt.Bc[q * (P + 1) + k], Gc = qt.Gc[q * (P + 1) + k];
            sx0[k] = __builtin_fma(Gc, k1, __builtin_fma(Bc, m0, sx0[k]));
            sxy[k] = __builtin_fma(-Bc, k2, sxy[k]);
            sy0[k] = __builtin_fma(-Gc, k0, __builtin_fma(Bc, m1, sy0[k]));
            syx[k] = __builtin_fma(Bc, k2, syx[k]);
          }
#pragma unroll
          for (int k = 0; k < P; k++)
          {
            const double Bo = qt.Bo[q * P + k];
            sz0[k] = __builtin_fma(Bo, m2, sz0[k]);
            szy[k] = __builtin_fma(Bo, k0, szy[k]);
            szx[k] = __builtin_fma(-Bo, k1, szx[k]);
          }
          phase();
        }
        if constexpr (P > 1)
          g0 = g1;
        if constexpr (FIRST)
        {
          // (the last layer loads itself again: a branch here would let the
          // compiler sink the points above past it and keep the loads alive there)
          const int64_t zn = z + 1 < z1 ? P : 0;
          load_layer(bx + zn * plx, by + zn * ply, bz + zn * plz, min(z + 1, z1 - 1));
          load_corners(min(z + 2, z1), nv);
        }
        phase();
        // transposed x, y stages
#pragma unroll
        for (int k = 0; k <= P; k++)
        {
          const double a = mm(sxy[k], bGc, mm(sx0[k], bBc, 0.0));
          yx[k] = mm(a, bBo, 0.0);
          const double b = mm(sy0[k], bBo, 0.0), c = mm(syx[k], bBo, 0.0);
          yy[k] = mm(c, bGc, mm(b, bBc, 0.0));
        }
#pragma unroll
        for (int k = 0; k < P; k++)
        {
          const double a = mm(szy[k], bGc, mm(sz0[k], bBc, 0.0)), b = mm(szx[k], bBc, 0.0);
          yz[k] = mm(b, bGc, mm(a, bBc, 0.0));
        }
      }
      else if constexpr (KIND == BOX_MASS)
      {
        const double kmx = mk0 * (sgN * wf), kmy = mk1 * (sgT * wf), kmz = mk2 * sgN;
#pragma unroll
        for (int q = 0; q < P; q++)
          yz[q] = tb.w[q] * mm(mm(kmz * uz[q], opM, 0.0), opM, 0.0);
#pragma unroll
        for (int k = 0; k <= P; k++)
        {
          double mx = 0.0, my = 0.0;
#pragma unroll
          for (int m = 0; m <= P; m++)
          {
            mx = __builtin_fma(tb.M[k][m], ux[m], mx);
            my = __builtin_fma(tb.M[k][m], uy[m], my);
          }
          yx[k] = mm(opM, kmx * mx, 0.0);
          yy[k] = mm(kmy * my, opM, 0.0);
        }
      }
      else
      {
        // In phases (the scheduler keeps to them: the order holds the number of
        // live registers below the 128 that four waves per SIMD leave each)
        auto phase = []() { __builtin_amdgcn_sched_barrier(0); };
        // curl components (c_y with reversed sign)
        const double kcx = ck0 * (nuT * wf), kcy = ck1 * (nuN * wf), kcz = ck2 * (nuN * wfs);
        const double kmx = mk0 * (sgN * wf), kmy = mk1 * (sgT * wf), kmz = mk2 * sgN;
        double cxs[P], cys[P], ut[P];
#pragma unroll
        for (int q = 0; q < P; q++)
          ut[q] = mm(uz[q], opI, 0.0); // u_z, T
#pragma unroll
        for (int q = 0; q < P; q++)
        {
          double dx = 0.0, dy = 0.0;
#pragma unroll
          for (int k = 0; k <= P; k++)
          {
            dx = __builtin_fma(-tb.D[q][k], ux[k], dx);
            dy = __builtin_fma(-tb.D[q][k], uy[k], dy);
          }
          cxs[q] = mm(uz[q], opD, dy); // T: D_y u_z - D_z u_y
          cys[q] = mm(ut[q], opD, dx); // N: D_x u_z - D_z u_x
        }
#pragma unroll
        for (int q = 0; q < P; q++)
        {
          cys[q] *= kcy;
          cxs[q] *= kcx;
          uz[q] *= kmz;
        }
        phase();
        // y_z = w (Mc_x Mc_y (sigma mk u_z) + D_x^T Mc_y cys + D_y^T Mc_x cxs),
        // and the z contractions that y_x and y_y take from u_x, u_y and the curl
#pragma unroll
        for (int q = 0; q < P; q++)
        {
          const double p1 = mm(uz[q], opM, 0.0);  // T
          const double p2 = mm(cys[q], opM, 0.0); // T
          const double p3 = mm(cxs[q], opM, 0.0); // N
          yz[q] = mm(p1, opM, 0.0);
          yz[q] = mm(p2, opDt, yz[q]);
          yz[q] = mm(opDt, p3, yz[q]);
        }
#pragma unroll
        for (int k = 0; k <= P; k++)
        {
          double mx = 0.0, my = 0.0, ax = 0.0, ay = 0.0;
#pragma unroll
          for (int m = 0; m <= P; m++)
          {
            mx = __builtin_fma(tb.M[k][m], ux[m], mx);
            my = __builtin_fma(tb.M[k][m], uy[m], my);
          }
#pragma unroll
          for (int q = 0; q < P; q++)
          {
            ax = __builtin_fma(-(tb.w[q] * tb.D[q][k]), cys[q], ax);
            ay = __builtin_fma(-(tb.w[q] * tb.D[q][k]), cxs[q], ay);
          }
          yx[k] = __builtin_fma(kmx, mx, ax);
          yy[k] = __builtin_fma(kmy, my, ay);
        }
#pragma unroll
        for (int q = 0; q < P; q++)
          yz[q] *= tb.w[q];
        phase();
        double cz[P + 1];
#pragma unroll
        for (int k = 0; k <= P; k++)
          cz[k] = mm(uy[k], opD, 0.0); // D_x u_y, N
#pragma unroll
        for (int k = 0; k <= P; k++)
          cz[k] = mm<1>(opD, ux[k], cz[k]); // - D_y u_x
        phase();
        double f[P + 1], ft[P + 1];
#pragma unroll
        for (int k = 0; k <= P; k++)
        {
          double fk = 0.0;
#pragma unroll
          for (int m = 0; m <= P; m++)
            fk = __builtin_fma(tb.M[k][m], cz[m], fk);
          f[k] = kcz * fk; // - f_z, N
        }
#pragma unroll
        for (int k = 0; k <= P; k++)
          ft[k] = mm(f[k], opI, 0.0); // - f_z, T
#pragma unroll
        for (int k = 0; k <= P; k++)
          f[k] = mm(opDt, f[k], 0.0); // - D_y^T f_z, N
#pragma unroll
        for (int k = 0; k <= P; k++)
          ft[k] = mm<1>(ft[k], opDt, 0.0); // D_x^T f_z, N
#pragma unroll
        for (int k = 0; k <= P; k++)
          yx[k] = mm(opM, yx[k], f[k]);
#pragma unroll
        for (int k = 0; k <= P; k++)
          yy[k] = mm(yy[k], opM, ft[k]);
      }
      };
      products(ux, uy, uz, cf, vN, std::true_type{});
      if constexpr (P == 1)
      {
        // A block holds 2 x 2 elements at order 1, and a zero of the block-diagonal
        // matrices times a value that is not finite is NaN for the elements beside
        // the one that has it.  Such a layer is done again element by element, the
        // others with zeros.  (The test and its registers: 64^3 18.3 -> 18.6 us,
        // trilinear 37.0 -> 38.0; nothing up to 31x37x29.)
        const bool finite = __builtin_isfinite(yx[0]) && __builtin_isfinite(yx[1]) && __builtin_isfinite(yy[0]) &&
                            __builtin_isfinite(yy[1]) && __builtin_isfinite(yz[0]);
        if (__any(!finite))
        {
          double rx[2] = {}, ry[2] = {}, rz = 0.0;
#pragma unroll 1
          for (int e = 0; e < 4; e++)
          {
            const bool inN = ef + 2 * es == e, inT = HEX ? inN : es + 2 * ef == e;
            const double vx[2] = {inN ? ux[0] : 0.0, inN ? ux[1] : 0.0}, vy[2] = {inT ? uy[0] : 0.0, inT ? uy[1] : 0.0};
            const double vz[1] = {inN ? uz[0] : 0.0};
            const Coef ce{inN ? cf.nuN : 0.0, inN ? cf.sgN : 0.0, inT ? cf.nuT : 0.0, inT ? cf.sgT : 0.0};
            products(vx, vy, vz, ce, vN && inN, std::false_type{});
            rx[0] = inN ? yx[0] : rx[0];
            rx[1] = inN ? yx[1] : rx[1];
            ry[0] = inN ? yy[0] : ry[0];
            ry[1] = inN ? yy[1] : ry[1];
            rz = inN ? yz[0] : rz;
          }
          yx[0] = rx[0];
          yx[1] = rx[1];
          yy[0] = ry[0];
          yy[1] = ry[1];
          yz[0] = rz;
        }
        if constexpr (HEX)
          g0 = g1;
      }
      yx[0] = yx[0] + carx;
      yy[0] = yy[0] + cary;
      carx = yx[P];
      cary = yy[P];
      // the top plane becomes the bottom plane of the next layer
      ux[0] = ux[P];
      uy[0] = uy[P];
      const int64_t cbx = bx, cby = by, cbz = bz;
      bx += P * plx;
      by += P * ply;
      bz += P * plz;
      // the lower halo layer of a chunk stores nothing (its top plane is
      // carried); no branch around the stores: on a path without them the next
      // layer's wait for its loads would have to wait for every store too
      const bool zout = z >= z0;
      const uint32_t jsx = (ownx && zout) ? ilx : OOB, jsy = (owny && zout) ? oyN : OOB;
      const uint32_t jsz = (ownz && zout) ? ilz : OOB;

      // face values to LDS; meanwhile b of the residual mode is on its way
      if (ps == P)
      {
#pragma unroll
        for (int k = 0; k < P; k++)
        {
          sX[buf][k][wR] = yx[k];
          sZR[buf][k][wR] = yz[k];
        }
      }
      if (pf == P)
      {
#pragma unroll
        for (int k = 0; k < P; k++)
        {
          sY[buf][k][wC] = yy[k];
          sZC[buf][k][wC] = yz[k];
        }
      }
      T rbx[P], rby[P], rbz[P];
      if constexpr (KIND == BOX_RESID || KIND == BOX_ADD)
      {
        const T * bv = (const T *)ad.resid + rof;
#pragma unroll
        for (int k = 0; k < P; k++)
        {
          rbx[k] = ldb(bv + cbx, jsx, k * spx);
          rby[k] = ldb(bv + cby, jsy, k * spy);
          rbz[k] = ldb(bv + cbz, jsz, k * spz);
        }
      }
      __syncthreads();
      // left, then diagonal, then below: a fixed order for every tile shape
#pragma unroll
      for (int k = 0; k < P; k++)
      {
        yx[k] += sX[buf][k][rB];
        yy[k] += sY[buf][k][rL];
        yz[k] = ((yz[k] + sZC[buf][k][rL]) + sZR[buf][k][rD]) + sZR[buf][k][rB];
      }
      if constexpr (KIND == BOX_ADD)
      {
#pragma unroll
        for (int k = 0; k < P; k++)
        {
          yx[k] = (double)rbx[k] + yx[k];
          yy[k] = (double)rby[k] + yy[k];
          yz[k] = (double)rbz[k] + yz[k];
        }
      }
      // PEC DOFs: y = x
      if (stash)
      {
        const bool zf = z == 0 && (pec & 16);
#pragma unroll
        for (int k = 0; k < P; k++)
        {
          const double vx = k ? sE[EX + (k ? k - 1 : 0)][eN] : sE[EX0 + (z & 1)][eN];
          const double vy = k ? sE[EY + (k ? k - 1 : 0)][eN] : sE[EY0 + (z & 1)][eN];
          const double vz = sE[EZ + k][eN];
          yx[k] = (essx || (zf && k == 0)) ? vx : yx[k];
          yy[k] = (essy || (zf && k == 0)) ? vy : yy[k];
          yz[k] = essz ? vz : yz[k];
        }
      }
      if constexpr (KIND == BOX_RESID)
      {
#pragma unroll
        for (int k = 0; k < P; k++)
        {
          yx[k] = (double)rbx[k] - yx[k];
          yy[k] = (double)rby[k] - yy[k];
          yz[k] = (double)rbz[k] - yz[k];
        }
      }
      T * yv = (T *)ad.y + rof;
#pragma unroll
      for (int k = 0; k < P; k++)
      {
        stb(yv + cbx, jsx, (T)yx[k], k * spx);
        stb(yv + cby, jsy, (T)yy[k], k * spy);
        stb(yv + cbz, jsz, (T)yz[k], k * spz);
      }
      buf ^= 1;
    }
    if (z1 == nz)
    {
      // top plane of the mesh (components x and y)
      const bool zf = (pec & 32) != 0;
      if (ps == P)
        sX[buf][0][wR] = carx;
      if (pf == P)
        sY[buf][0][wC] = cary;
      __syncthreads();
      carx += sX[buf][0][rB];
      cary += sY[buf][0][rL];
      T * yv = (T *)ad.y + rof;
      const uint32_t isx = ownx ? oxN : OOB, isy = owny ? oyN : OOB;
      const T vx = ldb(xv + bx, isx), vy = ldb(xv + by, isy);
      if constexpr (KIND == BOX_ADD)
      {
        const T * bv = (const T *)ad.resid + rof;
        carx = (double)ldb(bv + bx, isx) + carx;
        cary = (double)ldb(bv + by, isy) + cary;
      }
      carx = (essx || zf) ? (double)vx : carx;
      cary = (essy || zf) ? (double)vy : cary;
      if constexpr (KIND == BOX_RESID)
      {
        const T * bv = (const T *)ad.resid + rof;
        carx = (double)ldb(bv + bx, isx) - carx;
        cary = (double)ldb(bv + by, isy) - cary;
      }
      stb(yv + bx, isx, (T)carx);
      stb(yv + by, isy, (T)cary);
    }
    if (TABLE && rhs + 1 < r_end)
      __syncthreads(); // the next rhs starts over with buffer 0
  }
}

// P = 0: the instances of the table may have any order (one launch, and the
// small instances of one order run beside the large ones of another)
template <int P, typename T, int NS, bool TABLE, int KIND, bool HEX>
__global__ void __launch_bounds__(16 * NS, HEX ? 2 : 4)
k_apply_box(ApplyDesc d0, const ApplyDesc * __restrict__ descs, int ndesc)
{
  __shared__ double lds[box_lds<P == 0 ? PMAX : P, NS>()];
  const int wi = xcd_remap(blockIdx.x, gridDim.x);
  int di = 0;
  if constexpr (TABLE)
    di = __builtin_amdgcn_readfirstlane(find_instance(wi, ndesc, [&](int i) { return descs[i].w0; }));
  const ApplyDesc & ad = TABLE ? descs[di] : d0;
  const int rb = TABLE ? ad.rb : 1;
  const int ngrp = (ad.nrhs + rb - 1) / rb;
  const int wl = wi - ad.w0;
  const int r_begin = (wl % ngrp) * rb;
  const int r_end = TABLE ? min(ad.nrhs, r_begin + rb) : r_begin + 1;
  const int tile = wl / ngrp;
  if constexpr (P == 0)
  {
    if (ad.g.p == 1)
      box_body<1, T, NS, TABLE, KIND, HEX>(ad, tile, r_begin, r_end, lds);
    else if (ad.g.p == 2)
      box_body<2, T, NS, TABLE, KIND, HEX>(ad, tile, r_begin, r_end, lds);
    else
      box_body<3, T, NS, TABLE, KIND, HEX>(ad, tile, r_begin, r_end, lds);
  }
  else
    box_body<P, T, NS, TABLE, KIND, HEX>(ad, tile, r_begin, r_end, lds);
}

// ---------------------------------------------------------------------------
// tiles and launch
// ---------------------------------------------------------------------------

// Decomposition: for each number of slots the tile with the fewest tiles (ties:
// the widest rows) and the chunk of layers with the least modelled time.  A
// layer takes about 0.9 + 1.25 w us at order 3 with w waves per SIMD, so a mesh
// that leaves CUs idle takes small workgroups and short chunks (12^3 order 3:
// 7.8 us with 16 slots, 14.6 us with 64), one that fills them the fewest
// duplicated elements (48^3 order 3: 63 us with 64 slots, 78 us with 16).
// Measured, us a layer with 1, 2, 3, 4 waves (16 slots, one chunk):
//   box        order 1  0.91 1.26 1.53 1.96   2  1.35 1.96 2.56 3.17   3  2.11 3.04 4.29 5.53
//   trilinear  order 1  1.74 2.77             2  2.60 4.06             3  4.17 6.22
// Only the ratio of the two terms decides: 0.72 here, 0.85 to 1.2 measured for
// boxes (1.6 at order 1), 0.7 to 1.0 for the trilinear form, so that one pair
// serves all.  Against every pair of 16, 32, 64 slots and chunks of 2 to 48 layers
// on six meshes (17x23x41 to 48^3, 64x12x12, 9x9x63) the choice is within 2.5 % of
// the best, beyond that at 64x12x12 (order 2 boxes 4 %, order 3 5 %: chunks of 2)
// and 48^3 order 2 trilinear (6 %: 32 slots).
BoxTile
box_tile(const Geom & g, int nrhs, int ns_only, bool hex)
{
  const int ej = g.p == 1 ? 2 : 1;
  auto tiles = [&](int n, int c) { return n <= c * ej ? 1 : (n - 1 + c * ej - 2) / (c * ej - 1); };
  constexpr int CUS = 256;
  BoxTile best{};
  double cost = 1e300;
  for (int ns = 16; ns <= (hex ? 32 : 64); ns *= 2)
  {
    if (ns_only && ns != ns_only)
      continue;
    BoxTile b{};
    b.ns = ns;
    int64_t least = -1;
    for (int cy = 1; cy <= ns; cy++)
    {
      const int cx = ns / cy;
      if ((cy * ej < 2 && g.n[1] > 1) || (cx * ej < 2 && g.n[0] > 1))
        continue;
      const int ntx = tiles(g.n[0], cx), nty = tiles(g.n[1], cy);
      const int64_t t = (int64_t)ntx * nty;
      if (least < 0 || t < least || (t == least && cx > b.cx))
      {
        least = t;
        b.cx = cx;
        b.cy = cy;
        b.ntx = ntx;
        b.nty = nty;
      }
    }
    const int bpc = (hex ? 32 : 64) / ns, wpb = ns / 16; // workgroups per CU, waves per SIMD of one
    const int64_t cap = (int64_t)CUS * bpc;
    for (int zc = g.n[2];;)
    {
      const int nzc = (g.n[2] + zc - 1) / zc;
      const int64_t blocks = least * nrhs * nzc, rem = blocks % cap;
      double t = (double)(blocks / cap) * (0.9 + 1.25 * bpc * wpb);
      if (rem)
        t += 0.9 + 1.25 * wpb * (double)((rem + CUS - 1) / CUS);
      t *= zc + (nzc > 1 ? 1.8 : 0.8);
      if (t < cost)
      {
        cost = t;
        best = b;
        best.zc = zc;
        best.nzc = nzc;
      }
      if (zc == 1)
        break;
      zc = std::min(zc - 1, (g.n[2] + nzc) / (nzc + 1)); // the next chunk length with more chunks
    }
  }
  return best;
}

// The 32-bit offsets of the kernel: p planes of a component beyond a tile's
// first row.
bool
box_fits(const Geom & g)
{
  int64_t pl = 0;
  for (int c = 0; c < 3; c++)
    pl = std::max(pl, g.cd[c][0] * g.cd[c][1]);
  const int64_t vp = (int64_t)(g.n[0] + 1) * (g.n[1] + 1); // vertices of a plane (trilinear)
  return std::max((g.p + 1) * pl * (int64_t)sizeof(double), 24 * vp) < (int64_t)0xFFFFF000;
}

template <typename T>
hipError_t
apply_box(const ApplyDesc & d0, const ApplyDesc * descs, int ndesc, int nwork, int p, int ns, bool hex, hipStream_t st, BoxKind kind)
{
  if (nwork <= 0)
    return hipSuccess;
  const dim3 grid(nwork);
  auto go = [&](auto pc, auto nc) {
    constexpr int P = decltype(pc)::value, NS = decltype(nc)::value;
    const dim3 blk(16 * NS);
    auto run = [&](auto kern) { hipLaunchKernelGGL(kern, grid, blk, 0, st, d0, descs, ndesc); };
    if constexpr (P == 0)
      run(k_apply_box<0, T, NS, true, BOX_APPLY, false>);
    else
    {
      if constexpr (NS <= 32 && (sizeof(T) == 8 || P == 1))
      {
        if (hex)
          return descs ? run(k_apply_box<P, T, NS, true, BOX_APPLY, true>) : run(k_apply_box<P, T, NS, false, BOX_APPLY, true>);
      }
      if (descs)
        return run(k_apply_box<P, T, NS, true, BOX_APPLY, false>);
      if constexpr (sizeof(T) == 8)
      {
        if (kind == BOX_ADD)
          return run(k_apply_box<P, T, NS, false, BOX_ADD, false>);
        if (kind == BOX_MASS)
          return run(k_apply_box<P, T, NS, false, BOX_MASS, false>);
        if (kind == BOX_RESID)
          return run(k_apply_box<P, T, NS, false, BOX_RESID, false>);
      }
      run(k_apply_box<P, T, NS, false, BOX_APPLY, false>);
    }
  };
  auto by_ns = [&](auto pc) {
    if (ns == 16)
      go(pc, std::integral_constant<int, 16>{});
    else if (ns == 32)
      go(pc, std::integral_constant<int, 32>{});
    else
      go(pc, std::integral_constant<int, 64>{});
  };
  // residuals are formed for multigrid (FP64) and tables of several orders for
  // batches of box meshes only; FP32 vectors on trilinear meshes at order 1 only
  const bool with_y = kind == BOX_RESID || kind == BOX_ADD;
  if ((hex && (ns > 32 || kind != BOX_APPLY || p == 0)) || (p == 0 && !descs) || (descs && kind != BOX_APPLY) ||
      (sizeof(T) != 8 && (kind != BOX_APPLY || (hex && p != 1))) || (!descs && with_y != (d0.resid != nullptr)))
    return hipErrorInvalidValue;
  switch (p)
  {
  case 0:
    by_ns(std::integral_constant<int, 0>{});
    break;
  case 1:
    by_ns(std::integral_constant<int, 1>{});
    break;
  case 2:
    by_ns(std::integral_constant<int, 2>{});
    break;
  case 3:
    by_ns(std::integral_constant<int, 3>{});
    break;
  default:
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template hipError_t apply_box<double>(const ApplyDesc &, const ApplyDesc *, int, int, int, int, bool, hipStream_t, BoxKind);
template hipError_t apply_box<float>(const ApplyDesc &, const ApplyDesc *, int, int, int, int, bool, hipStream_t, BoxKind);

} // namespace hc
