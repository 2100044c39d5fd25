// Cell-loop assembly of the Ginzburg-Landau Jacobian J, its matrix-free form,
// and system_rhs = -R for FE_Q(k) x 18 on axis-aligned hexes, hand-written
// for gfx950.
//
// Reference: femgl/src/assemble.cc:177-280 (cell loop), residual.cc:152-232,
// the term functions of femgl/src/cell_mat_vec/, and the Robin face loops
// assemble.cc:286-348 / residual.cc:235-278.
//
// The reference evaluates about 170 3x3 products for each (cell, q, i, j).
// Because every FESystem(FE_Q(k),18) shape function is one-hot in the
// component, each term is a bilinear form evaluated at unit tensors, so the
// cell matrix factorises exactly as
//   J[(a,c),(b,d)] = sum_q JxW_q N_a N_b H_cd(q)
//                  + K1 delta_cd S_ab + (K2+K3) [same part and spin row] S^{k(c) l(d)}_ab
// with H(q) the 18x18 Hessian of the bulk density at the iterate
// (alpha + 2 sum beta_n m_n) and S the stiffness integrals; the residual
// factorises the same way.  H is evaluated in closed form from six 3x3 Gram
// matrices per quadrature point.
//
// A workgroup owns one cell of a colour, or a part of its node pairs.  Q2
// (k_assemble_q2) contracts the pair weights with H on the FP64 matrix cores,
// Q1 (k_assemble_q1) in registers; both write whole blocks, 16 bytes (FP64)
// per lane and consecutive lanes at consecutive entries.
// Cells of one colour share no node, so the read-modify-write scatter needs
// no atomics and the result is bit-deterministic; the first colour to touch
// a block stores instead of accumulating, so J needs no zero fill.
// Dirichlet rows/columns are condensed in the scatter (constrained entries
// 0, constrained diagonal += |local diagonal|, the documented behaviour of
// deal.II's AffineConstraints::distribute_local_to_global).
#include "glhip_dev.hpp"

#include <algorithm>
#include <climits>
#include <type_traits>

namespace glh {
namespace {

constexpr int NT = 192;   // threads per workgroup (3 wavefronts)
constexpr int GRAM = 57;  // per-q Gram data (see gram_entry)
constexpr int NUPAIR = 171;

// Gram layout per quadrature point:
//  [0,9) Auu = u^T u (orbital k,l)   [9,18) Avv = v^T v   [18,27) Auv = u^T v
//  [27,36) uut = u u^T (spin mu,nu)  [36,45) vvt          [45,54) uvt = u v^T
//  54 |u|^2  55 |v|^2  56 u:v
__device__ inline double gram_entry(const double *x, int g)
{
  const double *u = x, *v = x + 9;
  if (g < 54) {
    const int blk = g / 9, i = (g % 9) / 3, j = g % 3;
    const double *A = (blk == 0 || blk == 2 || blk == 3 || blk == 5) ? u : v;
    const double *B = (blk == 0 || blk == 3) ? u : v;
    double s = 0.0;
    if (blk < 3) {  // A^T B: sum over spin rows
      for (int m = 0; m < 3; ++m) s += A[3 * m + i] * B[3 * m + j];
    } else {        // A B^T: sum over orbital columns
      for (int k = 0; k < 3; ++k) s += A[3 * i + k] * B[3 * j + k];
    }
    return s;
  }
  double s = 0.0;
  if (g == 54) for (int a = 0; a < 9; ++a) s += u[a] * u[a];
  else if (g == 55) for (int a = 0; a < 9; ++a) s += v[a] * v[a];
  else for (int a = 0; a < 9; ++a) s += u[a] * v[a];
  return s;
}

// H_cd (c <= d) of the bulk density: alpha delta + 2 sum_n beta_n m_n(E_c, E_d).
__device__ inline double hess_entry(const double *__restrict__ G, const double *__restrict__ x, int c, int d,
                                    const Material &M)
{
  const double *u = x, *v = x + 9;
  const int pc = c / 9, pd = d / 9, ac = c % 9, ad = d % 9;
  const int mu = ac / 3, k = ac % 3, nu = ad / 3, l = ad % 3;
  const double dmn = (mu == nu) ? 1.0 : 0.0, dkl = (k == l) ? 1.0 : 0.0, dab = dmn * dkl;
  const double U2 = G[54], V2 = G[55], UV = G[56], D = U2 - V2, N = U2 + V2;
  const double b345 = M.b3 + M.b4 + M.b5;
  if (pc == pd) {
    // uu block, or vv block with the roles of u and v exchanged
    const double *p = pc ? v : u, *o = pc ? u : v;
    const double *App = pc ? G + 9 : G, *Aoo = pc ? G : G + 9;
    const double *Spp = pc ? G + 36 : G + 27, *Soo = pc ? G + 27 : G + 36;
    const double sD = pc ? -D : D;
    return dab * (M.al + 2.0 * M.b1 * sD + 2.0 * M.b2 * N) + 4.0 * (M.b1 + M.b2) * p[ac] * p[ad] +
           4.0 * M.b1 * o[ac] * o[ad] +
           2.0 * dmn * (b345 * App[3 * l + k] + (M.b3 + M.b4 - M.b5) * Aoo[3 * l + k]) +
           2.0 * b345 * p[3 * mu + l] * p[3 * nu + k] + 2.0 * (M.b3 - M.b4 + M.b5) * o[3 * mu + l] * o[3 * nu + k] +
           2.0 * dkl * (b345 * Spp[3 * mu + nu] + (-M.b3 + M.b4 + M.b5) * Soo[3 * mu + nu]);
  }
  // uv block: row (mu,k) in u, column (nu,l) in v
  const double Auv_lk = G[18 + 3 * l + k], Avu_lk = G[18 + 3 * k + l];
  const double uvt_mn = G[45 + 3 * mu + nu], uvt_nm = G[45 + 3 * nu + mu];
  const double Q = uvt_mn + uvt_nm, W = uvt_nm - uvt_mn;
  const double ua = u[ac], va = v[ac], ub = u[ad], vb = v[ad];
  const double uml = u[3 * mu + l], unk = u[3 * nu + k], vml = v[3 * mu + l], vnk = v[3 * nu + k];
  return dab * 4.0 * M.b1 * UV + 4.0 * M.b1 * (ub * va - vb * ua) + 4.0 * M.b2 * ua * vb +
         2.0 * M.b3 * (-dmn * Avu_lk - vml * unk + dmn * Auv_lk + uml * vnk + Q * dkl) +
         2.0 * M.b4 * (dmn * Avu_lk + vml * unk - dmn * Auv_lk + uml * vnk - W * dkl) +
         2.0 * M.b5 * (dmn * Avu_lk + vml * unk + dmn * Auv_lk - uml * vnk + W * dkl);
}

__device__ inline bool face_zeroed(int bid, int c) { return (c % 9) % 3 == bid - 2; }

__device__ inline double face_area(int lf, const double *h)
{
  return lf < 2 ? h[1] * h[2] : (lf < 4 ? h[0] * h[2] : h[0] * h[1]);
}

template <typename T> struct Vec2;
template <> struct Vec2<double> { using type = double2; };
template <> struct Vec2<float> { using type = float2; };

// Sizes of the cell contraction of Q2 assembly as a matrix product
//   OUT[p][col] = sum_k A[p][k] B[k][col]
// over node pairs p = (a <= b) and block entries col: the 171 entries c <= d,
// then the 18 entries [d][c] of the same part and spin (the only others that
// differ from their transposes); k: the NQ points (A = w N_a N_b, B = vol H_cd),
// the 9 derivative pairs (A = stiffness integrals, B = K1 and K23 factors) and
// the 6 faces (A = face masses, B = Robin factors; only cells that have one
// run those steps).  A is uniform over the cells, a table in the lane order of
// v_mfma_f64_16x16x4_f64 (RefTables::At).
struct AsmQ2 {
  static constexpr int NS = 27, NQ = NS, NPAIR = NS * (NS + 1) / 2;
  static constexpr int NTILE = (NPAIR + 15) / 16;               // row tiles of 16 pairs
  static constexpr int KB = (NQ + 9 + 3) / 4, KT = (NQ + 15 + 3) / 4;  // k steps of 4, without and with faces
  static constexpr int TS = 208;                                // LDS row stride of an output tile (192 columns)
  static constexpr int NW = 6, NTH = 64 * NW;                   // waves (2 column tiles each), threads
  // phase 0: U, X, Gram and half of B; then two output tiles
  static constexpr int P0 = NS * 18 + NQ * 18 + NQ * GRAM + 4 * KT * 96, LT = 2 * 16 * TS;
  static constexpr int LDS = P0 > LT ? P0 : LT;
};

// column of block entry [r][c] in OUT
__device__ inline int asm_col(int r, int c)
{
  if (r > c) {
    if (r / 3 == c / 3) return 171 + (r / 3) * 3 + (r % 3 == 1 ? 0 : 1 + c % 3);
    const int t = r;
    r = c;
    c = t;
  }
  return r * 18 - r * (r - 1) / 2 + (c - r);
}

typedef double f64x4 __attribute__((ext_vector_type(4)));

// The B operands of the cell: lane l of wave w gets B[4 s + l / 16][16 (w + 6 t)
// + l % 16] in Br[t][s].  S: AsmQ2::LDS doubles.
__device__ inline void asm_operands(const RefTables &T, const Material &M, const double *__restrict__ U,
                                    const int *__restrict__ cn, const double *h, uint32_t cface, bool rb, double *S,
                                    double (*Br)[AsmQ2::KT])
{
  using D = AsmQ2;
  constexpr int NS = D::NS, NQ = D::NQ;
  double *sU = S, *sX = sU + NS * 18, *sGram = sX + NQ * 18, *sB = sGram + NQ * GRAM;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const double ih[3] = {1.0 / h[0], 1.0 / h[1], 1.0 / h[2]}, vol = h[0] * h[1] * h[2];
  for (int i = tid; i < NS * 18; i += D::NTH) sU[i] = U[(size_t)cn[i / 18] * 18 + (i % 18)];
  __syncthreads();
  // the iterate at the quadrature points (s_vector2matrix.cc:116-217)
  for (int i = tid; i < NQ * 18; i += D::NTH) {
    const int q = i / 18, c = i % 18;
    double xv = 0;
    for (int a = 0; a < NS; ++a) xv += T.N[q * NS + a] * sU[a * 18 + c];
    sX[i] = xv;
  }
  __syncthreads();
#pragma unroll 1
  for (int i = tid; i < NQ * GRAM; i += D::NTH) {
    const int q = i / GRAM, g = i % GRAM;
    sGram[i] = gram_entry(sX + q * 18, g);
  }
  const int nk = 4 * (rb ? D::KT : D::KB);
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    // the entry [r][c] of this thread's column (192 columns, 189 used)
    const int lc = tid % 96, col = 96 * t + lc;
    int r = 0, c = 0;
    const bool used = col < 189;
    if (col < 171) {
      int k = col;
      while (k >= 18 - r) { k -= 18 - r; ++r; }
      c = r + k;
    } else if (used) {
      const int g = (col - 171) / 3, k = (col - 171) % 3;
      r = 3 * g + (k == 0 ? 1 : 2);
      c = 3 * g + (k == 2 ? 1 : 0);
    }
    const bool grad = r / 3 == c / 3;
    __syncthreads();  // Gram, or the first half of B has been read
#pragma unroll 1
    for (int k = tid / 96; k < nk; k += D::NTH / 96) {
      double v = 0.0;
      if (used && k < NQ) {
        v = vol * hess_entry(sGram + k * GRAM, sX + k * 18, r < c ? r : c, r < c ? c : r, M);
      } else if (used && k < NQ + 9) {
        const int kk = (k - NQ) / 3, kl = (k - NQ) % 3;
        if (r == c && kk == kl) v += M.K1 * (vol * ih[kk] * ih[kk]);
        if (grad && r % 3 == kk && c % 3 == kl) v += M.K23 * vol * ih[kk] * ih[kl];
      } else if (rb && used && r == c && k < NQ + 15) {
        const int lf = k - NQ - 9, bid = (int)((cface >> (3 * lf)) & 7u) - 1;
        if (bid >= 2 && bid <= 4 && !face_zeroed(bid, c)) v = M.robin * face_area(lf, h);
      }
      sB[k * 96 + lc] = v;
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < D::KT; ++s)
      Br[t][s] = 4 * s < nk ? sB[(4 * s + (lane >> 4)) * 96 + 16 * w + (lane & 15)] : 0.0;
  }
}

// One workgroup of 6 waves per cell of a colour (and per part blockIdx.y of
// its row tiles, where a colour has too few cells to fill the device).  The
// contraction of the bulk Hessian, the gradient terms and the Robin masses is
// one product on the FP64 matrix cores per 16 node pairs, whose result goes
// to LDS.  From there waves 0-2 write the pairs' blocks (a, b) and waves 3-5
// the transposed (b, a), 16 bytes per lane: a thread keeps its two entries
// of a block through all of them, so that the block's address and masks are
// scalar and its LDS offset constant (about 10 vector instructions a block,
// against 60 with the blocks' entries dealt over all threads).  The old
// values of blocks shared with earlier colours are requested before the
// product; one barrier per 16 pairs.  Jacobian of the 32^3 cube (82 GB moved,
// 44 GB of it the result: blocks shared between colours are read and written
// again): 34.4 -> 21.3 ms FP64 (3.9 TB/s), 28.0 -> 22.8 ms FP32, against one
// thread per component pair storing single values.
// UP: only the blocks on and above the diagonal (the products read no
// others): of a pair's two blocks the one whose row node is not the larger,
// waves 0-2 the even pairs and waves 3-5 the odd ones.  Half the bytes:
// colours of 287 cells 245 -> 182 us FP64.
template <typename TJ, bool HANG, bool UP>
__global__ __launch_bounds__(AsmQ2::NTH, 3) void k_assemble_q2(RefTables T, MeshDev Mh, Material M0,
                                                     const double *__restrict__ U, const int *__restrict__ cells,
                                                     TJ *__restrict__ J)
{
  using D = AsmQ2;
  using J2 = typename Vec2<TJ>::type;
  constexpr int NS = D::NS, NPAIR = D::NPAIR, KB = D::KB, KT = D::KT, TS = D::TS;
  __shared__ __attribute__((aligned(16))) double S[D::LDS];
  __shared__ int sBlk[NS * NS];
  __shared__ uint32_t sMask[NS];
  __shared__ int sNode[UP ? NS : 1];
  __shared__ uint16_t sPab[D::NTILE * 16];  // a | b << 8 of a pair, ~0 beyond the last
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int e = cells[blockIdx.x];
  if (Mh.inst_active && !Mh.inst_active[Mh.cell_inst[e]]) return;  // finished instance of a batch
  const Material M = Mh.mats ? Mh.mats[Mh.cell_mat[e]] : M0;       // per-instance (T, p) in a batch
  const int *cn = Mh.cell_nodes + (size_t)e * NS;
  double h[3];
  for (int k = 0; k < 3; ++k) h[k] = Mh.cell_h[3 * e + k];
  const uint32_t cface = Mh.cell_face[e];
  const bool rb = M.robin != 0.0 && cface != 0u;
  {
    const int *cb = Mh.cell_blk + (size_t)e * NS * NS;
    for (int i = tid; i < NS * NS; i += D::NTH) sBlk[i] = cb[i];
    for (int i = tid; i < NS; i += D::NTH) sMask[i] = Mh.node_mask[cn[i]];
    if (UP)
      for (int i = tid; i < NS; i += D::NTH) sNode[i] = cn[i];
    for (int i = tid; i < D::NTILE * 16; i += D::NTH)
      sPab[i] = i < NPAIR ? (uint16_t)(T.pa[i] | (T.pb[i] << 8)) : (uint16_t)0xffff;
  }
  double B[2][KT];
  asm_operands(T, M, U, cn, h, cface, rb, S, B);
  __syncthreads();  // B has been read: S takes the output tiles
  // this thread's entries [r][c], [r][c + 1] of a block, and their columns
  // in OUT: of (a, b), or transposed of (b, a)
  const bool tr = w >= 3;
  const int pos = 64 * (tr ? w - 3 : w) + lane;
  const bool own = pos < 162;
  const int r = own ? pos / 9 : 0, c = own ? 2 * (pos % 9) : 0;
  const int n0 = asm_col(r, c), n1 = asm_col(r, c + 1), r0 = asm_col(c, r), r1 = asm_col(c + 1, r);
  const int o0 = tr ? r0 : n0, o1 = tr ? r1 : n1;
  constexpr int NP = UP ? 8 : 16;  // pairs of a tile this wave stores
  const int t0 = D::NTILE * blockIdx.y / gridDim.y, t1 = D::NTILE * (blockIdx.y + 1) / gridDim.y;
  double A[KT];
  auto load_a = [&](int t) {
#pragma unroll
    for (int s = 0; s < KT; ++s) A[s] = (s < KB || rb) ? T.At[((size_t)t * KT + s) * 64 + lane] : 0.0;
  };
  load_a(t0);
  for (int t = t0; t < t1; ++t) {
    // lane p < 16: block code of pair 16 t + p for this wave's orientation
    // (no block: INT_MAX), its row and column masks, and whether a == b
    // (UP: lane i < 8 pair 16 t + 2 i, or + 1, and turn its orientation)
    int code = 0x7fffffff, mr = 0, mc = 0, dg = -1, turn = 0;
    if (lane < NP) {
      const int ab = sPab[16 * t + (UP ? 2 * lane + (tr ? 1 : 0) : lane)], a = ab & 255, b = ab >> 8;
      if (ab != 0xffff && (UP || !(tr && a == b))) {
        const bool x = UP ? sNode[a] > sNode[b] : tr;
        code = x ? sBlk[b * NS + a] : sBlk[a * NS + b];
        mr = (int)sMask[x ? b : a];
        mc = (int)sMask[x ? a : b];
        dg = a == b ? a : -1;
        turn = x;
      }
    }
    J2 old[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int cd = __builtin_amdgcn_readlane(code, p);
      old[p] = J2{0, 0};
      if (cd >= 0 && cd != 0x7fffffff && own) old[p] = reinterpret_cast<const J2 *>(J + (size_t)cd * 324)[pos];
    }
    f64x4 acc[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) acc[k] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < KB; ++s)
#pragma unroll
      for (int k = 0; k < 2; ++k) acc[k] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[s], B[k][s], acc[k], 0, 0, 0);
    if (rb)
#pragma unroll
      for (int s = KB; s < KT; ++s)
#pragma unroll
        for (int k = 0; k < 2; ++k) acc[k] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[s], B[k][s], acc[k], 0, 0, 0);
    if (t + 1 < t1) load_a(t + 1);
    double *O = S + (t & 1) * 16 * TS;
    // D layout: lane l holds rows 4 q + l / 16, column l % 16
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int q = 0; q < 4; ++q) O[(4 * q + (lane >> 4)) * TS + 16 * (w + 6 * k) + (lane & 15)] = acc[k][q];
    __syncthreads();
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int cd = __builtin_amdgcn_readlane(code, p);
      if (cd == 0x7fffffff) continue;
      const uint32_t ur = (uint32_t)__builtin_amdgcn_readlane(mr, p), uc = (uint32_t)__builtin_amdgcn_readlane(mc, p);
      const double *row = O + (UP ? 2 * p + (tr ? 1 : 0) : p) * TS;
      const bool x = UP && __builtin_amdgcn_readlane(turn, p);
      double v0 = row[UP ? (x ? r0 : n0) : o0], v1 = row[UP ? (x ? r1 : n1) : o1];
      if (ur | uc) {
        const int na = __builtin_amdgcn_readlane(dg, p);  // the node of a diagonal block
        // hanging nodes (adaptive meshes): the condensed row keeps the sum
        // over cells of |local diagonal|
        if (HANG && na >= 0 && (ur & HANG_BIT) && own && (c == r || c + 1 == r))
          Mh.hdiag[(size_t)cn[na] * 18 + r] += fabs(c == r ? v0 : v1);
        const bool rm = (ur >> r) & 1u;
        if (rm || ((uc >> c) & 1u)) v0 = (na >= 0 && rm && c == r) ? fabs(v0) : 0.0;
        if (rm || ((uc >> (c + 1)) & 1u)) v1 = (na >= 0 && rm && c + 1 == r) ? fabs(v1) : 0.0;
      }
      const int blk = cd < 0 ? -cd - 1 : cd;
      if (own)
        reinterpret_cast<J2 *>(J + (size_t)blk * 324)[pos] = J2{(TJ)((double)old[p].x + v0), (TJ)((double)old[p].y + v1)};
    }
  }
}

// The same for Q1 (8 points, 36 node pairs): one workgroup of 3 waves per
// cell and part of its pairs.  A thread owns entries [r][c], [r][c + 1] of
// every block, keeps their Hessian at the 8 points in registers and contracts
// it with the uniform node-pair weights; the block (a, b) and the transposed
// (b, a) take the same sums (the K2 + K3 term aside), so nothing goes through
// LDS after the Gram matrices, and a dozen cells run on a CU.  The block
// codes and masks of the cell sit in lanes, the old values of the next pairs
// are on their way.  48^3 cells: 11.3 -> 7.7 ms FP64, 9.5 -> 4.4 ms FP32;
// 8^3 cells (64 a colour): 0.37 -> 0.12 ms.
// UP: as k_assemble_q2 (batch of 48 slabs FP32, a colour: 156 -> 129 us).
template <typename TJ, bool HANG, bool UP>
__global__ __launch_bounds__(192, HANG && sizeof(TJ) == 8 ? 3 : 4) void k_assemble_q1(RefTables T, MeshDev Mh, Material M0,
                                                        const double *__restrict__ U, const int *__restrict__ cells,
                                                        TJ *__restrict__ J)
{
  using J2 = typename Vec2<TJ>::type;
  constexpr int NS = 8, NQ = 8, NPAIR = 36;
  __shared__ double sU[NS * 18], sX[NQ * 18], sGram[NQ * GRAM], sSp[NPAIR * 9], sH[NQ * NUPAIR];
  const int tid = threadIdx.x, lane = tid & 63;
  const int e = cells[blockIdx.x];
  if (Mh.inst_active && !Mh.inst_active[Mh.cell_inst[e]]) return;  // finished instance of a batch
  const Material M = Mh.mats ? Mh.mats[Mh.cell_mat[e]] : M0;       // per-instance (T, p) in a batch
  const int *cn = Mh.cell_nodes + (size_t)e * NS;
  double h[3], ih[3];
  for (int k = 0; k < 3; ++k) { h[k] = Mh.cell_h[3 * e + k]; ih[k] = 1.0 / h[k]; }
  const double vol = h[0] * h[1] * h[2];
  const uint32_t cface = Mh.cell_face[e];
  const bool rb = M.robin != 0.0 && cface != 0u;
  // lane l: the code of block (l / 8, l % 8), the mask of node l % 8
  const int codes = Mh.cell_blk[(size_t)e * NS * NS + lane];
  const int nodes = cn[lane & 7], masks = (int)Mh.node_mask[nodes];
  // UP: the block (a, b), or (b, a), of a pair is below the diagonal
  const auto low = [&](int a, int b) {
    return UP && __builtin_amdgcn_readlane(nodes, a) > __builtin_amdgcn_readlane(nodes, b);
  };
  if (tid < NS * 18) sU[tid] = U[(size_t)cn[tid / 18] * 18 + (tid % 18)];
  for (int i = tid; i < NPAIR * 9; i += 192) sSp[i] = T.Sp[i];
  __syncthreads();
  if (tid < NQ * 18) {  // the iterate at the quadrature points (s_vector2matrix.cc:116-217)
    const int q = tid / 18, c = tid % 18;
    double xv = 0;
#pragma unroll
    for (int a = 0; a < NS; ++a) xv += T.N[q * NS + a] * sU[a * 18 + c];
    sX[tid] = xv;
  }
  __syncthreads();
#pragma unroll 1
  for (int i = tid; i < NQ * GRAM; i += 192) {
    const int q = i / GRAM, g = i % GRAM;
    sGram[i] = gram_entry(sX + q * 18, g);
  }
  __syncthreads();
  // lanes beyond 162 repeat the last thread's work and store nothing (all
  // lanes stay active: the codes and masks are read across them)
  const bool own = tid < 162;
  const int pos = own ? tid : 161, r = pos / 9, c0 = 2 * (pos % 9);
  if (tid < NUPAIR) {  // H_cd, c <= d, once per cell
    int c = 0, t = tid;
    while (t >= 18 - c) { t -= 18 - c; ++c; }
#pragma unroll 2
    for (int q = 0; q < NQ; ++q)
      sH[q * NUPAIR + tid] = vol * hess_entry(sGram + q * GRAM, sX + q * 18, c, c + t, M);
  }
  __syncthreads();
  double H[2][NQ];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int c = c0 + k, lo = r < c ? r : c, hi = r < c ? c : r, i = lo * 18 - lo * (lo - 1) / 2 + hi - lo;
#pragma unroll
    for (int q = 0; q < NQ; ++q) H[k][q] = sH[q * NUPAIR + i];
  }
  const double lap0 = M.K1 * vol * ih[0] * ih[0], lap1 = M.K1 * vol * ih[1] * ih[1], lap2 = M.K1 * vol * ih[2] * ih[2];
  // K2 + K3 of [r][c] (the same part and spin) and where its integrals are:
  // of (a, b) and transposed of (b, a)
  double k23[2];
  int ks[2], kt[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int c = c0 + k;
    k23[k] = r / 3 == c / 3 ? M.K23 * vol * ih[r % 3] * ih[c % 3] : 0.0;
    ks[k] = 3 * (r % 3) + c % 3;
    kt[k] = 3 * (c % 3) + r % 3;
  }
  const bool d0 = c0 == r, d1 = c0 + 1 == r;
  constexpr int PD = 4;  // pairs whose old values are on their way
  J2 old[PD][2];
  const int p0 = NPAIR * blockIdx.y / gridDim.y, p1 = NPAIR * (blockIdx.y + 1) / gridDim.y;
  // pair p = (a, b), stepped in the order of the tables (uniform)
  struct Pair {
    int a, b;
    __device__ inline Pair(int p) : a(0)
    {
      while (p >= NS - a) { p -= NS - a; ++a; }
      b = a + p;
    }
    __device__ inline void next()
    {
      if (++b == NS) b = ++a;
    }
  };
  auto load_old = [&](const Pair &P, J2 *o) {
    const int cab = __builtin_amdgcn_readlane(codes, P.a * NS + P.b),
              cba = __builtin_amdgcn_readlane(codes, P.b * NS + P.a);
    o[0] = o[1] = J2{0, 0};
    if (cab >= 0 && !low(P.a, P.b)) o[0] = reinterpret_cast<const J2 *>(J + (size_t)cab * 324)[pos];
    if (P.a != P.b && cba >= 0 && !low(P.b, P.a)) o[1] = reinterpret_cast<const J2 *>(J + (size_t)cba * 324)[pos];
  };
  auto store = [&](int code, const J2 &o, double v0, double v1) {
    const int blk = code < 0 ? -code - 1 : code;
    const J2 v = {(TJ)((double)o.x + v0), (TJ)((double)o.y + v1)};
    if (own) reinterpret_cast<J2 *>(J + (size_t)blk * 324)[pos] = v;
  };
  Pair P(p0), F(p0);
#pragma unroll
  for (int k = 0; k < PD; ++k)
    if (p0 + k < p1) {
      load_old(F, old[k]);
      F.next();
    }
  // (rolled: 36 unrolled pairs are 40 KB of code, fetched once per wave)
#pragma unroll 1
  for (int pb = p0; pb < p1; pb += PD)
#pragma unroll
    for (int k = 0; k < PD; ++k) {
      const int p = pb + k;
      if (p >= p1) break;
      const int a = P.a, b = P.b;
      P.next();
      const J2 o0 = old[k][0], o1 = old[k][1];
      if (p + PD < p1) {
        load_old(F, old[k]);
        F.next();
      }
      double v0 = 0.0, v1 = 0.0;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const double wq = T.Wp[p * NQ + q];
        v0 += wq * H[0][q];
        v1 += wq * H[1][q];
      }
      double lap = T.Sp[p * 9] * lap0 + T.Sp[p * 9 + 4] * lap1 + T.Sp[p * 9 + 8] * lap2;
      if (rb)
        for (int lf = 0; lf < 6; ++lf) {
          const int bid = (int)((cface >> (3 * lf)) & 7u) - 1;
          if (bid >= 2 && bid <= 4 && !face_zeroed(bid, r))
            lap += M.robin * face_area(lf, h) * T.Mf[(lf * NS + a) * NS + b];
        }
      v0 += d0 ? lap : 0.0;
      v1 += d1 ? lap : 0.0;
      double t0 = v0 + k23[0] * sSp[p * 9 + kt[0]], t1 = v1 + k23[1] * sSp[p * 9 + kt[1]];  // of (b, a)
      v0 += k23[0] * sSp[p * 9 + ks[0]];
      v1 += k23[1] * sSp[p * 9 + ks[1]];
      const uint32_t ma = (uint32_t)__builtin_amdgcn_readlane(masks, a),
                     mb = (uint32_t)__builtin_amdgcn_readlane(masks, b);
      if (ma | mb) {
        // hanging nodes (adaptive meshes): the condensed row keeps the sum
        // over cells of |local diagonal|
        if (HANG && a == b && (ma & HANG_BIT) && own && (d0 || d1))
          Mh.hdiag[(size_t)cn[a] * 18 + r] += fabs(d0 ? v0 : v1);
        const bool ra = (ma >> r) & 1u, rbm = (mb >> r) & 1u;  // row r of node a, of node b
        if (ra || ((mb >> c0) & 1u)) v0 = (a == b && ra && d0) ? fabs(v0) : 0.0;
        if (ra || ((mb >> (c0 + 1)) & 1u)) v1 = (a == b && ra && d1) ? fabs(v1) : 0.0;
        if (rbm || ((ma >> c0) & 1u)) t0 = 0.0;
        if (rbm || ((ma >> (c0 + 1)) & 1u)) t1 = 0.0;
      }
      if (!low(a, b)) store(__builtin_amdgcn_readlane(codes, a * NS + b), o0, v0, v1);
      if (a != b && !low(b, a)) store(__builtin_amdgcn_readlane(codes, b * NS + a), o1, t0, t1);
    }
}

// ------------------------------------------------ matrix-free Jacobian
// J x without the assembled matrix (on a mesh with constraint lines applied
// to C x and condensed, gl_constraints.hip).  The Jacobian of the cell loop is
//   J_(a,c),(b,d) = vol sum_q w_q N_a N_b H_cd(q)             (bulk, H symmetric)
//                 + K1 delta_cd vol sum_q w_q grad N_a . grad N_b
//                 + K23 [c, d same part and spin] vol sum_q w_q d_kc N_a d_kd N_b
//                 + Robin face mass on the diagonal components,
// with kc, kd the orbital indices of c, d.  Per cell this is applied as
//   X_q = sum_b N_b(q) x_b, G_kq = sum_b d_k N_b(q) x_b / h_k,
//   y_a += sum_q w_q vol (N_a(q) H(q) X_q + sum_k d_k N_a(q) / h_k gamma_k(q)),
//   gamma_{c,k} = K1 G_kq[c] + K23 [k == kc] sum_kd G_kd,q[9 part + 3 mu + kd],
// sum-factorised, instead of streaming the cell's 729 blocks.  k_mf_setup
// stores the iterate at the quadrature points per cell (the only state of
// the operator besides the diagonal blocks; H(q) X(q) is formed from it in
// the product) and the cells' shares of the diagonal blocks for the
// point-block Jacobi preconditioner; Dirichlet columns are applied as a zero x
// in the product, Dirichlet rows keep only their diagonal (k_mf_gather).

// The diagonal blocks are symmetric: a cell's block of a node is its 171
// entries c <= d, those of the parts (u, u) and (v, v) first (their Hessian
// entries have one form, the (u, v) entries another, so that most wavefronts
// evaluate only one).
__device__ inline void diag_pair(int t, int &c, int &d)
{
  if (t >= 90) {
    c = (t - 90) / 9;
    d = 9 + (t - 90) % 9;
    return;
  }
  const int part = t / 45;
  int i = t - 45 * part;
  c = 0;
  while (i >= 9 - c) { i -= 9 - c; ++c; }
  d = 9 * part + c + i;
  c += 9 * part;
}

// 1D line of point values h -> sum_i w_i L_a(x_i)^2 h_i of its nodes
template <int DEG>
__device__ inline void square_line(double &a, double &b, double &c)
{
  if constexpr (DEG == 2) {
    constexpr double t = 0.38729833462074168852;  // sqrt(3/5) / 2, the outer points' distance from the middle
    constexpr double w = 5.0 / 18.0, p = w * (0.3 + t) * (0.3 + t), m = w * (0.3 - t) * (0.3 - t);
    const double h0 = a, h2 = c;
    a = p * h0 + m * h2;
    b = (8.0 / 18.0) * b + (w * 0.16) * (h0 + h2);
    c = m * h0 + p * h2;
  } else {
    constexpr double t = 0.28867513459481288225;  // 1 / (2 sqrt 3)
    constexpr double p = 0.5 * (0.5 + t) * (0.5 + t), m = 0.5 * (0.5 - t) * (0.5 - t);
    const double h0 = a;
    a = p * h0 + m * b;
    b = m * h0 + p * b;
  }
}
template <int DEG>
__device__ inline void square_lines(double *h)
{
  constexpr int N = DEG + 1;
#pragma unroll
  for (int s = 1, k = 0; k < 3; ++k, s *= N)
#pragma unroll
    for (int l = 0; l < N * N; ++l) {
      const int o = (l / s) * s * N + l % s;
      square_line<DEG>(h[o], h[o + s], h[o + (DEG == 2 ? 2 * s : s)]);
    }
}

// One workgroup per cell of a chunk of cells: the iterate at the quadrature
// points, and the cell's share of its nodes' diagonal blocks into slots
// ([cell][node][171], raw: no Dirichlet rule).  A thread holds one entry's
// Hessian at the points and contracts it with w N_a^2, a tensor product, by
// 1D lines (162 operations instead of 729 multiply-adds in Q2).  Bound by the
// Hessian entries' instructions and LDS reads (the vector unit busy 45% of the
// time, LDS about as much).  Per Newton step, setup and
// gather: 32^3 Q2 cells 10 x (114 + 39) us, against 8 colours of 280 us that
// read and rewrote the nodes' blocks; 5586 Q2 cells FP32 2 x (95 + 30) against
// 8 x 60; 22528 Q1 cells with hanging nodes 2 x (128 + 32) against 11 x 55.
// CON: a mesh with constraint lines (the raw local blocks X lists as well)
template <int DEG, typename TH, bool CON>
__global__ __launch_bounds__(NT) void k_mf_setup(RefTables T, MeshDev Mh, Material M0, const double *__restrict__ U,
                                                 int e0, TH *__restrict__ Uq, double *__restrict__ slots, MfCondDev X)
{
  constexpr int N1 = DEG + 1, NS = N1 * N1 * N1, NQ = NS;
  __shared__ double sU[NS * 18];
  __shared__ double sX[NQ * 18];
  __shared__ double sGram[NQ * GRAM];
  __shared__ double sSp[NS * 9];  // the gradient products of the node pairs (a, a)
  const int tid = threadIdx.x;
  const int e = e0 + blockIdx.x;
  // a finished instance of a batch keeps the iterate and blocks of its last
  // step (all of its cells are skipped together)
  if (Mh.inst_active && !Mh.inst_active[Mh.cell_inst[e]]) return;
  const Material M = Mh.mats ? Mh.mats[Mh.cell_mat[e]] : M0;
  const int *cn = Mh.cell_nodes + (size_t)e * NS;
  double h[3], ih[3];
  for (int k = 0; k < 3; ++k) { h[k] = Mh.cell_h[3 * e + k]; ih[k] = 1.0 / h[k]; }
  const double vol = h[0] * h[1] * h[2];
  const uint32_t cface = Mh.cell_face[e];
  for (int i = tid; i < NS * 18; i += NT) sU[i] = U[(size_t)cn[i / 18] * 18 + (i % 18)];
  for (int i = tid; i < NS * 9; i += NT) {
    const int a = i / 9;
    sSp[i] = T.Sp[(size_t)(a * NS - a * (a - 1) / 2) * 9 + i % 9];
  }
  __syncthreads();
  for (int i = tid; i < NQ * 18; i += NT) {
    const int q = i / 18, c = i % 18;
    double xv = 0;
    for (int a = 0; a < NS; ++a) xv += T.N[q * NS + a] * sU[a * 18 + c];
    sX[i] = xv;
    Uq[(size_t)e * NQ * 18 + c * NQ + q] = (TH)xv;  // the iterate at the points, the product's state
  }
  __syncthreads();
  for (int i = tid; i < NQ * GRAM; i += NT) {
    const int q = i / GRAM, g = i % GRAM;
    sGram[i] = gram_entry(sX + q * 18, g);
  }
  __syncthreads();
  if (tid >= NUPAIR) return;
  int c, d;
  diag_pair(tid, c, d);
  double Hv[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) Hv[q] = hess_entry(sGram + q * GRAM, sX + q * 18, c, d, M);
  const bool grad_cd = (c / 9 == d / 9) && ((c % 9) / 3 == (d % 9) / 3);
  const int kc = c % 3, kd = d % 3;
  const double lap0 = vol * ih[0] * ih[0], lap1 = vol * ih[1] * ih[1], lap2 = vol * ih[2] * ih[2];
  const double k23_cd = M.K23 * vol * ih[kc] * ih[kd];
  // the gradient and Robin terms of entry [c][d] of node pair (a, b), whose
  // gradient products are sp
  auto edge_terms = [&](const double *sp, int a, int b) {
    double v = 0.0;
    if (c == d) {
      v += M.K1 * (sp[0] * lap0 + sp[4] * lap1 + sp[8] * lap2);
      if (M.robin != 0.0)
        for (int lf = 0; lf < 6; ++lf) {
          const int bid = (int)((cface >> (3 * lf)) & 7u) - 1;
          if (bid >= 2 && bid <= 4 && !face_zeroed(bid, c))
            v += (M.robin * face_area(lf, h)) * T.Mf[(lf * NS + a) * NS + b];
        }
    }
    return v;
  };
  // constrained meshes: the raw local blocks that constraint lines fold into
  // the condensed diagonal blocks of masters (few cells have any)
  if (CON)
    for (int k = X.xptr[e]; k < X.xptr[e + 1]; ++k) {
      const int p = X.xpair[k], a = T.pa[p], b = T.pb[p];
      const double *wp = T.Wp + (size_t)p * NQ, *sp = T.Sp + (size_t)p * 9;
      double sym = 0.0;
#pragma unroll
      for (int q = 0; q < NQ; ++q) sym += wp[q] * Hv[q];
      sym = sym * vol + edge_terms(sp, a, b);
      double v1 = sym, v2 = sym;
      if (grad_cd) {
        v1 += k23_cd * sp[kc * 3 + kd];
        v2 += k23_cd * sp[kd * 3 + kc];
      }
      double *B = X.LB + (size_t)k * 324;
      B[c * 18 + d] = v1;
      if (c != d) B[d * 18 + c] = v2;
    }
  square_lines<DEG>(Hv);
  double *S = slots + (size_t)blockIdx.x * NS * NUPAIR + tid;
#pragma unroll
  for (int a = 0; a < NS; ++a) {
    double v = Hv[a] * vol + edge_terms(sSp + 9 * a, a, a);
    if (grad_cd) v += k23_cd * sSp[9 * a + 3 * kc + kd];
    S[a * NUPAIR] = v;
  }
}

// The diagonal blocks of the nodes n0 .. n1 - 1 (a range that holds the nodes
// of cells e0 .. e1 - 1) from their slots, in cell order: the first chunk that
// holds a cell of the node writes its block, later ones add.  A thread sums
// one of the 171 entries of DG nodes, 16 slots in flight; the blocks go out
// whole through LDS.  Dirichlet rows and columns are 0 but for the sum of
// |local diagonal|, which a hanging node also keeps in hdiag (CON).
constexpr int DG = 4;
template <int NS, bool CON>
__global__ __launch_bounds__(NT) void k_mf_diag_gather(int n0, int n1, int e0, int e1,
                                                       const int *__restrict__ n2c_ptr,
                                                       const int *__restrict__ n2c_idx,
                                                       const double *__restrict__ slots,
                                                       const uint32_t *__restrict__ node_mask,
                                                       const int *__restrict__ row_seg,
                                                       const int *__restrict__ inst_active, double *__restrict__ Jd,
                                                       double *__restrict__ hdiag)
{
  __shared__ double sB[DG][324];
  const int tid = threadIdx.x, base = n0 + blockIdx.x * DG;
  const int lo = e0 * NS, hi = e1 * NS;
  int c = 0, d = 0;
  if (tid < NUPAIR) diag_pair(tid, c, d);
  unsigned in = 0, first = 0;  // nodes of the chunk, and those written here first
#pragma unroll
  for (int j = 0; j < DG; ++j) {
    const int n = base + j;
    if (n >= n1 || (inst_active && !inst_active[row_seg[n]])) continue;
    const int p0 = n2c_ptr[n], p1 = n2c_ptr[n + 1];
    if (p0 == p1 || n2c_idx[p0] >= hi || n2c_idx[p1 - 1] < lo) continue;
    in |= 1u << j;
    if (n2c_idx[p0] >= lo) first |= 1u << j;
    if (tid >= NUPAIR) continue;
    const uint32_t m = node_mask[n];
    const bool rc = (m >> c) & 1u, rd = (m >> d) & 1u;
    double acc = 0.0, habs = 0.0;
    for (int p = p0; p < p1; p += 4) {
      double v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int k = p + u < p1 ? n2c_idx[p + u] : -1;
        v[u] = k >= lo && k < hi ? slots[(size_t)(k - lo) * NUPAIR + tid] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        acc += rc && c == d ? fabs(v[u]) : v[u];
        if (CON) habs += fabs(v[u]);
      }
    }
    if ((rc || rd) && c != d) acc = 0.0;
    sB[j][c * 18 + d] = acc;
    sB[j][d * 18 + c] = acc;
    if (CON && c == d && (m & HANG_BIT)) hdiag[(size_t)n * 18 + c] += habs;
  }
  if (!in) return;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < DG; ++j) {
    if (!((in >> j) & 1u)) continue;
    double *B = Jd + (size_t)(base + j) * 324;
    const bool f = (first >> j) & 1u;
    for (int i = tid; i < 324; i += NT) B[i] = f ? sB[j][i] : B[i] + sB[j][i];
  }
}

// The product in sum-factorised form: N_b(q) = L_bx(x_qx) L_by(x_qy) L_bz(x_qz),
// so x and its gradients at the quadrature points take 1D passes in the three
// directions, and the test against N_a and its gradients three more.  At the
// points, H(q) X(q) is formed as the derivative of rho at the stored iterate
// U(q) (18 values per point) in the direction X(q).
// TH: the stored iterate (FP64, or FP32 for the FP32 inner solve); TX: x.
// TA, the arithmetic, LDS and cell-slot type, is FP32 when both are FP32 (the
// FP32 inner solve, with FP32 accumulation) and FP64 otherwise.
// RES: the residual R(x) of the cell loop (residual.cc:164-232, the Robin
// faces :235-278) through the same passes: x is the iterate (no column
// masking), and rho(X(q)), the bulk residual density, takes the place of
// H(q) X(q); Uq is not read, and flag is the batch's instance_active.

// One 1D line of the tensor-product element FE_Q(DEG) x Gauss(DEG + 1), in
// Q2 in local polynomial coefficients: with tau = xi - 1/2 a quadratic is
// m + tau d + 2 tau^2 w (m = v1, d = v2 - v0, w = v0 - 2 v1 + v2).  The Gauss
// points are symmetric about the middle, so values and derivatives of a line
// at its points take 8 operations instead of 18 multiply-adds with the
// tables, and their transposes (the test passes) 12; the middle point's value
// is m and its derivative d.  (Q1 keeps the two node weights: the shorter
// v0 + xi d rounds worse in FP32.)  The
// transposes carry the 1D weights relative to the middle point's; the factor
// that is left per cell is W0 (the middle weight) cubed.
template <int DEG, typename T>
struct Line;

template <typename T>
struct Line<2, T> {
  static constexpr int N = 3;
  static constexpr double W0 = 8.0 / 18.0;
  static constexpr double h = 0.38729833462074168852;  // sqrt(3/5) / 2, the outer points' tau
  static constexpr double r = 0.625;                    // the outer points' weight over the middle one's
  // coefficients of the line (in place of its values)
  static __device__ inline void coef(T &a, T &b, T &c)
  {
    const T m = b, d = c - a, w = (a + c) - (T)2 * b;
    a = m;
    b = d;
    c = w;
  }
  static __device__ inline void uncoef(T &a, T &b, T &c)  // transpose of coef
  {
    const T m = a, d = b, w = c;
    a = w - d;
    b = m - (T)2 * w;
    c = w + d;
  }
  // point q (uniform) of the z lines: value and derivative from coefficients
  T v1, v2, d2, wq, wv1, wv2, wd2;
  __device__ inline void point(int q)
  {
    v1 = (T)(q == 0 ? -h : q == 1 ? 0.0 : h);
    v2 = (T)(q == 1 ? 0.0 : 2 * h * h);
    d2 = (T)(q == 0 ? -4 * h : q == 1 ? 0.0 : 4 * h);
    wq = (T)(q == 1 ? 1.0 : r);
    wv1 = (T)(q == 0 ? -r * h : q == 1 ? 0.0 : r * h);
    wv2 = (T)(q == 1 ? 0.0 : r * 2 * h * h);
    wd2 = (T)(q == 0 ? -r * 4 * h : q == 1 ? 0.0 : r * 4 * h);
  }
  __device__ inline T val(const T *k) const { return k[0] + v1 * k[1] + v2 * k[2]; }
  __device__ inline T der(const T *k) const { return k[1] + d2 * k[2]; }
  // transpose of both: k += val^T p + der^T g, with the weight of the point
  __device__ inline void back(T p, T g, T *k) const
  {
    k[0] += wq * p;
    k[1] += wv1 * p;
    k[1] += wq * g;
    k[2] += wv2 * p;
    k[2] += wd2 * g;
  }
  __device__ inline void back(T p, T *k) const
  {
    k[0] += wq * p;
    k[1] += wv1 * p;
    k[2] += wv2 * p;
  }
  // values (and derivatives) of a line at its points
  static __device__ inline void values(const T *v, T *p)
  {
    const T d = v[2] - v[0], w = (v[0] + v[2]) - (T)2 * v[1], e = v[1] + (T)(2 * h * h) * w;
    p[0] = e - (T)h * d;
    p[1] = v[1];
    p[2] = e + (T)h * d;
  }
  static __device__ inline void both(const T *v, T *p, T *g)
  {
    const T d = v[2] - v[0], w = (v[0] + v[2]) - (T)2 * v[1], e = v[1] + (T)(2 * h * h) * w;
    p[0] = e - (T)h * d;
    p[1] = v[1];
    p[2] = e + (T)h * d;
    g[0] = d - (T)(4 * h) * w;
    g[1] = d;
    g[2] = d + (T)(4 * h) * w;
  }
  // their transposes, with the points' weights
  static __device__ inline void test_v(const T *p, T *v)
  {
    const T a = p[0] + p[2], b = (T)(r * h) * (p[2] - p[0]), w = (T)(r * 2 * h * h) * a, m = p[1] + (T)r * a;
    v[0] = w - b;
    v[1] = m - (T)2 * w;
    v[2] = w + b;
  }
  static __device__ inline void test_d(const T *g, T *v)
  {
    const T d = g[1] + (T)r * (g[0] + g[2]), w = (T)(r * 4 * h) * (g[2] - g[0]);
    v[0] = w - d;
    v[1] = (T)-2 * w;
    v[2] = w + d;
  }
  static __device__ inline void test_vd(const T *p, const T *g, T *v)
  {
    const T a = p[0] + p[2], m = p[1] + (T)r * a;
    const T d = (T)(r * h) * (p[2] - p[0]) + (g[1] + (T)r * (g[0] + g[2]));
    const T w = (T)(r * 2 * h * h) * a + (T)(r * 4 * h) * (g[2] - g[0]);
    v[0] = w - d;
    v[1] = m - (T)2 * w;
    v[2] = w + d;
  }
  // 1D mass matrix of a unit edge times 30 (the Robin faces)
  static constexpr double M0 = 1.0 / 30.0;
  static __device__ inline void mass(const T *v, T *y)
  {
    y[0] = (T)4 * v[0] + (T)2 * v[1] - v[2];
    y[1] = (T)2 * v[0] + (T)16 * v[1] + (T)2 * v[2];
    y[2] = (T)-1 * v[0] + (T)2 * v[1] + (T)4 * v[2];
  }
};

template <typename T>
struct Line<1, T> {
  static constexpr int N = 2;
  static constexpr double W0 = 0.5;
  static constexpr double t0 = 0.21132486540518711775, t1 = 0.78867513459481288225;  // (1 -+ 1/sqrt(3)) / 2
  T a, b;  // of the z lines' point q: the weights of the two nodes
  __device__ inline void point(int q)
  {
    a = (T)(q == 0 ? t1 : t0);
    b = (T)(q == 0 ? t0 : t1);
  }
  __device__ inline T val(const T *k) const { return a * k[0] + b * k[1]; }
  __device__ inline T der(const T *k) const { return k[1] - k[0]; }
  __device__ inline void back(T p, T g, T *k) const
  {
    k[0] += a * p - g;
    k[1] += b * p + g;
  }
  __device__ inline void back(T p, T *k) const
  {
    k[0] += a * p;
    k[1] += b * p;
  }
  static __device__ inline void values(const T *v, T *p)
  {
    p[0] = (T)t1 * v[0] + (T)t0 * v[1];
    p[1] = (T)t0 * v[0] + (T)t1 * v[1];
  }
  static __device__ inline void both(const T *v, T *p, T *g)
  {
    values(v, p);
    g[0] = g[1] = v[1] - v[0];
  }
  static __device__ inline void test_v(const T *p, T *v)
  {
    v[0] = (T)t1 * p[0] + (T)t0 * p[1];
    v[1] = (T)t0 * p[0] + (T)t1 * p[1];
  }
  static __device__ inline void test_d(const T *g, T *v)
  {
    v[1] = g[0] + g[1];
    v[0] = -v[1];
  }
  static __device__ inline void test_vd(const T *p, const T *g, T *v)
  {
    const T d = g[0] + g[1];
    v[0] = ((T)t1 * p[0] + (T)t0 * p[1]) - d;
    v[1] = ((T)t0 * p[0] + (T)t1 * p[1]) + d;
  }
  static constexpr double M0 = 1.0 / 6.0;
  static __device__ inline void mass(const T *v, T *y)
  {
    y[0] = (T)2 * v[0] + v[1];
    y[1] = v[0] + (T)2 * v[1];
  }
};

// The bulk term at one point.  rho and its derivative are a symmetric 6 x 6
// matrix on the spin index of (u, v), rows mu, times the 6 x 3 matrix (u; v):
//   rho(A) = N(A) (u; v),   H(A) X = N(A) (a; b) + dN(A; X) (u; v),
//   N = [[E, C], [C^T, F]],
//   E = 2 (b3+b4+b5) u u^T + 2 (b4+b5-b3) v v^T + (al + 2 b1 p + 2 b2 s) 1,
//   F = 2 (b4+b5-b3) u u^T + 2 (b3+b4+b5) v v^T + (al - 2 b1 p + 2 b2 s) 1,
//   C = 2 (b3+b4-b5) u v^T + 2 (b3-b4+b5) v u^T + 4 b1 (u:v) 1,
// p = |u|^2 - |v|^2, s = |u|^2 + |v|^2: the terms of the reference's density
// collected by the Gram matrices u u^T, v v^T, u v^T, in which N is linear
// (dN is N of their derivatives, without al).  One thread forms the 18
// entries of a point from registers in about 500 operations (rho: 230),
// against 936 term by term.
template <typename T>
struct BulkMat {
  T E[6], F[6], C[9];  // symmetric entries 00 01 02 11 12 22
  __device__ inline void set(const T *uu, const T *vv, const T *uv, T al, T tb1, T tb2, T c1, T c2, T d1, T d2)
  {
    const T tu = uu[0] + uu[3] + uu[5], tv = vv[0] + vv[3] + vv[5], q = (T)2 * (uv[0] + uv[4] + uv[8]);
    const T p = tu - tv, s = tu + tv, i2 = al + tb2 * s;
    const T ei = i2 + tb1 * p, fi = i2 - tb1 * p, ci = tb1 * q;
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      const bool dg = i == 0 || i == 3 || i == 5;
      E[i] = c1 * uu[i] + c2 * vv[i];
      F[i] = c2 * uu[i] + c1 * vv[i];
      if (dg) {
        E[i] += ei;
        F[i] += fi;
      }
    }
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
      for (int n = 0; n < 3; ++n) {
        C[3 * m + n] = d1 * uv[3 * m + n] + d2 * uv[3 * n + m];
        if (m == n) C[3 * m + n] += ci;
      }
  }
  // (zu, zv) += N (a; b) for the orbital column k
  __device__ inline void add(const T *a, const T *b, int k, T *zu, T *zv) const
  {
    constexpr int id[9] = {0, 1, 2, 1, 3, 4, 2, 4, 5};
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
      for (int n = 0; n < 3; ++n) {
        zu[m] += E[id[3 * m + n]] * a[3 * n + k];
        zu[m] += C[3 * m + n] * b[3 * n + k];
        zv[m] += C[3 * n + m] * a[3 * n + k];
        zv[m] += F[id[3 * m + n]] * b[3 * n + k];
      }
  }
};

// u u^T, v v^T (symmetric entries) and u v^T of the 18 values s
template <typename T>
__device__ inline void gram(const T *s, T *uu, T *vv, T *uv)
{
  int i = 0;
#pragma unroll
  for (int m = 0; m < 3; ++m)
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      T a = s[3 * m] * s[9 + 3 * n];
      a += s[3 * m + 1] * s[9 + 3 * n + 1];
      a += s[3 * m + 2] * s[9 + 3 * n + 2];
      uv[3 * m + n] = a;
      if (n < m) continue;
      T b = s[3 * m] * s[3 * n], c = s[9 + 3 * m] * s[9 + 3 * n];
#pragma unroll
      for (int k = 1; k < 3; ++k) {
        b += s[3 * m + k] * s[3 * n + k];
        c += s[9 + 3 * m + k] * s[9 + 3 * n + k];
      }
      uu[i] = b;
      vv[i] = c;
      ++i;
    }
}

// their derivatives at s in the direction x
template <typename T>
__device__ inline void dgram(const T *s, const T *x, T *uu, T *vv, T *uv)
{
  int i = 0;
#pragma unroll
  for (int m = 0; m < 3; ++m)
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      T a = 0, b = 0, c = 0;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        a += x[3 * m + k] * s[9 + 3 * n + k];
        a += s[3 * m + k] * x[9 + 3 * n + k];
        if (n < m) continue;
        b += x[3 * m + k] * s[3 * n + k];
        c += x[9 + 3 * m + k] * s[9 + 3 * n + k];
        if (n == m) continue;
        b += s[3 * m + k] * x[3 * n + k];
        c += s[9 + 3 * m + k] * x[9 + 3 * n + k];
      }
      uv[3 * m + n] = a;
      if (n < m) continue;
      uu[i] = n == m ? (T)2 * b : b;
      vv[i] = n == m ? (T)2 * c : c;
      ++i;
    }
}

template <typename TH, typename TX>
using mf_arith = typename std::conditional<std::is_same<TH, float>::value && std::is_same<TX, float>::value, float,
                                           double>::type;
// Cells per workgroup: 7 on two waves (126 of 128 lanes hold a column, 189 Q2
// points fill three rounds of a wave), or for meshes of few cells, where the
// length of one thread's work counts, 1 on one wave with a thread per column
// and plane of points.
constexpr int MF_CELLS = 7;
template <int NCELL>
constexpr int mf_threads() { return NCELL == 1 ? 64 : 128; }

// waves per SIMD the register allocation aims at
template <int DEG, typename TA, int NCELL>
constexpr int mf_waves() { return NCELL == 1 ? 1 : std::is_same<TA, float>::value ? (DEG == 1 ? 4 : 3) : 2; }

// The product of NCELL cells per workgroup.  Two stages in registers with
// one exchange through LDS between them:
//   columns  a thread owns one component of one cell: its NS node values stay
//            in registers, and a plane of Gauss points at a time it forms X
//            and the three gradients (Line), the divergence with the two
//            other orbital components of its spin row (lane shuffles), the
//            fluxes K1 G_k + K23 [k == own] div, and tests them at once
//            (accumulators in registers).  Only X goes to LDS.
//   points   a thread owns one point: the 18 values of X from LDS, the iterate
//            from memory ([cell][component][point], so that the lanes read
//            consecutive points), H(q) X(q) in registers, back over X in LDS.
// and the columns then test it and write their NS values.  Before, a thread
// per pencil passed every 1D pass through LDS, with nine barriers per cell.
// XCD x works through the cells [x n8, (x+1) n8) in order, so neighbours
// share their nodes' x in that XCD's L2.  Bound by FP64 instructions and load
// latency at 1.75 waves per SIMD: a Q2 cell takes 40.8 k FP64 instructions by
// the algorithm and 42.3 k as counted (residual 33.1 k, 34.5 k), which keep
// the vector unit busy half of the 88 us of 32768 cells; FP32, at 2.5 waves,
// 88% of 52 us.
template <int DEG, typename TH, typename TX, bool RES, int NCELL>
__global__ __launch_bounds__(mf_threads<NCELL>(), (mf_waves<DEG, mf_arith<TH, TX>, NCELL>())) void k_mf_apply(
    MeshDev Mh, Material M0, const TH *__restrict__ Uq, const TX *__restrict__ x, int n_cells, int n8,
    const int *__restrict__ flag, mf_arith<TH, TX> *__restrict__ ycell)
{
  static_assert(!RES || (std::is_same<TH, double>::value && std::is_same<TX, double>::value), "FP64 residual");
  constexpr bool SPLIT = NCELL == 1;  // a thread per column and plane of points
  constexpr int MF_THREADS = mf_threads<NCELL>();
  static_assert(SPLIT || NCELL * 18 <= 126, "a column per lane of two waves");
  using TA = mf_arith<TH, TX>;
  using L = Line<DEG, TA>;
  constexpr int N = DEG + 1, N2 = N * N, NS = N2 * N, V = NS * 18;
  // per cell: fluxes' factors A_k (own gradient) and B_k (divergence), 1/h_k,
  // the bulk coefficients, Robin factor; A, B and the bulk ones with the
  // cell's volume and W0^3
  enum { CA = 0, CB = 3, CI = 6, CM = 9, CR = 16, NCONST = 17 };
  __shared__ __attribute__((aligned(16))) TA sX[NCELL * V];
  __shared__ TA sC[NCELL][NCONST];
  __shared__ int sE[NCELL];
  __shared__ int sNode[NCELL * NS];
  __shared__ uint32_t sMask[NCELL * NS];
  __shared__ TA sD[SPLIT ? 2 * V : 1];
  const int tid = threadIdx.x;
  const int in0 = NCELL * (blockIdx.x >> 3), e0 = (blockIdx.x & 7) * n8 + in0;  // this XCD's range
  const int n_in = min(min(NCELL, n8 - in0), n_cells - e0);                     // may be <= 0
  // the cells' nodes (and their masks) at once; a cell's instance flag beside
  constexpr int NL = (NCELL * NS + MF_THREADS - 1) / MF_THREADS;
  int nd[NL];
#pragma unroll
  for (int r = 0; r < NL; ++r) {
    const int t = tid + r * MF_THREADS;
    nd[r] = 0;
    if (t < n_in * NS) nd[r] = Mh.cell_nodes[(size_t)e0 * NS + t];
  }
  if (tid < NCELL) {
    int e = tid < n_in ? e0 + tid : -1;
    if (e >= 0 && flag && !flag[Mh.cell_inst[e]]) e = -1;  // instance not iterating: its rows are not read
    sE[tid] = e;
  }
  uint32_t mk[NL], mor = 0;
#pragma unroll
  for (int r = 0; r < NL; ++r) {
    const int t = tid + r * MF_THREADS;
    if (t < NCELL * NS) sNode[t] = nd[r];
    if constexpr (!RES) mk[r] = Mh.node_mask[nd[r]];
  }
  __syncthreads();
  bool any = false;
#pragma unroll
  for (int j = 0; j < NCELL; ++j) any = any || sE[j] >= 0;
  if (!any) return;  // uniform: padding, or instances that are not iterating
  // the column of this thread: component c of cell j; three neighbouring
  // lanes hold the orbital components of one spin row (63 = 21 triples per
  // wave; lane 63 repeats its neighbour and writes nothing)
  constexpr int NCOL = SPLIT ? 18 * N : 18 * NCELL;
  const int lane = tid & 63, col0 = 63 * (tid >> 6) + (lane < 63 ? lane : 62);
  const int col = min(col0, NCOL - 1);
  const int pl = SPLIT ? col / 18 : 0;  // SPLIT: the plane of points, and of nodes in the end
  const int j = SPLIT ? 0 : col / 18, c = col % 18, kc = c % 3;
  const int e = sE[j];
  const bool on = lane < 63 && col == col0 && e >= 0;
  TA v[NS];
#pragma unroll
  for (int a = 0; a < NS; ++a) v[a] = (TA)x[(size_t)sNode[j * NS + a] * 18 + c];
  // the cells' constants, while x is on its way
  constexpr int TC = SPLIT ? NCOL : 64;  // threads without a column, or the second wave's first
  if (tid >= TC && tid < TC + NCELL) {
    const int ec = max(sE[tid - TC], 0);
    const Material M = Mh.mats ? Mh.mats[Mh.cell_mat[ec]] : M0;
    double h[3], ih[3];
    for (int k = 0; k < 3; ++k) { h[k] = Mh.cell_h[3 * ec + k]; ih[k] = 1.0 / h[k]; }
    const double vol = h[0] * h[1] * h[2], s = vol * (L::W0 * L::W0 * L::W0);
    TA *C = sC[tid - TC];
    for (int k = 0; k < 3; ++k) {
      C[CA + k] = (TA)(s * M.K1 * ih[k] * ih[k]);
      C[CB + k] = (TA)(s * M.K23 * ih[k]);
      C[CI + k] = (TA)ih[k];
    }
    C[CM + 0] = (TA)(s * M.al);
    C[CM + 1] = (TA)(2.0 * s * M.b1);
    C[CM + 2] = (TA)(2.0 * s * M.b2);
    C[CM + 3] = (TA)(2.0 * s * (M.b3 + M.b4 + M.b5));
    C[CM + 4] = (TA)(2.0 * s * (M.b4 + M.b5 - M.b3));
    C[CM + 5] = (TA)(2.0 * s * (M.b3 + M.b4 - M.b5));
    C[CM + 6] = (TA)(2.0 * s * (M.b3 - M.b4 + M.b5));
    C[CR] = (TA)(M.robin * vol);
  }
  if constexpr (RES) {
    __syncthreads();
  } else {
    // Dirichlet components 0 (the masked columns): few cells have any
#pragma unroll
    for (int r = 0; r < NL; ++r) {
      const int t = tid + r * MF_THREADS;
      if (t < NCELL * NS) {
        sMask[t] = mk[r];
        mor |= mk[r];
      }
    }
    if (__syncthreads_or((int)(mor & 0x3ffffu))) {
#pragma unroll
      for (int a = 0; a < NS; ++a)
        if ((sMask[j * NS + a] >> c) & 1u) v[a] = (TA)0;
    }
  }
  // SPLIT: the point's iterate already now (registers are free there)
  TA s[18];
  const auto load_u = [&](int p, int ep) {
    const int q = p % NS;
    const TH *Up = Uq + (size_t)ep * V + q;
#pragma unroll
    for (int i = 0; i < 18; ++i) s[i] = (TA)Up[i * NS];
  };
  if constexpr (SPLIT && !RES) load_u(min(tid, NS - 1), e);
  const TA *Cj = sC[j];
  // z lines to coefficients: kz[b] of line b = by N + bx
  // acc: coefficients of the z lines of the result (SPLIT: the tested values
  // and z-derivatives of the own plane)
  TA kz[N2][N], acc[N2][SPLIT ? 2 : N];
#pragma unroll
  for (int b = 0; b < N2; ++b) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      kz[b][i] = v[i * N2 + b];
      if (i < (SPLIT ? 2 : N)) acc[b][i] = (TA)0;
    }
    if constexpr (DEG == 2) L::coef(kz[b][0], kz[b][1], kz[b][2]);
  }
  TA *const Xc = sX + j * V + c;
  {
    const TA a0 = Cj[CA], a1 = Cj[CA + 1], a2 = Cj[CA + 2];
    const TA b0 = kc == 0 ? Cj[CB] : (TA)0, b1 = kc == 1 ? Cj[CB + 1] : (TA)0, b2 = kc == 2 ? Cj[CB + 2] : (TA)0;
    const TA m0 = kc == 0 ? Cj[CI] : (TA)0, m1 = kc == 1 ? Cj[CI + 1] : (TA)0, m2 = kc == 2 ? Cj[CI + 2] : (TA)0;
    const int s1 = lane - kc + (kc + 1) % 3, s2 = lane - kc + (kc + 2) % 3;
#pragma unroll 1
    for (int qi = 0; qi < (SPLIT ? 1 : N); ++qi) {
      const int qz = SPLIT ? pl : qi;
      L ln;
      ln.point(qz);
      TA Y0[N][N], Yd[N][N], Y1[N][N];  // [qy][bx]
#pragma unroll
      for (int bx = 0; bx < N; ++bx) {
        TA z0[N], z1[N], p[N], g[N];
#pragma unroll
        for (int by = 0; by < N; ++by) {
          z0[by] = ln.val(kz[by * N + bx]);
          z1[by] = ln.der(kz[by * N + bx]);
        }
        L::both(z0, p, g);
#pragma unroll
        for (int q = 0; q < N; ++q) { Y0[q][bx] = p[q]; Yd[q][bx] = g[q]; }
        L::values(z1, p);
#pragma unroll
        for (int q = 0; q < N; ++q) Y1[q][bx] = p[q];
      }
      TA C0[N][N], C1[N][N], C2[N][N];  // [qy][ax]
#pragma unroll
      for (int qy = 0; qy < N; ++qy) {
        __builtin_amdgcn_sched_barrier(0);  // a row at a time: the rows' temporaries share registers
        TA X[N], g0[N], g1[N], g2[N];
        L::both(Y0[qy], X, g0);
        L::values(Yd[qy], g1);
        L::values(Y1[qy], g2);
#pragma unroll
        for (int qx = 0; qx < N; ++qx) {
          if (on) Xc[((qz * N + qy) * N + qx) * 18] = X[qx];
          const TA own = m0 * g0[qx] + m1 * g1[qx] + m2 * g2[qx];
          const TA div = own + __shfl(own, s1) + __shfl(own, s2);
          g0[qx] = a0 * g0[qx] + b0 * div;
          g1[qx] = a1 * g1[qx] + b1 * div;
          g2[qx] = a2 * g2[qx] + b2 * div;
        }
        L::test_d(g0, C0[qy]);
        L::test_v(g1, C1[qy]);
        L::test_v(g2, C2[qy]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ax = 0; ax < N; ++ax) {
        TA p[N], g[N], d0[N], d2[N];
#pragma unroll
        for (int q = 0; q < N; ++q) { p[q] = C0[q][ax]; g[q] = C1[q][ax]; }
        L::test_vd(p, g, d0);
#pragma unroll
        for (int q = 0; q < N; ++q) p[q] = C2[q][ax];
        L::test_v(p, d2);
#pragma unroll
        for (int ay = 0; ay < N; ++ay) {
          if constexpr (SPLIT) {
            acc[ay * N + ax][0] = d0[ay];
            acc[ay * N + ax][1] = d2[ay];
          } else {
            ln.back(d0[ay], d2[ay], acc[ay * N + ax]);
          }
        }
      }
    }
  }
  __syncthreads();
  // the points: vol w H(q) X(q) (the points' relative weights come with the
  // test passes), or rho(X(q)) for the residual
#pragma unroll 1
  for (int p = tid; p < NCELL * NS; p += MF_THREADS) {
    const int jp = p / NS, ep = sE[jp];
    if (ep < 0) continue;
    const TA *Cp = sC[jp] + CM;
    TA xp[18];
    if constexpr (!SPLIT && !RES) load_u(p, ep);
#pragma unroll
    for (int i = 0; i < 18; ++i) xp[i] = sX[p * 18 + i];
    BulkMat<TA> B;
    TA uu[6], vv[6], uv[9];
    gram(RES ? xp : s, uu, vv, uv);
    B.set(uu, vv, uv, Cp[0], Cp[1], Cp[2], Cp[3], Cp[4], Cp[5], Cp[6]);
    if constexpr (RES) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        TA zu[3] = {0, 0, 0}, zv[3] = {0, 0, 0};
        B.add(xp, xp + 9, k, zu, zv);
#pragma unroll
        for (int m = 0; m < 3; ++m) { sX[p * 18 + 3 * m + k] = zu[m]; sX[p * 18 + 9 + 3 * m + k] = zv[m]; }
      }
    } else {
      BulkMat<TA> D;
      __builtin_amdgcn_sched_barrier(0);
      dgram(s, xp, uu, vv, uv);
      D.set(uu, vv, uv, (TA)0, Cp[1], Cp[2], Cp[3], Cp[4], Cp[5], Cp[6]);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        __builtin_amdgcn_sched_barrier(0);
        TA zu[3] = {0, 0, 0}, zv[3] = {0, 0, 0};
        B.add(xp, xp + 9, k, zu, zv);
        D.add(s, s + 9, k, zu, zv);
#pragma unroll
        for (int m = 0; m < 3; ++m) { sX[p * 18 + 3 * m + k] = zu[m]; sX[p * 18 + 9 + 3 * m + k] = zv[m]; }
      }
    }
  }
  __syncthreads();
  if (!SPLIT && !on) return;
#pragma unroll 1
  for (int qi = 0; qi < (SPLIT ? 1 : N); ++qi) {
    const int qz = SPLIT ? pl : qi;
    L ln;
    ln.point(qz);
    TA C0[N][N];
#pragma unroll
    for (int qy = 0; qy < N; ++qy) {
      TA z[N];
#pragma unroll
      for (int qx = 0; qx < N; ++qx) z[qx] = Xc[((qz * N + qy) * N + qx) * 18];
      L::test_v(z, C0[qy]);
    }
#pragma unroll
    for (int ax = 0; ax < N; ++ax) {
      TA p[N], d[N];
#pragma unroll
      for (int q = 0; q < N; ++q) p[q] = C0[q][ax];
      L::test_v(p, d);
#pragma unroll
      for (int ay = 0; ay < N; ++ay) {
        if constexpr (SPLIT) acc[ay * N + ax][0] += d[ay];
        else ln.back(d[ay], acc[ay * N + ax]);
      }
    }
  }
  // the node values of the column (SPLIT: of its plane pl of nodes, summed
  // over the planes of points through LDS)
  TA out[N2][SPLIT ? 1 : N];
  if constexpr (SPLIT) {
    if (on) {
#pragma unroll
      for (int b = 0; b < N2; ++b) {
        sD[(2 * pl * N2 + b) * 18 + c] = acc[b][0];
        sD[((2 * pl + 1) * N2 + b) * 18 + c] = acc[b][1];
      }
    }
    __syncthreads();
    if (!on) return;
#pragma unroll
    for (int b = 0; b < N2; ++b) out[b][0] = (TA)0;
#pragma unroll
    for (int q = 0; q < N; ++q) {
      TA p[N] = {}, g[N] = {}, one[N], wv, wd;  // weight times value and derivative of L_pl at point q
      p[q] = g[q] = (TA)1;
      L::test_v(p, one);
      wv = pl == 0 ? one[0] : pl == 1 ? one[1] : one[N - 1];
      L::test_d(g, one);
      wd = pl == 0 ? one[0] : pl == 1 ? one[1] : one[N - 1];
#pragma unroll
      for (int b = 0; b < N2; ++b) {
        out[b][0] += wv * sD[(2 * q * N2 + b) * 18 + c];
        out[b][0] += wd * sD[((2 * q + 1) * N2 + b) * 18 + c];
      }
    }
  } else {
#pragma unroll
    for (int b = 0; b < N2; ++b) {
#pragma unroll
      for (int i = 0; i < N; ++i) out[b][i] = acc[b][i];
      if constexpr (DEG == 2) L::uncoef(out[b][0], out[b][1], out[b][2]);
    }
  }
  // Robin faces: robin * area * (1D masses along the face) on the components
  // that the wall does not hold at zero
  const TA rob = Cj[CR];
  if (rob != (TA)0) {
    const uint32_t cface = Mh.cell_face[e];
#pragma unroll
    for (int lf = 0; lf < 6; ++lf) {
      const int bid = (int)((cface >> (3 * lf)) & 7u) - 1;
      if (bid < 2 || bid > 4 || face_zeroed(bid, c)) continue;
      // nodes of the face: f0 + i s0 + k s1 in the lexicographic order
      const int s0 = lf < 2 ? N : 1, s1 = lf < 4 ? N2 : N;
      const int f0 = (lf & 1) ? (N - 1) * (lf < 2 ? 1 : (lf < 4 ? N : N2)) : 0;
      TA t[N][N];
#pragma unroll
      for (int i = 0; i < N; ++i) {
        TA u[N];
#pragma unroll
        for (int k = 0; k < N; ++k) {
          const int a = j * NS + f0 + i * s0 + k * s1;
          u[k] = (TA)x[(size_t)sNode[a] * 18 + c];
          if constexpr (!RES)
            if ((sMask[a] >> c) & 1u) u[k] = (TA)0;
        }
        L::mass(u, t[i]);
      }
      const TA f = rob * Cj[CI + lf / 2] * (TA)(L::M0 * L::M0);
#pragma unroll
      for (int k = 0; k < N; ++k) {
        TA u[N], y[N];
#pragma unroll
        for (int i = 0; i < N; ++i) u[i] = t[i][k];
        L::mass(u, y);
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const int a = f0 + i * s0 + k * s1;
          if constexpr (!SPLIT) out[a % N2][a / N2] += f * y[i];
          else if (a / N2 == pl) out[a % N2][0] += f * y[i];
        }
      }
    }
  }
  TA *const Y = ycell + (size_t)e * V + c;  // Dirichlet rows are replaced in the gather
  if constexpr (SPLIT) {
#pragma unroll
    for (int b = 0; b < N2; ++b) Y[(pl * N2 + b) * 18] = out[b][0];
  } else {
#pragma unroll
    for (int a = 0; a < NS; ++a) Y[a * 18] = out[a % N2][a / N2];
  }
}

// The sums over a node's cell slots of components c and c + 1, in the
// node's cell order: four slot indices, then their four loads in flight.
template <typename TY>
__device__ __forceinline__ void slot_pair_sum(const int *__restrict__ ptr, const int *__restrict__ idx,
                                              const TY *__restrict__ ycell, int node, int c, TY &s0, TY &s1)
{
  using Y2 = typename Vec2<TY>::type;
  const int k1 = ptr[node + 1];
  int k = ptr[node];
  for (; k + 4 <= k1; k += 4) {
    int j[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) j[u] = idx[k + u];
    Y2 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = *reinterpret_cast<const Y2 *>(ycell + (size_t)j[u] * 18 + c);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      s0 += v[u].x;
      s1 += v[u].y;
    }
  }
  for (; k < k1; ++k) {
    const Y2 v = *reinterpret_cast<const Y2 *>(ycell + (size_t)idx[k] * 18 + c);
    s0 += v.x;
    s1 += v.y;
  }
}

// y = sum over the cells of each node of their contributions (fixed cell
// order), and for the Dirichlet rows their diagonal entry (the sum over cells
// of |local diagonal|) times x; with b != null the residual y = b - J x.  One
// thread per node and component pair (c, c + 1): two slot values per load.
// TY, the slot and accumulation type, is that of the product (FP32 for the
// FP32 inner solve).
template <typename TX, typename TY>
__global__ void k_mf_gather(int n_nodes, const int *__restrict__ ptr, const int *__restrict__ idx,
                            const TY *__restrict__ ycell, const uint32_t *__restrict__ mask,
                            const double *__restrict__ Jd, const double *__restrict__ sh, const TX *__restrict__ x,
                            const TX *__restrict__ b, const int *__restrict__ row_seg, const int *__restrict__ flag,
                            TX *__restrict__ y)
{
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long long)n_nodes * 9) return;
  const int node = (int)(i / 9), c = 2 * (int)(i % 9);
  if (flag && !flag[row_seg[node]]) return;  // instance not iterating: its rows are left as they are
  TY s0 = 0, s1 = 0;
  slot_pair_sum(ptr, idx, ycell, node, c, s0, s1);
  const uint32_t mk = mask[node];
  const size_t o = (size_t)node * 18 + c;
  double r0 = ((mk >> c) & 1u) ? Jd[(size_t)node * 324 + c * 19] * (double)x[o] : (double)s0;
  double r1 = ((mk >> (c + 1)) & 1u) ? Jd[(size_t)node * 324 + (c + 1) * 19] * (double)x[o + 1] : (double)s1;
  if (sh) {  // zero on the Dirichlet and hanging rows
    r0 += sh[o] * (double)x[o];
    r1 += sh[o + 1] * (double)x[o + 1];
  }
  y[o] = b ? (TX)((double)b[o] - r0) : (TX)r0;
  y[o + 1] = b ? (TX)((double)b[o + 1] - r1) : (TX)r1;
}

// system_rhs = -R from the residual's cell contributions: each node's sum in
// the fixed cell order, negated; 0 on the Dirichlet components and on the
// rows of a batch instance that is not active (whose cells were skipped).
// Every row is written, so the output needs no fill.  One workgroup per
// reduction chunk (ch: instance, first dof, end dof; even bounds, so a pair
// of components stays in one chunk), which also leaves the chunk's sum of
// squares in partial (unless null): the norm costs no pass of its own over
// rhs (14 us of 107 per residual of the 32^3 Q2 cube, 28 of 182 on 256
// slabs).  8 waves per workgroup: a chunk of 4096 takes 4 rounds of pairs,
// one of 1024 one.
constexpr int GT = 512;
typedef double pair8 __attribute__((ext_vector_type(2), aligned(8)));  // rhs may be the caller's: aligned to a double
__global__ __launch_bounds__(GT) void k_res_gather(const long long *__restrict__ ch, const int *__restrict__ ptr,
                                                   const int *__restrict__ idx, const double *__restrict__ ycell,
                                                   const uint32_t *__restrict__ mask,
                                                   const int *__restrict__ active, double *__restrict__ rhs,
                                                   double *__restrict__ partial)
{
  __shared__ double sh[GT / 64];
  const long long sg = ch[3 * blockIdx.x], beg = ch[3 * blockIdx.x + 1], end = ch[3 * blockIdx.x + 2];
  const bool on = !active || active[sg];
  double acc = 0.0;
  for (long long o = beg + 2 * threadIdx.x; o < end; o += 2 * GT) {
    const int node = (int)(o / 18), c = (int)(o - 18LL * node);
    pair8 r = {0.0, 0.0};
    if (on) {
      double s0 = 0.0, s1 = 0.0;
      slot_pair_sum(ptr, idx, ycell, node, c, s0, s1);
      const uint32_t mk = mask[node];
      r.x = ((mk >> c) & 1u) ? 0.0 : -s0;
      r.y = ((mk >> (c + 1)) & 1u) ? 0.0 : -s1;
    }
    *reinterpret_cast<pair8 *>(rhs + o) = r;
    acc += r.x * r.x;
    acc += r.y * r.y;
  }
  if (!partial) return;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
#pragma unroll
    for (int i = 0; i < GT / 64; ++i) t += sh[i];
    partial[blockIdx.x] = t;
  }
}

template <int DEG>
__global__ __launch_bounds__(NT) void k_energy(RefTables T, MeshDev Mh, Material M0, const double *__restrict__ U,
                                               int n_cells, double *__restrict__ Fcell)
{
  constexpr int N1 = DEG + 1, NS = N1 * N1 * N1, NQ = NS;
  __shared__ double sU[NS * 18];
  __shared__ double sX[NQ * 18];
  __shared__ double sG[NQ * 54];
  __shared__ double sF[NT];
  const int tid = threadIdx.x, e = blockIdx.x;
  if (e >= n_cells) return;
  const Material M = Mh.mats ? Mh.mats[Mh.cell_mat[e]] : M0;
  const int *cn = Mh.cell_nodes + (size_t)e * NS;
  double h[3], ih[3];
  for (int k = 0; k < 3; ++k) { h[k] = Mh.cell_h[3 * e + k]; ih[k] = 1.0 / h[k]; }
  const double vol = h[0] * h[1] * h[2];
  for (int i = tid; i < NS * 18; i += NT) sU[i] = U[(size_t)cn[i / 18] * 18 + (i % 18)];
  __syncthreads();
  for (int i = tid; i < NQ * 18; i += NT) {
    const int q = i / 18, c = i % 18;
    double xv = 0, g0 = 0, g1 = 0, g2 = 0;
    for (int a = 0; a < NS; ++a) {
      const double Ua = sU[a * 18 + c];
      xv += T.N[q * NS + a] * Ua;
      g0 += T.dN[(q * NS + a) * 3 + 0] * Ua;
      g1 += T.dN[(q * NS + a) * 3 + 1] * Ua;
      g2 += T.dN[(q * NS + a) * 3 + 2] * Ua;
    }
    sX[i] = xv;
    sG[q * 54 + c] = g0 * ih[0];
    sG[q * 54 + 18 + c] = g1 * ih[1];
    sG[q * 54 + 36 + c] = g2 * ih[2];
  }
  __syncthreads();
  double acc = 0.0;
  for (int q = tid; q < NQ; q += NT) {
    const double *x = sX + q * 18, *u = x, *v = x + 9, *g = sG + q * 54;
    double uut[9], vvt[9], uvt[9];
    for (int i = 0; i < 3; ++i)
      for (int j = 0; j < 3; ++j) {
        double a1 = 0, a2 = 0, a3 = 0;
        for (int k = 0; k < 3; ++k) {
          a1 += u[3 * i + k] * u[3 * j + k];
          a2 += v[3 * i + k] * v[3 * j + k];
          a3 += u[3 * i + k] * v[3 * j + k];
        }
        uut[3 * i + j] = a1; vvt[3 * i + j] = a2; uvt[3 * i + j] = a3;
      }
    double U2 = 0, V2 = 0, UV = 0;
    for (int a = 0; a < 9; ++a) { U2 += u[a] * u[a]; V2 += v[a] * v[a]; UV += u[a] * v[a]; }
    double trP2 = 0, trQ2 = 0, trS2 = 0, trW2 = 0;
    for (int i = 0; i < 3; ++i)
      for (int j = 0; j < 3; ++j) {
        const double P = uut[3 * i + j] - vvt[3 * i + j], S = uut[3 * i + j] + vvt[3 * i + j];
        const double Q = uvt[3 * i + j] + uvt[3 * j + i];
        const double Wij = uvt[3 * j + i] - uvt[3 * i + j], Wji = uvt[3 * i + j] - uvt[3 * j + i];
        trP2 += P * P; trQ2 += Q * Q; trS2 += S * S; trW2 += Wij * Wji;
      }
    const double D = U2 - V2, N = U2 + V2;
    double f = M.al * N + M.b1 * (D * D + 4 * UV * UV) + M.b2 * N * N + M.b3 * (trP2 + trQ2) +
               M.b4 * (trS2 - trW2) + M.b5 * (trS2 + trW2);
    double g2 = 0;
    for (int i = 0; i < 54; ++i) g2 += g[i] * g[i];
    double dv = 0;
    for (int part = 0; part < 2; ++part)
      for (int m = 0; m < 3; ++m) {
        const double dd = g[9 * part + 3 * m] + g[18 + 9 * part + 3 * m + 1] + g[36 + 9 * part + 3 * m + 2];
        dv += dd * dd;
      }
    f += M.K1 * g2 + M.K23 * dv;
    acc += T.w[q] * vol * f;
  }
  // Robin wall energy: (K1/bt) sum_faces U^T M_f U over unzeroed components
  if (M.robin != 0.0) {
    const uint32_t cface = Mh.cell_face[e];
    for (int lf = 0; lf < 6; ++lf) {
      const int bid = (int)((cface >> (3 * lf)) & 7u) - 1;
      if (bid < 2 || bid > 4) continue;
      for (int i = tid; i < NS * 18; i += NT) {
        const int a = i / 18, c = i % 18;
        if (face_zeroed(bid, c)) continue;
        double s = 0;
        for (int b = 0; b < NS; ++b) s += T.Mf[(lf * NS + a) * NS + b] * sU[b * 18 + c];
        acc += M.robin * face_area(lf, h) * sU[a * 18 + c] * s;
      }
    }
  }
  sF[tid] = acc;
  __syncthreads();
  // fixed-order tree: fold 192 -> 128, then halve
  if (tid < NT - 128) sF[tid] += sF[tid + 128];
  __syncthreads();
  for (int st = 64; st > 0; st >>= 1) {
    if (tid < st) sF[tid] += sF[tid + st];
    __syncthreads();
  }
  if (tid == 0) Fcell[e] = sF[0];
}

}  // namespace

hipError_t launch_assemble(int deg, bool jfp32, const RefTables &T, const MeshDev &M, const Material &mat,
                           const double *U, const int *cells, int n, void *J, bool upper, hipStream_t s)
{
  if (n <= 0) return hipSuccess;
  // a colour of few cells: the pairs of a cell go to several workgroups, which
  // each form H again (Q2 colours of 287 cells: 253 us in one part, 245 in
  // three; Q1 of 64: 15.9 us in four parts, 15.5 in six)
  const int parts = std::max(1, std::min(deg == 1 ? 6 : AsmQ2::NTILE / 3, 1024 / n));
  const dim3 g(n, parts);
  // the hanging-node variant (adaptive meshes) also gathers the constrained diagonals
  const bool hang = M.hdiag != nullptr;
  if (upper && hang) return hipErrorInvalidValue;  // the condensation reads both halves
#define GLH_ASM(K, TJ, HG, UP, B) hipLaunchKernelGGL((K<TJ, HG, UP>), g, dim3(B), 0, s, T, M, mat, U, cells, (TJ *)J)
#define GLH_ASM2(K, B)                                                                                   \
  if (hang) { if (jfp32) GLH_ASM(K, float, true, false, B); else GLH_ASM(K, double, true, false, B); }    \
  else if (upper) { if (jfp32) GLH_ASM(K, float, false, true, B); else GLH_ASM(K, double, false, true, B); } \
  else { if (jfp32) GLH_ASM(K, float, false, false, B); else GLH_ASM(K, double, false, false, B); }
  if (deg == 1) { GLH_ASM2(k_assemble_q1, 192) }
  else { GLH_ASM2(k_assemble_q2, AsmQ2::NTH) }
#undef GLH_ASM2
#undef GLH_ASM
  return hipGetLastError();
}

size_t mf_setup_slots(int deg) { return (size_t)(deg == 1 ? 8 : 27) * NUPAIR; }

hipError_t launch_mf_setup(int deg, bool u32, const RefTables &T, const MeshDev &M, const Material &mat,
                           const double *U, int n_cells, int chunk, const int *node_range, const int *n2c_ptr,
                           const int *n2c_idx, const int *row_seg, double *slots, void *Uq, double *Jd,
                           const MfCondDev &X, hipStream_t s)
{
  if (n_cells <= 0) return hipSuccess;
  if (chunk < 1 || (X.xptr && !M.hdiag)) return hipErrorInvalidValue;  // the constrained setup writes hdiag
  for (int e0 = 0; e0 < n_cells; e0 += chunk) {
    const int n = n_cells - e0 < chunk ? n_cells - e0 : chunk;
    int n0 = INT_MAX, n1 = 0;
    for (int k = e0 / MF_RANGE; k <= (e0 + n - 1) / MF_RANGE; ++k) {
      n0 = std::min(n0, node_range[2 * k]);
      n1 = std::max(n1, node_range[2 * k + 1]);
    }
#define GLH_MFS(D, TH, CON)                                                                                          \
  hipLaunchKernelGGL((k_mf_setup<D, TH, CON>), dim3(n), dim3(NT), 0, s, T, M, mat, U, e0, (TH *)Uq, slots, X);       \
  hipLaunchKernelGGL((k_mf_diag_gather<(D + 1) * (D + 1) * (D + 1), CON>), dim3((n1 - n0 + DG - 1) / DG), dim3(NT),  \
                     0, s, n0, n1, e0, e0 + n, n2c_ptr, n2c_idx, slots, M.node_mask, row_seg, M.inst_active, Jd, M.hdiag)
#define GLH_MFS2(D, TH) \
  if (X.xptr) { GLH_MFS(D, TH, true); } else { GLH_MFS(D, TH, false); }
    if (deg == 1) { if (u32) { GLH_MFS2(1, float) } else { GLH_MFS2(1, double) } }
    else { if (u32) { GLH_MFS2(2, float) } else { GLH_MFS2(2, double) } }
#undef GLH_MFS2
#undef GLH_MFS
  }
  return hipGetLastError();
}

namespace {
// workgroups of nc cells: XCD x (workgroup index mod 8) takes the cells
// [x n8, (x + 1) n8)
inline int mf_range(int n_cells) { return (n_cells + 7) / 8; }
inline int mf_grid(int n_cells, int nc) { return 8 * ((mf_range(n_cells) + nc - 1) / nc); }
// Up to this many cells a thread takes one plane of one column (NCELL = 1):
// its work is a third as long, but it reads and transforms the column once
// per plane.  Measured, us per launch, NCELL 1 against 7: Q2 FP64 product
// 7.6 / 12.4 at 8^3 cells, 10.1 / 13.4 at 10^3, 15.2 / 14.5 at 11^3 (residual
// 11.4 / 12.0), 16.3 / 15.1 at 12^3 (12.8 / 13.6): the line between the last
// two; Q2 FP32 9.4 / 12.8 at 12^3, 12.8 / 14.4 at 14^3, 15.4 / 15.8 at 15^3;
// Q1 FP64 5.3 / 6.1 at 5^3 (residual 4.5 / 5.4), 5.9 / 6.1 at 8^3 (5.0 / 5.2),
// 6.4 / 6.3 at 10^3 (5.6 / 5.6), 8.2 / 6.6 at 12^3 (6.9 / 5.9).
template <int DEG, typename TA>
constexpr int mf_small_mesh() { return DEG == 1 ? 512 : std::is_same<TA, float>::value ? 3072 : 1536; }

template <int DEG, typename TH, typename TX, bool RES>
hipError_t mf_launch(const MeshDev &M, const Material &mat, const void *Uq, const void *x, int n_cells,
                     const int *flag, void *ycell, hipStream_t s)
{
  using TA = mf_arith<TH, TX>;
  if (n_cells <= mf_small_mesh<DEG, TA>())
    hipLaunchKernelGGL((k_mf_apply<DEG, TH, TX, RES, 1>), dim3(mf_grid(n_cells, 1)), dim3(mf_threads<1>()), 0, s, M,
                       mat, (const TH *)Uq, (const TX *)x, n_cells, mf_range(n_cells), flag, (TA *)ycell);
  else
    hipLaunchKernelGGL((k_mf_apply<DEG, TH, TX, RES, MF_CELLS>), dim3(mf_grid(n_cells, MF_CELLS)),
                       dim3(mf_threads<MF_CELLS>()), 0, s, M, mat, (const TH *)Uq, (const TX *)x, n_cells, mf_range(n_cells), flag, (TA *)ycell);
  return hipGetLastError();
}
}  // namespace

hipError_t launch_mf_apply(int deg, bool u32, bool x32, const MeshDev &M, const Material &mat, const void *Uq,
                           const void *x, int n_cells, const int *flag, void *ycell, hipStream_t s)
{
  if (n_cells <= 0) return hipSuccess;
  if (x32 && !u32) return hipErrorInvalidValue;  // an FP64 operator is applied to FP64 vectors only
  if (deg == 1) {
    if (x32) return mf_launch<1, float, float, false>(M, mat, Uq, x, n_cells, flag, ycell, s);
    if (u32) return mf_launch<1, float, double, false>(M, mat, Uq, x, n_cells, flag, ycell, s);
    return mf_launch<1, double, double, false>(M, mat, Uq, x, n_cells, flag, ycell, s);
  }
  if (x32) return mf_launch<2, float, float, false>(M, mat, Uq, x, n_cells, flag, ycell, s);
  if (u32) return mf_launch<2, float, double, false>(M, mat, Uq, x, n_cells, flag, ycell, s);
  return mf_launch<2, double, double, false>(M, mat, Uq, x, n_cells, flag, ycell, s);
}

hipError_t launch_res_apply(int deg, const MeshDev &M, const Material &mat, const double *U, int n_cells,
                            double *ycell, hipStream_t s)
{
  if (n_cells <= 0) return hipSuccess;
  if (deg == 1) return mf_launch<1, double, double, true>(M, mat, nullptr, U, n_cells, M.inst_active, ycell, s);
  return mf_launch<2, double, double, true>(M, mat, nullptr, U, n_cells, M.inst_active, ycell, s);
}

hipError_t launch_res_gather(const SegInfo &S, const int *ptr, const int *idx, const double *ycell,
                             const uint32_t *mask, const int *active, double *rhs, double *partial, hipStream_t s)
{
  if (S.n_chunks <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_res_gather, dim3(S.n_chunks), dim3(GT), 0, s, S.chunks, ptr, idx, ycell, mask, active, rhs,
                     partial);
  return hipGetLastError();
}

template <typename TX>
hipError_t launch_mf_gather(int n_nodes, const int *ptr, const int *idx, const void *ycell, const uint32_t *mask,
                            const double *Jd, const double *sh, const TX *x, const TX *b, const int *row_seg,
                            const int *flag, TX *y, hipStream_t s)
{
  if (n_nodes <= 0) return hipSuccess;
  const long long n = (long long)n_nodes * 9;
  // the slots are FP32 exactly when x is (the product's arithmetic type)
  using TY = typename std::conditional<std::is_same<TX, float>::value, float, double>::type;
  hipLaunchKernelGGL((k_mf_gather<TX, TY>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n_nodes, ptr, idx,
                     (const TY *)ycell, mask, Jd, sh, x, b, row_seg, flag, y);
  return hipGetLastError();
}
template hipError_t launch_mf_gather<double>(int, const int *, const int *, const void *, const uint32_t *,
                                             const double *, const double *, const double *, const double *,
                                             const int *, const int *, double *, hipStream_t);
template hipError_t launch_mf_gather<float>(int, const int *, const int *, const void *, const uint32_t *,
                                            const double *, const double *, const float *, const float *,
                                            const int *, const int *, float *, hipStream_t);

hipError_t launch_energy(int deg, const RefTables &T, const MeshDev &M, const Material &mat, const double *U,
                         int n_cells, double *Fcell, hipStream_t s)
{
  if (n_cells <= 0) return hipSuccess;
  if (deg == 1) hipLaunchKernelGGL(k_energy<1>, dim3(n_cells), dim3(NT), 0, s, T, M, mat, U, n_cells, Fcell);
  else hipLaunchKernelGGL(k_energy<2>, dim3(n_cells), dim3(NT), 0, s, T, M, mat, U, n_cells, Fcell);
  return hipGetLastError();
}

}  // namespace glh
