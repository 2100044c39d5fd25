// C ABI of the MI355X Ginzburg-Landau Newton-step library: context, per-cycle
// upload, assembly, GMRES + point-block Jacobi, damped Newton line search and
// free energy.  Host orchestration of the HIP kernels in gl_assemble.hip and
// gl_linalg.hip.  See include/glhip.h for the reference methods each entry
// point replaces.
//
// Every context solves a batch of independent instances (a single mesh is a
// batch of one).  Instances own disjoint node/cell ranges of one concatenated
// mesh, so assembly, SpMV and the block-Jacobi preconditioner run unchanged on
// the block-diagonal system; dot products, Gram-Schmidt coefficients, Givens
// rotations, convergence tests and the Newton line search are per instance.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "glhip.h"
#include "glhip_dev.hpp"
#include "amr.hpp"
#include "handles.hpp"
#include "mesh.hpp"

using glh::NC;


namespace {

// device buffer owned by a context (or a scope); freed with it
template <typename T>
struct DBuf {
  T *p = nullptr;
  size_t n = 0;
  DBuf() = default;
  DBuf(const DBuf &) = delete;
  DBuf &operator=(const DBuf &) = delete;
  ~DBuf() { release(); }
  hipError_t alloc(size_t count)
  {
    if (count <= n && p) return hipSuccess;
    release();
    hipError_t e = hipMalloc((void **)&p, std::max<size_t>(count, 1) * sizeof(T));
    if (e != hipSuccess) {
      (void)hipGetLastError();  // reported here: the next launch would find it again
      p = nullptr;
      return e;
    }
    n = count;
    return hipSuccess;
  }
  void release()
  {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
};

// pinned host staging for the small per-instance arrays exchanged every
// GMRES iteration
template <typename T>
struct HBuf {
  T *p = nullptr;
  size_t n = 0;
  HBuf() = default;
  HBuf(const HBuf &) = delete;
  HBuf &operator=(const HBuf &) = delete;
  ~HBuf() { release(); }
  hipError_t alloc(size_t count)
  {
    if (count <= n && p) return hipSuccess;
    release();
    hipError_t e = hipHostMalloc((void **)&p, std::max<size_t>(count, 1) * sizeof(T), hipHostMallocDefault);
    if (e != hipSuccess) {
      (void)hipGetLastError();  // reported here: the next launch would find it again
      p = nullptr;
      return e;
    }
    n = count;
    return hipSuccess;
  }
  void release()
  {
    if (p) (void)hipHostFree(p);
    p = nullptr;
    n = 0;
  }
};

// dofs per reduction chunk (one workgroup each): 1024, or 4096 for instances
// of 2^20 dofs and more, where fewer and longer workgroups still fill the
// device (3% less GMRES time on the 4.9 M-dof Q2 cube)
constexpr long long CHUNK = 1024, CHUNK_LARGE = 4096, LARGE_INSTANCE = 1 << 20;
// the Gram-Schmidt kernels read value pairs: chunk bounds must stay even
static_assert(CHUNK % 2 == 0 && CHUNK_LARGE % 2 == 0 && NC % 2 == 0, "reduction chunks must have even bounds");
static_assert(CHUNK <= glh::GS_MAX_CHUNK && CHUNK_LARGE <= glh::GS_MAX_CHUNK, "chunks the segmented kernels accept");

}  // namespace

struct glh_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  bool have_mat = false, have_mesh = false;
  glh::Material mat{};
  std::vector<glh::Material> mats_host;  // per instance when set by glh_set_materials
  // mesh
  int deg = 1, ns = 8, nq = 8, npair = 36;
  int n_cells = 0, n_nodes = 0, nnzb = 0;
  std::vector<int> color_ptr;
  std::vector<int> node_off, cell_off;  // instance ranges
  int n_seg = 1, n_chunks = 0;
  int max_seg_chunks = 0;  // reduction chunks of the largest instance
  int chunk_len = (int)glh::GS_MAX_CHUNK;  // the longest chunk
  // reference tables
  DBuf<double> tN, tdN, tw, tWp, tSp, tMf, tAt;
  DBuf<int> tpa, tpb;
  // mesh arrays
  DBuf<int> cell_nodes, row_ptr, col, diag, cell_blk, color_cells, cell_mat, seg_chunk;
  // hanging-node constraints: the cell loop assembles Jf (nnzb_a blocks over
  // the unconstrained cell pattern) and rf, which are then condensed into the
  // system matrix J and rhs
  bool constrained = false;
  int nnzb_a = 0, n_hang = 0;
  // upper-triangle products of the assembled Jacobian: 1 usable, -1 not,
  // 0 not looked at on this mesh
  int sym_state = 0;
  bool j_upper = false;  // the assembled values stop at the diagonal
  DBuf<int> sym_lo;
  DBuf<double> sym_T;
  glh::ConstraintDev cons;
  DBuf<int> c_gptr, c_gsrc, c_brow, c_rptr, c_rsrc, c_hnode, c_hptr, c_hm;
  DBuf<double> c_gw, c_rw, c_hw, hdiag, rfull;
  DBuf<unsigned char> c_gfl, c_rfl;
  DBuf<double> Jf64;
  DBuf<float> Jf32;
  DBuf<long long> chunks;
  DBuf<glh::Material> mats;
  DBuf<double> cell_h;
  DBuf<uint32_t> cell_face, node_mask;
  // state vectors (FP64)
  DBuf<double> U, U0, dU, X, rhs, res, Fcell;
  // per-instance small device arrays
  DBuf<double> s_norm, s_alpha, s_part;
  DBuf<int> s_flag;
  // Jacobian and preconditioner
  DBuf<double> J64, D64;
  DBuf<float> J32, D32;
  bool j_fp32 = false, j_valid = false, d_valid = false;
  // matrix-free Jacobian (glh_set_matrix_free): per cell the iterate at the
  // quadrature points, and the diagonal blocks, in place of the BSR values
  bool matfree = false, j_mf = false;
  DBuf<double> Uq64, Jd64;
  DBuf<float> Uq32;  // the stored iterate of an FP32 matrix-free Jacobian
  DBuf<int> diag_id;  // node -> its block in Jd64 (the identity, hanging nodes aside)
  DBuf<int> n2c_ptr, n2c_idx;  // node -> its (cell * ns + local node) entries
  DBuf<double> mf_ycell;       // per-cell contributions of a product [n_cells][ns][18] (FP32 in an FP32 product)
  // constrained meshes: the lists of glh::MfCondDev (raw local blocks folded
  // into the masters' diagonal blocks), node -> hanging index, and the C x and
  // J C x of a product
  DBuf<int> mfx_ptr, mfx_pair, mft_node, mft_ptr, mft_slot, mft_A, mft_B, c_hidx;
  DBuf<double> mfx_LB, mft_w, mf_xf, mf_yf, mf_diag;
  std::vector<int> mf_range;  // nodes of every MF_RANGE cells (first, one past the last)
  DBuf<unsigned char> mft_fl;
  glh::MfCondDev mfc;
  size_t mfx_slots = 0;
  // continuation shift of a matrix-free Jacobian (sigma |diag| per value),
  // used by the product while mf_sh_on
  DBuf<double> mf_sh;
  bool mf_sh_on = false;
  DBuf<int> status;
  // GMRES workspace
  DBuf<double> gV64, gZ64, gW64, gh64, gp64, gy64, gs64, gq64, gn64;
  DBuf<float> gV32, gZ32, gW32, gh32, gp32, gy32, gs32, gq32, gb32, gx32, gn32;
  HBuf<double> pin64, pinv;
  // device-side GMRES control (per instance)
  DBuf<double> gmH, gmcs, gmsn, gmg, gmbeta, gmtarget;
  DBuf<int> gmcyc, gmconv, gmjseg, gmits, gmro, gmfrozen, gmjlast, row_seg;
  // active set of a batched GMRES cycle (instances still iterating)
  DBuf<int> d_node_off, act_counts, act_seg, act_rpref, act_chunk;
  // one restart cycle as graphs: head (true residual, start of cycle), body
  // blocks of Arnoldi steps, tail (update of x), a single instance's second
  // Gram-Schmidt passes
  struct Graph {
    std::vector<hipGraphExec_t> exec;  // head; tail and blocks of each grid size; second passes
    std::vector<const void *> key;
    int q = 1;
  } graph64, graph32;
  HBuf<float> pin32;
  HBuf<int> pin_st;  // status of each step of a single instance's cycle, written by the device
  hipEvent_t ev_step[2] = {nullptr, nullptr};  // the two last steps enqueued
  HBuf<int> pin_i, pin_fl;  // pinned staging of the per-instance flags and counters
  DBuf<double> ir_r;
  // per-instance results of the last Newton solve: 8 values per instance
  std::vector<double> inst_stats;
  // timing
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  double asm_ms = 0.0, asm_launches = 0;
  // live kernel timing (glh_set_timing): event pairs around each SpMV launch
  // on the context stream, read back when the pool fills or a solve ends
  bool timing = false;
  int verbose = 0;
  double ptc_sigma0 = 0.0;  // pseudo-transient continuation in glh_newton_solve (0: off)
  bool ew_forcing = false;  // Eisenstat-Walker forcing terms in glh_newton_solve
  // schedule of the batched GMRES (set by glh_autotune or glh_set_schedule):
  // Arnoldi steps per replayed block, grid caps of the active-set launches,
  // restart used when glh_newton_solve is called with restart <= 0
  int q_block = 0, row_cap = 0, chunk_cap = 0, tuned_restart = 100;
  int gs_tile = 8;  // Gram-Schmidt tile (glh::SegInfo::gs)
  // The second classical Gram-Schmidt pass runs for a column whose norm falls
  // below 10% of its norm before the projection (||w'||^2 < 0.01 ||w||^2),
  // that is, when cancellation has cost about a digit.  Measured on the 32^3
  // Q2 cube and the 256-slab batch (FP64 and FP32): the iteration counts and
  // free energies are those of the classic 1/sqrt(2) threshold, which
  // re-projected nearly every column and cost 6% of the solve
  // (glh_set_reorth sets another ratio).
  double dgks = 0.01;
  const int *asm_active = nullptr;  // device flags: assemble only these instances (inside glh_newton_solve)
  DBuf<int> asm_flag;
  std::vector<double> r_ref;  // per-instance stopping reference (empty: ||R0|| of the solve)
  long reorth_count = 0;
  double *scratch = nullptr;  // device address of the library's scratch array on this device
  std::vector<hipEvent_t> ev_pool;
  int ev_used = 0;
  double spmv_ms_total = 0.0, spmv_count = 0;
  double jasm_ms_total = 0.0, jasm_count = 0, rasm_ms_total = 0.0, rasm_count = 0;

  glh::RefTables tables() const
  {
    return glh::RefTables{tN.p, tdN.p, tw.p, tWp.p, tSp.p, tMf.p, tpa.p, tpb.p, tAt.p};
  }
  glh::MeshDev meshdev() const
  {
    const bool per = !mats_host.empty();
    return glh::MeshDev{per ? cell_mat.p : nullptr, per ? mats.p : nullptr, cell_nodes.p, cell_h.p,
                        cell_face.p,          node_mask.p,                  cell_blk.p,
                        constrained ? hdiag.p : nullptr, cell_mat.p, asm_active};
  }
  glh::SegInfo seg() const
  {
    glh::SegInfo S{chunks.p, seg_chunk.p, n_chunks, n_seg};
    S.gs = gs_tile;
    S.len = chunk_len;
    return S;
  }
};

namespace {

int fail(glh_ctx *c, int code, const std::string &msg)
{
  if (c) c->err = msg;
  return code;
}

// Captured GMRES graphs hold kernel arguments by value: the buffers, and the
// material (K1, K2 + K3 and the Robin coefficient of the matrix-free product)
// together with the device pointer of the per-instance materials.  Whatever
// changes those must drop the graphs; the next solve records them again.
void drop_graphs(glh_ctx *c)
{
  for (auto *g : {&c->graph64, &c->graph32}) {
    for (auto e : g->exec)
      if (e) (void)hipGraphExecDestroy(e);
    g->exec.clear();
    g->key.clear();
  }
}

#define HIPCHK(ctx, ...)                                                                         \
  do {                                                                                           \
    hipError_t e_ = (__VA_ARGS__);                                                               \
    if (e_ != hipSuccess)                                                                        \
      return fail((ctx), GLH_ERR_HIP, std::string(#__VA_ARGS__) + ": " + hipGetErrorString(e_)); \
  } while (0)

#define RCHK(expr)       \
  do {                   \
    int rc_ = (expr);    \
    if (rc_) return rc_; \
  } while (0)

// Device memory that the context holds only to be faster: the upper-triangle
// products' map and scratch (the whole matrix serves as well, its blocks below
// the diagonal filled in) and the matrix-free setup's shares (taken again at
// the next setup).  Returns whether there was any to give back.
bool give_back(glh_ctx *c)
{
  if (!c->mf_diag.p && !c->sym_T.p && !c->sym_lo.p) return false;
  if (c->sym_state == 1) {
    hipError_t e = hipSuccess;
    if (c->j_valid && !c->j_mf && c->j_upper && c->j_fp32)
      e = glh::launch_sym_fill<float>(c->n_nodes, c->row_ptr.p, c->diag.p, c->sym_lo.p, c->J32.p, c->stream);
    else if (c->j_valid && !c->j_mf && c->j_upper)
      e = glh::launch_sym_fill<double>(c->n_nodes, c->row_ptr.p, c->diag.p, c->sym_lo.p, c->J64.p, c->stream);
    if (e != hipSuccess) return false;
    c->j_upper = false;
    c->sym_state = -1;
  }
  if (hipStreamSynchronize(c->stream) != hipSuccess) return false;
  drop_graphs(c);  // the recorded products read the scratch
  c->mf_diag.release();
  c->sym_T.release();
  c->sym_lo.release();
  return true;
}

// n values of device memory for b, which may be had by giving those back: what
// fits the card without them does not fail for them
template <typename T>
hipError_t take(glh_ctx *c, DBuf<T> &b, size_t n)
{
  hipError_t e = b.alloc(n);
  if (e == hipErrorOutOfMemory && give_back(c)) e = b.alloc(n);
  return e;
}

template <typename T>
hipError_t upload(glh_ctx *c, DBuf<T> &b, const T *src, size_t n, hipStream_t s)
{
  hipError_t e = take(c, b, n);
  if (e != hipSuccess) return e;
  if (n == 0) return hipSuccess;
  return hipMemcpyAsync(b.p, src, n * sizeof(T), hipMemcpyHostToDevice, s);
}

double now_s()
{
  return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

// 1D Gauss points on [0,1] and Lagrange basis on equispaced support points
void gauss01(int n, double *x, double *w)
{
  if (n == 2) {
    const double d = 0.5 / std::sqrt(3.0);
    x[0] = 0.5 - d; x[1] = 0.5 + d; w[0] = w[1] = 0.5;
  } else {
    const double d = 0.5 * std::sqrt(0.6);
    x[0] = 0.5 - d; x[1] = 0.5; x[2] = 0.5 + d;
    w[0] = w[2] = 5.0 / 18.0; w[1] = 8.0 / 18.0;
  }
}
void lagrange(int deg, double x, double *L, double *dL)
{
  if (deg == 1) {
    L[0] = 1 - x; L[1] = x; dL[0] = -1; dL[1] = 1;
  } else {
    L[0] = 2 * (x - 0.5) * (x - 1); L[1] = -4 * x * (x - 1); L[2] = 2 * x * (x - 0.5);
    dL[0] = 4 * x - 3; dL[1] = 4 - 8 * x; dL[2] = 4 * x - 1;
  }
}

int build_tables(glh_ctx *c, int deg)
{
  const int n1 = deg + 1, ns = n1 * n1 * n1, nq = ns, npair = ns * (ns + 1) / 2;
  c->deg = 0;  // of no degree until all of them are there
  double gx[3], gw[3], L[3][3], dL[3][3];
  gauss01(n1, gx, gw);
  for (int i = 0; i < n1; ++i) lagrange(deg, gx[i], L[i], dL[i]);
  std::vector<double> N(nq * ns), dN(nq * ns * 3), w(nq);
  for (int q = 0; q < nq; ++q) {
    const int qx = q % n1, qy = (q / n1) % n1, qz = q / (n1 * n1);
    w[q] = gw[qx] * gw[qy] * gw[qz];
    for (int a = 0; a < ns; ++a) {
      const int ax = a % n1, ay = (a / n1) % n1, az = a / (n1 * n1);
      N[q * ns + a] = L[qx][ax] * L[qy][ay] * L[qz][az];
      dN[(q * ns + a) * 3 + 0] = dL[qx][ax] * L[qy][ay] * L[qz][az];
      dN[(q * ns + a) * 3 + 1] = L[qx][ax] * dL[qy][ay] * L[qz][az];
      dN[(q * ns + a) * 3 + 2] = L[qx][ax] * L[qy][ay] * dL[qz][az];
    }
  }
  std::vector<double> Wp((size_t)npair * nq), Sp((size_t)npair * 9);
  std::vector<int> pa(npair), pb(npair);
  int p = 0;
  for (int a = 0; a < ns; ++a)
    for (int b = a; b < ns; ++b, ++p) {
      pa[p] = a; pb[p] = b;
      for (int q = 0; q < nq; ++q) Wp[(size_t)p * nq + q] = w[q] * N[q * ns + a] * N[q * ns + b];
      for (int k = 0; k < 3; ++k)
        for (int l = 0; l < 3; ++l) {
          double s = 0;
          for (int q = 0; q < nq; ++q) s += w[q] * dN[(q * ns + a) * 3 + k] * dN[(q * ns + b) * 3 + l];
          Sp[(size_t)p * 9 + k * 3 + l] = s;
        }
    }
  // face mass on each unit face: QGauss<2>(k+1) (assemble.cc:124)
  std::vector<double> Mf((size_t)6 * ns * ns, 0.0);
  for (int f = 0; f < 6; ++f) {
    const int dn = f / 2;
    int t0 = (dn + 1) % 3, t1 = (dn + 2) % 3;
    if (t0 > t1) std::swap(t0, t1);
    for (int i0 = 0; i0 < n1; ++i0)
      for (int i1 = 0; i1 < n1; ++i1) {
        double xi[3];
        xi[dn] = (f & 1) ? 1.0 : 0.0;
        xi[t0] = gx[i0];
        xi[t1] = gx[i1];
        const double wf = gw[i0] * gw[i1];
        double Lx[3][3], dLx[3][3];
        for (int k = 0; k < 3; ++k) lagrange(deg, xi[k], Lx[k], dLx[k]);
        std::vector<double> Ns(ns);
        for (int a = 0; a < ns; ++a) Ns[a] = Lx[0][a % n1] * Lx[1][(a / n1) % n1] * Lx[2][a / (n1 * n1)];
        for (int a = 0; a < ns; ++a)
          for (int b = 0; b < ns; ++b) Mf[((size_t)f * ns + a) * ns + b] += wf * Ns[a] * Ns[b];
      }
  }
  hipStream_t s = c->stream;
  HIPCHK(c, upload(c, c->tN, N.data(), N.size(), s));
  HIPCHK(c, upload(c, c->tdN, dN.data(), dN.size(), s));
  HIPCHK(c, upload(c, c->tw, w.data(), w.size(), s));
  HIPCHK(c, upload(c, c->tWp, Wp.data(), Wp.size(), s));
  HIPCHK(c, upload(c, c->tSp, Sp.data(), Sp.size(), s));
  HIPCHK(c, upload(c, c->tMf, Mf.data(), Mf.size(), s));
  HIPCHK(c, upload(c, c->tpa, pa.data(), pa.size(), s));
  HIPCHK(c, upload(c, c->tpb, pb.data(), pb.size(), s));
  // the pair tables as matrix-core operands: row tile t, k step s, lane l hold
  // pair 16 t + l % 16 and k = 4 s + l / 16 (points, derivative pairs, faces)
  // (Q2; the Q1 assembly reads the pair tables themselves)
  const int nt = deg == 2 ? (npair + 15) / 16 : 0, kt = (nq + 15 + 3) / 4;
  std::vector<double> At((size_t)nt * kt * 64, 0.0);
  for (int t = 0; t < nt; ++t)
    for (int k4 = 0; k4 < kt; ++k4)
      for (int l = 0; l < 64; ++l) {
        const int pr = 16 * t + l % 16, k = 4 * k4 + l / 16;
        if (pr >= npair) continue;
        double v = 0.0;
        if (k < nq) v = Wp[(size_t)pr * nq + k];
        else if (k < nq + 9) v = Sp[(size_t)pr * 9 + k - nq];
        else if (k < nq + 15) v = Mf[((size_t)(k - nq - 9) * ns + pa[pr]) * ns + pb[pr]];
        At[((size_t)t * kt + k4) * 64 + l] = v;
      }
  HIPCHK(c, upload(c, c->tAt, At.data(), At.size(), s));
  HIPCHK(c, hipStreamSynchronize(s));
  c->deg = deg; c->ns = ns; c->nq = nq; c->npair = npair;
  return GLH_OK;
}

int check_ready(glh_ctx *c, bool need_mat = true)
{
  if (!c) return GLH_ERR_ARG;
  if (!c->have_mesh) return fail(c, GLH_ERR_STATE, "no mesh uploaded");
  if (need_mat && !c->have_mat) return fail(c, GLH_ERR_STATE, "material not set");
  if (need_mat && !c->mats_host.empty() && (int)c->mats_host.size() != c->n_seg)
    return fail(c, GLH_ERR_STATE, "per-instance materials do not match the uploaded batch");
  HIPCHK(c, hipSetDevice(c->device));
  return GLH_OK;
}

size_t ndofs(const glh_ctx *c) { return (size_t)c->n_nodes * NC; }
// values between two vectors of the Krylov basis: every vector starts at 16 bytes
size_t basis_stride(const glh_ctx *c) { return (ndofs(c) + 3) / 4 * 4; }

// per-instance ||v_s||^2 of an FP64 device vector into out (host, n_seg values)
int seg_norm2(glh_ctx *c, const double *v, std::vector<double> &out)
{
  const size_t n = ndofs(c);
  HIPCHK(c, take(c, c->s_part, (size_t)std::max(1, c->n_chunks)));
  HIPCHK(c, take(c, c->s_norm, c->n_seg));
  HIPCHK(c, c->pinv.alloc(c->n_seg));
  HIPCHK(c, glh::launch_seg_mdot<double>(c->seg(), 1, v, n, v, c->s_part.p, c->s_norm.p, 1, 0, false, c->stream));
  HIPCHK(c, hipMemcpyAsync(c->pinv.p, c->s_norm.p, c->n_seg * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  out.assign(c->pinv.p, c->pinv.p + c->n_seg);
  return GLH_OK;
}

int norm64(glh_ctx *c, const double *v, double *out)
{
  std::vector<double> s;
  RCHK(seg_norm2(c, v, s));
  double t = 0;
  for (double x : s) t += x;
  *out = std::sqrt(t);
  return GLH_OK;
}

// system_rhs = -R at U into out, condensed on a constrained mesh: the cell
// loop of compute_residual (residual.cc:164-289) in the cell slots, summed
// per node in a fixed order (no colours, no fill: every row is written).
// With norm2 (device, n_seg values) also ||R_s||^2, through the chunk
// partials part.
int residual_cells(glh_ctx *c, const double *U, double *out, double *part = nullptr, double *norm2 = nullptr)
{
  const glh::MeshDev M = c->meshdev();
  const glh::SegInfo S = c->seg();
  hipStream_t s = c->stream;
  HIPCHK(c, glh::launch_res_apply(c->deg, M, c->mat, U, c->n_cells, c->mf_ycell.p, s));
  HIPCHK(c, glh::launch_res_gather(S, c->n2c_ptr.p, c->n2c_idx.p, c->mf_ycell.p, c->node_mask.p, M.inst_active,
                                   c->constrained ? c->rfull.p : out, c->constrained ? nullptr : part, s));
  if (c->constrained) {
    HIPCHK(c, glh::launch_condense_rhs(c->cons, c->rfull.p, out, s));
    if (norm2) HIPCHK(c, glh::launch_seg_mdot<double>(S, 1, out, ndofs(c), out, part, norm2, 1, 0, false, s));
  } else if (norm2) {
    HIPCHK(c, glh::launch_seg_final(S, part, norm2, s));
  }
  return GLH_OK;
}

// -R at U into out and its per-instance ||R_s||^2 on the host
int residual_norms(glh_ctx *c, const double *U, double *out, std::vector<double> &n2)
{
  HIPCHK(c, take(c, c->s_part, (size_t)std::max(1, c->n_chunks)));
  HIPCHK(c, take(c, c->s_norm, c->n_seg));
  HIPCHK(c, c->pinv.alloc(c->n_seg));
  if (c->timing) HIPCHK(c, hipEventRecord(c->ev0, c->stream));
  RCHK(residual_cells(c, U, out, c->s_part.p, c->s_norm.p));
  if (c->timing) HIPCHK(c, hipEventRecord(c->ev1, c->stream));
  HIPCHK(c, hipMemcpyAsync(c->pinv.p, c->s_norm.p, c->n_seg * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  n2.assign(c->pinv.p, c->pinv.p + c->n_seg);
  if (c->timing) {
    float ms = 0;
    HIPCHK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->asm_ms = ms;
    c->asm_launches = 2;
    c->rasm_ms_total += ms;
    c->rasm_count += 1;
  }
  return GLH_OK;
}

// From this many blocks of the assembled matrix on the products read its upper
// triangle (launch_spmv_sym).  A second launch costs 3 us: 1000 blocks 8.1 us
// against 5.5 whole; 4913 (rows of up to 125) 23 against 43, 6859 9.1 against
// 10.7.
constexpr int SYM_MIN_BLOCKS = 4096;

// the upper-triangle product's map and scratch, once per mesh, at its first
// assembly (without constraint lines only the blocks it reads are assembled);
// without the memory for them, here or for what is taken later (give_back), or
// on a pattern that is not symmetric, the products read the whole matrix
int ensure_sym(glh_ctx *c)
{
  if (c->sym_state || c->nnzb < SYM_MIN_BLOCKS) return GLH_OK;
  HIPCHK(c, take(c, c->status, 1));  // (may give back what the scratch held on the last mesh)
  c->sym_state = -1;
  if (c->sym_lo.alloc(c->nnzb) != hipSuccess || c->sym_T.alloc((size_t)c->nnzb * NC) != hipSuccess) {
    c->sym_lo.release();
    c->sym_T.release();
    return GLH_OK;
  }
  HIPCHK(c, glh::launch_fill<int>(1, 0, c->status.p, c->stream));
  HIPCHK(c, glh::launch_sym_map(c->n_nodes, c->row_ptr.p, c->col.p, c->sym_lo.p, c->status.p, c->stream));
  int bad = 0;
  HIPCHK(c, hipMemcpyAsync(&bad, c->status.p, sizeof(int), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->sym_state = bad ? -1 : 1;
  return GLH_OK;
}
// values of the cells' diagonal-block shares held at a time (128 MB)
constexpr size_t MF_SETUP_VALUES = (size_t)16 << 20;

// assemble (J and/or -R) at state Ustate into (J, rhs_out)
int assemble_at(glh_ctx *c, const double *Ustate, bool do_j, bool do_r, bool fp32, double *rhs_out, bool timed,
                bool mf = false)
{
  void *J = nullptr;
  int mf_chunk = 0;
  if (do_j && mf) {  // matrix-free: H at the quadrature points and the diagonal blocks
    const size_t un = (size_t)c->n_cells * c->nq * NC;
    if (fp32) HIPCHK(c, take(c, c->Uq32, un));
    else HIPCHK(c, take(c, c->Uq64, un));
    HIPCHK(c, take(c, c->mf_ycell, (size_t)c->n_cells * c->ns * NC));
    // one block per node, and on a constrained mesh one more per hanging node
    // (its condensed row for the point-block Jacobi, diag_id points there)
    HIPCHK(c, take(c, c->Jd64, ((size_t)c->n_nodes + (c->constrained ? c->n_hang : 0)) * 324));
    if (c->constrained) {
      HIPCHK(c, take(c, c->mfx_LB, c->mfx_slots * 324));
      c->mfc.LB = c->mfx_LB.p;
      HIPCHK(c, take(c, c->mf_xf, ndofs(c)));
      HIPCHK(c, take(c, c->mf_yf, ndofs(c)));
    }
    c->mf_sh_on = false;
    // the cells' shares of the diagonal blocks, a chunk of cells at a time:
    // large enough to fill the device, small enough to stay in the caches;
    // smaller chunks where the memory is not to be had
    const size_t per = glh::mf_setup_slots(c->deg);
    const int most = std::max(1, (int)(MF_SETUP_VALUES / per)), parts = (c->n_cells + most - 1) / most;
    mf_chunk = (c->n_cells + parts - 1) / parts;
    hipError_t e = take(c, c->mf_diag, (size_t)mf_chunk * per);
    while (e == hipErrorOutOfMemory && mf_chunk > 1) {
      mf_chunk = (mf_chunk + 1) / 2;
      e = c->mf_diag.alloc((size_t)mf_chunk * per);
    }
    HIPCHK(c, e);
  } else if (do_j) {
    const size_t nv = (size_t)c->nnzb * 324;
    if (fp32) { HIPCHK(c, take(c, c->J32, nv)); J = c->J32.p; }
    else { HIPCHK(c, take(c, c->J64, nv)); J = c->J64.p; }
  }
  // with hanging nodes the cell loop writes Jf, condensed afterwards
  void *Jcell = J;
  if (c->constrained) {
    if (do_j && !mf) {
      const size_t nv = (size_t)c->nnzb_a * 324;
      if (fp32) { HIPCHK(c, take(c, c->Jf32, nv)); Jcell = c->Jf32.p; }
      else { HIPCHK(c, take(c, c->Jf64, nv)); Jcell = c->Jf64.p; }
    }
    if (do_j) HIPCHK(c, glh::launch_fill<double>(ndofs(c), 0.0, c->hdiag.p, c->stream));
  }
  if (do_j && !mf) RCHK(ensure_sym(c));  // after the matrix, which comes first where the memory is short
  const glh::RefTables T = c->tables();
  const glh::MeshDev M = c->meshdev();
  timed = timed || c->timing;
  if (timed) HIPCHK(c, hipEventRecord(c->ev0, c->stream));
  int launches = 0;
  const bool upper = c->sym_state == 1 && !c->constrained;
  if (do_j && mf) {
    HIPCHK(c, glh::launch_mf_setup(c->deg, fp32, T, M, c->mat, Ustate, c->n_cells, mf_chunk, c->mf_range.data(),
                                   c->n2c_ptr.p, c->n2c_idx.p, c->row_seg.p, c->mf_diag.p,
                                   fp32 ? (void *)c->Uq32.p : (void *)c->Uq64.p, c->Jd64.p,
                                   c->constrained ? c->mfc : glh::MfCondDev{}, c->stream));
    launches = 2 * ((c->n_cells + mf_chunk - 1) / mf_chunk);
  } else if (do_j) {
    launches = (int)c->color_ptr.size() - 1;
    c->j_upper = upper;
    for (int k = 0; k < launches; ++k) {
      const int off = c->color_ptr[k], n = c->color_ptr[k + 1] - off;
      HIPCHK(c, glh::launch_assemble(c->deg, fp32, T, M, c->mat, Ustate, c->color_cells.p + off, n, Jcell, upper,
                                     c->stream));
    }
  }
  if (c->constrained) {
    if (do_j && mf) HIPCHK(c, glh::launch_mf_cond_diag(c->cons, c->mfc, c->n_nodes, c->hdiag.p, c->Jd64.p, c->stream));
    else if (do_j) {
      if (fp32) HIPCHK(c, glh::launch_condense<float>(c->cons, c->Jf32.p, c->J32.p, c->hdiag.p, c->stream));
      else HIPCHK(c, glh::launch_condense<double>(c->cons, c->Jf64.p, c->J64.p, c->hdiag.p, c->stream));
    }
  }
  if (do_r) RCHK(residual_cells(c, Ustate, rhs_out));
  if (timed) {
    HIPCHK(c, hipEventRecord(c->ev1, c->stream));
    HIPCHK(c, hipEventSynchronize(c->ev1));
    float ms = 0;
    HIPCHK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->asm_ms = ms;
    c->asm_launches = launches + (do_r ? 2 : 0);
    if (c->timing) {
      if (do_j) { c->jasm_ms_total += ms; c->jasm_count += 1; }
      else { c->rasm_ms_total += ms; c->rasm_count += 1; }
    }
  }
  if (do_j) {
    c->j_fp32 = fp32;
    c->j_mf = mf;
    c->j_valid = true;
    c->d_valid = false;
  }
  return GLH_OK;
}

// constraints distribute: Dirichlet components to 0, hanging values from
// their masters (AffineConstraints::distribute)
int distribute(glh_ctx *c, double *v)
{
  HIPCHK(c, glh::launch_mask_zero(c->n_nodes, c->node_mask.p, v, c->stream));
  if (c->constrained) HIPCHK(c, glh::launch_distribute(c->cons, v, c->stream));
  return GLH_OK;
}

int ensure_precond(glh_ctx *c)
{
  if (c->d_valid) return GLH_OK;
  HIPCHK(c, take(c, c->status, 1));
  HIPCHK(c, hipMemsetAsync(c->status.p, 0, sizeof(int), c->stream));
  const size_t nv = (size_t)c->n_nodes * 171;  // the inverses' upper triangles
  if (c->j_fp32 && c->j_mf) {  // FP64 inverses of the FP64 diagonal blocks, rounded to FP32
    HIPCHK(c, take(c, c->D64, nv));
    HIPCHK(c, take(c, c->D32, nv));
    HIPCHK(c, glh::launch_bj_invert<double>(c->n_nodes, c->diag_id.p, c->Jd64.p, c->D64.p, c->status.p, c->stream));
    HIPCHK(c, (glh::launch_convert<double, float>(nv, c->D64.p, c->D32.p, c->stream)));
  } else if (c->j_fp32) {
    HIPCHK(c, take(c, c->D32, nv));
    HIPCHK(c, glh::launch_bj_invert<float>(c->n_nodes, c->diag.p, c->J32.p, c->D32.p, c->status.p, c->stream));
  } else {
    HIPCHK(c, take(c, c->D64, nv));
    if (c->j_mf)
      HIPCHK(c, glh::launch_bj_invert<double>(c->n_nodes, c->diag_id.p, c->Jd64.p, c->D64.p, c->status.p, c->stream));
    else
      HIPCHK(c, glh::launch_bj_invert<double>(c->n_nodes, c->diag.p, c->J64.p, c->D64.p, c->status.p, c->stream));
  }
  int st = 0;
  HIPCHK(c, hipMemcpyAsync(&st, c->status.p, sizeof(int), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  if (st) return fail(c, GLH_ERR_SINGULAR, "singular 18x18 diagonal block in point-block Jacobi");
  c->d_valid = true;
  return GLH_OK;
}

template <typename TV>
struct Work;
template <>
struct Work<double> {
  static DBuf<double> &V(glh_ctx *c) { return c->gV64; }
  static DBuf<double> &Z(glh_ctx *c) { return c->gZ64; }
  static DBuf<double> &W(glh_ctx *c) { return c->gW64; }
  static DBuf<double> &h(glh_ctx *c) { return c->gh64; }
  static DBuf<double> &hp(glh_ctx *c) { return c->gq64; }
  static DBuf<double> &part(glh_ctx *c) { return c->gp64; }
  static DBuf<double> &npart(glh_ctx *c) { return c->gn64; }
  static DBuf<double> &y(glh_ctx *c) { return c->gy64; }
  static DBuf<double> &sc(glh_ctx *c) { return c->gs64; }
  static HBuf<double> &pin(glh_ctx *c) { return c->pin64; }
  static glh_ctx::Graph &graph(glh_ctx *c) { return c->graph64; }
};
template <>
struct Work<float> {
  static DBuf<float> &V(glh_ctx *c) { return c->gV32; }
  static DBuf<float> &Z(glh_ctx *c) { return c->gZ32; }
  static DBuf<float> &W(glh_ctx *c) { return c->gW32; }
  static DBuf<float> &h(glh_ctx *c) { return c->gh32; }
  static DBuf<float> &hp(glh_ctx *c) { return c->gq32; }
  static DBuf<float> &part(glh_ctx *c) { return c->gp32; }
  static DBuf<float> &npart(glh_ctx *c) { return c->gn32; }
  static DBuf<float> &y(glh_ctx *c) { return c->gy32; }
  static DBuf<float> &sc(glh_ctx *c) { return c->gs32; }
  static HBuf<float> &pin(glh_ctx *c) { return c->pin32; }
  static glh_ctx::Graph &graph(glh_ctx *c) { return c->graph32; }
};

int flush_events(glh_ctx *c)
{
  if (c->ev_used == 0) return GLH_OK;
  HIPCHK(c, hipEventSynchronize(c->ev_pool[2 * c->ev_used - 1]));
  for (int i = 0; i < c->ev_used; ++i) {
    float ms = 0;
    HIPCHK(c, hipEventElapsedTime(&ms, c->ev_pool[2 * i], c->ev_pool[2 * i + 1]));
    c->spmv_ms_total += ms;
    c->spmv_count += 1;
  }
  c->ev_used = 0;
  return GLH_OK;
}

// y = J x (b == null) or y = b - J x with the matrix-free Jacobian: every cell
// at once into its own slot, then a fixed-order gather per node (no colours:
// one launch, no read-modify-write of y).  The stored iterate is FP32 for an
// FP32 Jacobian, whatever the vector type.
template <typename TV>
int mf_product(glh_ctx *c, const TV *x, const TV *b, TV *y, const int *flag = nullptr)
{
  const glh::MeshDev M = c->meshdev();
  const bool u32 = c->j_fp32, x32 = std::is_same<TV, float>::value;
  const double *sh = c->mf_sh_on ? c->mf_sh.p : nullptr;
  // constrained meshes: y = C^T Jf (C x), hanging rows hdiag x
  const bool con = c->constrained;
  TV *xf = con ? reinterpret_cast<TV *>(c->mf_xf.p) : nullptr, *yf = con ? reinterpret_cast<TV *>(c->mf_yf.p) : y;
  const TV *xin = con ? xf : x;
  if (con) HIPCHK(c, glh::launch_mf_distribute<TV>(c->cons, c->n_nodes, x, xf, c->row_seg.p, flag, c->stream));
  HIPCHK(c, glh::launch_mf_apply(c->deg, u32, x32, M, c->mat, u32 ? (const void *)c->Uq32.p : (const void *)c->Uq64.p,
                                 xin, c->n_cells, flag, c->mf_ycell.p, c->stream));
  HIPCHK(c, glh::launch_mf_gather<TV>(c->n_nodes, c->n2c_ptr.p, c->n2c_idx.p, c->mf_ycell.p, c->node_mask.p,
                                      c->Jd64.p, sh, xin, con ? nullptr : b, c->row_seg.p, flag, yf, c->stream));
  if (con)
    HIPCHK(c, glh::launch_mf_condense<TV>(c->cons, c->n_nodes, c->hdiag.p, yf, x, b, y, c->row_seg.p, flag,
                                          c->stream));
  return GLH_OK;
}

template <typename TJ, typename TV>
int apply_j(glh_ctx *c, const TJ *J, const TV *x, TV *y, const int *flag, glh::ActiveSet act)
{
  if (c->j_mf) {  // every cell of the iterating instances (flag); act only narrows the SpMV's grid
    static_assert(std::is_same<TJ, TV>::value, "the matrix-free product keeps x and y in one type");
    RCHK(mf_product<TV>(c, x, nullptr, y, flag));
    return GLH_OK;
  }
  if (c->sym_state == 1)
    HIPCHK(c, (glh::launch_spmv_sym<TJ, TV>(c->n_nodes, c->row_ptr.p, c->diag.p, c->col.p, c->sym_lo.p, J, x, nullptr,
                                            y, c->sym_T.p, c->stream, c->row_seg.p, flag, act)));
  else
    HIPCHK(c, glh::launch_spmv<TJ, TV>(c->n_nodes, c->row_ptr.p, c->col.p, J, x, y, c->stream, c->row_seg.p, flag,
                                       act));
  return GLH_OK;
}

template <typename TJ, typename TV>
int spmv(glh_ctx *c, const TJ *J, const TV *x, TV *y, const int *flag = nullptr, glh::ActiveSet act = {})
{
  const bool t = c->timing && !c->ev_pool.empty();
  if (t) {
    if (2 * c->ev_used >= (int)c->ev_pool.size()) RCHK(flush_events(c));
    HIPCHK(c, hipEventRecord(c->ev_pool[2 * c->ev_used], c->stream));
  }
  RCHK((apply_j<TJ, TV>(c, J, x, y, flag, act)));
  if (t) {
    HIPCHK(c, hipEventRecord(c->ev_pool[2 * c->ev_used + 1], c->stream));
    ++c->ev_used;
  }
  return GLH_OK;
}

// batches whose instances have at most this many reduction chunks let each
// Gram-Schmidt update workgroup sum its instance's multi-dot partials
constexpr int FOLD_MAX_CHUNKS = 64;

// Right-preconditioned restarted GMRES(m) with 18x18 point-block Jacobi and
// classical Gram-Schmidt with selective (DGKS) reorthogonalisation, batched
// over the instances of the context: every instance has its own Krylov
// coefficients, Givens rotations and stopping test
// ||b_s - J x_s|| <= rtol[s] ||b_s||.  The Hessenberg updates, rotations and
// tests run on the device (k_gmres_ctl), and every kernel skips the instances
// that have stopped, so the host needs no values of a step: a batch's cycle is
// enqueued in blocks of steps, between which the host only asks whether any
// instance still iterates; a single instance goes step by step, its status
// read after each and the next one already enqueued.  The pieces are captured
// in HIP graphs and replayed (or launched directly when kernel timing is on).
// its_out: lockstep iterations; its_seg: iterations each instance used.
template <typename TJ, typename TV>
int enqueue_cycle(glh_ctx *c, const TJ *J, const TJ *Dinv, const TV *b, TV *x, int m, const glh::GmresCtl<TV> &C,
                  bool timed, int part, int j0 = 0, int j1 = 0, int shift = 0)
{
  const size_t n = ndofs(c), ldv = basis_stride(c);
  const int ldh = m + 2;
  const glh::SegInfo SI = c->seg();
  hipStream_t s = c->stream;
  auto &V = Work<TV>::V(c);
  auto &Z = Work<TV>::Z(c);
  auto &W = Work<TV>::W(c);
  auto &pt = Work<TV>::part(c);
  TV *nrm2 = const_cast<TV *>(C.nrm2);
  TV *hs = const_cast<TV *>(C.hs), *hq = const_cast<TV *>(C.hq);
  const int *rs = c->row_seg.p, *cyc = C.cyc, *ro = C.ro;
  // batches: the body and tail visit only the instances that iterate in this
  // cycle (active set built at the end of the head)
  const bool use_act = c->n_seg > 1;
  glh::ActiveSet act{};
  if (use_act)
    act = glh::ActiveSet{c->act_counts.p, c->act_seg.p, c->act_rpref.p, c->act_chunk.p, c->d_node_off.p, shift,
                         c->row_cap, c->chunk_cap};
  glh::SegInfo SA = SI;
  SA.act = act;
  // the second Gram-Schmidt pass rarely runs (its flag is usually off): a
  // capped grid keeps the skipped multi-dot launch cheap
  glh::SegInfo SR = SA;
  SR.cap = 256;
  const bool fold = c->n_seg > 1 && c->max_seg_chunks <= FOLD_MAX_CHUNKS;
  TV *np = Work<TV>::npart(c).p;  // the norm partials beside the multi-dot partials (fold)
  auto mv = [&](const TV *in, TV *out, const int *flag, glh::ActiveSet a) -> int {
    if (timed) return spmv<TJ, TV>(c, J, in, out, flag, a);
    (void)rs;
    return apply_j<TJ, TV>(c, J, in, out, flag, a);
  };
  if (part == 0) {  // head: V0 = b - J x, beta_s, cycle flags
    RCHK(mv(x, W.p, nullptr, glh::ActiveSet{}));
    HIPCHK(c, glh::launch_seg_residual<TV>(SI, b, W.p, V.p, pt.p, nrm2, s));
    HIPCHK(c, glh::launch_gmres_ctl<TV>(C, 0, 0, s));
    if (use_act)
      HIPCHK(c, glh::launch_build_active(SI, cyc, c->d_node_off.p, c->act_counts.p, c->act_seg.p, c->act_rpref.p,
                                         c->act_chunk.p, s));
    return GLH_OK;
  }
  if (part == 2) {  // tail: x += M^-1 V y
    HIPCHK(c, glh::launch_gmres_ctl<TV>(C, 3, 0, s));
    HIPCHK(c, glh::launch_seg_lincomb<TV>(SA, m, V.p, ldv, C.y, ldh, W.p, s, C.jseg));
    HIPCHK(c, (glh::launch_bj_apply<TJ, TV>(c->n_nodes, Dinv, W.p, Z.p, s, rs, nullptr, act)));
    if (use_act) HIPCHK(c, glh::launch_seg_add<TV>(SA, Z.p, x, s));
    else HIPCHK(c, (glh::launch_axpy<TV, TV>(n, 1.0, Z.p, x, s)));
    return GLH_OK;
  }
  if (c->n_seg == 1) {
    // one step (part 1), or the second Gram-Schmidt pass of step j0 (part 3),
    // which a column rarely needs: the host enqueues it when the step's
    // status asks for it.  The updates of a small instance sum the multi-dot
    // partials themselves.
    const int j = j0;
    TV *wv = V.p + ldv * (j + 1);
    int *st = c->pin_st.p + j;
    const bool small = c->n_chunks <= FOLD_MAX_CHUNKS;
    if (part == 3) {
      HIPCHK(c, glh::launch_seg_mdot<TV>(SI, j + 1, V.p, ldv, wv, pt.p, hq, ldh, 0, false, s, ro, !small));
      HIPCHK(c, glh::launch_seg_sub_lincomb_norm<TV>(SI, j + 1, V.p, ldv, hq, ldh, wv, np, nrm2, 1, 0, s, ro, nullptr,
                                                     0, j, small ? pt.p : nullptr, small ? j + 1 : 0, false));
      HIPCHK(c, (glh::launch_step_end<TJ, TV>(SI, np, nrm2, C, j, c->n_nodes, Dinv, wv, Z.p, true, st, s)));
      return GLH_OK;
    }
    // Z = D^-1 V_j: of the cycle's first vector here, of the others by the
    // end of the step that normalises them
    if (j == 0) {
      HIPCHK(c, glh::launch_seg_scale<TV>(SI, V.p, nrm2, 1, V.p, s, cyc, true));
      HIPCHK(c, (glh::launch_bj_apply<TJ, TV>(c->n_nodes, Dinv, V.p, Z.p, s, rs, cyc, act)));
    }
    RCHK(mv(Z.p, wv, cyc, act));
    HIPCHK(c, glh::launch_seg_mdot<TV>(SI, j + 2, V.p, ldv, wv, pt.p, hs, ldh, 0, false, s, cyc, !small));
    HIPCHK(c, glh::launch_seg_sub_lincomb_norm<TV>(SI, j + 1, V.p, ldv, hs, ldh, wv, np, nrm2, 1, 0, s, cyc, nullptr,
                                                   0, j, small ? pt.p : nullptr, small ? j + 2 : 0, false));
    HIPCHK(c, (glh::launch_step_end<TJ, TV>(SI, np, nrm2, C, j, c->n_nodes, Dinv, wv, Z.p, false, st, s)));
    return GLH_OK;
  }
  // body block: Arnoldi steps j0 <= j < j1
  if (j0 == 0) HIPCHK(c, glh::launch_seg_scale<TV>(SA, V.p, nrm2, 1, V.p, s, cyc, true));
  for (int j = j0; j < j1; ++j) {
    TV *vj = V.p + ldv * j, *wv = V.p + ldv * (j + 1);
    HIPCHK(c, (glh::launch_bj_apply<TJ, TV>(c->n_nodes, Dinv, vj, Z.p, s, rs, cyc, act)));
    RCHK(mv(Z.p, wv, cyc, act));
    // each pass's norm reduction runs the control op of its instance
    // (op 1: second-pass flag; op 2: Givens update and stopping test), so an
    // instance that stops here keeps V_{j+1} unnormalised: it is not used
    // (batches of small instances: each update workgroup sums its instance's
    // multi-dot partials itself, instead of a reduction launch per pass)
    if (fold) {
      HIPCHK(c, glh::launch_seg_mdot<TV>(SA, j + 2, V.p, ldv, wv, pt.p, hs, ldh, 0, false, s, cyc, false));
      HIPCHK(c, glh::launch_seg_sub_lincomb_norm<TV>(SA, j + 1, V.p, ldv, hs, ldh, wv, np, nrm2, 1, 0, s, cyc, nullptr,
                                                     0, j, pt.p, j + 2, false));
      // op 1 (the second pass's flag) formed by the second pass's multi-dot
      // workgroups from the first pass's norm partials: no launch of its own
      glh::Op1In<TV> o1;
      o1.npart = np;
      o1.norm2 = nrm2;
      o1.seg_chunk = SR.seg_chunk;
      o1.C = C;
      o1.j = j;
      HIPCHK(c, glh::launch_seg_mdot<TV>(SR, j + 1, V.p, ldv, wv, pt.p, hq, ldh, 0, false, s, ro, false, o1));
      HIPCHK(c, glh::launch_seg_sub_lincomb_norm<TV>(SA, j + 1, V.p, ldv, hq, ldh, wv, np, nrm2, 1, 0, s, ro, nullptr, 0,
                                                     j, pt.p, j + 1, false));
      // the pass's norm reduction, op 2 and the normalisation in one launch
      HIPCHK(c, glh::launch_seg_ctl2_scale<TV>(SA, np, nrm2, C, j, wv, s));
    } else {
      HIPCHK(c, glh::launch_seg_mdot<TV>(SA, j + 2, V.p, ldv, wv, pt.p, hs, ldh, 0, false, s, cyc));
      HIPCHK(c, glh::launch_seg_sub_lincomb_norm<TV>(SA, j + 1, V.p, ldv, hs, ldh, wv, pt.p, nrm2, 1, 0, s, cyc, &C, 1, j));
      HIPCHK(c, glh::launch_seg_mdot<TV>(SR, j + 1, V.p, ldv, wv, pt.p, hq, ldh, 0, false, s, ro));
      HIPCHK(c, glh::launch_seg_sub_lincomb_norm<TV>(SA, j + 1, V.p, ldv, hq, ldh, wv, pt.p, nrm2, 1, 0, s, ro, nullptr,
                                                     0, j, nullptr, 0, false));
      // as above: the pass's norm reduction (its partials where it ran), op 2
      // and the normalisation in one launch
      HIPCHK(c, glh::launch_seg_ctl2_scale<TV>(SA, pt.p, nrm2, C, j, wv, s));
    }
  }
  return GLH_OK;
}

template <typename TJ, typename TV>
int gmres(glh_ctx *c, const TJ *J, const TJ *Dinv, const TV *b, TV *x, const std::vector<double> &rtol, int maxit,
          int m, int *its_out, std::vector<double> &rel_out, std::vector<int> &its_seg)
{
  if (m > 126) m = 126;
  const size_t n = ndofs(c);
  const int S = c->n_seg, ldh = m + 2;
  const glh::SegInfo SI = c->seg();
  hipStream_t s = c->stream;
  auto &V = Work<TV>::V(c);
  auto &Z = Work<TV>::Z(c);
  auto &W = Work<TV>::W(c);
  auto &hs = Work<TV>::h(c);
  auto &hq = Work<TV>::hp(c);
  auto &pt = Work<TV>::part(c);
  auto &yb = Work<TV>::y(c);
  auto &sc = Work<TV>::sc(c);
  HIPCHK(c, take(c, V, basis_stride(c) * (m + 1)));
  HIPCHK(c, take(c, Z, n));
  HIPCHK(c, take(c, W, n));
  HIPCHK(c, take(c, hs, (size_t)S * ldh));
  HIPCHK(c, take(c, hq, (size_t)S * ldh));
  HIPCHK(c, take(c, yb, (size_t)S * ldh));
  HIPCHK(c, take(c, sc, (size_t)S * 2));
  HIPCHK(c, take(c, pt, (size_t)std::max(1, c->n_chunks) * (m + 2)));
  HIPCHK(c, take(c, Work<TV>::npart(c), (size_t)std::max(1, c->n_chunks)));
  HIPCHK(c, take(c, c->gmH, (size_t)S * (m + 1) * m));
  HIPCHK(c, take(c, c->gmcs, (size_t)S * m));
  HIPCHK(c, take(c, c->gmsn, (size_t)S * m));
  HIPCHK(c, take(c, c->gmg, (size_t)S * (m + 1)));
  HIPCHK(c, take(c, c->gmbeta, S));
  HIPCHK(c, take(c, c->gmtarget, S));
  DBuf<int> *ib[] = {&c->gmcyc, &c->gmconv, &c->gmjseg, &c->gmits, &c->gmro, &c->gmfrozen, &c->gmjlast};
  for (auto *q : ib) HIPCHK(c, take(c, *q, S));
  HIPCHK(c, c->pinv.alloc((size_t)4 * S));
  HIPCHK(c, take(c, c->act_counts, 4));
  // every host <-> device copy of the loop below goes through pinned memory
  HIPCHK(c, c->pin_i.alloc(2 * (size_t)S + 4));
  HIPCHK(c, c->pin_st.alloc(128));
  HIPCHK(c, Work<TV>::pin(c).alloc(S));
  HIPCHK(c, take(c, c->act_seg, S));
  HIPCHK(c, take(c, c->act_rpref, S + 1));
  HIPCHK(c, take(c, c->act_chunk, std::max(1, c->n_chunks)));
  glh::GmresCtl<TV> C{S,        m,          ldh,        hs.p,         hq.p,         sc.p,        yb.p,
                      c->gmH.p, c->gmcs.p,  c->gmsn.p,  c->gmg.p,     c->gmbeta.p,  c->gmtarget.p, c->gmcyc.p,
                      c->gmconv.p, c->gmjseg.p, c->gmits.p, c->gmro.p, c->gmfrozen.p, c->gmjlast.p,
                      c->dgks};
  // ||b_s|| and the absolute targets
  HIPCHK(c, glh::launch_seg_mdot<TV>(SI, 1, b, n, b, pt.p, sc.p, 1, 0, false, s));
  TV *bn2 = Work<TV>::pin(c).p;
  HIPCHK(c, hipMemcpyAsync(bn2, sc.p, S * sizeof(TV), hipMemcpyDeviceToHost, s));
  HIPCHK(c, hipStreamSynchronize(s));
  std::vector<double> bn(S);
  for (int i = 0; i < S; ++i) {
    bn[i] = std::sqrt(std::max(0.0, (double)bn2[i]));
    c->pinv.p[i] = rtol[i] * bn[i];
  }
  HIPCHK(c, hipMemcpyAsync(c->gmtarget.p, c->pinv.p, S * sizeof(double), hipMemcpyHostToDevice, s));
  HIPCHK(c, glh::launch_fill<int>(S, 0, c->gmits.p, s));
  HIPCHK(c, glh::launch_fill<int>(S, 0, c->gmjseg.p, s));
  HIPCHK(c, glh::launch_fill<int>(S, 0, c->gmfrozen.p, s));
  HIPCHK(c, glh::launch_fill<TV>(n, (TV)0, x, s));
  HIPCHK(c, hipStreamSynchronize(s));
  // Graphs of one restart cycle, rebuilt whenever their buffers change.  The
  // Arnoldi steps go in blocks of q; the host checks between blocks whether
  // any instance still iterates, so at most q - 1 steps of a cycle run as
  // skipped launches.  A single instance (q = 1) runs one skipped step where
  // a cycle stops before its last column, and one at each second pass: the
  // step enqueued ahead.  Batches record
  // the body and tail at three grid sizes (shift 0, 3, 6) and replay the
  // one that fits the number of rows still iterating, so that a few
  // straggling instances do not pay for the workgroups of the full batch.
  const bool timed = c->timing && !c->ev_pool.empty();
  const int q = S == 1 ? 1 : std::min(m, c->q_block > 0 ? c->q_block : 8);
  const int nblk = (m + q - 1) / q;
  constexpr int NLEV = 3;
  auto &gc = Work<TV>::graph(c);
  // The buffers and sizes the captured launches use and the product they run,
  // beside what an upload sets (it drops the graphs).
  const std::vector<const void *> key = {J,           Dinv,          b,           x,            V.p,
                                         Z.p,         W.p,           pt.p,        hs.p,         hq.p, Work<TV>::npart(c).p,
                                         yb.p,        sc.p,          c->gmH.p,    c->gmcs.p,    c->gmsn.p,
                                         c->gmg.p,    c->gmbeta.p,   c->gmtarget.p, c->gmcyc.p, c->gmconv.p,
                                         c->gmjseg.p, c->gmits.p,    c->gmro.p,   c->gmfrozen.p, c->gmjlast.p,
                                         c->row_seg.p, c->d_node_off.p, c->act_counts.p, c->act_seg.p,
                                         c->act_rpref.p, c->act_chunk.p, c->chunks.p, c->seg_chunk.p,
                                         c->row_ptr.p, c->col.p, c->diag.p, c->sym_lo.p, c->sym_T.p,
                                         (const void *)(size_t)(c->sym_state == 1), c->pin_st.p,
                                         c->Uq64.p, c->Uq32.p, c->Jd64.p,
                                         c->mf_xf.p, c->mf_yf.p, c->mf_sh_on ? c->mf_sh.p : nullptr,
                                         (const void *)(size_t)c->j_mf,
                                         (const void *)(size_t)m, (const void *)(size_t)S,
                                         (const void *)(size_t)c->n_chunks, (const void *)(size_t)c->n_nodes,
                                         (const void *)(size_t)q, (const void *)(size_t)c->row_cap,
                                         (const void *)(size_t)c->chunk_cap};
  if (!timed && gc.key != key) {
    for (auto e : gc.exec)
      if (e) (void)hipGraphExecDestroy(e);
    gc.exec.assign(1 + NLEV * (1 + nblk) + nblk, nullptr);
    gc.key = key;
    gc.q = q;
  }
  // graph slot: 0 head; per level L: tail, then the body blocks; then the
  // second passes of a single instance's steps
  auto slot = [&](int part, int lev, int blk) {
    return part == 0 ? 0 : part == 3 ? 1 + NLEV * (1 + nblk) + blk : 1 + lev * (1 + nblk) + (part == 2 ? 0 : 1 + blk);
  };
  auto launch = [&](int part, int lev, int blk) -> int {
    const int j0 = blk * q, j1 = std::min(m, j0 + q), shift = 3 * lev;
    if (timed) return enqueue_cycle<TJ, TV>(c, J, Dinv, b, x, m, C, true, part, j0, j1, shift);
    hipGraphExec_t &ge = gc.exec[slot(part, lev, blk)];
    if (!ge) {
      hipGraph_t graph = nullptr;
      HIPCHK(c, hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
      const int rc = enqueue_cycle<TJ, TV>(c, J, Dinv, b, x, m, C, false, part, j0, j1, shift);
      hipError_t e = hipStreamEndCapture(s, &graph);
      if (rc) {
        if (graph) (void)hipGraphDestroy(graph);
        return rc;
      }
      HIPCHK(c, e);
      e = hipGraphInstantiate(&ge, graph, nullptr, nullptr, 0);
      (void)hipGraphDestroy(graph);
      HIPCHK(c, e);
    }
    HIPCHK(c, hipGraphLaunch(ge, s));
    return GLH_OK;
  };
  // cycle loop
  int it = 0;
  bool conv = false;
  int *hconv = c->pin_i.p, *hj = hconv + S, *hcnt = hj + S;
  while (true) {
    RCHK(launch(0, 0, 0));
    HIPCHK(c, hipMemcpyAsync(hconv, c->gmconv.p, S * sizeof(int), hipMemcpyDeviceToHost, s));
    HIPCHK(c, hipMemcpyAsync(hj, c->gmjlast.p, S * sizeof(int), hipMemcpyDeviceToHost, s));
    if (S > 1) HIPCHK(c, hipMemcpyAsync(hcnt, c->act_counts.p, 3 * sizeof(int), hipMemcpyDeviceToHost, s));
    HIPCHK(c, hipStreamSynchronize(s));
    bool all = true;
    int jmax = 0;
    for (int i = 0; i < S; ++i) {
      all = all && hconv[i];
      jmax = std::max(jmax, hj[i]);
    }
    it += jmax;
    if (all) {
      conv = true;
      break;
    }
    if (it >= maxit) break;
    int lev = 0;
    if (S > 1) {
      const double f = (double)hcnt[2] / std::max(1, c->n_nodes);
      lev = f > 1.0 / 8 ? 0 : f > 1.0 / 64 ? 1 : 2;
    }
    if (S == 1) {
      // A step ahead: while step j runs, step j + 1 is enqueued (it skips
      // itself if j turns out to be the last, or to need its second pass), so
      // the device does not wait for the host to read j's status.  With
      // kernel timing on, each step is waited for, so that no skipped product
      // is counted.
      for (auto &e : c->ev_step)
        if (!e) HIPCHK(c, hipEventCreateWithFlags(&e, hipEventDisableTiming));
      volatile int *st = c->pin_st.p;
      auto step = [&](int j) -> int {
        RCHK(launch(1, lev, j));
        HIPCHK(c, hipEventRecord(c->ev_step[j & 1], s));
        return GLH_OK;
      };
      RCHK(step(0));
      for (int j = 0; j < nblk; ++j) {
        const bool ahead = !timed && j + 1 < nblk;
        if (ahead) RCHK(step(j + 1));
        HIPCHK(c, hipEventSynchronize(c->ev_step[j & 1]));
        int v = st[j];
        if (v == 2) {
          RCHK(launch(3, lev, j));
          HIPCHK(c, hipStreamSynchronize(s));
          v = st[j];
          if (v == 1 && ahead) RCHK(step(j + 1));  // the one enqueued before has skipped itself
        }
        if (v != 1) break;
        if (!ahead && j + 1 < nblk) RCHK(step(j + 1));
      }
      RCHK(launch(2, lev, 0));
      continue;
    }
    for (int blk = 0; blk < nblk; ++blk) {
      RCHK(launch(1, lev, blk));
      if (blk + 1 == nblk) break;
      HIPCHK(c, hipMemcpyAsync(hconv, c->gmcyc.p, S * sizeof(int), hipMemcpyDeviceToHost, s));
      HIPCHK(c, hipStreamSynchronize(s));
      bool any = false;
      for (int i = 0; i < S && !any; ++i) any = hconv[i] != 0;
      if (!any) break;
    }
    RCHK(launch(2, lev, 0));
  }
  RCHK(flush_events(c));
  // the last head computed the true residual norms of the final iterate
  HIPCHK(c, hipMemcpyAsync(c->pinv.p, c->gmbeta.p, S * sizeof(double), hipMemcpyDeviceToHost, s));
  HIPCHK(c, hipMemcpyAsync(hconv, c->gmits.p, S * sizeof(int), hipMemcpyDeviceToHost, s));
  HIPCHK(c, hipStreamSynchronize(s));
  *its_out = it;
  its_seg.assign(hconv, hconv + S);
  rel_out.assign(S, 0.0);
  for (int i = 0; i < S; ++i) {
    const double r = c->pinv.p[i];
    rel_out[i] = bn[i] > 0 ? r / bn[i] : 0.0;
    if (!std::isfinite(rel_out[i]) || !std::isfinite(bn[i]))
      return fail(c, GLH_ERR_NOCONV, "GMRES: non-finite residual in instance " + std::to_string(i));
  }
  return conv ? GLH_OK : fail(c, GLH_ERR_NOCONV, "GMRES reached the maximum iteration number");
}

// J dU = rhs per instance to ||r_s|| <= rtol ||rhs_s||.  stats: [0] lockstep
// iterations, [1] worst relative residual.
int solve_impl(glh_ctx *c, const std::vector<double> &rtolv, int maxit, int restart, double stats[2],
               std::vector<int> *its_seg_out)
{
  if (!c->j_valid) return fail(c, GLH_ERR_STATE, "no Jacobian assembled");
  if (restart < 1 || maxit < 1 || (int)rtolv.size() != c->n_seg) return fail(c, GLH_ERR_ARG, "bad solver parameters");
  for (double r : rtolv)
    if (!(r > 0)) return fail(c, GLH_ERR_ARG, "bad solver parameters");
  RCHK(ensure_precond(c));
  const size_t n = ndofs(c);
  const int S = c->n_seg;
  hipStream_t s = c->stream;
  int its = 0, rc = GLH_OK;
  std::vector<double> rel;
  std::vector<int> its_seg(S, 0);
  if (!c->j_fp32) {
    rc = gmres<double, double>(c, c->J64.p, c->D64.p, c->rhs.p, c->dU.p, rtolv, maxit, restart, &its, rel, its_seg);
  } else {
    // FP32 GMRES inside FP64 iterative refinement, per instance:
    //   r = rhs - J32 dU (FP64 arithmetic), solve J32 c = r in FP32, dU += c
    HIPCHK(c, take(c, c->gb32, n));
    HIPCHK(c, take(c, c->gx32, n));
    HIPCHK(c, take(c, c->ir_r, n));
    HIPCHK(c, take(c, c->s_flag, S));
    HIPCHK(c, hipMemsetAsync(c->dU.p, 0, n * sizeof(double), s));
    std::vector<double> bn2, rn2;
    RCHK(seg_norm2(c, c->rhs.p, bn2));
    HIPCHK(c, hipMemcpyAsync(c->ir_r.p, c->rhs.p, n * sizeof(double), hipMemcpyDeviceToDevice, s));
    rn2 = bn2;
    std::vector<int> flag(S);
    for (int sweep = 0; sweep < 20 && its < maxit; ++sweep) {
      bool any = false;
      std::vector<double> rt(S, 1.0);
      for (int i = 0; i < S; ++i) {
        const double bn = std::sqrt(bn2[i]), rn = std::sqrt(rn2[i]);
        const double inner = std::max(rtolv[i], 1e-4);
        flag[i] = rn > rtolv[i] * bn;
        any = any || flag[i];
        if (flag[i]) rt[i] = std::max(inner, rtolv[i] * bn / rn);
      }
      if (!any) break;
      HIPCHK(c, c->pin_fl.alloc(S));
      std::copy(flag.begin(), flag.end(), c->pin_fl.p);
      HIPCHK(c, hipMemcpyAsync(c->s_flag.p, c->pin_fl.p, S * sizeof(int), hipMemcpyHostToDevice, s));
      HIPCHK(c, (glh::launch_convert<double, float>(n, c->ir_r.p, c->gb32.p, s)));
      HIPCHK(c, glh::launch_seg_zero<float>(c->seg(), c->s_flag.p, c->gb32.p, s));
      int it2 = 0;
      std::vector<double> rel2;
      std::vector<int> is2;
      rc = gmres<float, float>(c, c->J32.p, c->D32.p, c->gb32.p, c->gx32.p, rt, maxit - its, restart, &it2, rel2, is2);
      its += it2;
      for (int i = 0; i < S; ++i) its_seg[i] += is2[i];
      if (rc && rc != GLH_ERR_NOCONV) return rc;
      HIPCHK(c, (glh::launch_axpy<float, double>(n, 1.0, c->gx32.p, c->dU.p, s)));
      if (c->j_mf) RCHK(mf_product<double>(c, c->dU.p, c->rhs.p, c->ir_r.p));
      else if (c->sym_state == 1)
        HIPCHK(c, (glh::launch_spmv_sym<float, double>(c->n_nodes, c->row_ptr.p, c->diag.p, c->col.p, c->sym_lo.p,
                                                       c->J32.p, c->dU.p, c->rhs.p, c->ir_r.p, c->sym_T.p, s)));
      else
        HIPCHK(c, glh::launch_residual_spmv<float>(c->n_nodes, c->row_ptr.p, c->col.p, c->J32.p, c->dU.p, c->rhs.p,
                                                   c->ir_r.p, s));
      RCHK(seg_norm2(c, c->ir_r.p, rn2));
    }
    rel.assign(S, 0.0);
    bool ok = true;
    for (int i = 0; i < S; ++i) {
      const double bn = std::sqrt(bn2[i]), rn = std::sqrt(rn2[i]);
      rel[i] = bn > 0 ? rn / bn : 0.0;
      ok = ok && rel[i] <= rtolv[i];
    }
    rc = ok ? GLH_OK : fail(c, GLH_ERR_NOCONV, "mixed-precision GMRES did not reach the tolerance");
  }
  if (stats) {
    stats[0] = its;
    stats[1] = rel.empty() ? 0.0 : *std::max_element(rel.begin(), rel.end());
  }
  if (its_seg_out) *its_seg_out = its_seg;
  if (rc) return rc;
  // constraints_newton_update.distribute (solve.cc:181)
  RCHK(distribute(c, c->dU.p));
  return GLH_OK;
}

// damped back-tracking line search of iteration.cc:170-206 per instance.
// active[s] == 0: the instance is frozen (its update is zero).
// prev/cur: per-instance ||rhs|| before, ||R|| after; alpha, trials per instance.
int newton_step_impl(glh_ctx *c, double step, int damped, const std::vector<char> &active, std::vector<double> &prev,
                     std::vector<double> &cur, std::vector<double> &alpha, std::vector<int> &trials)
{
  const int S = c->n_seg;
  std::vector<double> p2, c2;
  RCHK(seg_norm2(c, c->rhs.p, p2));  // previous_residual = ||system_rhs|| (iteration.cc:130)
  prev.resize(S);
  for (int i = 0; i < S; ++i) prev[i] = std::sqrt(p2[i]);
  std::vector<char> acc(S);
  alpha.assign(S, 0.0);
  trials.assign(S, 0);
  for (int i = 0; i < S; ++i) acc[i] = !active[i];
  HIPCHK(c, take(c, c->s_alpha, S));
  HIPCHK(c, c->pinv.alloc(S));
  const int n_try = damped ? 100 : 1;
  cur.assign(S, 0.0);
  for (int t = 0; t < n_try; ++t) {
    for (int i = 0; i < S; ++i)
      if (!acc[i]) {
        alpha[i] = damped ? std::pow(step, (double)t) : 1.0;
        trials[i] = t + 1;
      }
    std::copy(alpha.begin(), alpha.end(), c->pinv.p);
    HIPCHK(c, hipMemcpyAsync(c->s_alpha.p, c->pinv.p, S * sizeof(double), hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, glh::launch_seg_trial(c->seg(), c->U.p, c->dU.p, c->s_alpha.p, c->node_mask.p, c->X.p, c->stream));
    if (c->constrained) HIPCHK(c, glh::launch_distribute(c->cons, c->X.p, c->stream));  // iteration.cc:180
    RCHK(residual_norms(c, c->X.p, c->res.p, c2));
    bool all = true;
    for (int i = 0; i < S; ++i) {
      cur[i] = std::sqrt(c2[i]);
      if (!acc[i] && cur[i] < prev[i]) acc[i] = 1;
      all = all && acc[i];
    }
    if (all) break;
  }
  HIPCHK(c, hipMemcpyAsync(c->U.p, c->X.p, ndofs(c) * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return GLH_OK;
}

int instance_energy(glh_ctx *c, std::vector<double> &F)
{
  HIPCHK(c, glh::launch_energy(c->deg, c->tables(), c->meshdev(), c->mat, c->U.p, c->n_cells, c->Fcell.p,
                               c->stream));
  std::vector<double> fc(c->n_cells);
  HIPCHK(c, hipMemcpyAsync(fc.data(), c->Fcell.p, c->n_cells * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  F.assign(c->n_seg, 0.0);
  for (int s = 0; s < c->n_seg; ++s)
    for (int e = c->cell_off[s]; e < c->cell_off[s + 1]; ++e) F[s] += fc[e];  // fixed order
  return GLH_OK;
}

bool make_material(const double *co, glh::Material &m)
{
  // co: alpha, beta1..5, K1, K2, K3, bt
  if (!(co[9] > 0)) return false;
  m.al = co[0];
  m.b1 = co[1]; m.b2 = co[2]; m.b3 = co[3]; m.b4 = co[4]; m.b5 = co[5];
  m.K1 = co[6];
  m.K23 = co[7] + co[8];
  m.robin = (co[9] < 1e10) ? co[6] / co[9] : 0.0;
  return true;
}

int get_vec(glh_ctx *c, const double *src, double *dst)
{
  RCHK(check_ready(c, false));
  if (!dst) return fail(c, GLH_ERR_ARG, "null output");
  HIPCHK(c, hipMemcpyAsync(dst, src, ndofs(c) * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return GLH_OK;
}

}  // namespace

// ===================================================================== ABI
extern "C" {

int glh_create(int device, glh_ctx **out)
{
  if (!out) return GLH_ERR_ARG;
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return GLH_ERR_HIP;
  if (device < 0 || device >= ndev) return GLH_ERR_ARG;
  glh_ctx *c = new glh_ctx();
  c->device = device;
  if (hipSetDevice(device) != hipSuccess || hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreate(&c->ev0) != hipSuccess || hipEventCreate(&c->ev1) != hipSuccess ||
      glh::scratch_address(device, &c->scratch) != hipSuccess) {
    glh_destroy(c);  // releases whatever was created
    return GLH_ERR_HIP;
  }
  *out = c;
  return GLH_OK;
}

int glh_destroy(glh_ctx *c)
{
  if (!c) return GLH_OK;
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  DBuf<double> *dbs[] = {&c->tN,     &c->tdN,  &c->tw,   &c->tWp,  &c->tSp,   &c->tMf,   &c->tAt,   &c->cell_h,
                         &c->U,      &c->U0,   &c->dU,   &c->X,    &c->rhs,   &c->res,   &c->Fcell,
                         &c->s_norm, &c->s_alpha, &c->s_part, &c->J64, &c->D64, &c->gV64, &c->gZ64,
                         &c->gW64,   &c->gh64, &c->gp64, &c->gy64, &c->gs64,  &c->gq64,  &c->ir_r, &c->gn64, &c->sym_T};
  for (auto *b : dbs) b->release();
  DBuf<float> *fbs[] = {&c->J32,  &c->D32,  &c->gV32, &c->gZ32, &c->gW32, &c->gh32,
                        &c->gp32, &c->gy32, &c->gs32, &c->gq32, &c->gb32, &c->gx32, &c->gn32};
  for (auto *b : fbs) b->release();
  DBuf<int> *ibs[] = {&c->tpa,      &c->tpb,         &c->cell_nodes, &c->row_ptr,  &c->col,       &c->diag,
                      &c->cell_blk, &c->color_cells, &c->status,     &c->cell_mat, &c->seg_chunk, &c->s_flag, &c->sym_lo};
  for (auto *b : ibs) b->release();
  for (auto *g : {&c->graph64, &c->graph32})
    for (auto e : g->exec)
      if (e) (void)hipGraphExecDestroy(e);
  DBuf<double> *gd[] = {&c->gmH, &c->gmcs, &c->gmsn, &c->gmg, &c->gmbeta, &c->gmtarget};
  for (auto *b : gd) b->release();
  DBuf<int> *gi[] = {&c->gmcyc,   &c->gmconv,     &c->gmjseg,     &c->gmits,    &c->gmro,     &c->gmfrozen,
                     &c->gmjlast, &c->row_seg,    &c->d_node_off, &c->act_counts, &c->act_seg, &c->act_rpref,
                     &c->act_chunk};
  for (auto *b : gi) b->release();
  DBuf<int> *ci[] = {&c->c_gptr,  &c->c_gsrc,   &c->c_brow,   &c->c_rptr,  &c->c_rsrc,  &c->c_hnode, &c->c_hptr,
                     &c->c_hm,    &c->c_hidx,   &c->mfx_ptr,  &c->mfx_pair, &c->mft_node, &c->mft_ptr, &c->mft_slot,
                     &c->mft_A,   &c->mft_B};
  for (auto *b : ci) b->release();
  DBuf<double> *cd[] = {&c->c_gw, &c->c_rw, &c->c_hw, &c->hdiag, &c->rfull, &c->Jf64, &c->mfx_LB, &c->mft_w, &c->mf_diag,
                        &c->mf_xf, &c->mf_yf, &c->mf_sh};
  for (auto *b : cd) b->release();
  c->mft_fl.release();
  c->c_gfl.release();
  c->c_rfl.release();
  c->asm_flag.release();
  c->Jf32.release();
  c->chunks.release();
  c->mats.release();
  c->cell_face.release();
  c->node_mask.release();
  c->pin64.release();
  c->pinv.release();
  c->pin32.release();
  c->pin_i.release();
  c->pin_st.release();
  for (auto e : c->ev_step)
    if (e) (void)hipEventDestroy(e);
  c->pin_fl.release();
  for (auto e : c->ev_pool)
    if (e) (void)hipEventDestroy(e);
  if (c->ev0) (void)hipEventDestroy(c->ev0);
  if (c->ev1) (void)hipEventDestroy(c->ev1);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
  return GLH_OK;
}

const char *glh_last_error(const glh_ctx *c) { return c ? c->err.c_str() : "null context"; }

int glh_set_material(glh_ctx *c, double alpha, const double beta[5], const double K[3], double bt)
{
  if (!c || !beta || !K) return GLH_ERR_ARG;
  const double co[10] = {alpha, beta[0], beta[1], beta[2], beta[3], beta[4], K[0], K[1], K[2], bt};
  glh::Material mt{};
  if (!make_material(co, mt)) return fail(c, GLH_ERR_ARG, "AdGR diffuse length must be positive");
  HIPCHK(c, hipSetDevice(c->device));
  if (c->stream) HIPCHK(c, hipStreamSynchronize(c->stream));
  drop_graphs(c);  // the matrix-free product's graphs carry the old material by value
  c->mat = mt;
  c->mats_host.clear();
  c->have_mat = true;
  c->j_valid = c->d_valid = false;
  return GLH_OK;
}

int glh_set_materials(glh_ctx *c, int n_inst, const double *coef)
{
  if (!c || !coef || n_inst < 1) return GLH_ERR_ARG;
  std::vector<glh::Material> ms(n_inst);
  for (int i = 0; i < n_inst; ++i)
    if (!make_material(coef + 10 * i, ms[i])) return fail(c, GLH_ERR_ARG, "AdGR diffuse length must be positive");
  HIPCHK(c, hipSetDevice(c->device));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  drop_graphs(c);  // recorded products read the old materials (and possibly the old buffer)
  HIPCHK(c, upload(c, c->mats, ms.data(), ms.size(), c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->mats_host = ms;
  c->mat = ms[0];
  c->have_mat = true;
  c->j_valid = c->d_valid = false;
  return GLH_OK;
}

namespace {
// message of the last failed mesh-building call on this thread (the mesh
// functions have no context to keep it in)
thread_local std::string mesh_err;
}  // namespace

const char *glh_mesh_last_error(void) { return mesh_err.c_str(); }

int glh_mesh_box(int degree, int nx, int ny, int nz, const double lo[3], const double hi[3], const int side_id[6],
                 glh_mesh **out)
{
  if (!out || !lo || !hi || !side_id) return GLH_ERR_ARG;
  *out = nullptr;
  glh_mesh *m = new glh_mesh();
  if (glh::make_box(m->m, degree, nx, ny, nz, lo, hi, side_id, mesh_err)) {
    delete m;
    return GLH_ERR_ARG;
  }
  *out = m;
  return GLH_OK;
}

int glh_mesh_from_arrays(const glh_mesh_desc *d, glh_mesh **out)
{
  if (!d || !out) return GLH_ERR_ARG;
  *out = nullptr;
  glh::ArrayMesh a;
  a.degree = d->degree; a.n_cells = d->n_cells; a.n_nodes = d->n_nodes; a.order = d->local_order;
  a.cell_nodes = d->cell_nodes; a.cell_lo = d->cell_lo; a.cell_h = d->cell_h; a.node_xyz = d->node_xyz;
  a.n_faces = d->n_faces; a.faces = d->faces; a.node_mask = d->node_mask;
  a.n_lines = d->n_lines; a.line_node = d->line_node; a.line_ptr = d->line_ptr; a.line_master = d->line_master;
  a.line_w = d->line_w;
  glh_mesh *m = new glh_mesh();
  if (glh::from_arrays(m->m, a, mesh_err)) {
    delete m;
    return GLH_ERR_ARG;
  }
  *out = m;
  return GLH_OK;
}

int glh_mesh_concat(const glh_mesh *const *ms, int n, glh_mesh **out)
{
  if (!ms || !out || n < 1) return GLH_ERR_ARG;
  *out = nullptr;
  std::vector<const glh::Mesh *> v(n);
  for (int i = 0; i < n; ++i) {
    if (!ms[i]) return GLH_ERR_ARG;
    v[i] = &ms[i]->m;
  }
  glh_mesh *m = new glh_mesh();
  std::string err;
  if (glh::concat(m->m, v, err)) {
    delete m;
    return GLH_ERR_ARG;
  }
  *out = m;
  return GLH_OK;
}

int glh_mesh_destroy(glh_mesh *m)
{
  delete m;
  return GLH_OK;
}

int glh_mesh_sizes(const glh_mesh *mm, int64_t sizes[8])
{
  if (!mm || !sizes) return GLH_ERR_ARG;
  const glh::Mesh &m = mm->m;
  sizes[0] = m.deg; sizes[1] = m.n_cells; sizes[2] = m.n_nodes; sizes[3] = (int64_t)m.faces.size() / 3;
  sizes[4] = m.row_ptr.empty() ? 0 : m.row_ptr.back(); sizes[5] = (int64_t)m.color_ptr.size() - 1;
  sizes[6] = (int64_t)m.node_off.size() - 1; sizes[7] = 0;
  return GLH_OK;
}

int glh_mesh_get(const glh_mesh *mm, int *cell_nodes, double *cell_h, double *node_xyz, int *faces,
                 uint32_t *node_mask, int *color_ptr, int *color_cells, int *row_ptr, int *col)
{
  if (!mm) return GLH_ERR_ARG;
  const glh::Mesh &m = mm->m;
  auto cp = [](auto *dst, const auto &v) {
    if (dst && !v.empty()) std::memcpy(dst, v.data(), v.size() * sizeof(v[0]));
  };
  cp(cell_nodes, m.cell_nodes); cp(cell_h, m.cell_h); cp(node_xyz, m.node_xyz); cp(faces, m.faces);
  cp(node_mask, m.node_mask); cp(color_ptr, m.color_ptr); cp(color_cells, m.color_cells); cp(row_ptr, m.row_ptr);
  cp(col, m.col);
  return GLH_OK;
}

int glh_forest_create(int nx, int ny, int nz, const double lo[3], const double hi[3], const int side_id[6],
                      glh_forest **out)
{
  if (!lo || !hi || !side_id || !out) return GLH_ERR_ARG;
  *out = nullptr;
  auto *f = new glh_forest();
  std::string err;
  if (glh::forest_init(f->f, nx, ny, nz, lo, hi, side_id, err)) {
    delete f;
    return GLH_ERR_ARG;
  }
  *out = f;
  return GLH_OK;
}

int glh_forest_destroy(glh_forest *f)
{
  delete f;
  return GLH_OK;
}

int64_t glh_forest_n_cells(const glh_forest *f) { return f ? (int64_t)f->f.leaves.size() : -1; }

int glh_forest_set_degree(glh_forest *f, int deg)
{
  if (!f || (deg != 1 && deg != 2)) return GLH_ERR_ARG;
  f->deg = deg;
  return GLH_OK;
}

int glh_forest_refine(const glh_forest *f, const uint8_t *flags, glh_forest **out)
{
  if (!f || !flags || !out) return GLH_ERR_ARG;
  *out = nullptr;
  auto *g = new glh_forest(*f);
  std::vector<char> fl(flags, flags + f->f.leaves.size());
  std::string err;
  if (glh::forest_refine(g->f, fl, err)) {
    delete g;
    return GLH_ERR_ARG;
  }
  *out = g;
  return GLH_OK;
}

int glh_forest_mesh(const glh_forest *f, glh_mesh **out)
{
  if (!f || !out) return GLH_ERR_ARG;
  *out = nullptr;
  auto *mm = new glh_mesh();
  std::string err;
  if (glh::forest_mesh(f->f, mm->m, err, f->deg)) {
    delete mm;
    return GLH_ERR_ARG;
  }
  *out = mm;
  return GLH_OK;
}

int glh_forest_transfer(const glh_forest *fo, const glh_mesh *mo, const double *Uo, const glh_forest *fn,
                        const glh_mesh *mn, double *Un)
{
  if (!fo || !mo || !Uo || !fn || !mn || !Un) return GLH_ERR_ARG;
  std::string err;
  return glh::forest_transfer(fo->f, mo->m, Uo, fn->f, mn->m, Un, err) ? GLH_ERR_ARG : GLH_OK;
}

int glh_transfer_solution(glh_ctx *c, const glh_forest *fo, const glh_mesh *mo, const glh_forest *fn,
                          const glh_mesh *mn)
{
  RCHK(check_ready(c, false));
  if (!fo || !mo || !fn || !mn) return fail(c, GLH_ERR_ARG, "null forest or mesh");
  if (c->n_nodes != mo->m.n_nodes || c->n_cells != mo->m.n_cells || c->n_seg != 1 || mo->m.deg != c->deg)
    return fail(c, GLH_ERR_STATE, "the context does not hold the old mesh");
  if (mn->m.deg != mo->m.deg) return fail(c, GLH_ERR_ARG, "old and new mesh of different degree");
  std::string err;
  std::vector<int> cell;
  std::vector<float> t;
  if (glh::forest_transfer_map(fo->f, mo->m, fn->f, mn->m, cell, t, err)) return fail(c, GLH_ERR_ARG, err);
  hipStream_t s = c->stream;
  // the old field and cell corners outlive the upload of the new mesh
  DBuf<double> Uo;
  DBuf<int> cno, dcell;
  DBuf<float> dt;
  auto release = [&]() {
    Uo.release();
    cno.release();
    dcell.release();
    dt.release();
  };
  const size_t no = (size_t)mo->m.n_nodes * NC, nco = (size_t)mo->m.n_cells * mo->m.ns;
  hipError_t e = take(c, Uo, no);
  if (e == hipSuccess) e = take(c, cno, nco);
  if (e == hipSuccess) e = hipMemcpyAsync(Uo.p, c->U.p, no * sizeof(double), hipMemcpyDeviceToDevice, s);
  if (e == hipSuccess) e = hipMemcpyAsync(cno.p, c->cell_nodes.p, nco * sizeof(int), hipMemcpyDeviceToDevice, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) {
    release();
    return fail(c, GLH_ERR_HIP, std::string("transfer staging: ") + hipGetErrorString(e));
  }
  int rc = glh_upload_mesh(c, mn);
  if (rc) {
    release();
    return rc;
  }
  e = upload(c, dcell, cell.data(), cell.size(), s);
  if (e == hipSuccess) e = upload(c, dt, t.data(), t.size(), s);
  if (e == hipSuccess) e = glh::launch_transfer(mn->m.n_nodes, mn->m.deg, dcell.p, dt.p, cno.p, Uo.p, c->U.p, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  release();
  if (e != hipSuccess) return fail(c, GLH_ERR_HIP, std::string("transfer: ") + hipGetErrorString(e));
  // constraints_solution.distribute (refine.cc:173)
  RCHK(distribute(c, c->U.p));
  HIPCHK(c, hipStreamSynchronize(s));
  return GLH_OK;
}

int glh_kelly(const glh_forest *f, const glh_mesh *m, const double *U, float *eta)
{
  if (!f || !m || !U || !eta) return GLH_ERR_ARG;
  std::string err;
  return glh::kelly_estimate(f->f, m->m, U, eta, err) ? GLH_ERR_ARG : GLH_OK;
}

int glh_flag_fixed_number(int64_t n, const float *eta, double frac, uint8_t *flags)
{
  if (n < 0 || n > INT32_MAX || (n > 0 && (!eta || !flags)) || !(frac >= 0.0 && frac <= 1.0)) return GLH_ERR_ARG;
  std::vector<char> fl;
  glh::flag_fixed_number((int)n, eta, frac, fl);
  for (int64_t i = 0; i < n; ++i) flags[i] = (uint8_t)fl[i];
  return GLH_OK;
}

int glh_flag_refine_coarsen(int64_t n, const float *eta, double refine_frac, double coarsen_frac, uint8_t *flags)
{
  if (n < 0 || n > INT32_MAX || (n > 0 && (!eta || !flags)) || !(refine_frac >= 0.0 && refine_frac <= 1.0) ||
      !(coarsen_frac >= 0.0 && coarsen_frac <= 1.0) || refine_frac + coarsen_frac > 1.0)
    return GLH_ERR_ARG;
  std::vector<char> fl;
  glh::flag_refine_coarsen((int)n, eta, refine_frac, coarsen_frac, fl);
  for (int64_t i = 0; i < n; ++i) flags[i] = (uint8_t)fl[i];
  return GLH_OK;
}

int glh_mesh_constraint_sizes(const glh_mesh *mm, int64_t sizes[3])
{
  if (!mm || !sizes) return GLH_ERR_ARG;
  const glh::Mesh &m = mm->m;
  int64_t nh = 0;
  if (m.has_hanging())
    for (int v = 0; v < m.n_nodes; ++v) nh += m.hang_ptr[v + 1] > m.hang_ptr[v];
  sizes[0] = nh;
  sizes[1] = (int64_t)m.hang_m.size();
  sizes[2] = m.arow_ptr.empty() ? (m.row_ptr.empty() ? 0 : m.row_ptr.back()) : m.arow_ptr.back();
  return GLH_OK;
}

int glh_mesh_constraints(const glh_mesh *mm, int *hang_ptr, int *hang_m, double *hang_w, int *arow_ptr, int *acol)
{
  if (!mm) return GLH_ERR_ARG;
  const glh::Mesh &m = mm->m;
  const bool h = m.has_hanging();
  if (hang_ptr) {
    if (h) std::memcpy(hang_ptr, m.hang_ptr.data(), m.hang_ptr.size() * sizeof(int));
    else std::fill(hang_ptr, hang_ptr + m.n_nodes + 1, 0);
  }
  if (hang_m && h) std::memcpy(hang_m, m.hang_m.data(), m.hang_m.size() * sizeof(int));
  if (hang_w && h) std::memcpy(hang_w, m.hang_w.data(), m.hang_w.size() * sizeof(double));
  const std::vector<int> &rp = m.arow_ptr.empty() ? m.row_ptr : m.arow_ptr;
  const std::vector<int> &cl = m.arow_ptr.empty() ? m.col : m.acol;
  if (arow_ptr) std::memcpy(arow_ptr, rp.data(), rp.size() * sizeof(int));
  if (acol) std::memcpy(acol, cl.data(), cl.size() * sizeof(int));
  return GLH_OK;
}

int glh_mesh_instances(const glh_mesh *mm, int *node_off, int *cell_off)
{
  if (!mm) return GLH_ERR_ARG;
  const glh::Mesh &m = mm->m;
  if (node_off) std::memcpy(node_off, m.node_off.data(), m.node_off.size() * sizeof(int));
  if (cell_off) std::memcpy(cell_off, m.cell_off.data(), m.cell_off.size() * sizeof(int));
  return GLH_OK;
}

namespace {

// Gather lists of the condensation Jc = C^T Jf C, rc = C^T rf and the
// hanging lines, built on the host from the mesh's closed constraint lines.
int upload_constraints(glh_ctx *c, const glh::Mesh &m, const std::vector<int> &diag)
{
  hipStream_t s = c->stream;
  const int nn = m.n_nodes;
  auto hanging = [&](int a) { return m.hang_ptr[a + 1] > m.hang_ptr[a]; };
  // Jc block t gathers Jf block (A,B) with weight wA*wB for every master pair
  // (r in T(A), s in T(B)); T(A) = {A} or the line of a hanging A
  std::vector<std::vector<int>> tsrc(c->nnzb);
  std::vector<std::vector<double>> tw(c->nnzb);
  std::vector<std::vector<unsigned char>> tfl(c->nnzb);
  for (int A = 0; A < nn; ++A)
    for (int sb = m.arow_ptr[A]; sb < m.arow_ptr[A + 1]; ++sb) {
      const int B = m.acol[sb];
      const bool ha = hanging(A), hb = hanging(B);
      const int ka0 = ha ? m.hang_ptr[A] : 0, ka1 = ha ? m.hang_ptr[A + 1] : 1;
      const int kb0 = hb ? m.hang_ptr[B] : 0, kb1 = hb ? m.hang_ptr[B + 1] : 1;
      for (int ka = ka0; ka < ka1; ++ka)
        for (int kb = kb0; kb < kb1; ++kb) {
          const int r = ha ? m.hang_m[ka] : A, cc = hb ? m.hang_m[kb] : B;
          const double w = (ha ? m.hang_w[ka] : 1.0) * (hb ? m.hang_w[kb] : 1.0);
          const int t = glh::find_block(m, r, cc);
          if (t < 0) return fail(c, GLH_ERR_ARG, "condensed pattern lacks a constrained coupling");
          tsrc[t].push_back(sb);
          tw[t].push_back(w);
          tfl[t].push_back((unsigned char)((ha ? 1 : 0) | (hb ? 2 : 0)));
        }
    }
  std::vector<int> gptr(c->nnzb + 1, 0), gsrc, brow(c->nnzb);
  std::vector<double> gw;
  std::vector<unsigned char> gfl;
  for (int t = 0; t < c->nnzb; ++t) {
    gptr[t + 1] = gptr[t] + (int)tsrc[t].size();
    gsrc.insert(gsrc.end(), tsrc[t].begin(), tsrc[t].end());
    gw.insert(gw.end(), tw[t].begin(), tw[t].end());
    gfl.insert(gfl.end(), tfl[t].begin(), tfl[t].end());
    std::vector<int>().swap(tsrc[t]);
    std::vector<double>().swap(tw[t]);
    std::vector<unsigned char>().swap(tfl[t]);
  }
  for (int r = 0; r < nn; ++r)
    for (int t = m.row_ptr[r]; t < m.row_ptr[r + 1]; ++t) brow[t] = r;
  // rhs: row r gathers itself and every hanging node whose line holds r
  std::vector<std::vector<int>> rs(nn);
  std::vector<std::vector<double>> rwv(nn);
  std::vector<int> hnode, hptr(1, 0), hm;
  std::vector<double> hw;
  for (int a = 0; a < nn; ++a) {
    if (!hanging(a)) {
      rs[a].push_back(a);
      rwv[a].push_back(1.0);
      continue;
    }
    hnode.push_back(a);
    for (int k = m.hang_ptr[a]; k < m.hang_ptr[a + 1]; ++k) {
      hm.push_back(m.hang_m[k]);
      hw.push_back(m.hang_w[k]);
    }
    hptr.push_back((int)hm.size());
  }
  for (int a = 0; a < nn; ++a)
    if (hanging(a))
      for (int k = m.hang_ptr[a]; k < m.hang_ptr[a + 1]; ++k) {
        rs[m.hang_m[k]].push_back(-(a + 1));  // marks a constraint contribution
        rwv[m.hang_m[k]].push_back(m.hang_w[k]);
      }
  std::vector<int> rptr(nn + 1, 0), rsrc;
  std::vector<double> rw;
  std::vector<unsigned char> rfl;
  for (int r = 0; r < nn; ++r) {
    for (size_t k = 0; k < rs[r].size(); ++k) {
      const int v = rs[r][k];
      rsrc.push_back(v >= 0 ? v : -v - 1);
      rfl.push_back(v >= 0 ? 0 : 1);
      rw.push_back(rwv[r][k]);
    }
    rptr[r + 1] = (int)rsrc.size();
  }
  HIPCHK(c, upload(c, c->c_gptr, gptr.data(), gptr.size(), s));
  HIPCHK(c, upload(c, c->c_gsrc, gsrc.data(), gsrc.size(), s));
  HIPCHK(c, upload(c, c->c_gw, gw.data(), gw.size(), s));
  HIPCHK(c, upload(c, c->c_gfl, gfl.data(), gfl.size(), s));
  HIPCHK(c, upload(c, c->c_brow, brow.data(), brow.size(), s));
  HIPCHK(c, upload(c, c->c_rptr, rptr.data(), rptr.size(), s));
  HIPCHK(c, upload(c, c->c_rsrc, rsrc.data(), rsrc.size(), s));
  HIPCHK(c, upload(c, c->c_rw, rw.data(), rw.size(), s));
  HIPCHK(c, upload(c, c->c_rfl, rfl.data(), rfl.size(), s));
  c->n_hang = (int)hnode.size();
  HIPCHK(c, upload(c, c->c_hnode, hnode.data(), hnode.size(), s));
  HIPCHK(c, upload(c, c->c_hptr, hptr.data(), hptr.size(), s));
  HIPCHK(c, upload(c, c->c_hm, hm.data(), hm.size(), s));
  HIPCHK(c, upload(c, c->c_hw, hw.data(), hw.size(), s));
  std::vector<int> hidx(nn, -1);
  for (size_t j = 0; j < hnode.size(); ++j) hidx[hnode[j]] = (int)j;
  HIPCHK(c, upload(c, c->c_hidx, hidx.data(), hidx.size(), s));
  HIPCHK(c, take(c, c->hdiag, (size_t)nn * NC));
  HIPCHK(c, take(c, c->rfull, (size_t)nn * NC));
  // Matrix-free Jacobian: the condensed diagonal block of a master n holds,
  // besides the (n, n) blocks of its cells, w_A(n) w_B(n) J_K(a, b) for every
  // cell K and local pair (a, b) with A = cn[a], B = cn[b] both reaching n
  // through T(A) = {A} or the line of a hanging A (the gather of Jc's
  // diagonal blocks above, cell by cell).  Slots: local pairs (a <= b) whose
  // raw block some term uses, per cell in pair order.
  {
    const int ns = m.ns;
    struct Term {
      int n, slot, A, B;
      double w;
      unsigned char fl;
    };
    std::vector<Term> terms;
    std::vector<int> xptr(m.n_cells + 1, 0), xpair;
    for (int e = 0; e < m.n_cells; ++e) {
      const int *cn = &m.cell_nodes[(size_t)e * ns];
      int p = 0;
      for (int a = 0; a < ns; ++a)
        for (int b = a; b < ns; ++b, ++p) {
          const int A = cn[a], B = cn[b];
          if (!hanging(A) && !hanging(B)) continue;
          const int slot = (int)xpair.size();
          bool used = false;
          for (int o = 0; o < (a == b ? 1 : 2); ++o) {  // (a, b), then (b, a): the transposed block
            const int P = o ? B : A, Q = o ? A : B;
            const bool hp = hanging(P), hq = hanging(Q);
            const int kp0 = hp ? m.hang_ptr[P] : 0, kp1 = hp ? m.hang_ptr[P + 1] : 1;
            const int kq0 = hq ? m.hang_ptr[Q] : 0, kq1 = hq ? m.hang_ptr[Q + 1] : 1;
            for (int kp = kp0; kp < kp1; ++kp)
              for (int kq = kq0; kq < kq1; ++kq) {
                const int np = hp ? m.hang_m[kp] : P, nq = hq ? m.hang_m[kq] : Q;
                if (np != nq) continue;
                const double w = (hp ? m.hang_w[kp] : 1.0) * (hq ? m.hang_w[kq] : 1.0);
                terms.push_back(Term{np, slot, P, Q, w,
                                     (unsigned char)((hp ? 1 : 0) | (hq ? 2 : 0) | (o ? 4 : 0) | (a == b ? 8 : 0))});
                used = true;
              }
          }
          if (used) xpair.push_back(p);
        }
      xptr[e + 1] = (int)xpair.size();
    }
    std::stable_sort(terms.begin(), terms.end(), [](const Term &x, const Term &y) { return x.n < y.n; });
    std::vector<int> tnode, tptr(1, 0), tslot, tA, tB;
    std::vector<double> tw;
    std::vector<unsigned char> tfl;
    for (size_t k = 0; k < terms.size(); ++k) {
      if (k == 0 || terms[k].n != terms[k - 1].n) {
        if (k) tptr.push_back((int)k);
        tnode.push_back(terms[k].n);
      }
      tslot.push_back(terms[k].slot);
      tA.push_back(terms[k].A);
      tB.push_back(terms[k].B);
      tw.push_back(terms[k].w);
      tfl.push_back(terms[k].fl);
    }
    if (!terms.empty()) tptr.push_back((int)terms.size());
    HIPCHK(c, upload(c, c->mfx_ptr, xptr.data(), xptr.size(), s));
    HIPCHK(c, upload(c, c->mfx_pair, xpair.data(), xpair.size(), s));
    HIPCHK(c, upload(c, c->mft_node, tnode.data(), tnode.size(), s));
    HIPCHK(c, upload(c, c->mft_ptr, tptr.data(), tptr.size(), s));
    HIPCHK(c, upload(c, c->mft_slot, tslot.data(), tslot.size(), s));
    HIPCHK(c, upload(c, c->mft_A, tA.data(), tA.size(), s));
    HIPCHK(c, upload(c, c->mft_B, tB.data(), tB.size(), s));
    HIPCHK(c, upload(c, c->mft_w, tw.data(), tw.size(), s));
    HIPCHK(c, upload(c, c->mft_fl, tfl.data(), tfl.size(), s));
    c->mfx_slots = xpair.size();
    c->mfc = glh::MfCondDev{c->mfx_ptr.p, c->mfx_pair.p, nullptr, (int)tnode.size(), c->mft_node.p, c->mft_ptr.p,
                            c->mft_slot.p, c->mft_A.p, c->mft_B.p, c->mft_w.p, c->mft_fl.p};
    HIPCHK(c, hipStreamSynchronize(s));  // the host vectors go out of scope
  }
  HIPCHK(c, hipStreamSynchronize(s));
  return GLH_OK;
}

}  // namespace

int glh_upload_mesh(glh_ctx *c, const glh_mesh *mm)
{
  if (!c || !mm) return GLH_ERR_ARG;
  const glh::Mesh &m = mm->m;
  HIPCHK(c, hipSetDevice(c->device));
  // until all of it is there: an allocation that fails has given up the
  // previous mesh's buffer
  c->have_mesh = c->j_valid = c->d_valid = false;
  if (c->deg != m.deg || !c->tN.p) RCHK(build_tables(c, m.deg));
  hipStream_t s = c->stream;
  drop_graphs(c);  // captured GMRES graphs refer to the previous mesh's buffers
  c->sym_state = 0;
  c->n_cells = m.n_cells;
  c->n_nodes = m.n_nodes;
  c->nnzb = m.row_ptr.back();
  c->color_ptr = m.color_ptr;
  c->node_off = m.node_off.empty() ? std::vector<int>{0, m.n_nodes} : m.node_off;
  c->cell_off = m.cell_off.empty() ? std::vector<int>{0, m.n_cells} : m.cell_off;
  c->n_seg = (int)c->node_off.size() - 1;
  c->r_ref.clear();
  // per-cell face codes (boundary id + 1, 3 bits per local face)
  std::vector<uint32_t> cface(m.n_cells, 0u);
  for (size_t f = 0; f + 2 < m.faces.size(); f += 3) {
    const int e = m.faces[f], lf = m.faces[f + 1], bid = m.faces[f + 2];
    const uint32_t code = (uint32_t)std::min(bid, 6) + 1u;
    cface[e] |= code << (3 * lf);
  }
  std::vector<int> diag(m.n_nodes);
  for (int r = 0; r < m.n_nodes; ++r) {
    diag[r] = glh::find_block(m, r, r);
    if (diag[r] < 0) return fail(c, GLH_ERR_ARG, "pattern lacks a diagonal block");
  }
  c->constrained = m.has_hanging();
  c->nnzb_a = c->constrained ? m.arow_ptr.back() : c->nnzb;
  c->n_hang = 0;
  if (c->constrained) RCHK(upload_constraints(c, m, diag));
  // the matrix-free Jacobian's diagonal block of each node: its own, or for a
  // hanging node block n_nodes + j (hanging nodes in node order)
  std::vector<int> did(m.n_nodes);
  for (int i = 0, j = 0; i < m.n_nodes; ++i)
    did[i] = (c->constrained && m.hang_ptr[i + 1] > m.hang_ptr[i]) ? m.n_nodes + j++ : i;
  HIPCHK(c, upload(c, c->diag_id, did.data(), did.size(), s));
  // cell -> block map (cell-loop pattern) with first-writer marks in colour order
  const int ns = m.ns;
  std::vector<int> cblk((size_t)m.n_cells * ns * ns);
  std::vector<uint8_t> touched(c->nnzb_a, 0);
  for (size_t k = 0; k + 1 < m.color_ptr.size(); ++k)
    for (int i = m.color_ptr[k]; i < m.color_ptr[k + 1]; ++i) {
      const int e = m.color_cells[i];
      const int *cn = &m.cell_nodes[(size_t)e * ns];
      for (int a = 0; a < ns; ++a)
        for (int b = 0; b < ns; ++b) {
          const int blk = glh::find_ablock(m, cn[a], cn[b]);
          if (blk < 0) return fail(c, GLH_ERR_ARG, "pattern lacks a cell coupling");
          const bool first = !touched[blk];
          touched[blk] = 1;
          cblk[((size_t)e * ns + a) * ns + b] = first ? -(blk + 1) : blk;
        }
    }
  // instance of each cell, and reduction chunks that never straddle instances
  std::vector<int> cmat(m.n_cells);
  for (int sg = 0; sg < c->n_seg; ++sg)
    for (int e = c->cell_off[sg]; e < c->cell_off[sg + 1]; ++e) cmat[e] = sg;
  std::vector<long long> ch;
  std::vector<int> segch(1, 0);
  for (int sg = 0; sg < c->n_seg; ++sg) {
    const long long b0 = (long long)c->node_off[sg] * NC, b1 = (long long)c->node_off[sg + 1] * NC;
    const long long len = b1 - b0 >= LARGE_INSTANCE ? CHUNK_LARGE : CHUNK;
    for (long long b = b0; b < b1; b += len) {
      ch.push_back(sg);
      ch.push_back(b);
      ch.push_back(std::min(b1, b + len));
    }
    segch.push_back((int)(ch.size() / 3));
  }
  c->n_chunks = (int)(ch.size() / 3);
  long long clen = 2;
  for (int i = 0; i < c->n_chunks; ++i) clen = std::max(clen, ch[3 * i + 2] - ch[3 * i + 1]);
  c->chunk_len = (int)clen;
  c->max_seg_chunks = 0;
  for (int sg = 0; sg < c->n_seg; ++sg) c->max_seg_chunks = std::max(c->max_seg_chunks, segch[sg + 1] - segch[sg]);
  HIPCHK(c, upload(c, c->cell_nodes, m.cell_nodes.data(), m.cell_nodes.size(), s));
  // node -> (cell * ns + local node) lists in cell order, for the gather of
  // the matrix-free product, and the nodes' range of every MF_RANGE cells
  c->mf_range.clear();
  for (int e = 0; e < m.n_cells; e += glh::MF_RANGE) {
    const auto b = m.cell_nodes.begin() + (size_t)e * ns,
               l = m.cell_nodes.begin() + (size_t)std::min(m.n_cells, e + glh::MF_RANGE) * ns;
    const auto nr = std::minmax_element(b, l);
    c->mf_range.push_back(*nr.first);
    c->mf_range.push_back(*nr.second + 1);
  }
  std::vector<int> n2c_ptr(m.n_nodes + 1, 0), n2c_idx(m.cell_nodes.size());
  for (int v : m.cell_nodes) ++n2c_ptr[v + 1];
  for (int i = 0; i < m.n_nodes; ++i) n2c_ptr[i + 1] += n2c_ptr[i];
  {
    std::vector<int> fill(n2c_ptr.begin(), n2c_ptr.end() - 1);
    for (size_t k = 0; k < m.cell_nodes.size(); ++k) n2c_idx[fill[m.cell_nodes[k]]++] = (int)k;
  }
  HIPCHK(c, upload(c, c->n2c_ptr, n2c_ptr.data(), n2c_ptr.size(), s));
  HIPCHK(c, upload(c, c->n2c_idx, n2c_idx.data(), n2c_idx.size(), s));
  HIPCHK(c, upload(c, c->cell_h, m.cell_h.data(), m.cell_h.size(), s));
  HIPCHK(c, upload(c, c->cell_face, cface.data(), cface.size(), s));
  HIPCHK(c, upload(c, c->node_mask, m.node_mask.data(), m.node_mask.size(), s));
  HIPCHK(c, upload(c, c->row_ptr, m.row_ptr.data(), m.row_ptr.size(), s));
  HIPCHK(c, upload(c, c->col, m.col.data(), m.col.size(), s));
  HIPCHK(c, upload(c, c->diag, diag.data(), diag.size(), s));
  c->cons = glh::ConstraintDev{};
  if (c->constrained) {
    glh::ConstraintDev &C = c->cons;
    C.n_nodes = m.n_nodes;
    C.nnzb = c->nnzb;
    C.n_hang = c->n_hang;
    C.gptr = c->c_gptr.p; C.gsrc = c->c_gsrc.p; C.gw = c->c_gw.p; C.gfl = c->c_gfl.p;
    C.brow = c->c_brow.p; C.col = c->col.p; C.mask = c->node_mask.p; C.diag = c->diag.p;
    C.rptr = c->c_rptr.p; C.rsrc = c->c_rsrc.p; C.rw = c->c_rw.p; C.rfl = c->c_rfl.p;
    C.hnode = c->c_hnode.p; C.hptr = c->c_hptr.p; C.hm = c->c_hm.p; C.hw = c->c_hw.p;
    C.hidx = c->c_hidx.p;
  }
  HIPCHK(c, upload(c, c->cell_blk, cblk.data(), cblk.size(), s));
  HIPCHK(c, upload(c, c->color_cells, m.color_cells.data(), m.color_cells.size(), s));
  HIPCHK(c, upload(c, c->cell_mat, cmat.data(), cmat.size(), s));
  HIPCHK(c, upload(c, c->chunks, ch.data(), ch.size(), s));
  HIPCHK(c, upload(c, c->seg_chunk, segch.data(), segch.size(), s));
  std::vector<int> rseg(m.n_nodes);
  for (int sg = 0; sg < c->n_seg; ++sg)
    for (int r = c->node_off[sg]; r < c->node_off[sg + 1]; ++r) rseg[r] = sg;
  HIPCHK(c, upload(c, c->row_seg, rseg.data(), rseg.size(), s));
  HIPCHK(c, upload(c, c->d_node_off, c->node_off.data(), c->node_off.size(), s));
  const size_t n = (size_t)m.n_nodes * NC;
  HIPCHK(c, take(c, c->U, n));
  HIPCHK(c, take(c, c->dU, n));
  HIPCHK(c, take(c, c->X, n));
  HIPCHK(c, take(c, c->rhs, n));
  HIPCHK(c, take(c, c->res, n));
  HIPCHK(c, take(c, c->Fcell, m.n_cells));
  // the cell slots of the residual (and of the matrix-free product)
  HIPCHK(c, take(c, c->mf_ycell, (size_t)m.n_cells * c->ns * NC));
  HIPCHK(c, hipMemsetAsync(c->U.p, 0, n * sizeof(double), s));
  HIPCHK(c, hipMemsetAsync(c->dU.p, 0, n * sizeof(double), s));
  HIPCHK(c, hipMemsetAsync(c->rhs.p, 0, n * sizeof(double), s));
  HIPCHK(c, hipStreamSynchronize(s));
  c->have_mesh = true;
  c->inst_stats.assign((size_t)c->n_seg * 8, 0.0);
  return GLH_OK;
}

int glh_set_solution(glh_ctx *c, const double *Uh)
{
  RCHK(check_ready(c, false));
  if (!Uh) return fail(c, GLH_ERR_ARG, "null solution");
  HIPCHK(c, hipMemcpyAsync(c->U.p, Uh, ndofs(c) * sizeof(double), hipMemcpyHostToDevice, c->stream));
  // constraints_solution.distribute (setup_uniform_B-phase.cc:262)
  RCHK(distribute(c, c->U.p));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return GLH_OK;
}

int glh_store_initial(glh_ctx *c)
{
  RCHK(check_ready(c, false));
  HIPCHK(c, take(c, c->U0, ndofs(c)));
  HIPCHK(c, hipMemcpyAsync(c->U0.p, c->U.p, ndofs(c) * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return GLH_OK;
}

int glh_restore_initial(glh_ctx *c)
{
  RCHK(check_ready(c, false));
  if (!c->U0.p || c->U0.n < ndofs(c)) return fail(c, GLH_ERR_STATE, "no stored initial state");
  HIPCHK(c, hipMemcpyAsync(c->U.p, c->U0.p, ndofs(c) * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return GLH_OK;
}

int glh_get_solution(glh_ctx *c, double *Uh) { return c ? get_vec(c, c->U.p, Uh) : GLH_ERR_ARG; }
int glh_get_update(glh_ctx *c, double *d) { return c ? get_vec(c, c->dU.p, d) : GLH_ERR_ARG; }
int glh_get_rhs(glh_ctx *c, double *r) { return c ? get_vec(c, c->rhs.p, r) : GLH_ERR_ARG; }

int glh_apply_jacobian(glh_ctx *c, const double *x, double *y)
{
  RCHK(check_ready(c));
  if (!x || !y) return fail(c, GLH_ERR_ARG, "null vector");
  if (!c->j_valid) return fail(c, GLH_ERR_STATE, "no Jacobian assembled");
  const size_t n = ndofs(c);
  HIPCHK(c, take(c, c->gW64, n));
  HIPCHK(c, take(c, c->gZ64, n));
  HIPCHK(c, hipMemcpyAsync(c->gZ64.p, x, n * sizeof(double), hipMemcpyHostToDevice, c->stream));
  if (c->j_fp32) {
    HIPCHK(c, take(c, c->gW32, n));
    HIPCHK(c, take(c, c->gZ32, n));
    HIPCHK(c, (glh::launch_convert<double, float>(n, c->gZ64.p, c->gZ32.p, c->stream)));
    RCHK((apply_j<float, float>(c, c->J32.p, c->gZ32.p, c->gW32.p, nullptr, glh::ActiveSet{})));
    HIPCHK(c, (glh::launch_convert<float, double>(n, c->gW32.p, c->gW64.p, c->stream)));
  } else {
    RCHK((apply_j<double, double>(c, c->J64.p, c->gZ64.p, c->gW64.p, nullptr, glh::ActiveSet{})));
  }
  HIPCHK(c, hipMemcpyAsync(y, c->gW64.p, n * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return GLH_OK;
}

int glh_diagonal_blocks(glh_ctx *c, double *out)
{
  RCHK(check_ready(c, false));
  if (!out) return fail(c, GLH_ERR_ARG, "null output");
  if (!c->j_valid) return fail(c, GLH_ERR_STATE, "no Jacobian assembled");
  const size_t nv = (size_t)c->n_nodes * 324;
  DBuf<double> tmp;
  HIPCHK(c, take(c, tmp, nv));
  if (c->j_mf) HIPCHK(c, glh::launch_gather_blocks<double>(c->n_nodes, c->diag_id.p, c->Jd64.p, tmp.p, c->stream));
  else if (c->j_fp32) HIPCHK(c, glh::launch_gather_blocks<float>(c->n_nodes, c->diag.p, c->J32.p, tmp.p, c->stream));
  else HIPCHK(c, glh::launch_gather_blocks<double>(c->n_nodes, c->diag.p, c->J64.p, tmp.p, c->stream));
  HIPCHK(c, hipMemcpyAsync(out, tmp.p, nv * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return GLH_OK;
}

int glh_apply_block_jacobi(glh_ctx *c, const double *x, double *y)
{
  RCHK(check_ready(c));
  if (!x || !y) return fail(c, GLH_ERR_ARG, "null vector");
  if (!c->j_valid) return fail(c, GLH_ERR_STATE, "no Jacobian assembled");
  RCHK(ensure_precond(c));
  const size_t n = ndofs(c);
  HIPCHK(c, take(c, c->gW64, n));
  HIPCHK(c, take(c, c->gZ64, n));
  HIPCHK(c, hipMemcpyAsync(c->gZ64.p, x, n * sizeof(double), hipMemcpyHostToDevice, c->stream));
  if (c->j_fp32) {  // the FP32 inverses the FP32 inner solve applies, on FP32 vectors
    HIPCHK(c, take(c, c->gW32, n));
    HIPCHK(c, take(c, c->gZ32, n));
    HIPCHK(c, (glh::launch_convert<double, float>(n, c->gZ64.p, c->gZ32.p, c->stream)));
    HIPCHK(c, (glh::launch_bj_apply<float, float>(c->n_nodes, c->D32.p, c->gZ32.p, c->gW32.p, c->stream, nullptr,
                                                  nullptr, glh::ActiveSet{})));
    HIPCHK(c, (glh::launch_convert<float, double>(n, c->gW32.p, c->gW64.p, c->stream)));
  } else {
    HIPCHK(c, (glh::launch_bj_apply<double, double>(c->n_nodes, c->D64.p, c->gZ64.p, c->gW64.p, c->stream, nullptr,
                                                    nullptr, glh::ActiveSet{})));
  }
  HIPCHK(c, hipMemcpyAsync(y, c->gW64.p, n * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return GLH_OK;
}

int glh_get_jacobian(glh_ctx *c, double *val)
{
  RCHK(check_ready(c, false));
  if (!c->j_valid) return fail(c, GLH_ERR_STATE, "no Jacobian assembled");
  if (c->j_mf) return fail(c, GLH_ERR_STATE, "the last Jacobian is matrix-free: no assembled values (glh_assemble)");
  const size_t nv = (size_t)c->nnzb * 324;
  if (c->j_upper && c->j_fp32)
    HIPCHK(c, glh::launch_sym_fill<float>(c->n_nodes, c->row_ptr.p, c->diag.p, c->sym_lo.p, c->J32.p, c->stream));
  else if (c->j_upper)
    HIPCHK(c, glh::launch_sym_fill<double>(c->n_nodes, c->row_ptr.p, c->diag.p, c->sym_lo.p, c->J64.p, c->stream));
  if (!c->j_fp32) {
    HIPCHK(c, hipMemcpyAsync(val, c->J64.p, nv * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
  } else {
    std::vector<float> tmp(nv);
    HIPCHK(c, hipMemcpyAsync(tmp.data(), c->J32.p, nv * sizeof(float), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    for (size_t i = 0; i < nv; ++i) val[i] = tmp[i];
  }
  return GLH_OK;
}

int glh_assemble(glh_ctx *c, int flags)
{
  RCHK(check_ready(c));
  const bool dj = flags & GLH_ASM_J, dr = flags & GLH_ASM_R, f32 = flags & GLH_ASM_FP32;
  const bool mf = flags & GLH_ASM_MATRIX_FREE;
  if (!dj && !dr) return fail(c, GLH_ERR_ARG, "nothing to assemble");
  if (mf && !dj) return fail(c, GLH_ERR_ARG, "the matrix-free form is a Jacobian form");
  RCHK(assemble_at(c, c->U.p, dj, dr, f32, c->rhs.p, true, mf));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return GLH_OK;
}

int glh_rhs_norm(glh_ctx *c, double *nrm)
{
  RCHK(check_ready(c));
  return norm64(c, c->rhs.p, nrm);
}

int glh_residual(glh_ctx *c, double *nrm)
{
  RCHK(check_ready(c));
  std::vector<double> r2;
  RCHK(residual_norms(c, c->U.p, c->res.p, r2));
  double t = 0;
  for (double x : r2) t += x;
  *nrm = std::sqrt(t);
  return GLH_OK;
}

int glh_residual_into(glh_ctx *c, const double *U, double *R, double *norm2)
{
  RCHK(check_ready(c));
  if (!U || !R || !norm2) return fail(c, GLH_ERR_ARG, "null device pointer");
  if ((long long)c->n_chunks > glh::SCRATCH_DOUBLES)
    return fail(c, GLH_ERR_ARG,
                "the mesh needs " + std::to_string(c->n_chunks) + " reduction chunks; glh_residual_into holds " +
                    std::to_string(glh::SCRATCH_DOUBLES) + " (use glh_residual)");
  // the residual at U into R (through the context's cell slots, allocated
  // with the mesh) and per-instance ||R_s||^2 with the chunk partials in the
  // scratch array
  return residual_cells(c, U, R, c->scratch, norm2);
}

int glh_solve(glh_ctx *c, double rtol, int maxit, int restart, double stats[2])
{
  RCHK(check_ready(c));
  return solve_impl(c, std::vector<double>(c->n_seg, rtol), maxit, restart, stats, nullptr);
}

int glh_newton_step(glh_ctx *c, double step, int damped, double out[4])
{
  RCHK(check_ready(c));
  if (damped && !(step > 0 && step < 1)) return fail(c, GLH_ERR_ARG, "line-search step must be in (0,1)");
  std::vector<double> prev, cur, alpha;
  std::vector<int> trials;
  RCHK(newton_step_impl(c, step, damped, std::vector<char>(c->n_seg, 1), prev, cur, alpha, trials));
  if (out) {
    double p2 = 0, c2 = 0;
    for (int i = 0; i < c->n_seg; ++i) { p2 += prev[i] * prev[i]; c2 += cur[i] * cur[i]; }
    out[0] = std::sqrt(p2);
    out[1] = std::sqrt(c2);
    out[2] = alpha[0];
    out[3] = *std::max_element(trials.begin(), trials.end());
  }
  return GLH_OK;
}

int glh_free_energy(glh_ctx *c, double *F)
{
  RCHK(check_ready(c));
  if (!F) return fail(c, GLH_ERR_ARG, "null output");
  std::vector<double> f;
  RCHK(instance_energy(c, f));
  double t = 0;
  for (double v : f) t += v;
  *F = t;
  return GLH_OK;
}

int glh_instance_energy(glh_ctx *c, double *F)
{
  RCHK(check_ready(c));
  if (!F) return fail(c, GLH_ERR_ARG, "null output");
  std::vector<double> f;
  RCHK(instance_energy(c, f));
  std::copy(f.begin(), f.end(), F);
  return GLH_OK;
}

int glh_instance_residuals(glh_ctx *c, double *R)
{
  RCHK(check_ready(c));
  if (!R) return fail(c, GLH_ERR_ARG, "null output");
  std::vector<double> r2;
  RCHK(residual_norms(c, c->U.p, c->res.p, r2));
  for (int i = 0; i < c->n_seg; ++i) R[i] = std::sqrt(r2[i]);
  return GLH_OK;
}

int glh_newton_solve(glh_ctx *c, double rtol, int max_newton, double lin_tol, int lin_maxit, int restart,
                     double ls_step, int damped, int fp32, double stats[10])
{
  RCHK(check_ready(c));
  if (!(rtol >= 0) || max_newton < 0 || !(lin_tol > 0) || lin_maxit < 1 || (damped && !(ls_step > 0 && ls_step < 1)))
    return fail(c, GLH_ERR_ARG, "bad Newton controls (rtol >= 0, max_newton >= 0, lin_tol > 0, lin_maxit >= 1, "
                                "line-search step in (0,1))");
  if (restart <= 0) restart = c->tuned_restart;
  // the instance filter of the assembly lives only inside this solve
  struct FilterReset {
    glh_ctx *c;
    ~FilterReset() { c->asm_active = nullptr; }
  } filter_reset{c};
  const int S = c->n_seg;
  double t_asm = 0, t_sol = 0, t_ls = 0;
  int lin_total = 0, k = 0, trials_total = 0;
  const double t_start = now_s();
  double t0 = t_start;
  std::vector<double> r0(S), rcur(S), r2;
  RCHK(residual_norms(c, c->U.p, c->rhs.p, r2));
  for (int i = 0; i < S; ++i) r0[i] = rcur[i] = std::sqrt(r2[i]);
  t_asm += now_s() - t0;
  std::vector<double> &st = c->inst_stats;
  st.assign((size_t)S * 8, 0.0);
  for (int i = 0; i < S; ++i) { st[8 * i + 2] = r0[i]; st[8 * i + 4] = -1.0; }
  std::vector<char> active(S), stalled(S, 0);
  HIPCHK(c, take(c, c->s_flag, S));
  const bool f32 = fp32 != 0;
  // the matrix-free operator when switched on (FP64 or FP32, with or without
  // the continuation shift; a batch, or one instance on a constrained mesh);
  // the assembled BSR Jacobian otherwise
  const bool mf = c->matfree && !(c->constrained && S > 1);
  std::vector<int> flag(S);
  // batches only: an instance whose ||R|| has fallen by less than 10% over the
  // last STALL_WINDOW steps is stopped and reported as not converged, so that
  // it cannot hold the others in lockstep until max_newton
  constexpr int STALL_WINDOW = 10;
  std::vector<double> hist;  // [k][S] ||R|| after step k
  hist.insert(hist.end(), rcur.begin(), rcur.end());
  // stopping reference: ||R0|| of this solve, or the caller's per-instance norms
  std::vector<double> rref = r0;
  if ((int)c->r_ref.size() == S) rref = c->r_ref;
  std::vector<double> rprev(S, 0.0), eta_prev(S, lin_tol);
  for (k = 0; k <= max_newton; ++k) {
    bool any = false;
    const double tnow = now_s() - t_start;
    for (int i = 0; i < S; ++i) {
      if (S > 1 && k >= STALL_WINDOW && rcur[i] > rtol * rref[i] &&
          rcur[i] > 0.9 * hist[(size_t)(k - STALL_WINDOW) * S + i])
        stalled[i] = 1;
      active[i] = !stalled[i] && rcur[i] > rtol * rref[i];
      if (!active[i] && st[8 * i + 4] < 0) st[8 * i + 4] = tnow;
      any = any || active[i];
    }
    if (!any || k == max_newton) break;
    t0 = now_s();
    // finished instances are skipped by the assembly kernels from here on:
    // their rows keep the last Jacobian and get a zero right-hand side
    // (a buffer of its own: solve_impl reuses s_flag for its refinement sweeps)
    for (int i = 0; i < S; ++i) flag[i] = active[i];
    HIPCHK(c, take(c, c->asm_flag, S));
    HIPCHK(c, c->pin_fl.alloc(S));
    HIPCHK(c, hipStreamSynchronize(c->stream));  // the pinned flags of the last step are no longer read
    std::copy(flag.begin(), flag.end(), c->pin_fl.p);
    HIPCHK(c, hipMemcpyAsync(c->asm_flag.p, c->pin_fl.p, S * sizeof(int), hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipMemcpyAsync(c->s_flag.p, c->pin_fl.p, S * sizeof(int), hipMemcpyHostToDevice, c->stream));
    c->asm_active = S > 1 ? c->asm_flag.p : nullptr;
    RCHK(assemble_at(c, c->U.p, true, true, f32, c->rhs.p, false, mf));
    // pseudo-transient continuation: J + sigma_k |diag J|, sigma_k =
    // sigma0 ||R_k|| / ||R_0|| per instance (switched evolution relaxation)
    if (c->ptc_sigma0 > 0) {
      HIPCHK(c, c->pin64.alloc(S));
      HIPCHK(c, hipStreamSynchronize(c->stream));
      double *sg = c->pin64.p;  // pinned: the copy below is asynchronous
      for (int i = 0; i < S; ++i) sg[i] = active[i] ? c->ptc_sigma0 * rcur[i] / std::max(r0[i], 1e-300) : 0.0;
      HIPCHK(c, take(c, c->s_norm, S));
      HIPCHK(c, hipMemcpyAsync(c->s_norm.p, sg, S * sizeof(double), hipMemcpyHostToDevice, c->stream));
      if (mf) {  // on the diagonal blocks, and as a diagonal term of the product
        HIPCHK(c, take(c, c->mf_sh, ndofs(c)));
        HIPCHK(c, glh::launch_mf_shift(c->n_nodes, c->node_mask.p, c->row_seg.p, c->s_norm.p, c->Jd64.p, c->mf_sh.p,
                                       c->stream));
        c->mf_sh_on = true;
      } else if (f32)
        HIPCHK(c, glh::launch_diag_shift<float>(c->n_nodes, c->diag.p, c->node_mask.p, c->row_seg.p, c->s_norm.p,
                                                c->J32.p, c->stream));
      else
        HIPCHK(c, glh::launch_diag_shift<double>(c->n_nodes, c->diag.p, c->node_mask.p, c->row_seg.p, c->s_norm.p,
                                                 c->J64.p, c->stream));
      HIPCHK(c, hipStreamSynchronize(c->stream));
    }
    // frozen instances see a zero right-hand side, so GMRES leaves them at dU = 0
    HIPCHK(c, glh::launch_seg_zero<double>(c->seg(), c->s_flag.p, c->rhs.p, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    const double t1 = now_s();
    t_asm += t1 - t0;
    double sst[2] = {0, 0};
    std::vector<int> its_seg;
    // an inexact solve that hit lin_maxit still gives a usable update: the
    // line search below decides whether it lowers ||R||
    // forcing terms: the fixed lin_tol of the reference (solve.cc:119-128), or
    // Eisenstat-Walker (choice 2, gamma 0.9, alpha 2) capped at lin_tol
    std::vector<double> eta(S, lin_tol);
    if (c->ew_forcing)
      for (int i = 0; i < S; ++i) {
        if (k == 0 || !(rprev[i] > 0)) continue;
        double e = 0.9 * (rcur[i] / rprev[i]) * (rcur[i] / rprev[i]);
        const double safe = 0.9 * eta_prev[i] * eta_prev[i];
        if (safe > 0.1) e = std::max(e, safe);
        // no tighter than needed to reach the stopping test this step
        e = std::max(e, 0.5 * rtol * rref[i] / std::max(rcur[i], 1e-300));
        eta[i] = std::min(lin_tol, std::max(e, 1e-8));
      }
    eta_prev = eta;
    const int src = solve_impl(c, eta, lin_maxit, restart, sst, &its_seg);
    if (src == GLH_ERR_NOCONV) {
      RCHK(distribute(c, c->dU.p));
    } else if (src) {
      return src;
    }
    if (its_seg.size() != (size_t)S) its_seg.assign(S, 0);
    lin_total += (int)sst[0];
    const double t2 = now_s();
    t_sol += t2 - t1;
    std::vector<double> prev, cur, alpha;
    std::vector<int> trials;
    RCHK(newton_step_impl(c, ls_step, damped, active, prev, cur, alpha, trials));
    for (int i = 0; i < S; ++i)
      if (active[i]) {
        rprev[i] = rcur[i];
        rcur[i] = cur[i];
        st[8 * i + 0] += 1;
        st[8 * i + 6] += trials[i];
        st[8 * i + 7] += its_seg[i];
      }
    trials_total += *std::max_element(trials.begin(), trials.end());
    hist.insert(hist.end(), rcur.begin(), rcur.end());
    t_ls += now_s() - t2;
    if (c->verbose) {
      int na = 0;
      double rmax = 0;
      for (int i = 0; i < S; ++i)
        if (active[i]) {
          ++na;
          rmax = std::max(rmax, rcur[i] / std::max(r0[i], 1e-300));
        }
      int ns = 0;
      for (int i = 0; i < S; ++i) ns += stalled[i];
      fprintf(stderr, "glhip: newton %d: %d active, %d stalled, worst ||R||/||R0|| %.3e, gmres %d%s, %.2f s\n", k + 1,
              na, ns, rmax, (int)sst[0], src == GLH_ERR_NOCONV ? " (maxit)" : "", now_s() - t_start);
      fflush(stderr);
    }
  }
  std::vector<double> F;
  RCHK(instance_energy(c, F));
  bool all = true;
  double r0t = 0, rft = 0, Ft = 0;
  for (int i = 0; i < S; ++i) {
    const bool ok = rcur[i] <= rtol * rref[i];
    all = all && ok;
    st[8 * i + 1] = ok ? 1.0 : 0.0;
    st[8 * i + 3] = rcur[i];
    st[8 * i + 5] = F[i];
    r0t += r0[i] * r0[i];
    rft += rcur[i] * rcur[i];
    Ft += F[i];
  }
  if (stats) {
    stats[0] = k; stats[1] = lin_total; stats[2] = std::sqrt(r0t); stats[3] = std::sqrt(rft);
    stats[4] = t_asm; stats[5] = t_sol; stats[6] = t_ls; stats[7] = Ft;
    stats[8] = trials_total; stats[9] = all ? 1.0 : 0.0;
  }
  return GLH_OK;
}

int glh_instance_stats(glh_ctx *c, double *out)
{
  if (!c || !out) return GLH_ERR_ARG;
  std::copy(c->inst_stats.begin(), c->inst_stats.end(), out);
  return GLH_OK;
}

int glh_last_assembly_ms(glh_ctx *c, double ms[2])
{
  if (!c || !ms) return GLH_ERR_ARG;
  ms[0] = c->asm_ms;
  ms[1] = c->asm_launches;
  return GLH_OK;
}

int glh_set_schedule(glh_ctx *c, int restart, int q_block, int row_cap, int chunk_cap, int gs_tile)
{
  if (!c || restart < 1 || restart > 126 || q_block < 0 || row_cap < 0 || chunk_cap < 0) return GLH_ERR_ARG;
  if (gs_tile != 0 && gs_tile != 4 && gs_tile != 8 && gs_tile != 16) return GLH_ERR_ARG;
  c->tuned_restart = restart;
  c->q_block = q_block;
  c->row_cap = row_cap;
  c->chunk_cap = chunk_cap;
  c->gs_tile = gs_tile ? gs_tile : 8;
  return GLH_OK;
}

int glh_set_reorth(glh_ctx *c, double ratio)
{
  if (!c || !(ratio >= 0.0) || !std::isfinite(ratio)) return GLH_ERR_ARG;
  c->dgks = ratio;
  drop_graphs(c);  // recorded control ops carry the ratio by value
  return GLH_OK;
}

int glh_autotune(glh_ctx *c, int fp32, int trial_newton, double lin_tol, int lin_maxit, double out[7])
{
  RCHK(check_ready(c));
  if (trial_newton < 1 || trial_newton > 8 || !(lin_tol > 0) || lin_maxit < 1 || !out)
    return fail(c, GLH_ERR_ARG, "bad autotune parameters");
  struct Cand {
    int m, q, rc, cc, gs;
  };
  RCHK(glh_store_initial(c));
  const int old_verbose = c->verbose;
  c->verbose = 0;
  int rc = GLH_OK, tried = 0;
  // one untimed step records the candidate's graphs, then the timed trial
  auto trial = [&](const Cand &k, double tol, double &t) {
    c->q_block = k.q;
    c->row_cap = k.rc;
    c->chunk_cap = k.cc;
    c->gs_tile = k.gs;
    double st[10];
    ++tried;
    if ((rc = glh_restore_initial(c)) != GLH_OK) return;
    if ((rc = glh_newton_solve(c, 1e-300, 1, tol, lin_maxit, k.m, 0.83, 1, fp32, st)) != GLH_OK) return;
    if ((rc = glh_restore_initial(c)) != GLH_OK) return;
    const double t0 = now_s();
    if ((rc = glh_newton_solve(c, 1e-300, trial_newton, tol, lin_maxit, k.m, 0.83, 1, fp32, st)) != GLH_OK) return;
    t = now_s() - t0;
  };
  // The restart length is not tuned: it changes the Krylov iteration, and
  // a trial of a few Newton steps does not predict its effect on the later,
  // harder linear systems of a solve (measured on 256 slabs: short trials
  // picked restart 30 or 60, and the full solve then took up to 2.7x as long
  // as with 100).  The candidates leave the arithmetic as it is: the launch
  // schedule of a batch (Arnoldi steps per replayed graph block, grid caps),
  // then, with the best schedule, the Gram-Schmidt tile (basis vectors per
  // multi-dot workgroup, loads in flight per update thread; every tile sums in
  // the same order, so the iterates are the same bits).
  const bool batch = c->n_seg > 1;
  const int m = c->tuned_restart;
  Cand best{m, batch ? 8 : 0, batch ? 8192 : 0, batch ? 2048 : 0, 8};
  double tbest = 1e300;
  // a candidate replaces the best so far only when it is faster by more than
  // 2% (shorter differences are within the run-to-run spread of a trial)
  auto consider = [&](const Cand &k) {
    double t = 1e300;
    trial(k, lin_tol, t);
    if (!rc && t < 0.98 * tbest) {
      tbest = t;
      best = k;
    }
  };
  if (batch) {
    for (int q : {4, 8, 16}) {
      for (int cap : {2048, 8192}) {
        consider(Cand{m, q, cap, cap / 4, 8});
        if (rc) break;
      }
      if (rc) break;
    }
  } else {
    consider(best);
  }
  for (int gs : {4, 16}) {
    if (rc) break;
    Cand k = best;
    k.gs = gs;
    consider(k);
  }
  c->verbose = old_verbose;
  c->tuned_restart = best.m;
  c->q_block = best.q;
  c->row_cap = best.rc;
  c->chunk_cap = best.cc;
  c->gs_tile = best.gs;
  RCHK(rc);
  RCHK(glh_restore_initial(c));
  out[0] = best.m; out[1] = best.q; out[2] = best.rc; out[3] = best.cc; out[4] = tbest;
  out[5] = (double)tried;
  out[6] = best.gs;
  return GLH_OK;
}

int glh_set_forcing(glh_ctx *c, int eisenstat_walker)
{
  if (!c) return GLH_ERR_ARG;
  c->ew_forcing = eisenstat_walker != 0;
  return GLH_OK;
}

int glh_set_residual_reference(glh_ctx *c, int n, const double *r_ref)
{
  if (!c || n < 0 || (n > 0 && !r_ref)) return GLH_ERR_ARG;
  c->r_ref.assign(r_ref, r_ref + n);
  for (double r : c->r_ref)
    if (!(r > 0)) {
      c->r_ref.clear();
      return fail(c, GLH_ERR_ARG, "reference residual norms must be positive");
    }
  return GLH_OK;
}

int glh_set_matrix_free(glh_ctx *c, int on)
{
  if (!c) return GLH_ERR_ARG;
  c->matfree = on != 0;
  return GLH_OK;
}

int glh_set_continuation(glh_ctx *c, double sigma0)
{
  if (!c || !(sigma0 >= 0.0)) return GLH_ERR_ARG;
  c->ptc_sigma0 = sigma0;
  return GLH_OK;
}

int glh_set_verbose(glh_ctx *c, int level)
{
  if (!c) return GLH_ERR_ARG;
  c->verbose = level;
  return GLH_OK;
}

int glh_set_timing(glh_ctx *c, int on)
{
  if (!c) return GLH_ERR_ARG;
  HIPCHK(c, hipSetDevice(c->device));
  if (on && c->ev_pool.empty()) {
    c->ev_pool.resize(2 * 1024, nullptr);
    for (auto &e : c->ev_pool) HIPCHK(c, hipEventCreate(&e));
  }
  c->timing = on != 0;
  c->ev_used = 0;
  c->spmv_ms_total = c->spmv_count = 0;
  c->jasm_ms_total = c->jasm_count = c->rasm_ms_total = c->rasm_count = 0;
  return GLH_OK;
}

int glh_timing(glh_ctx *c, double out[6])
{
  if (!c || !out) return GLH_ERR_ARG;
  RCHK(flush_events(c));
  out[0] = c->spmv_ms_total; out[1] = c->spmv_count;
  out[2] = c->jasm_ms_total; out[3] = c->jasm_count;
  out[4] = c->rasm_ms_total; out[5] = c->rasm_count;
  return GLH_OK;
}

int glh_bench_spmv(glh_ctx *c, int k, double *ms_avg)
{
  RCHK(check_ready(c));
  if (!c->j_valid || k < 1 || !ms_avg) return fail(c, GLH_ERR_STATE, "no Jacobian assembled");
  if (c->j_fp32) {
    HIPCHK(c, take(c, c->gW32, ndofs(c)));
    HIPCHK(c, take(c, c->gZ32, ndofs(c)));
    HIPCHK(c, (glh::launch_convert<double, float>(ndofs(c), c->U.p, c->gZ32.p, c->stream)));
  }
  HIPCHK(c, hipEventRecord(c->ev0, c->stream));
  for (int i = 0; i < k; ++i) {
    if (c->j_fp32)
      RCHK((apply_j<float, float>(c, c->J32.p, c->gZ32.p, c->gW32.p, nullptr, glh::ActiveSet{})));
    else
      RCHK((apply_j<double, double>(c, c->J64.p, c->U.p, c->res.p, nullptr, glh::ActiveSet{})));
  }
  HIPCHK(c, hipEventRecord(c->ev1, c->stream));
  HIPCHK(c, hipEventSynchronize(c->ev1));
  float ms = 0;
  HIPCHK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
  *ms_avg = ms / k;
  return GLH_OK;
}

int glh_bench_read(glh_ctx *c, size_t nbytes, int k, double *ms_avg)
{
  if (!c || !ms_avg || k < 1 || nbytes % 16 || nbytes == 0) return GLH_ERR_ARG;
  HIPCHK(c, hipSetDevice(c->device));
  constexpr int grid = 1024;
  DBuf<unsigned char> a;
  DBuf<float> out;
  hipError_t e = take(c, a, nbytes);
  if (e == hipSuccess) e = take(c, out, (size_t)grid * 256);
  if (e == hipSuccess) e = hipMemsetAsync(a.p, 0, nbytes, c->stream);
  if (e == hipSuccess) e = hipEventRecord(c->ev0, c->stream);
  for (int i = 0; i < k && e == hipSuccess; ++i) e = glh::launch_read(nbytes, a.p, out.p, grid, c->stream);
  if (e == hipSuccess) e = hipEventRecord(c->ev1, c->stream);
  if (e == hipSuccess) e = hipEventSynchronize(c->ev1);
  float ms = 0;
  if (e == hipSuccess) e = hipEventElapsedTime(&ms, c->ev0, c->ev1);
  a.release();
  out.release();
  if (e != hipSuccess) return fail(c, GLH_ERR_HIP, std::string("read benchmark: ") + hipGetErrorString(e));
  *ms_avg = ms / k;
  return GLH_OK;
}

int glh_bench_copy(glh_ctx *c, size_t nbytes, int k, double *ms_avg)
{
  if (!c || !ms_avg || k < 1 || nbytes % 16 || nbytes == 0) return GLH_ERR_ARG;
  HIPCHK(c, hipSetDevice(c->device));
  DBuf<unsigned char> a, b;
  hipError_t e = take(c, a, nbytes);
  if (e == hipSuccess) e = take(c, b, nbytes);
  if (e == hipSuccess) e = hipMemsetAsync(a.p, 0, nbytes, c->stream);
  if (e == hipSuccess) e = hipEventRecord(c->ev0, c->stream);
  for (int i = 0; i < k && e == hipSuccess; ++i) e = glh::launch_copy(nbytes, a.p, b.p, c->stream);
  if (e == hipSuccess) e = hipEventRecord(c->ev1, c->stream);
  if (e == hipSuccess) e = hipEventSynchronize(c->ev1);
  float ms = 0;
  if (e == hipSuccess) e = hipEventElapsedTime(&ms, c->ev0, c->ev1);
  a.release();
  b.release();
  if (e != hipSuccess) return fail(c, GLH_ERR_HIP, std::string("copy benchmark: ") + hipGetErrorString(e));
  *ms_avg = ms / k;
  return GLH_OK;
}

}  // extern "C"
