// HIP kernels of the hex8 solve path (gfx950) and their host launchers.
//
// Data layout in HBM (one multigrid level):
//   * vectors: node-major, 3 dofs interleaved (u_x, u_y, u_z) per independent
//     node, nodes in forest order (Morton order of the node positions);
//   * elements are processed in batches of up to 256 consecutive (Morton
//     order) elements of one stiffness class; a batch stages the distinct
//     nodes it touches ("slots") in LDS.  Slot ids are global:
//     wg_node_ptr[b] .. wg_node_ptr[b+1] belong to batch b;
//   * element -> slot connectivity is 8 x uint16 local indices per element;
//   * the element pass writes one partial sum per slot; the assembly pass
//     gathers, for every independent node, its slots (weight 1) and the slots
//     of the hanging nodes that depend on it (hanging-node weight), so there
//     are no atomics and the summation order is fixed.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace tmrx {

constexpr int WG_ELEMS = 256;
constexpr int MAX_COLORS = 32;

// launch errors: noted after every launch, reported by the next
// synchronising call of the problem
void note_launch(hipError_t e);
hipError_t take_launch_error();
#define TMRX_LAUNCH_CHECK() ::tmrx::note_launch(hipGetLastError())

struct ElemBatches {
  int n_wg = 0;
  int n_elem = 0;
  int ncolors = 0;
  int max_wg_nodes = 0;
  const int *wg_node_ptr = nullptr;  // [n_wg + 1]
  const int *wg_nodes = nullptr;     // [nslots]: >= 0 node, < 0 -(hanging + 1)
  const int *wg_elem_ptr = nullptr;  // [n_wg + 1]
  const int *wg_class = nullptr;     // [n_wg]
  const uint16_t *lconn = nullptr;   // [n_elem * 8]
  const uint8_t *color = nullptr;    // [n_elem]
  const int4 *dep4 = nullptr;        // hanging nodes' parents (load_node)
  const uint8_t *bcmask = nullptr;   // [n_nodes], bit d set = dof d clamped
};

// Owner tiles: tile t owns the contiguous independent nodes
// [node0[t], node0[t+1]) and holds every element touching them (or touching a
// hanging node one of them supports).  LDS slots: owned nodes, then the
// hanging nodes whose sums the tile needs ("accumulated"), then halo nodes.
constexpr int TILE_NODES = 512;
constexpr int MFMA_WAVES = 4;  // waves of a matrix-core tile, each owning a share of its nodes
constexpr int TILE_THREADS = 256;

// LDS position of tile slot s: an XOR of higher bits into the low three bits
// (a permutation inside each aligned group of 8), so that the corner slots of
// same-colour elements -- Morton strides of 8, 64, 512 -- spread over banks.
__host__ __device__ inline int tile_pos(int s) {
  return s ^ (((s >> 3) ^ (s >> 6) ^ (s >> 9)) & 7);
}
inline int round8(int n) { return (n + 7) & ~7; }

struct TileElem {       // 24 bytes
  uint16_t lc[8];       // LDS slot of each corner
  int32_t elem;         // global element index (stiffness scale)
  uint8_t mask;         // corners whose slot is accumulated
  uint8_t color;        // conflict-free accumulation phase
  uint8_t cls;          // stiffness class
  uint8_t pad;
};
static_assert(sizeof(TileElem) == 24, "tile element record is 24 bytes");

struct Tiles {
  int n_tiles = 0;
  bool single_class = true;
  int max_slots = 0, max_acc = 0;
  int max_rec = 0, max_mrec = 0;  // records per tile (plain, matrix-core padded)
  int ncolors = 0;
  const int *node0 = nullptr;     // [n_tiles + 1]
  // slots: owned, then the hanging ones (accumulated first) by the LDS
  // positions of their parents (four uint16: two parents of weight 1/2, third
  // 0xffff, or four of 1/4), then the halo nodes (those corners and parents
  // of the tile that it does not own), clamped dofs in the top three bits
  const int *extd_ptr = nullptr;  // [n_tiles + 1]
  const uint2 *extd = nullptr;
  const int *ext_ptr = nullptr;   // [n_tiles + 1]
  const uint32_t *ext = nullptr;
  bool masked = true;             // false: every dof free (bcmask all zero)
  const int *nacc_dep = nullptr;  // [n_tiles] accumulated hanging slots
  const int *el_ptr = nullptr;    // [n_tiles + 1]
  const TileElem *el = nullptr;
  // the same records for the FP32 element-density apply, with the element
  // word holding the element's FP32 scale (refreshed with the design)
  TileElem *el32 = nullptr;
  const int *el_elem = nullptr;  // element of each record
  int n_rec = 0;
  // owned node <- hanging slots of its tile, groups of four packed entries:
  // LDS position | 2^16 (weight 1/2) or 2^17 (weight 1/4), 0 pads
  const int *comb_ptr = nullptr;  // [n_nodes + 1] in groups
  const uint4 *comb = nullptr;
  const uint8_t *bcmask = nullptr;
  // matrix-core (FP32) form: per tile and wave, records of the elements
  // touching the wave's share of the nodes, in batches of 16 of one colour
  // and class (padded with mask-0 records); K0 of every class split into
  // bf16 hi/mid/lo MFMA A fragments
  const int *mb_ptr = nullptr;    // [n_tiles * (MFMA_WAVES + 1)] batch offsets
  TileElem *mel = nullptr;        // [16 * batches]; elem word holds the FP32 scale
  const int *mel_elem = nullptr;  // [16 * batches] element of each record
  int n_mrec = 0;
  const uint4 *afrag = nullptr;   // [n_classes][hi, lo][row block][64 lanes]
  // FP32-input matrix-core form: K0 fragments [n_classes][row block][step][64]
  const float *afrag32 = nullptr;
  bool use_mfma = false;
  bool mfma_f32 = false;  // matrix cores with FP32 inputs (else bf16 three-way split)
  // nodal design: the element stiffness is sum_g s_eg K_g over the 8 Gauss
  // points (K0 holds the gradient tables, s_elem 8 scales per element)
  bool nodal = false;
  // threads per tile of the vector-ALU form (256 or 512)
  int threads = TILE_THREADS;
  // when set, launches return at once while *run == 0 (no segment of a
  // batched solve is still running)
  const int *run = nullptr;
};

// Per stiffness class, the nodal-design element tables: dN_a/dx_d at the 8
// Gauss points of the full-block element (G[24 g + 3 a + d], 192 entries),
// then lambda and mu times the Gauss weight |J| (= volume / 8), then 2 pads.
constexpr int NODAL_TABLE = 196;
// Per stiffness class, the element stiffness in the reflection-symmetric
// basis: 8 blocks of 3 x 3 (row-major), block s coupling the Walsh-Hadamard
// coefficients X_0[s^1], X_1[s^2], X_2[s^4], scaled by 1/64.  The
// element-density tile apply takes this table in place of K0.
constexpr int REFL_TABLE = 72;
// Structural non-zeros of those blocks (bit 3 r + c for row r, column c of
// block s) for a box element of an isotropic material, any aspect ratio:
// the rigid translations X_0[0], X_1[0], X_2[0] span the null rows and
// columns of blocks 1, 2 and 4, and blocks 3, 5 and 6 decouple one of their
// three coefficients.  45 of the 72 entries remain.
constexpr unsigned short REFL_NZ[8] = {0x1FF, 0x1B0, 0x145, 0x11B, 0x01B, 0x155, 0x1B1, 0x1FF};
__host__ __device__ constexpr bool refl_nz(int s, int k) { return (REFL_NZ[s] >> k) & 1; }


struct AsmCSR {
  int n_nodes = 0;
  const int *ptr = nullptr;   // [n_nodes + 1]
  const int *slot = nullptr;  // [nnz]
  const float *w = nullptr;   // [nnz]
};

struct TransferCSR {  // rows = output nodes
  int n_rows = 0;
  const int *ptr = nullptr;
  const int *col = nullptr;
  const float *w = nullptr;
  const int *run = nullptr;  // as Tiles::run
  // per fine node: 1 + e when its prolongation row has 2^e equal weights
  // 2^-e (the weights are then not read), 0 otherwise; indexed by row for
  // P and by column for R = P^T
  const uint8_t *wexp = nullptr;
};

// y-side operation performed by the assembly pass
enum AsmMode {
  ASM_STORE = 0,   // y = A x
  ASM_RESID = 1,   // y = b - A x
  ASM_CHEB = 2,    // r = b - A x; d = a d + c Dinv r; x += d
  ASM_DIAG = 3,    // Dinv = 1 / diag(A)   (partials hold element diagonals)
  ASM_DOT = 4,     // y = A x and block partials of x . y
  ASM_GATHER = 5,  // y = sum of the slot partials (clamped rows zero): Z^T g
  ASM_POWER = 6,   // y = Dinv A x (power iteration)
  ASM_CHEBDOT = 7, // ASM_CHEB and per-tile partials of x_out . dr, x_out . dq
};

// Chebyshev-step flags: read the previous direction d, take d = x (the step
// after a first step from a zero guess, where x = d), store the new d
enum { CHEB_D_READ = 1, CHEB_D_IS_X = 2, CHEB_D_STORE = 4 };

struct AsmArgs {
  const void *b = nullptr;
  void *y = nullptr;
  void *x = nullptr;       // input of the product (read) or iterate (CHEB)
  void *x_out = nullptr;   // CHEB iterate output of the tile kernel
  void *d = nullptr;       // Chebyshev direction
  const void *dinv = nullptr;
  // ASM_CHEB: device pair (a, c) of the step in the vectors' type, so that a
  // captured iteration outlives a new set-up's eigenvalue bounds
  const void *cf = nullptr;
  int cflags = CHEB_D_READ | CHEB_D_STORE;  // tile apply, ASM_CHEB
  double *partials = nullptr;
  const double *dr = nullptr, *dq = nullptr;  // ASM_CHEBDOT
};

// single-pass apply with fused epilogue (modes as AsmMode, except ASM_DIAG);
// K0 is the REFL_TABLE table (element densities) or the NODAL_TABLE table
// (tl.nodal) on the vector ALUs, unused by the matrix-core form
template <class T>
void launch_tile_apply(const Tiles &tl, const T *K0, const T *s_elem, const T *x, int mode,
                       const AsmArgs &args, hipStream_t st, int nrhs = 1, int64_t vs = 0);
template <class T>
void launch_elem_diag(const ElemBatches &eb, const T *K0, const T *s_elem, T *partial,
                      hipStream_t st, bool nodal = false);
// Dinv of the nodes with corner-pair terms: dinv = 1 / (1 / dinv + sum_k
// w_k K_e[a][b]) per direction, K_e = s_e K0[cls] (element design) or
// sum_g s_g K_g (nodal design, K0 the NODAL_TABLE tables); clamped dofs kept
void launch_diag_cross(int n, const int *ptr, const int *node, const int *code, const double *w,
                       const int *cls, const double *K0, const double *s, bool nodal,
                       const uint8_t *bcmask, double *dinv, hipStream_t st);
void launch_assemble(const AsmCSR &a, const uint8_t *bcmask, const double *partial, int mode,
                     double *y, hipStream_t st);
int assemble_num_blocks(int n_nodes);

template <class T>
void launch_prolong_add(const TransferCSR &P, const uint8_t *bcmask_f, const T *xc, T *xf,
                        hipStream_t st, int nrhs = 1, int64_t vsc = 0, int64_t vsf = 0);
// rc = R rf (clamped rows zero); with x1, also the coarse level's first
// Chebyshev step from zero, x1 = *c0 Dinv_c rc
template <class T>
void launch_restrict(const TransferCSR &R, const uint8_t *bcmask_c, const T *rf, T *rc,
                     hipStream_t st, int nrhs = 1, int64_t vsf = 0, int64_t vsc = 0,
                     const T *dinv_c = nullptr, const double *c0 = nullptr, T *x1 = nullptr);
// x = *c Dinv b (and d = x when d is not null)
template <class T>
void launch_cheb_first(int ndof, const T *b, const T *dinv, const double *c, T *d, T *x,
                       hipStream_t st, int nrhs = 1, const int *run = nullptr);
// one dense SPD matrix of a batched inversion: n rows padded to nblk blocks
// of 64 (leading dimension 64 nblk), at `off` in both buffers
struct GJProb {
  int n, nblk;
  int64_t off;
};
// C (M x N) = A (M x K) B^T (N x K), row-major at the given offsets; ct >= 0:
// also C^T
struct GemmProb {
  int M, N, K;
  int64_t a, b, c, ct;
};
// row of the substructured solve: segments [seg0, seg1), output dof and
// position in the work vector
struct CoarseRow {
  int seg0, seg1, dof, pos;
};
struct CoarseSeg {
  int64_t a;
  int len, idx;
};
// coarsest-level solve: explicit inverses (per row of a whole component:
// first column, block size (0: not such a row), row offset) and
// substructured components (three stages of rows)
struct CoarseBlocks {
  int n = 0;
  bool direct = true;             // some rows have an explicit inverse
  const double *Ainv = nullptr;
  const float *Ainv32 = nullptr;  // the same in FP32 (FP32 V-cycles read it when set)
  const int *col0 = nullptr;
  const int *nb = nullptr;
  const int64_t *aoff = nullptr;
  int nrow[3] = {0, 0, 0};
  const CoarseRow *row[3] = {nullptr, nullptr, nullptr};
  const CoarseSeg *seg = nullptr;
  const int *idx = nullptr;
  double *tmp = nullptr, *xs = nullptr;  // [nrhs][ntmp], [nrhs][nxs]
  int ntmp = 0, nxs = 0;
  const int *run = nullptr;  // as Tiles::run
};
template <class T>
void launch_dense_solve(const CoarseBlocks &cb, const T *b, T *x, hipStream_t st, int nrhs = 1);
// the substructured components' part of it
template <class T>
void launch_coarse_schur(const CoarseBlocks &cb, const T *b, T *x, hipStream_t st, int nrhs);
// explicit inverses of nprob dense SPD matrices (largest first): matrix p
// starts in A1 when its nblk is odd, else in A0, padding rows zero, and ends
// in A0; both buffers are overwritten.  Step k works on the first active[k]
// matrices, tiles[k] blocks; fac: 4 x 64 x 64 words per matrix; *bad |= 1 on a
// non-positive pivot
void launch_gj_inverse(const GJProb *pr, const int *tile0, int nprob, const int *active,
                       const int *tiles, int nsteps, double *A0, double *A1, double *fac,
                       int *bad, hipStream_t st);
void launch_gemm_nt(int nprob, int ntiles, const GemmProb *pr, const int *tile0, const double *A,
                    const double *B, double *C, double *Ct, hipStream_t st);
void launch_coarse_scatter(int nnzb, const double *val, const uint8_t *which, const int64_t *dst,
                           const int *ld, double *A0, double *A1, double *Et, hipStream_t st);
void launch_schur_sum(int m, int lds, int nleaf, const int *loc, const int64_t *coff,
                      const int *ldc, const double *C, double *S, hipStream_t st);

// Galerkin coarse operator of one level: 3 x 3 blocks over the independent
// nodes (block row i = node i), row-major blocks, clamped rows and columns
// identity
template <class T>
struct BSR {
  int n = 0;     // block rows
  int nnzb = 0;  // blocks
  const int *ptr = nullptr;  // [n + 1]
  const int *col = nullptr;  // [nnzb] column node, ascending within a row
  const T *val = nullptr;    // [nnzb][9]
  const uint8_t *bcmask = nullptr;
  const int *run = nullptr;  // as Tiles::run
};
using BSR64 = BSR<double>;
// coarse element matrices K_E = sum_e (Q_e x I3)^T K_e (Q_e x I3) over the
// children e of every coarse element (CSR ptr/child over coarse elements;
// place = level difference << 24 | z offset << 16 | y offset << 8 | x
// offset of the child inside E, in child widths).  mode 0: K_e = s_e
// Ktab[cls_e] (finest level, element densities); 1: K_e = Kin[e]; 2:
// K_e = sum_g s_eg Ktab[cls_e][g] (finest level, nodal design)
void launch_galerkin_elem(int mode, int nE, const int *ptr, const int *child, const int *place,
                          const int *cls, const double *s, const double *Ktab, const double *Kin,
                          double *Kout, hipStream_t st);
// BSR values from the element matrices: block k collects the terms
// [tptr[k], tptr[k+1]) (code 64 E + 8 a + b, weight w: w K_E[a][b]); brow[k]
// is its row
// element matrices of one level from its scales: KE[e] = s_e K0[cls_e]
// (element design, Ktab 576 per class) or sum_g s_eg K_g[cls_e] (nodal
// design, Ktab 8 x 576 per class)
void launch_elem_matrices(int ne, const int *cls, const double *s, const double *Ktab, bool nodal,
                          double *KE, hipStream_t st);
void launch_bsr_assemble(const BSR64 &A, const int *tptr, const int *tcode, const double *tw,
                         const int *brow, const double *KE, double *val, hipStream_t st);
// dinv = 1 / diagonal of the blocks at diag[i]
template <class T>
void launch_bsr_dinv(int n, const int *diag, const double *val, T *dinv, hipStream_t st);
// y = A x with the tile apply's epilogues (ASM_STORE, ASM_RESID, ASM_CHEB)
template <class T>
void launch_bsr_apply(const BSR<T> &A, const T *x, int mode, const AsmArgs &g, hipStream_t st,
                      int nrhs = 1, int64_t vs = 0);

// out[k] = val[map[k]] per 3 x 3 block
void launch_bsr_gather(int nnzb, const int *map, const double *val, double *out, hipStream_t st);
// One symmetric point SOR sweep (forward, then in reverse) over the colours
// of a node colouring of A's graph: nodes[cptr[c] .. cptr[c + 1]) hold colour
// c (cptr on the host, ncolors + 1 entries) and A's block row k is node
// nodes[k] (colour-major rows, node-index columns); x updated in place
template <class T>
void launch_sor_symmetric(const BSR<T> &A, const int *nodes, const int *cptr, int ncolors,
                          const T *b, T *x, double omega, hipStream_t st, int nrhs = 1,
                          int64_t vs = 0);

// dst[0..n) = dst32[0..n) = v (n <= 32), from kernel arguments
void launch_set_words(int n, const double *v, double *dst, float *dst32, hipStream_t st);
template <class TI, class TO>
void launch_convert(int64_t n, const TI *a, TO *b, hipStream_t st);
template <class T>
void launch_fill(int64_t n, T v, T *a, hipStream_t st);
// v[r][i] += alpha y[i] for every right-hand side r (vectors of n values)
void launch_axpy_bcast(int64_t n, int nrhs, double alpha, const double *y, double *v,
                       hipStream_t st);
// y[r][v] = sum_j w_j x[col_j][v] over CSR rows (nv values per node)
void launch_interp_nodal(int nrows, const int *ptr, const int *col, const double *w, int nv,
                         const double *x, double *y, hipStream_t st);
// power-iteration start vector: 0.5 + a hash-drawn U[0, 1) per free dof,
// 0 on clamped dofs
void launch_start_vector(int64_t n, const uint8_t *bcmask, uint64_t seed, double *x,
                         hipStream_t st);
// *bad |= 1 if any of v[0..n) is not finite or outside [lo, hi]
void launch_check_range(int64_t n, const double *v, double lo, double hi, int *bad,
                        hipStream_t st);
// zero the clamped components of a node-major 3-dof vector
void launch_zero_clamped(int n_nodes, const uint8_t *bcmask, double *v, hipStream_t st,
                         int nrhs = 1, int64_t vs = 0);

// word 4 of every matrix-core record <- s32[its element]
void launch_rec_scale(int nrec, const int *rec_elem, const float *s32, uint32_t *rec_words,
                      hipStream_t st);
// element stiffness scales for a level: s = penalty(rho) * 2^-level
void launch_simp_scale(int n, const double *rho, const int16_t *level, double q, double k0,
                       int penalty_type, double *s64, float *s32, hipStream_t st);
// coarse element scales: volume-weighted mean of the material factor of the
// fine elements inside each coarse element (CSR over coarse elements)
void launch_restrict_scale(int nc, const int *ptr, const int *child, const float *vw,
                           const double *s_fine, const int16_t *lev_fine,
                           const int16_t *lev_coarse, double *s64, float *s32, hipStream_t st);

// nodal design (TMROctConstitutive with one design variable per node,
// src/topology/TMROctConstitutive.cpp:498-551): rho at the 8 Gauss points of
// every element from its corner values (hanging corners interpolated from
// their parents), s = penalty(rho) * 2^-level per point; rho_gp (may be null)
// receives the point densities
void launch_nodal_scale(int nelem, const int *conn, const int4 *dep4, const double *xn, const int16_t *level, double q,
                        double k0, int penalty_type, double *rho_gp, double *s64, float *s32,
                        hipStream_t st);
// design vector to the next coarser level: x_c = (R x_f) / (R 1), R = P^T
// (TACSBVecInterp::multWeightTranspose as used by TMRConformFilter::setDesignVars,
// src/topology/TMRConformFilter.cpp:154-167)
void launch_weight_restrict(const TransferCSR &R, const double *xf, double *xc, hipStream_t st);
// v_e^T K_g u_e at every Gauss point of every element (full-block tables)
void launch_nodal_energy(int nelem, const int *conn, const int4 *dep4, const uint8_t *bcmask, const int *cls,
                         const double *G, const double *u, const double *v, double *out,
                         hipStream_t st);
// nodal design gradient into slot partials (element batches, component 0):
// t_a = sum_g N_a(g) (ex_g - dpenalty(rho_g) 2^-level e_g), ex may be null
void launch_nodal_grad(const ElemBatches &eb, const int16_t *lev, const double *rho_gp, double q,
                       int penalty_type, const double *e_gp, const double *ex_gp,
                       double *partial, hipStream_t st);
// out[i] = in[3 i]
void launch_take_comp0(int n, const double *in, double *out, hipStream_t st);

// FP64 PCG helpers (scalars live on the device)
// SC_XIT: the iteration whose alpha p is still to be added to x (-1: none)
enum { SC_RZ = 0, SC_PQ, SC_ALPHA, SC_RR, SC_ZQ, SC_BETA, SC_BB, SC_RZNEW, SC_TRR, SC_XIT, SC_N };
int reduce_blocks(int64_t n);
void launch_dot1(int64_t ndof, const double *a, const double *b, double *partials,
                 hipStream_t st);
void launch_dinv_dots(int64_t n, const double *dinv, double *y, const double *x,
                      double *partials, hipStream_t st);
// sc[SC_BB] = sum of the partials; or of the pairs of launch_dinv_dots,
// |y|^2 into sc[SC_ZQ] and |x|^2 into sc[SC_RZNEW]
void launch_finalize(int nparts, const double *partials, double *sc, hipStream_t st);
void launch_finalize_pairs(int nparts, const double *partials, double *sc, hipStream_t st);

// Batched PCG over nrhs right-hand sides (vectors [nrhs][n]) whose dofs split
// into independent segments (components) with their own scalars
// sc[(rhs * nseg + seg) * SC_N + k], running flags act[rhs * nseg + seg] and
// fixed reduction blocks that never straddle a segment.
struct SegPlan {
  int nrhs = 1, nseg = 1, nblk = 0, ntiles = 0;
  int64_t n = 0;                 // dofs per right-hand side
  const int *blk_lo = nullptr;   // [nblk + 1] block b = dofs [blk_lo[b], blk_lo[b+1])
  const int *blk_seg = nullptr;  // [nblk]
  const int *seg_blk = nullptr;  // [nseg + 1]
  const int *seg_tile = nullptr; // [nseg + 1] finest-level owner tiles of each segment
};
// FIN_BETA sums the pairs of launch_b_dot2, FIN_BETA_TILE those of ASM_CHEBDOT
enum { FIN_BB = 0, FIN_RZ, FIN_PQ, FIN_RR, FIN_BETA, FIN_TRUE, FIN_BETA_TILE };
void launch_b_dot1(const SegPlan &pl, const double *a, const double *b, const int *act,
                   double *partials, hipStream_t st);
// r -= alpha q, the FP32 copy r32 of r and, with x1, the finest level's
// first Chebyshev step from zero x1 = c0 Dinv32 r32 (x += alpha p follows in
// the same iteration's p update, which reads p anyway)
void launch_b_update_xr(const SegPlan &pl, double *r, const double *q, float *r32,
                        const double *sc, const int *act, double *partials, hipStream_t st,
                        const float *dinv32 = nullptr, const double *c0 = nullptr,
                        float *x1 = nullptr);
template <class TZ>
void launch_b_dot2(const SegPlan &pl, const TZ *z, const double *r, const double *q,
                   const int *act, double *partials, hipStream_t st);
// x += alpha p for segments whose alpha was formed in the iteration before
// *iter (SC_XIT), then p = z + beta p for running segments
template <class TZ>
void launch_b_update_p(const SegPlan &pl, double *p, const TZ *z, const double *sc,
                       const int *act, double *x, const int *iter, hipStream_t st);
void launch_b_copy(const SegPlan &pl, const double *a, double *b, const int *act,
                   hipStream_t st);
// FIN_BB also sets the stop threshold max(rtol2 |b|^2, atol2) and the flags;
// FIN_RR stops a segment at the threshold (itconv = iteration, negative on
// breakdown) and, with nact, its last block does launch_b_tick's work
void launch_b_finalize(const SegPlan &pl, int mode, const double *partials, double *sc, int *act,
                       double *thr2, int *iter, int *itconv, double rtol2, double atol2,
                       hipStream_t st, int *nact = nullptr, int *host = nullptr);
// count the running segments into nact[0] and the pinned *host, advance the
// iteration counter (nact[1]: arrival counter of FIN_RR, zero between launches)
void launch_b_tick(int *iter, const int *act, int nidx, int *nact, int *host, hipStream_t st);

// per-element compliance density and its design derivative (element mode)
// K: the REFL_TABLE blocks of every class
void launch_elem_energy(int nelem, const int *conn, const int4 *dep4, const uint8_t *bcmask, const int *cls,
                        const double *K0, const double *u, double *energy, hipStream_t st);
// p-norm of the relaxed von Mises failure (TMROctConstitutive::evalFailure,
// src/topology/TMROctConstitutive.cpp:1056-1104; TACS "pnorm-continuous"
// aggregation): S = sum_e sum_g (V_e / 8) (r(rho_e) vm(C0 B_g u_e) / ys)^P,
// the stress formed from grad u at the point; vol: per class block volume.
struct StressArgs {
  double P = 8.0, eps = 0.3, ys = 1.0;
  const double *G = nullptr;    // NODAL_TABLE tables
  const double *vol = nullptr;
};
// rho_gp (nodal design, may be null): densities at the Gauss points, used
// in place of the element densities rho
void launch_stress_sum(int nelem, const int *conn, const int4 *dep4, const uint8_t *bcmask, const int *cls,
                       const int16_t *lev, const double *rho, const double *rho_gp,
                       const double *u, const StressArgs &sa, double *partials, hipStream_t st);
// element dfdu into slot partials (element batches) and the explicit
// d f / d rho_e (or, with rho_gp, d f / d rho_g per Gauss point);
// coef = S^(1/P - 1) read from sc[SC_ZQ]
void launch_stress_grad(const ElemBatches &eb, const int16_t *lev, const int *cls,
                        const double *rho, const double *rho_gp, const double *u,
                        const StressArgs &sa, const double *sc, double *partial,
                        double *dfdrho, hipStream_t st);
// psi_e^T K0 u_e per element (adjoint-residual product without the factor)
void launch_elem_energy2(int nelem, const int *conn, const int4 *dep4, const uint8_t *bcmask, const int *cls,
                         const double *K0, const double *u, const double *v, double *out,
                         hipStream_t st);
// g = dfdrho_explicit - dpenalty(rho) 2^-level * prod
void launch_adjoint_grad(int n, const double *rho, const int16_t *lev, double q, int ptype,
                         const double *prod, const double *explicit_part, double *g,
                         hipStream_t st);

// SIMP/RAMP derivative (src/topology/TMROctConstitutive.cpp:597-619) times
// -2^-level times the element energy
void launch_compliance_grad(int n, const double *rho, const int16_t *lev, double q, int ptype,
                            const double *energy, double *g, hipStream_t st);

}  // namespace tmrx
