// Internal declarations shared by the gfx950 kernels and the C ABI layer.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

namespace pyiid {

// Atom record in HBM: float32 input positions widened exactly to double (the
// sampler integrates them in double), and the element index stored in w.
// 32 B per atom, one vector load.
struct alignas(32) AtomRec {
  double x, y, z, w;
};

// Q bins per wave of the fused F + gradient kernel (the larger of its two shapes).
constexpr int kGradM = 32;
constexpr int kFqM = 64;  // default Q bins per wave of the F-only kernel
constexpr int kWaves = 4;      // waves per block in the contracted-force kernel
constexpr int kJTile = 256;    // atoms staged in LDS per j tile

// Work item of the Debye kernels.  Structures ("chains") are stored back to
// back; an item is a 64-atom i tile [i_base, i_end) of one chain against the
// j range [jbeg, jend) of the same chain.  `split` indexes the gradient
// partial buffer, `tile` the chain-global i tile (for force reduction).
struct Item {
  int i_base, i_end, jbeg, jend;
  int split, chain, tile, pad;
};

// Items [item_begin, item_end) of one i tile (or of one chain, for F).
struct Range {
  int begin, end, i_base, i_end;
};

// ---- launch wrappers (debye.hip) ----
// Ordered-pair F + gradient, m = 16 or 32 Q bins per wave (compensated
// sums: m = 16 only):
// gpart[item.split][i][c][q] (float) for i in the item's tile and
// fpart[item][q] (F partial, double).  Weighted: the j indices of an item are
// positions in jperm and item.pad is the element of the item's j range;
// unweighted: atom indices.
hipError_t launch_fused_grad(hipStream_t st, int m, bool compensated, const AtomRec* pos,
                             const int32_t* jperm, int n_total, const float* ftab, int nq,
                             double dq, const Item* items, int n_items, bool weighted,
                             float* gpart, double* fpart);
// Work item of the symmetric F + gradient kernel: 64-position tiles [g0, g1)
// against tiles [r0, r1) of one element, pairs (I, J) with J <= I.  The I
// rows of tile I go to slot islot0 + (I - max(g0, r0)), the J rows of tile J
// to slot jslot0 + (J - r0).
struct SymItem {
  int g0, g1, r0, r1, islot0, jslot0, pad0, pad1;
};
// Unordered-pair F + gradient: slots[slot][c][q][64] (float; tiles[t] =
// {slot list begin, end, position begin, end}, positions in perm) and
// fpart[item][q] (F partial, double).  Weighted: tile_el[t] is the element
// of tile t.
// m = 16 (8 waves, 128 bins per block) or 12 (12 waves, 144 bins).
hipError_t launch_sym_grad(hipStream_t st, int m, const AtomRec* pos, const int32_t* perm,
                           const Range* tiles, const int* tile_el, const float* ftab, int nq,
                           double dq, const SymItem* items, int n_items, bool weighted,
                           float* slots, double* fpart);
// out[perm[p]][c][q] = gscale[q] * sum_{e in tile} slots[entries[e]][c][q][row]
// (FP64, list order), float or double output.
hipError_t launch_reduce_slots(hipStream_t st, const float* slots, const int* entries,
                               const Range* tiles, int n_tiles, const int32_t* perm, int nq,
                               const double* gscale, void* out, bool out_f64);
// Contracted forces over unordered pairs: items are tile pairs (I, J), J <= I,
// of at most 64 positions of one chain in perm (Item.tile = I's and Item.pad =
// J's chain-global tile index; weighted: Item.split = e_I | e_J << 16, each
// tile of one element); n_groups Q groups of `span` bins (a multiple of 32)
// each.  part[(item * n_groups + g)][side][64][3], side 0 = I, 1 = J.
constexpr size_t kPairForceLds = 64 * 1024;
hipError_t launch_pair_force(hipStream_t st, const AtomRec* pos, const int32_t* perm,
                             const float* ftab, int nq, double dq, const Item* items, int n_items,
                             int n_groups, int span, bool weighted, const float* u,
                             const float* uq, float* part);
// force[perm[p]][c] = conv * sum_{e in entries[tile]} part[e][row][c] (FP64)
// for the tile's positions p = i_base + row, where an entry is work * 2 +
// side; tiles[t] = {entry begin, end, i_base, i_end}.
hipError_t launch_reduce_pair_force(hipStream_t st, const float* part, const int* entries,
                                    const Range* tiles, int n_tiles, const int32_t* perm,
                                    double conv, double* out);
// uq[b][q] = u[b][q] * float32(q dq)
hipError_t launch_uq(hipStream_t st, const float* u, int n_chain, int nq, double dq, float* uq);
// Unordered-pair F only: fpart[item][q] (double), m Q bins per wave (64, 72,
// 80, 88, 96 or 112; compensated sums: 64 only).  Item indices are positions
// in perm; weighted: item.split is the element of the item's i tile and
// item.pad that of its j range.  forms (nullable): forms[0], forms[1] gain
// the (wave, j atom) steps run in the three-term and in the Reinsch form.
hipError_t launch_fq(hipStream_t st, int m, bool compensated, const AtomRec* pos,
                     const int32_t* perm, const float* ftab, int nq, double dq, const Item* items,
                     int n_items, bool weighted, double* fpart, unsigned long long* forms);
// out[r][q] = scale[r][q] * sum_{p in ranges[r]} part[p][q], r < n_rows (FP64)
hipError_t launch_reduce_ranges(hipStream_t st, const double* part, const Range* ranges,
                                int n_rows, int nq, const double* scale, double* out_f64,
                                float* out_f32);
// grad[i][c][q] = gscale[q] * sum_s gpart[s][i][c][q]
hipError_t launch_reduce_grad(hipStream_t st, const float* gpart, int n_split, int64_t n,
                              int nq, const double* gscale, void* out, bool out_f64);
// per-chain normalisation: na, 2w/na, w/na, -w/na  ([chain][q])
hipError_t launch_norm(hipStream_t st, const float* ftab, const int64_t* counts, int n_elem,
                       int nq, const int64_t* n_atoms, int n_chain, bool weighted, double* na,
                       double* fscale_unordered, double* fscale_ordered, double* gscale);
hipError_t launch_pair_geometry(hipStream_t st, const AtomRec* pos, int64_t k_offset,
                                int64_t k_count, float* d, float* r);

// ---- F(Q) by spreading (spread.hip) ----
// Item: positions [i0, i1) (at most 64) against positions [j0, j1), pairs
// j < i.  Unit: items [begin, end) of one chain and element pair, added to
// grid `grid`.
struct SpreadItem {
  int i0, i1, j0, j1;
};
struct SpreadUnit {
  int begin, end, grid, pad;
};
constexpr size_t kSpreadLds = 160 * 1024 - 256;  // a block's grid lives in LDS
int fq_grid_points(int nq);
int fq_grid_stride(int nq);  // 64-bit words per grid (points, close-contact nodes, flag)
// Bits of the grid's fixed point for distances up to about r_max.
int fq_scale_bits(int nq, double dq, double r_max);
// Spreads every unit's pairs and adds them to grids[unit.grid] (zero before
// the first call; launch_transform_fq clears them again).  shift: right shift
// of a unit's sums (0 up to 2^32 pairs).
hipError_t launch_spread_fq(hipStream_t st, const AtomRec* pos, const SpreadUnit* units,
                            int n_units, const SpreadItem* items, int nq, double dq, int shift,
                            int scale_bits, unsigned long long* grids);
// out[b][q] = scale[b][q] * sum over the chain's element pairs (grid index
// b * n_pair + e_i (e_i + 1) / 2 + e_j, e_j <= e_i) of f_i f_j times the pair's
// sum of sin(Q r) / r; clears the grids.  part: n_chain * n_pair *
// fq_transform_parts * nq doubles.  one_part (single grids only): in one launch,
// without part, and the grids stay as they are.
int fq_transform_parts(int nq, int n_chain, int n_pair);
hipError_t launch_transform_fq(hipStream_t st, unsigned long long* grids, int n_chain, int n_pair,
                               bool weighted, const float* ftab, int nq, double dq, int shift,
                               int scale_bits, const double* scale, double* part, double* out_f64,
                               float* out_f32, bool one_part);
// F of chains of at most kSmallAtoms atoms (off: n_chain + 1 offsets) in one
// launch; the grids must fit kSmallFqLds.
constexpr int kSmallAtoms = 128, kSmallAtoms2 = 85, kSmallAtoms3 = 70;  // by elements
constexpr size_t kSmallFqLds = 80 * 1024;
size_t small_fq_lds(int nq, int n_pair);
hipError_t launch_small_fq(hipStream_t st, const AtomRec* pos, const int* off, int n_chain,
                           int n_pair, bool weighted, const float* ftab, int nq, double dq,
                           int scale_bits, const double* scale, double* out_f64, float* out_f32);
// Atom records from float positions and elements; keep (nullable) takes a copy
// of the positions, reach (nullable) a bound of their distances (one block
// then: for at most kReachAtoms atoms); with place (nullable) ordered[place[i]]
// takes the record too.
constexpr int64_t kReachAtoms = 4096;
hipError_t launch_pack(hipStream_t st, const float* p, const int32_t* e, int64_t n, AtomRec* out,
                       float* keep, double* reach, const int32_t* place, AtomRec* ordered);
// *reach: a bound of the distances within pos (its bounding sphere's diameter;
// infinite where a position is not finite)
hipError_t launch_reach(hipStream_t st, const AtomRec* pos, int64_t n, double* reach);
// out[p] = pos[perm[p]]
hipError_t launch_gather(hipStream_t st, const AtomRec* pos, const int32_t* perm, int64_t n,
                         AtomRec* out);

// ---- gradient by spreading (gradspread.hip) ----
constexpr size_t kGradLds = 160 * 1024 - 512;   // a block's three grids live in LDS
int grad_row_len(int nq);                     // points per row (a multiple of 32)
size_t grad_lds_bytes(int nq);
double grad_reach(int nq, double dq, double r_max);  // points of a row that r_max reaches
// bytes of a split operand: tiles of 128 rows, two halves for every point
inline size_t split_bytes(int64_t rows, int row_len) {
  return static_cast<size_t>((rows + 127) / 128) * 128 * row_len * 4;
}
// w: split_bytes(nq, grad_row_len(nq)); inv_phihat: nq floats
hipError_t launch_sine_matrix(hipStream_t st, int nq, void* w, float* inv_phihat);
// Grids of positions [p0, p0 + n_atoms) against each of the n_run element
// runs [runs[e], runs[e + 1]): rows 3 (p - p0) + c of a split operand for each e,
// and row_scale (e * 3 n_atoms + 3 (p - p0) + c).  Points used: k_fixed, or those that
// distances up to *reach need.
hipError_t launch_spread_grad(hipStream_t st, const AtomRec* pos, int p0, int n_atoms, int64_t n,
                              const int* runs, int n_run, int nq, double dq, double r_max,
                              int k_fixed, const double* reach, void* rows, float* row_scale);
// out[perm[p]][c][m] = gs[m] f_p(m) sum_e f_e(m) sum_k rows w / phihat
// (single element: without f).  perm null: identity.  clear (nullable): an even
// number of words that blocks of the launch set to zero.
hipError_t launch_gemm_split(hipStream_t st, const void* rows, const float* row_scale, int n_atoms,
                             int n_run, const void* w, const float* inv_phihat, int nq, double dq,
                             int k_fixed, const double* reach, const double* gs, const float* ftab,
                             const int* run_elem, bool weighted, const AtomRec* pos,
                             const int32_t* perm, int p0, void* out, bool out_f64,
                             unsigned long long* clear, int64_t clear_words);
// The rows of all atoms and the F grids of launch_spread_fq's units (shift 0)
// in one launch.
hipError_t launch_spread_both(hipStream_t st, const AtomRec* pos, int n_atoms, const int* runs,
                              int n_run, int nq, double dq, double r_max, int k_fixed,
                              const double* reach, void* rows, float* row_scale,
                              const SpreadUnit* units, int n_units, const SpreadItem* items,
                              int scale_bits, unsigned long long* grids);

// ---- contracted forces from a pair-force table (forcetab.hip) ----
// Unit: positions [i0, i1) in `tiles` (1, 2, 4, 8 or 16) tiles of 64 against
// positions [j0, j1), all of elements ei, ej (-1: single element) of one
// chain, with table `table`; its sums go to plane `plane`.
struct ForceUnit {
  int i0, i1, j0, j1;
  int tiles, plane, table, chain;
  int ei, ej, pad0, pad1;
};
constexpr size_t kForceLds = 160 * 1024;
double force_cell(int nq, double dq);       // cell width of the table
size_t force_lds_bytes(int64_t n_cell);     // LDS of a block
// t4 / t2 [table][n_cell]: coefficients 0..3 / 4, 5; coef[table][q] (table =
// chain * n_pair + pair) as launch_adjoint_sum writes it
hipError_t launch_force_table(hipStream_t st, const double2* coef, int nq, double dq, int n_table,
                              int n_cell, float4* t4, float2* t2);
// part[plane][position][3], or with out the forces themselves (a single plane):
// out[perm[p]][c] = conv * sum; *far_seen (nullable, host
// memory) becomes 1 when a pair lies past the table
hipError_t launch_table_force(hipStream_t st, const AtomRec* pos, const ForceUnit* units,
                              int n_units, int n_cell, const float4* t4, const float2* t2,
                              const float* u, const float* ftab, int nq, double dq, int64_t n,
                              double* part, const int32_t* perm, double conv, double* out,
                              double* far_seen);
// out[perm[p]][c] = conv * sum_{k < planes[p]} part[k][p][c] (perm null: identity)
hipError_t launch_reduce_force(hipStream_t st, const double* part, int64_t n,
                               const int32_t* planes, const int32_t* perm, double conv,
                               double* out);

// ---- transform / potential (transform.hip) ----
// C[m][ldc] = A[m][K] . B[n][K]^T in FP32 MFMA; A float or double.
hipError_t launch_gemm_nt(hipStream_t st, const void* a, bool a_f64, int64_t m, int k,
                          const float* b, int n, double* c_f64, float* c_f32);
// The same for rows of the gradient, on split operands (split_bytes(rows,
// split_row_len(k)) and a scale per row) of both factors; a: the rows themselves,
// t: T.  From kSplitBins bins and kSplitWork entries on, where the split's
// launch is worth it (us, 4,000 points, against launch_gemm_nt: 96 rows of 330 bins
// 25 and 29, 129 of 330 22 and 29, 192 of 128 14 and 12, 258 of 128 14 and 14, 960 of
// 330 24 and 66).
constexpr int kSplitBins = 128;
constexpr int64_t kSplitWork = 32768;
inline int split_row_len(int k) { return (k + 31) / 32 * 32; }
hipError_t launch_split_rows(hipStream_t st, const void* a, bool a_f64, int64_t m, int k, void* rows,
                             float* scale);
hipError_t launch_gemm_grad(hipStream_t st, const void* rows, const float* row_scale, const void* a,
                            bool a_f64, int m, int k, const void* ts, const float* t_scale,
                            const float* t, int n, double* out);
// Potential value/scale and the adjoint w[t] (FP64) of one array.
// out5 = {value, scale, a_opt, res.res, g.res}.
hipError_t launch_potential(hipStream_t st, int potential, const double* gobs,
                            const double* gcalc, int n, double* out5, double* w);
// y[row] = sum_t X[row][t] * w[t]  (FP64), one wave per row
hipError_t launch_gemv_rows(hipStream_t st, const double* x, int64_t rows, int n,
                            const double* w, double* y);
// The potential of every chain (out5[b]) and what the adjoint of all needs: mix[b]
// and, unless part is null, the products of o and g with T (kAdjointSlices * 2 *
// n_chain * nq doubles).  clear (nullable): an even number of words that blocks of
// the launch set to zero.
constexpr int kAdjointSlices = 4;
hipError_t launch_score(hipStream_t st, int potential, const double* gobs, const double* gcalc,
                        int n_r, int n_chain, double* out5, double2* mix, const float* t, int nq,
                        double* part, unsigned long long* clear, int64_t clear_words);
// u[b][q] = gscale[b][q] * sum_t T[t][q] w[b][t] (FP64) from these and, unless null,
// coef[b][pair][q] = (u f_I f_J q dq, u f_I f_J) for the force table
hipError_t launch_adjoint_sum(hipStream_t st, const double* part, const double2* mix, int n_chain,
                              int nq, const double* gscale, double dq, const float* ftab,
                              bool weighted, int n_pair, float* u, double2* coef);
// the same from u[q] = gscale[q] * w[q - q_first] (0 below q_first), one chain
hipError_t launch_adjoint_fq(hipStream_t st, int nq, int q_first, const double* w,
                             const double* gscale, double dq, const float* ftab, bool weighted,
                             int n_pair, float* u, double2* coef);
hipError_t launch_f64_to_f32(hipStream_t st, const double* x, int64_t n, float* y);
hipError_t launch_f32_to_f64(hipStream_t st, const float* x, int64_t n, double* y);

// ---- sampler (hmc.hip) ----
struct HmcChain {
  int atom_begin, atom_end;
};
// Start of a proposal: save positions, draw momenta p ~ N(0, m/beta) from the
// counter-based generator (seed, proposal counter), kinetic energy K0[b],
// first half kick p += eps/2 F.
hipError_t launch_hmc_begin(hipStream_t st, AtomRec* pos, double* pos_save, double* mom,
                            const double* force, const double* mass, const HmcChain* chains,
                            int n_chain, double beta, double eps, uint64_t seed,
                            const int64_t* counter, double* kin0);
// x += eps p / m
hipError_t launch_hmc_drift(hipStream_t st, AtomRec* pos, const double* mom, const double* mass,
                            int64_t n, double eps);
// p += h F, then x += eps p / m: the end of one step and the start of the next
hipError_t launch_hmc_kick_drift(hipStream_t st, AtomRec* pos, double* mom, const double* force,
                                 const double* mass, int64_t n, double h, double eps);
// p += h F
hipError_t launch_hmc_kick(hipStream_t st, double* mom, const double* force, int64_t n, double h);
// End of a proposal: K1, Metropolis with exp(beta (H0 - H1)), restore or
// accept (positions, force, energy), record energy/acceptance, bump counter.
// force_cur null: no force copy.  viol (nullable): chains flagged there are
// rejected, counted in viol_count and their flag cleared.
hipError_t launch_hmc_end(hipStream_t st, AtomRec* pos, const double* pos_save, const double* mom,
                          const double* mass, double* force_cur, const double* force_new,
                          double* e_cur, const double* out5_new, double conv,
                          const HmcChain* chains, int n_chain, double beta, uint64_t seed,
                          int64_t* counter, const double* kin0, double* e_hist,
                          int32_t* acc_hist, int64_t hist_cap, int* viol, int* viol_count);
// e_cur[b] = conv * out5[b].value
hipError_t launch_energy_from_out5(hipStream_t st, const double* out5, int n_chain, double conv,
                                   double* e);

// ---- learned integrator (surrogate.hip) ----
// Network parameter block: bf16 W1[16][64], bf16 W2[64][64], f32 b1[64],
// b2[64], descriptor mean[16], inv_scale[16].
constexpr int kSurNetBytes = 16 * 64 * 2 + 64 * 64 * 2 + 64 * 4 * 2 + 16 * 4 * 2;
constexpr int kSurHidden = 64;
constexpr int kSurRbf = 16;
constexpr int kSurGram = 64 * 64 + 64 + 1;  // Phi Phi^T, Phi y, y.y per chain
// tiles: Item{i_base, i_end, jbeg, jend = the chain's atoms, chain}.
hipError_t launch_nbr_build(hipStream_t st, const AtomRec* pos, int n, const Item* tiles,
                            int n_tiles, float rl, int max_nbr, int* nbr, int* cnt, int* viol);
// rbf = {rc, mu0, dmu, eta}
hipError_t launch_descriptors(hipStream_t st, const AtomRec* pos, int n, const int* nbr,
                              const int* cnt, const float* rbf, float* d);
hipError_t launch_mlp(hipStream_t st, const float* d, int n, const Item* tiles, int n_tiles,
                      const void* net, const unsigned short* w3, int w3_stride, float* c,
                      float* e_atom);
hipError_t launch_sur_force(hipStream_t st, const AtomRec* pos, int n, const int* nbr,
                            const int* cnt, const float* rbf, const float* c, double* force,
                            float* phi);
// chunks: Item{jbeg, jend = flat column range, split = partial slot, chain};
// ranges[b] = {first slot, end slot}.  out[b] (FP64, kSurGram values).
hipError_t launch_gram(hipStream_t st, const float* phi, int64_t n3, const double* y,
                       const Item* chunks, int n_chunks, float* part, const Range* ranges,
                       int n_chain, double* out);
// out[b][k] = sum_{a in chain b} e_atom[k * n + a] (FP64), off: chain offsets (n_chain + 1).
hipError_t launch_chain_feature_energy(hipStream_t st, const float* e_atom, int64_t n,
                                       const int64_t* off, int n_chain, double* out);
hipError_t launch_disp_check(hipStream_t st, const AtomRec* pos, const double* pos_save,
                             const int* atom_chain, int64_t n, double lim, int* viol);

// Records the calling thread's message for pyiid_last_error and returns code.
int set_error(int code, const char* fmt, ...);

}  // namespace pyiid
