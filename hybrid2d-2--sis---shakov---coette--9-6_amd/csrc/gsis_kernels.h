// gsis_kernels.h -- launch wrappers of the gfx950 kernels (gsis_kernels.hip).
#pragma once
#include "gsis_device.h"

namespace gsis {

constexpr int kMaxV1 = 512;  // max discrete velocities per direction (LDS tables)

// up to kMaxWalls subfaces launched together (diffuse walls; periodic subfaces
// of one direction); start[k] is the first block of subface k
constexpr int kMaxWalls = 16;
struct BcSet {
  int n;
  int start[kMaxWalls + 1];
  BcDev b[kMaxWalls];
};
template <typename T> void launch_walls(const Dev &d, const BcSet &ws, T *FG, T *FH, T *slot, hipStream_t s);
template <typename T> void launch_farfield(const Dev &d, const BcDev &b, T *FG, T *FH, hipStream_t s);
template <typename T> void launch_periodic(const Dev &d, const BcSet &bs, T *FG, T *FH, hipStream_t s);
// inner-face exchange of LAP = 2 layers, FRD(1:2) and S_GKUA(1:10); n1 cells along the face
template <typename T>
void launch_inner(const Dev &dd, const BcDev &bd, T *FGd, T *FHd, const Dev &ds, const BcDev &bs, const T *FGs,
                  const T *FHs, int n1, int orient, hipStream_t s);
template <typename T> void launch_rhs(const Dev &d, const T *FG, const T *FH, const T *slot, T *RG, T *RH, hipStream_t s);
template <typename T> void launch_sweep(const Dev &d, T *FG, T *FH, const T *RG, const T *RH, hipStream_t s);
template <typename T> void launch_moments(const Dev &d, T *FG, T *FH, hipStream_t s);
constexpr int kNCellPar = 20;  // per-cell constants of the fused kinetic kernel
// Fused kinetic step over F = [G plane | H plane] (and R likewise); false when
// the mesh does not fit the fused kernel.
template <typename T> bool launch_walk(const Dev &d, double *cpar, T *F, const T *slot, T *R, int store_rhs, int tiles, hipStream_t s);
// Buffers of the column-pair kernel (k_strip): seam messages
// [seam][tile][row][4][64] (elements of the working precision), every word
// strip_empty_word() outside a launch, a word set when a wait for a message timed
// out, and a counter per tile (strip_counters of them) that the tile's workgroups
// draw their strips from.
constexpr int kNextStride = 16;  // words from one tile's counter to the next
struct StripBufs {
  void *msg = nullptr;
  int *err = nullptr, *next = nullptr;
  // face-override words: ny+2 rows (bit 0 i-face 1, bit 1 i-face nx), then
  // nx+2 columns (bit 0 j-face 1, bit 1 j-face ny)
  const int *oflags = nullptr;
  size_t msg_elems = 0;
  // when set, recorded on the stream just before and after k_strip itself
  hipEvent_t ev_before = nullptr, ev_after = nullptr;
};
// seam rows (seam x tile x row) of a mesh with nw columns per workgroup
size_t strip_rows(const Dev &d, int nw);
inline size_t strip_counters(const Dev &d) { return (size_t)((d.nv + 63) / 64) * kNextStride; }
// the word a seam message is filled with before its first use
uint32_t strip_empty_word(bool fp32);
// Column-pair kinetic step with nw (8 or 16) columns per workgroup; false when
// the mesh or the buffers do not fit.
template <typename T> bool launch_strip(const Dev &d, double *cpar, T *F, const T *slot, T *R, int store_rhs, int nw, StripBufs &b, hipStream_t s);
template <typename T> void launch_res4(const Dev &d, const T *RG, const T *RH, hipStream_t s);
// Columns per workgroup: 16 where the mesh has more than 8 and the launch's
// strips of 16 still give every CU a workgroup, else 8, whose shorter pipelines
// fill more CUs.  Measured, 16 against 8 columns: 128^2 x 64^2 (512 strips of 16)
// 0.73 and 0.74 ms, FP32 0.39 and 0.49, 256^2 x 96^2 (2304) 6.1 and 6.6; 96^2 x 48^2
// (216) 0.342 and 0.336, 101^2 x 37^2 (154) 0.35 and 0.33, 64^2 x 32^2 (64) 0.21 and
// 0.17, 12^2 x 24^2 (9) 43 and 39 us.
constexpr long long kWideStrips = 256;
inline int strip_columns(const Dev &d, long long strips16) { return d.nx - 1 > 8 && strips16 >= kWideStrips ? 16 : 8; }
// workgroups of a mesh's strips with nw columns
int strip_blocks(const Dev &d, int nw);

// One instance of a batched step: its device state and the first workgroup
// of its share of each batched launch.  Jobs with strips of 16 columns come
// before those with 8.
template <typename T>
struct StripJob {
  Dev d;
  const T *cp;  // cell constants in T (k_cellpar), by cell
  T *F, *R;
  const T *slot;
  T *msg;
  int *next;
  const int *oflags;
  const int *wall_list;  // DETFPwall nodes (k_det_wall)
  double *swall;
  int nwall;
  int ntiles;
  int strip0, cell0, mom0, mom1, det0, conv0, hot0;
};
// Subfaces of one instance in a batched boundary launch.
struct BcJob {
  enum { kWalls, kPeriodic, kFarfield };
  int job, start, kind;
  BcSet bs;
};
// jobs (the first wide of them with strips of 16 columns) and workgroups of
// each batched launch
struct BatchBlocks {
  int jobs = 0, wide = 0, strip16 = 0, strip8 = 0, cell = 0, mom0 = 0, mom1 = 0, det = 0, conv = 0, hot = 0;
};
template <typename T> void batch_blocks(StripJob<T> &j, bool wide, bool hot, BatchBlocks &n);
// Batched launches over a device table of jobs (scheme and T shared by all):
// boundary subfaces, S0 + cell constants + one column-pair launch per strip
// width over all jobs' strips (no RHS kept), moments + DETFPwall, Convert_NS +
// HoT.
template <typename T>
void launch_bc_batch(const StripJob<T> *djobs, const BcJob *dbcs, int n, int blocks, hipStream_t s);
template <typename T>
void launch_strip_batch(const StripJob<T> *djobs, const BatchBlocks &n, int scheme, int *werr, hipStream_t s);
template <typename T> void launch_moments_batch(const StripJob<T> *djobs, const BatchBlocks &n, hipStream_t s);
template <typename T> void launch_convert_batch(const StripJob<T> *djobs, const BatchBlocks &n, hipStream_t s);
// every cell's distribution set to g[v] (G) and h[v] (H), wall slots zero
template <typename T>
void launch_fill_uniform(const Dev &d, const double *g, const double *h, T *FG, T *FH, T *slot, hipStream_t s);
// FRD (Fortran layout) to and from the device layout for velocities v0..v0+nvc-1 through a stage holding that
// contiguous slice of the Fortran FRD array (2(nx+7)(ny+7) doubles per velocity)
template <typename T>
void launch_frd_out_chunk(const Dev &d, double *stage, int v0, int nvc, const T *FG, const T *FH, const T *slot,
                          hipStream_t s);
template <typename T>
void launch_frd_in_chunk(const Dev &d, const double *stage, int v0, int nvc, T *FG, T *FH, T *slot, hipStream_t s);
void launch_save_s0(const Dev &d, hipStream_t s);
// out_mass (sum of S_GKUA(1)*vol over interior cells) into out[0]
void launch_out_mass(const Dev &d, double *out, hipStream_t s);
// MassCorrect: out_mass into work[0], then S_GKUA(1) scaled by init/out_mass
void launch_mass_correct(const Dev &d, double *work, double init, hipStream_t s);
void launch_det_wall(const Dev &d, const int *list, int n, double *swall, hipStream_t s);
void launch_convert(const Dev &d, hipStream_t s);
void launch_hot(const Dev &d, hipStream_t s);
// ncomp plane-major fields of the padded cells into [ny1][nx1][nf] (zero where there is none)
void launch_fields_out(const Dev &d, const double *src, int ncomp, int nf, int nx1, int ny1, int o, double *out,
                       hipStream_t s);
void launch_residual(const Dev &d, double *out, hipStream_t s);

}  // namespace gsis
