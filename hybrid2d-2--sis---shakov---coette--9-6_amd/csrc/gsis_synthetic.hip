// gsis_synthetic.hip -- the GSIS synthetic NS solve (mode M1) on one MI355X.
//
// Restates the block of Hybrid_Time_advance_LU_SGS that the reference ships
// commented out (src/Hybrid_Sub.f90:45-153) and its inner loop
// NS_Time_advance_LU_SGS (src/sub_NS_singlegrid.f90:4-40) with the options of
// the shipped control.in: original-variable NND2 reconstruction
// (src/sub_Residual.f90:387-397,476-546), Van Leer splitting
// (src/sub_flux_split.f90:141-192), viscous terms plus the kinetic HoT
// correction (src/sub_Residual.f90:176-193,309-326), local time step
// (src/sub_NS_singlegrid.f90:160-221) and the plane-by-plane LU-SGS
// (src/sub_LU_SGS.f90:4-143).
//
// The inner loop is one cooperative launch that iterates on the device until
// the max |energy residual| drops to ns_tol or ns_maxit is reached.  Its
// recurrence sets its time: dU of a cell needs dU of (i-1,j) and (i,j-1)
// (forward; (i+1,j) and (i,j+1) backward), so an iteration is two chains of
// nx+ny-11 plane steps, however many CUs there are.  Everything else is
// arranged around the chain:
//  * a sweep workgroup per band of 64 swept rows, each on a CU of its own.  One
//    wavefront sweeps, a row per lane, a plane per step; the band's edge row
//    goes to the next band through memory (0.3 us one way on one XCD, which
//    costs a lag of a few steps per band, not time per step).  The other
//    wavefronts of the workgroup do what would hold it up: three fetch the
//    records of coming planes and form what does not depend on dU, one brings
//    the neighbouring band's values, one keeps the books;
//  * flux workgroups compute tile after tile what the sweeps need: primitives,
//    viscosity, face fluxes (inviscid, viscous, HoT), Res, Lc, Lv, dt, stored
//    by anti-diagonal plane.  A tile of the next iteration is computed as soon
//    as the backward sweep has passed its cells, and the next forward sweep
//    starts when the first tiles are done: the decision that there is a next
//    iteration is taken from the residual before the backward sweep begins.
// One lane per row and one plane per step give the order of the reference's
// sweeps, so the inner iteration counts are the reference's.  The loop ends by
// the reference's rule: iteration k+1 runs when max |Res_4| of iteration k
// exceeds ns_tol and k < ns_maxit.  Every wait between workgroups is bounded;
// a timeout ends the loop and is reported by the host.
//
// Measured per inner iteration (mesh cells, sweeps of all bands in one
// workgroup with separate flux phases before): 64^2 102 -> 64 us, 128^2
// 238 -> 127 us, 256^2 607 -> 255-266 us; 40 instances of side 64-256 in one
// launch 4.5 -> 0.42 ms (one workgroup each before).  Between these meshes (234,
// 490 and 1002 plane steps) a step costs 0.25 us, and an iteration 6 us besides.
// A step of which everything it waits for is there already takes 0.2 us (450-480
// cycles, about 400 of them the arithmetic): a fifth of the step in the loop is
// waiting that has not been told apart.
#include <algorithm>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "gsis_ns_common.h"
#include "gsis_synthetic.h"
#include "gsis_wait.h"

namespace gsis {

namespace {
std::string g_syn_err;
}

const char *synthetic_error() { return g_syn_err.c_str(); }

// A flux tile: kTI x kTJ cells.  A workgroup's 384 threads take each phase of
// a tile of 8 x 16 at once (240 cells with halo, 280 faces, 128 cells), so it
// has the latency of 8 x 8 and less halo; 16 x 16 takes two rounds of faces.
constexpr int kTI = 8, kTJ = 16;
constexpr int kCI = kTI + 4, kCJ = kTJ + 4;  // with two halo rings each side
constexpr int kTC = kCI * kCJ;
constexpr int kLev = kTJ / kTI;  // tile (a, b) is of level a + kLev b: it holds the planes from 6 + kTI level on
constexpr int kBand = 64;                    // swept rows of a sweep workgroup, one per lane of its sweep wavefront
constexpr int kBandTiles = kBand / kTJ;      // tile rows of a band
constexpr int kMaxBands = 16;                // rows <= 1024
constexpr int kThreads = 384;                // a workgroup of the inner loop: six wavefronts
constexpr int kLoaders = 3;                  // wavefronts of a sweep workgroup that fetch records
constexpr int kGroup = 4;                    // plane steps a loader fetches and hands over at a time
constexpr int kGroups = 2;                   // groups of prepared records in LDS
constexpr int kPad = kGroup - 1;             // planes before the first and after the last one that steps store to
constexpr int kHand = 64;                    // received neighbour values in LDS (a power of two)
constexpr long long kWaitTicks = 200000000;  // bounded waits: 2 s of the 100 MHz wall clock
// a batched gang's wait for its last workgroup: 120 s without an iteration of an earlier gang
constexpr long long kStartTicks = 12000000000;

// ctl words
enum { kCtlGo = 1, kCtlErr = 3, kCtlBad = 4, kCtlStop = 5, kCtlLast = 6, kCtlArrived = 7 };

// Sweep records are blocked by (plane, band): block ((p-6)*nw + w) holds the
// 64 rows 3+64w .. 3+64w+63, pair q of row 3+64w+l at q*128 + 2l, so each pair
// of fields of a plane is one contiguous 1 KiB load per wavefront.  dU*, the
// updated state and the geometry weights use the same blocks with 2, 2 and
// geo_pairs pairs.  Every array stays below 2 GiB (synthetic_init), so byte
// offsets fit the 32-bit buffer offsets.
constexpr int kBlk = kNRec * 64;      // doubles per block
constexpr int kBlk4 = 4 * 64;         // the same of dU* and of the updated state
__host__ __device__ inline int geo_pairs(bool axis) { return axis ? 2 : 6; }
static_assert(kRecRes == 0 && kRecU == 4 && kRecRa == 8 && kRecCbi == 9 && kRecCbj == 10 && kRecRr == 11 &&
                  kNRec == 12,
              "the loaders' pair loads and the flux workgroups' pair stores assume this field order");
// block and row-in-block of a cell
__device__ __forceinline__ int blk_of(int i, int j, int nw) { return (i + j - 6) * nw + ((j - 3) >> 6); }

// Record, dU*, state and hand-off arrays as raw buffers; loads and stores
// through them carry sc1, the cache policy of ld_agent / st_agent, so they are
// coherent across the device's XCDs.
constexpr int kBufWord3 = 0x00020000;  // gfx9-family descriptor word 3 (raw buffer, stride 0)
constexpr int kCoherent = 16;          // buffer instruction cache policy: sc1
constexpr unsigned kOff = 0x80000000u;  // past every buffer's range: a store there is discarded
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// Global-memory views of the mesh arrays: loads through them are global
// loads also where the compiler cannot infer the address space of a Dev
// field (the flux workgroups' function, the batched kernel's job table)
typedef const __attribute__((address_space(1))) double gdbl;
__device__ __forceinline__ gdbl *gp(const double *p) { return (gdbl *)p; }
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(double *p, size_t doubles) {
  return __builtin_amdgcn_make_buffer_rsrc(p, (short)0, (int)(doubles * sizeof(double)), kBufWord3);
}
__device__ __forceinline__ size_t nblocks(const SyntheticState &st) { return (size_t)st.np * st.nw; }
// dU* and the updated state have kPad more planes at either end, which the
// steps of a last group past the band's last plane store to
__device__ __forceinline__ size_t padded_blocks(const SyntheticState &st) { return (size_t)(st.np + 2 * kPad) * st.nw; }
__device__ __forceinline__ int pblk_of(int i, int j, int nw) { return (i + j - 6 + kPad) * nw + ((j - 3) >> 6); }
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rec_rsrc(const SyntheticState &st) {
  return rsrc_of(st.rec, nblocks(st) * kBlk);
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t ub_rsrc(const SyntheticState &st) {
  return rsrc_of(st.ub, padded_blocks(st) * kBlk4);
}
__device__ __forceinline__ void st_pair(__amdgpu_buffer_rsrc_t r, unsigned voff, int soff, double a, double b) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, double2{a, b}), r, voff, soff, kCoherent);
}
__device__ __forceinline__ double2 ld_pair(__amdgpu_buffer_rsrc_t r, unsigned voff, int soff) {
  return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, kCoherent));
}
// hand-off slots [2 directions][nw bands][nx-5+kPad][4]: the values that the
// edge row of a band passes to the next band, in the order they are made (the
// last kPad are not read).  A slot
// whose doubles hold kEmpty has not been written: a signalling NaN, which no
// arithmetic returns, so each double of a slot says by itself whether it is
// there, and no flag has to follow the data.
constexpr unsigned long long kEmpty = 0x7FF4A5A5A5A5A5A5ull;
constexpr unsigned kEmptyHi = (unsigned)(kEmpty >> 32);
__host__ __device__ inline int hand_len(int nx) { return nx - 5 + kPad; }
__device__ __forceinline__ double *hand_of(const Dev &d, const SyntheticState &st, bool fwd, int band) {
  return st.hand + (size_t)((fwd ? 0 : st.nw) + band) * hand_len(d.nx) * 4;
}

// Every record slot's density and its reciprocal to 1 (the rest stays zero):
// the slots of cells that are not swept keep this finite state for good.  The
// geometry that a cell's terms take, which does not change.  Forward: half
// lengths and normals of the faces towards i+1 and j+1.  Backward: half
// lengths of the cell's own lower faces, and the normals of the lower faces of
// (i-1,j) and (i,j-1), which the reference takes there (src/sub_LU_SGS.f90:82-96).
__global__ void k_rec_init(Dev d, SyntheticState st) {
  const size_t nslot = nblocks(st) * 64;
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nslot) return;
  const size_t blk = t / 64, l = t % 64;
  st.rec[blk * kBlk + (kRecU / 2) * 128 + 2 * l] = 1.0;
  st.rec[blk * kBlk + (kRecRr / 2) * 128 + 2 * l + 1] = 1.0;
  const int p = (int)(blk / st.nw) + 6, j = 3 + 64 * (int)(blk % st.nw) + (int)l, i = p - j;
  if (j > d.ny - 3 || i < 3 || i > d.nx - 3) return;
  const int gpn = geo_pairs(st.axis), g0 = gidx(d, i, j), gi = gidx(d, i + 1, j), gj = gidx(d, i, j + 1);
  double2 *g = reinterpret_cast<double2 *>(st.geo + blk * gpn * 128) + l;
  g[0] = {0.5 * d.si[gi], 0.5 * d.sj[gj]};
  g[64] = {0.5 * d.si[g0], 0.5 * d.sj[g0]};
  if (st.axis) return;
  g[128] = {d.ni1[gi], d.ni2[gi]};
  g[192] = {d.nj1[gj], d.nj2[gj]};
  const int hi = gidx(d, i - 1, j), hj = gidx(d, i, j - 1);
  g[256] = {d.ni1[hi], d.ni2[hi]};
  g[320] = {d.nj1[hj], d.nj2[hj]};
}

// every hand-off slot empty, by the threads t, t + nt, ... of a launch
__device__ void clear_hands(const Dev &d, const SyntheticState &st, size_t t, size_t nt) {
  const size_t n = (size_t)2 * st.nw * hand_len(d.nx) * 4;
  for (; t < n; t += nt) st.hand[t] = __longlong_as_double((long long)kEmpty);
}

// S0 <- S - S0, S00 <- S on interior cells; the kinetic increment added to the
// synthetic state of the previous step on cells 3..n-3 (src/Hybrid_Sub.f90:45-94).
// Also resets the inner loop's control words.
__global__ void k_ns_prepare(Dev d, SyntheticState st) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t == 0) {
    st.ctl[kCtlGo] = (1.0 > st.tol && st.maxit > 0) ? 1 : -1;  // the reference starts from res = 1
    st.ctl[kCtlErr] = 0;
    st.ctl[kCtlBad] = 0;
    st.ctl[kCtlStop] = 0;
    st.ctl[kCtlLast] = 0;
    st.ctl[kCtlArrived] = 0;
    st.iters[0] = 0;
    st.iters[1] = 0;
    st.iters[2] = 0;
  }
  if (t < st.ntx * st.nty) st.ready[t] = 0;      // no iteration's fluxes done
  if (t < st.nw) st.prog[kProgStride * t] = 0;   // no plane of a backward sweep done
  clear_hands(d, st, t, (size_t)gridDim.x * blockDim.x);
  const int nc = (d.nx - 1) * (d.ny - 1);
  if (t >= nc) return;
  const int i = t % (d.nx - 1) + 1, j = t / (d.nx - 1) + 1;
  const int N = d.ncell, c = cidx(d, i, j);
  for (int k = 0; k < 10; k++) d.S0[k * N + c] = d.S[k * N + c] - d.S0[k * N + c];
  for (int k = 0; k < 4; k++) st.s00[k * N + c] = d.S[k * N + c];
  if (i < 3 || i > d.nx - 3 || j < 3 || j > d.ny - 3) return;
  const double sq = sqrt(2.0 / d.gamma), cv = d.cv;
  const double trho = d.S0[c], tu = d.S0[N + c] / d.ma * sq, tv = d.S0[2 * N + c] / d.ma * sq, tt = d.S0[3 * N + c];
  const double *U0 = d.U0;
  double rns = U0[c];
  double uns = U0[N + c] / U0[c], vns = U0[2 * N + c] / U0[c];
  double tns = (U0[3 * N + c] - 0.5 * U0[c] * (uns * uns + vns * vns)) / (cv * U0[c]);
  rns = rns + trho; uns = uns + tu; vns = vns + tv; tns = tns + tt;
  d.U[c] = rns;
  d.U[N + c] = rns * uns;
  d.U[2 * N + c] = rns * vns;
  d.U[3 * N + c] = cv * tns * rns + 0.5 * rns * (uns * uns + vns * vns);
  for (int m = 0; m < 4; m++) d.U2[m * N + c] = d.U[m * N + c];
}

__device__ __forceinline__ double minmod_ns(double a, double b) {  // src/sub_Residual.f90:357-368
  if (a * b <= 0.0) return 0.0;
  return (fabs(a) <= fabs(b)) ? a : b;
}

// Flux_Van_Leer_1Da, src/sub_flux_split.f90:141-192
__device__ void van_leer(const double ql[4], const double qr[4], double g, double f[4]) {
  const double dl = ql[0], uul = ql[1], vvl = ql[2], pl = ql[3];
  const double dr = qr[0], uur = qr[1], vvr = qr[2], pr = qr[3];
  const double al = sqrt(g * pl / dl), ar = sqrt(g * pr / dr);
  const double ml = uul / al, mr = uur / ar;
  double fp[4] = {0, 0, 0, 0}, fm[4] = {0, 0, 0, 0};
  if (ml >= 1.0) {
    fp[0] = dl * uul;
    fp[1] = dl * uul * uul + pl;
    fp[2] = dl * uul * vvl;
    fp[3] = uul * (g * pl / (g - 1.0) + 0.5 * dl * (uul * uul + vvl * vvl));
  } else if (fabs(ml) < 1.0) {
    const double mp = 0.25 * (1.0 + ml) * (1.0 + ml);
    const double t0 = dl * al * mp;
    fp[0] = t0;
    fp[1] = t0 * ((g - 1.0) * uul + 2.0 * al) / g;
    fp[2] = t0 * vvl;
    fp[3] = t0 * (((g - 1.0) * uul + 2.0 * al) * ((g - 1.0) * uul + 2.0 * al) * 0.5 / (g * g - 1.0) + 0.5 * (vvl * vvl));
  }
  if (mr >= 1.0) {
  } else if (fabs(mr) < 1.0) {
    const double mm = -0.25 * (mr - 1.0) * (mr - 1.0);
    const double t0 = dr * ar * mm;
    fm[0] = t0;
    fm[1] = t0 * ((g - 1.0) * uur - 2.0 * ar) / g;
    fm[2] = t0 * vvr;
    fm[3] = t0 * (((g - 1.0) * uur - 2.0 * ar) * ((g - 1.0) * uur - 2.0 * ar) * 0.5 / (g * g - 1.0) + 0.5 * (vvr * vvr));
  } else {
    fm[0] = dr * uur;
    fm[1] = dr * uur * uur + pr;
    fm[2] = dr * uur * vvr;
    fm[3] = uur * (g * pr / (g - 1.0) + 0.5 * dr * (uur * uur + vvr * vvr));
  }
  for (int m = 0; m < 4; m++) f[m] = fp[m] + fm[m];
}

// comput_DFn (src/sub_LU_SGS.f90:122-143): DF = F.n(U + dU) - F.n(U) on the
// unit normal (n1, n2).  F.n is linear in n: F.n = Fx n1 + Fy n2 with the
// Euler fluxes Fx, Fy of the state, so a cell's DF on any normal is
// (Fx(U+dU) - Fx(U)) n1 + (Fy(U+dU) - Fy(U)) n2.  The first components of the
// two differences are dU(2) and dU(3), and Fx(3) = Fy(2), so five components
// are left to form.

// 1/a: the hardware reciprocal (23 bits) and one step r(1 + e + e^2), e =
// 1 - a r, whose error is e^3: about 1 ulp
__device__ __forceinline__ double rcp_nr(double a) {
  const double r = __builtin_amdgcn_rcp(a);
  const double e = fma(-a, r, 1.0);
  return fma(r, fma(e, e, e), r);
}
// velocities, pressure and pressure + energy of a state with r = 1/u[0]
struct Euler {
  double vx, vy, p, e;
  __device__ Euler(const double u[4], double r, double g1) {
    const double kin = fma(u[1], u[1], u[2] * u[2]);
    const double ei = fma(-0.5 * kin, r, u[3]);
    p = g1 * ei;
    e = fma(g1, ei, u[3]);
    vx = u[1] * r;
    vy = u[2] * r;
  }
};

// a flux workgroup's tile
struct FluxShared {
  double U[4][kTC];    // tile + halo
  double pr[5][kTC];   // d, u, v, T, p (comput_duvtpckw)
  double mu[kTC];      // amu_of
  double fi[4][(kTI + 1) * kTJ];  // i-face fluxes, face (i0+a, j0+b) at b*(kTI+1)+a
  double fj[4][kTI * (kTJ + 1)];  // j-face fluxes, face (i0+a, j0+b) at b*kTI+a
  double red[kThreads / 64];
  int word;
};
// a sweep workgroup's records and words (see sweep_pass)
constexpr int kLdsPairs = 9;  // pairs of a prepared record, without the normals
template <bool kAxis>
struct SweepShared {
  static constexpr int kPairs = kAxis ? kLdsPairs : kLdsPairs + 2;
  static constexpr int kStep = kPairs * 128;  // doubles of a step's records
  double ring[kGroups * kGroup][kPairs * 128];  // prepared records, pair q of lane l at q*128 + 2l
  double hand[kHand + 2][4];         // values received from the neighbouring band; two that stay zero
  int avail[kGroups];  // 1 + the running number of the group of steps that a ring slot holds
  int used;            // half groups whose records the sweep has read
  int hand_n;          // values received
  int fwd_done, bwd_done;  // iterations whose sweeps are complete, their stores at memory
  int bgo;             // iterations whose backward sweep may begin
  int clr;             // iterations after whose backward sweep its hand-off slots are empty again
  int quit;            // a wait timed out, or the loop has ended
};

// the tile's cell fields for ns_face_of
struct TileCells {
  const FluxShared &sh;
  int ib, jb;  // cell (ib, jb) is LDS cell 0
  __device__ int l(int i, int j) const { return (j - jb) * kCI + (i - ib); }
  __device__ double u(int i, int j) const { return sh.pr[1][l(i, j)]; }
  __device__ double v(int i, int j) const { return sh.pr[2][l(i, j)]; }
  __device__ double T(int i, int j) const { return sh.pr[3][l(i, j)]; }
  __device__ double mu(int i, int j) const { return sh.mu[l(i, j)]; }
};
struct MeshCells {
  const Dev &d;
  __device__ double x1(int i, int j) const { return gp(d.x1)[cidx(d, i, j)]; }
  __device__ double y1(int i, int j) const { return gp(d.y1)[cidx(d, i, j)]; }
};

// What a thread's part of a tile takes from the mesh, read before the wait for
// the tile's state: a face (threads below kFaceThreads), or kCells cells.
constexpr int kFaceThreads = kThreads - 64;                 // the last wavefront has the cells
constexpr int kCells = (kTI * kTJ + 63) / 64;
static_assert((kTI + 1) * kTJ + kTI * (kTJ + 1) <= kFaceThreads, "a face per thread");
struct TileGeo {
  int i0, j0, nci, ncj;
  int dir, i, j;  // face; dir < 0: none
  double s, n1, n2, t11, t22, t12, qx, qy;
  NsMetric m;
  double vol[kCells], si[kCells], sj[kCells], ni1[kCells], ni2[kCells], nj1[kCells], nj2[kCells];
};
// cell t of a tile: threads run along wrapped anti-diagonals, whose cells are
// consecutive in the blocked arrays
__device__ __forceinline__ int cell_b(int t) { return t % kTJ; }
__device__ __forceinline__ int cell_a(int t) { return (t / kTJ - t % kTJ) & (kTI - 1); }

__device__ __forceinline__ void tile_geo(const Dev &d, const SyntheticState &st, int tile, TileGeo &g) {
  const int tid = threadIdx.x;
  g.i0 = 3 + (tile % st.ntx) * kTI;
  g.j0 = 3 + (tile / st.ntx) * kTJ;
  g.nci = min(kTI, d.nx - 3 - g.i0 + 1);
  g.ncj = min(kTJ, d.ny - 3 - g.j0 + 1);
  g.dir = -1;
  if (tid < kFaceThreads) {
    const int nfi = (g.nci + 1) * g.ncj, nfj = g.nci * (g.ncj + 1);
    if (tid >= nfi + nfj) return;
    g.dir = tid < nfi ? 0 : 1;
    g.i = g.i0 + (g.dir == 0 ? tid % (g.nci + 1) : (tid - nfi) % g.nci);
    g.j = g.j0 + (g.dir == 0 ? tid / (g.nci + 1) : (tid - nfi) / g.nci);
    const int q = gidx(d, g.i, g.j), c = cidx(d, g.i, g.j), N = d.ncell;
    g.s = gp(g.dir == 0 ? d.si : d.sj)[q];
    g.n1 = gp(g.dir == 0 ? d.ni1 : d.nj1)[q];
    g.n2 = gp(g.dir == 0 ? d.ni2 : d.nj2)[q];
    if (!st.if_viscous) return;
    gdbl *tg = gp(g.dir == 0 ? d.taoi : d.taoj), *qg = gp(g.dir == 0 ? d.qi : d.qj);
    g.t11 = tg[c];
    g.t22 = tg[N + c];
    g.t12 = tg[2 * N + c];
    g.qx = qg[c];
    g.qy = qg[N + c];
    g.m = ns_metric_of(MeshCells{d}, g.dir, g.i, g.j);
    return;
  }
#pragma unroll
  for (int r = 0; r < kCells; r++) {
    const int t = tid - kFaceThreads + 64 * r, i = g.i0 + min(cell_a(t), g.nci - 1), j = g.j0 + min(cell_b(t), g.ncj - 1);
    const int g0 = gidx(d, i, j), gi = gidx(d, i + 1, j), gj = gidx(d, i, j + 1);
    g.vol[r] = gp(d.vol)[g0];
    g.si[r] = 0.5 * (gp(d.si)[g0] + gp(d.si)[gi]);
    g.ni1[r] = 0.5 * (gp(d.ni1)[g0] + gp(d.ni1)[gi]);
    g.ni2[r] = 0.5 * (gp(d.ni2)[g0] + gp(d.ni2)[gi]);
    g.sj[r] = 0.5 * (gp(d.sj)[g0] + gp(d.sj)[gj]);
    g.nj1[r] = 0.5 * (gp(d.nj1)[g0] + gp(d.nj1)[gj]);
    g.nj2[r] = 0.5 * (gp(d.nj2)[g0] + gp(d.nj2)[gj]);
  }
}

// Residual_FVM face flux (src/sub_Residual.f90:68-202, :210-338) of the
// thread's face, primitives from the tile in LDS
__device__ __forceinline__ void face_flux(const Dev &d, const FluxShared &sh, const TileGeo &g, bool visc,
                                          double fl[4]) {
  const TileCells tc{sh, g.i0 - 2, g.j0 - 2};
  const int c0 = tc.l(g.i, g.j), step = g.dir == 0 ? 1 : kCI;
  double ul[4], ur[4];
  for (int m = 0; m < 4; m++) {
    const double *q = sh.pr[m < 3 ? m : 4] + c0;  // d, u, v, p
    const double u1 = q[-2 * step], u2 = q[-step], u3 = q[0], u4 = q[step];
    ul[m] = u2 + 0.5 * minmod_ns(u2 - u1, u3 - u2);
    ur[m] = u3 - 0.5 * minmod_ns(u3 - u2, u4 - u3);
  }
  const double s = g.s, n1 = g.n1, n2 = g.n2;
  const double ql[4] = {ul[0], ul[1] * n1 + ul[2] * n2, -ul[1] * n2 + ul[2] * n1, ul[3]};
  const double qr[4] = {ur[0], ur[1] * n1 + ur[2] * n2, -ur[1] * n2 + ur[2] * n1, ur[3]};
  double f0[4];
  van_leer(ql, qr, d.gamma, f0);
  fl[0] = -f0[0] * s;
  fl[1] = -(f0[1] * n1 - f0[2] * n2) * s;
  fl[2] = -(f0[1] * n2 + f0[2] * n1) * s;
  fl[3] = -f0[3] * s;
  if (!visc) return;
  double o[8];
  ns_face_of(tc, d, g.m, g.dir, g.i, g.j, o);
  const double t11 = o[0] + g.t11, t22 = o[1] + g.t22, t12 = o[2] + g.t12;
  const double qx = o[4] + g.qx, qy = o[5] + g.qy;
  const double u1 = o[6], v1 = o[7];
  const double e1 = u1 * t11 + v1 * t12 + qx;
  const double e2 = u1 * t12 + v1 * t22 + qy;
  fl[1] = fl[1] + (t11 * n1 + t12 * n2) * s;
  fl[2] = fl[2] + (t12 * n1 + t22 * n2) * s;
  fl[3] = fl[3] + (e1 * n1 + e2 * n2) * s;
}

// One tile of Comput_Residual_one_mesh (src/sub_NS_singlegrid.f90:45-114):
// comput_duvtpckw with its T<0.1 stop, get_viscous, the face fluxes, Res,
// comput_Lvc, comput_dt and the LU-SGS diagonal (src/sub_LU_SGS.f90:34-36),
// stored as sweep records.  Returns the thread's max |Res_4| and T<0.1 flag.
// The time of a tile is the chain of its phases (state, faces, residual), not
// their work: the last wavefront forms what the cells need besides the fluxes
// beside the faces.
__device__ __forceinline__ void flux_tile(const Dev &d, const SyntheticState &st, FluxShared &sh, const TileGeo &tg,
                                          bool first, double &rmax, int &bad) {
  const int nx = d.nx, ny = d.ny, N = d.ncell, i0 = tg.i0, j0 = tg.j0;
  const int tid = threadIdx.x, nw = st.nw;
  const double g = d.gamma;
  const bool visc = st.if_viscous != 0;
  const TileCells tc{sh, i0 - 2, j0 - 2};
  // U of the loop's start is in the mesh array; later iterations read the
  // swept cells from the sweeps' blocked array
  const __amdgpu_buffer_rsrc_t ru = ub_rsrc(st);
  static_assert(kTC <= kThreads, "a cell with halo per thread");
  if (tid < kTC) {
    const int b = tid % kCJ, a = (tid / kCJ + 2 * kCI - b) % kCI;
    const int i = i0 - 2 + a, j = j0 - 2 + b, l = b * kCI + a;
    if (i <= nx + 1 && j <= ny + 1) {
      double u[4];
      if (!first && i >= 3 && i <= nx - 3 && j >= 3 && j <= ny - 3) {
        const unsigned o = (unsigned)pblk_of(i, j, nw) * (kBlk4 * 8u) + 16u * ((j - 3) & 63);
        const double2 u01 = ld_pair(ru, o, 0), u23 = ld_pair(ru, o + 1024u, 0);
        u[0] = u01.x; u[1] = u01.y; u[2] = u23.x; u[3] = u23.y;
      } else {
        const int c = cidx(d, i, j);
        for (int m = 0; m < 4; m++) u[m] = gp(d.U)[m * N + c];
      }
      for (int m = 0; m < 4; m++) sh.U[m][l] = u[m];
      const double dd = u[0], uu = u[1] / dd, vv = u[2] / dd;
      const double T = (u[3] - 0.5 * dd * (uu * uu + vv * vv)) / (d.cv * dd);
      sh.pr[0][l] = dd;
      sh.pr[1][l] = uu;
      sh.pr[2][l] = vv;
      sh.pr[3][l] = T;
      sh.pr[4][l] = (1. / (g * d.ma * d.ma)) * dd * T;
      sh.mu[l] = visc ? 1. / d.re * pow(T, 0.8100000023841858) : 0.0;
      if (i >= 1 && i <= nx - 1 && j >= 1 && j <= ny - 1 && T < 0.10000000149011612) bad = 1;
    }
  }
  __syncthreads();
  const __amdgpu_buffer_rsrc_t rr = rec_rsrc(st);
  if (tid < kFaceThreads) {
    if (tg.dir >= 0) {
      double fl[4];
      face_flux(d, sh, tg, visc, fl);
      const int a = tg.i - i0, b = tg.j - j0;
      if (tg.dir == 0)
        for (int m = 0; m < 4; m++) sh.fi[m][b * (kTI + 1) + a] = fl[m];
      else
        for (int m = 0; m < 4; m++) sh.fj[m][b * kTI + a] = fl[m];
    }
  } else {
#pragma unroll
    for (int r = 0; r < kCells; r++) {
      const int t = tid - kFaceThreads + 64 * r, a = cell_a(t), b = cell_b(t), i = i0 + a, j = j0 + b;
      if (t >= kTI * kTJ || a >= tg.nci || b >= tg.ncj) continue;
      // comput_Lvc and comput_dt (src/sub_NS_singlegrid.f90:160-221)
      const int lc = tc.l(i, j);
      const double s0 = tg.vol[r], si = tg.si[r], sj = tg.sj[r];
      const double uu = sh.pr[1][lc], vv = sh.pr[2][lc];
      const double uni = uu * tg.ni1[r] + vv * tg.ni2[r], unj = uu * tg.nj1[r] + vv * tg.nj2[r];
      const double cc = sqrt(sh.pr[3][lc]) / d.ma;
      const double lci = (fabs(uni) + cc) * si, lcj = (fabs(unj) + cc) * sj;
      const double tmp1 = g / sh.pr[0][lc] * (sh.mu[lc] / d.pr + 0.0 / 0.9);
      const double lvi = visc ? tmp1 * si * si / s0 : 0.0, lvj = visc ? tmp1 * sj * sj / s0 : 0.0;
      double dt;
      if (!st.local_dt) dt = d.dt;
      else {
        dt = st.cfl * s0 / (lci + lcj + 1.0 * (lvi + lvj));
        if (dt > st.dtmax) dt = st.dtmax;
        if (dt < st.dtmin) dt = st.dtmin;
      }
      double alfa = s0 / dt + 1.0 * (lci + lcj);
      if (visc) alfa = alfa + 2.0 * (lvi + lvj);
      const unsigned o = (unsigned)blk_of(i, j, nw) * (kBlk * 8u) + 16u * ((j - 3) & 63);
      st_pair(rr, o + (kRecU / 2) * 1024u, 0, sh.U[0][lc], sh.U[1][lc]);
      st_pair(rr, o + (kRecU / 2 + 1) * 1024u, 0, sh.U[2][lc], sh.U[3][lc]);
      st_pair(rr, o + (kRecRa / 2) * 1024u, 0, 1.0 / alfa, 0.5 * lci + lvi);            // ra, cbi
      st_pair(rr, o + (kRecCbj / 2) * 1024u, 0, 0.5 * lcj + lvj, rcp_nr(sh.U[0][lc]));  // cbj, 1/rho
    }
  }
  __syncthreads();
  if (tid < kTI * kTJ) {
    const int a = cell_a(tid), b = cell_b(tid), i = i0 + a, j = j0 + b;
    if (a < tg.nci && b < tg.ncj) {
      double res[4];
      for (int m = 0; m < 4; m++)
        res[m] = sh.fi[m][b * (kTI + 1) + a + 1] - sh.fi[m][b * (kTI + 1) + a] + sh.fj[m][(b + 1) * kTI + a] -
                 sh.fj[m][b * kTI + a];
      rmax = fabs(res[3]);
      const unsigned o = (unsigned)blk_of(i, j, nw) * (kBlk * 8u) + 16u * ((j - 3) & 63);
      st_pair(rr, o + (kRecRes / 2) * 1024u, 0, res[0], res[1]);
      st_pair(rr, o + (kRecRes / 2 + 1) * 1024u, 0, res[2], res[3]);
    }
  }
}

// x of lane l-1 (FWD, wave_shr:1) or l+1 (wave_shl:1) of the wavefront; edge
// in the lane that has no such neighbour (lane 0, or lane 63)
template <bool FWD>
__device__ __forceinline__ double lane_shift(double x, double edge) {
  const unsigned long long b = __double_as_longlong(x), e = __double_as_longlong(edge);
  const int lo = (int)(unsigned)b, hi = (int)(unsigned)(b >> 32), el = (int)(unsigned)e, eh = (int)(unsigned)(e >> 32);
  constexpr int kCtrl = FWD ? 0x138 : 0x130;
  const int l = __builtin_amdgcn_update_dpp(el, lo, kCtrl, 0xf, 0xf, false);
  const int h = __builtin_amdgcn_update_dpp(eh, hi, kCtrl, 0xf, 0xf, false);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)h << 32) | (unsigned)l));
}

// LDS words read and written by several wavefronts of a workgroup; values
// are wavefront-uniform
__device__ __forceinline__ int lds_get(int *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
__device__ __forceinline__ void lds_put(int *p, int v) {
  if ((threadIdx.x & 63) == 0) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ void mem_order() { asm volatile("" ::: "memory"); }  // no compiler reordering
__device__ __forceinline__ void vm_wait() {  // this wavefront's stores are at memory
  mem_order();
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  mem_order();
}

// A bounded wait's bookkeeping: every 64 polls it looks for the end of the
// loop (the error word; for the waits of a sweep, the stop word too) and for
// the time; a timeout sets the error word.
struct Patience {
  int *ctl;
  long long t0 = 0;
  int n = 0;
  __device__ explicit Patience(int *c) : ctl(c) {}
  __device__ bool over(bool stop_too) {
    if ((++n & 63) != 0) return false;
    if (uniform(ld_agent(ctl + kCtlErr)) != 0 || (stop_too && uniform(ld_agent(ctl + kCtlStop)) != 0)) return true;
    if (n == 64) t0 = wall_clock64();
    if (wall_clock64() - t0 > kWaitTicks) {
      st_agent(ctl + kCtlErr, 1);
      return true;
    }
    return false;
  }
};

// Waits until the LDS word *p has reached want (in wrapping order); false
// when the loop has ended instead.
template <class Sh>
__device__ bool wait_lds(int *p, int want, Sh &sh, int *ctl) {
  Patience pt(ctl);
  while (uniform(lds_get(p)) - want < 0) {
    if (uniform(lds_get(&sh.quit))) return false;
    __builtin_amdgcn_s_sleep(1);
    if (pt.over(true)) {
      lds_put(&sh.quit, 1);
      return false;
    }
  }
  mem_order();
  return true;
}
// Waits for the word after iteration k: whether iteration k+1 runs.
template <class Sh>
__device__ bool next_iteration(int k, Sh &sh, int *ctl) {
  Patience pt(ctl);
  int go;
  while ((go = uniform(ld_agent(ctl + kCtlGo))) == k) {
    if (uniform(lds_get(&sh.quit))) return false;
    __builtin_amdgcn_s_sleep(4);
    if (pt.over(true)) {
      lds_put(&sh.quit, 1);
      return false;
    }
  }
  mem_order();
  return go == k + 1;
}

// the plane steps of a band: rows j0 .. j0+rows-1, planes first .. last
struct Band {
  int w, j0, rows, first, last, n, groups;
  int links;  // values handed from band to band in a sweep

  __device__ Band(const Dev &d, int band) : w(band), j0(3 + kBand * band) {
    rows = min(kBand, d.ny - 3 - j0 + 1);
    first = j0 + 3;
    last = d.nx - 3 + j0 + rows - 1;
    n = last - first + 1;
    groups = (n + kGroup - 1) / kGroup;
    links = d.nx - 5;
  }
};

// A prepared record of a lane's cell: Res/alfa (forward) or dU* (backward),
// U, the inverse diagonal, the weights towards the cells that use this one as
// their neighbour (hi, hj negated in a backward sweep), and those components
// of the Euler fluxes of U that are not U's own: f = Fx(2), Fx(3) = Fy(2),
// Fx(4), Fy(3), Fy(4); ni, nj: the normals of the faces towards those cells.
struct Rec {
  double r[4], u[4], ra, cbi, cbj, hi, hj, f[5], ni[2], nj[2];
};
template <bool kAxis>
__device__ __forceinline__ void read_rec(const double *slot, int lane, Rec &x) {
  const double2 *s = reinterpret_cast<const double2 *>(slot) + lane;
  const double2 a = s[0], b = s[64], c = s[128], e = s[192], f = s[256], g = s[320], h = s[384], k = s[448], l = s[512];
  x.r[0] = a.x; x.r[1] = a.y; x.r[2] = b.x; x.r[3] = b.y;
  x.u[0] = c.x; x.u[1] = c.y; x.u[2] = e.x; x.u[3] = e.y;
  x.ra = f.x; x.cbi = f.y;
  x.cbj = g.x; x.hi = g.y;
  x.hj = h.x; x.f[0] = h.y;
  x.f[1] = k.x; x.f[2] = k.y;
  x.f[3] = l.x; x.f[4] = l.y;
  if (!kAxis) {
    const double2 o = s[576], q = s[640];
    x.ni[0] = o.x; x.ni[1] = o.y;
    x.nj[0] = q.x; x.nj[1] = q.y;
  }
}

// One sweep of a band by its sweep wavefront: du_LU_SGS_2D
// (src/sub_LU_SGS.f90:4-113), forward dU* = (Res + dui + duj)/alfa on planes
// first .. last (:26-69) or backward dU = dU* + (dui + duj)/alfa on planes
// last .. first (:73-111) and U + dU.  Lane l owns row j0 + l; a step visits
// one plane.  The off-diagonal term that cell (i,j) adds to (i+1,j) (forward;
// (i-1,j) backward) stays in the lane, the one for (i,j+1) moves to the next
// lane, or through memory to the next band:
//   forward:  dui = 0.5 (DF si(i,j) + Lci(i-1,j) dU) + Lvi(i-1,j) dU      (:44-49)
//   backward: dui = -0.5 (DF si(i+1,j) - Lci(i+1,j) dU) + Lvi(i+1,j) dU   (:82-86)
// with DF = F.n(U+dU) - F.n(U) of the neighbour (comput_DFn, :122-143): all
// of a term's factors belong to the neighbour and to the face between, so the
// neighbour forms the whole term and four values move, not eleven.  Terms
// across faces to cells that are not swept (src/sub_LU_SGS.f90:44-56) vanish
// without a test: the slots of such cells hold U = (1,0,0,0) and zero weights.
//
// What bounds a step is the number of the wavefront's instructions: a lone
// wavefront issues one in about 5 cycles, of whatever kind, and a step takes
// about 42 FP64 operations in about 75.  Nothing it executes waits for memory.
// Records come through LDS, prepared by the loader wavefronts; the
// neighbouring band's values come through LDS, brought by the receiver; both
// are read a step before they are used, and the words that say that they are
// there are looked at once in kGroup steps.  Its only memory instructions are
// stores, whose completion it waits for once per sweep (and, eight steps
// late, where it publishes the progress that the flux workgroups follow).
template <bool FWD, bool kAxis>
__device__ __forceinline__ bool sweep_pass(const Dev &d, const SyntheticState &st, SweepShared<kAxis> &sh,
                                           const Band &bd, int k, int &group, int &hseq) {
  static_assert(kGroup == 4 && kGroups == 2, "the loop below");
  const int lane = threadIdx.x & 63, nw = st.nw;
  const double g1 = d.gamma - 1.0;
  const bool has_from = FWD ? bd.w > 0 : bd.w < nw - 1, has_to = FWD ? bd.w < nw - 1 : bd.w > 0;
  const int n_in = has_from ? bd.links : 0;
  int *ctl = st.ctl;
  const __amdgpu_buffer_rsrc_t rs = rsrc_of(FWD ? st.dstar : st.ub, padded_blocks(st) * kBlk4);
  const __amdgpu_buffer_rsrc_t rh = rsrc_of(hand_of(d, st, FWD, bd.w), (size_t)hand_len(d.nx) * 4);
  // the edge row's values go out from the step of its first cell to the last step
  const unsigned v_out = lane == (FWD ? kBand - 1 : 0) ? 0u : kOff;
  const int out_from = has_to ? (FWD ? kBand - 1 : bd.rows - 1) : 0x7fffffff;
  int h_out = 0;
  // every lane stores every step: a slot without a cell gets zeros (forward) or is not read (backward)
  constexpr int kBlkBytes = kBlk4 * 8;
  const unsigned v_st = (unsigned)lane * 16u;
  int soff = (((FWD ? bd.first : bd.last) - 6 + kPad) * nw + bd.w) * kBlkBytes;  // block of the step's plane
  const int dsoff = (FWD ? nw : -nw) * kBlkBytes;
  // of the lane's previous cell: dU, DF across the i-face and their weights; the term for the next lane
  double du[4] = {0, 0, 0, 0}, fi[4] = {0, 0, 0, 0}, hi = 0.0, cbi = 0.0, to[4] = {0, 0, 0, 0}, t[4];
  double in0[4], in1[4];  // values from the neighbouring band for the next two steps
  int hn = 0;
  // (zeros without a neighbour; past the last value any finite value does, as
  // the edge lane has no cell there)
  const double *hands = sh.hand[has_from ? 0 : kHand];
  const int hmask = has_from ? kHand - 1 : 0;
  auto fetch_hands = [&](int s) {
    const double2 *h = reinterpret_cast<const double2 *>(hands + 4 * (s & hmask));
    const double2 a = h[0], b = h[1], c = h[2], e = h[3];  // kHand is even: no wrap
    in0[0] = a.x; in0[1] = a.y; in0[2] = b.x; in0[3] = b.y;
    in1[0] = c.x; in1[1] = c.y; in1[2] = e.x; in1[3] = e.y;
  };
  // the word, then the values: LDS performs a wavefront's operations in order
  auto fetch_next_hands = [&](int s) {
    hn = lds_get(&sh.hand_n);
    mem_order();
    fetch_hands(s);
  };
  auto gather = [&](const double in[4]) {  // the off-diagonal terms of this step's cells
    for (int m = 0; m < 4; m++) t[m] = fma(hi, fi[m], fma(cbi, du[m], lane_shift<FWD>(to[m], in[m])));
  };
  auto step = [&](int s, const Rec &x) {
    double u[4];
    for (int m = 0; m < 4; m++) {
      du[m] = fma(t[m], x.ra, x.r[m]);
      u[m] = x.u[m] + du[m];
    }
    const double *q = FWD ? du : u;  // dU* or the updated state
    st_pair(rs, v_st, soff, q[0], q[1]);
    st_pair(rs, v_st + 1024u, soff, q[2], q[3]);
    soff += dsoff;
    const Euler w(u, rcp_nr(u[0]), g1);
    const double dx[4] = {du[1], fma(u[1], w.vx, w.p) - x.f[0], fma(u[2], w.vx, -x.f[1]), fma(w.e, w.vx, -x.f[2])};
    const double dy[4] = {du[2], dx[2], fma(u[2], w.vy, w.p) - x.f[3], fma(w.e, w.vy, -x.f[4])};
    for (int m = 0; m < 4; m++) {
      const double fj = kAxis ? dy[m] : fma(dy[m], x.nj[1], dx[m] * x.nj[0]);
      fi[m] = kAxis ? dx[m] : fma(dy[m], x.ni[1], dx[m] * x.ni[0]);
      to[m] = fma(x.hj, fj, x.cbj * du[m]);
    }
    hi = x.hi;
    cbi = x.cbi;
    if (s >= out_from) {
      st_pair(rh, v_out, h_out, to[0], to[1]);
      st_pair(rh, v_out + 16u, h_out, to[2], to[3]);
      h_out += 32;
    }
  };
  Rec x, y;
  if (!wait_lds(&sh.avail[group & 1], group + 1, sh, ctl)) return false;
  read_rec<kAxis>(sh.ring[(group & 1) * kGroup], lane, x);
  mem_order();
  fetch_next_hands(0);
  for (int q = 0; q < bd.groups; q++) {
    const int s = kGroup * q;
    const double *ring = sh.ring[(group & 1) * kGroup];
    if (s < n_in) {
      const int need = hseq + min(s + kGroup, n_in);
      if (uniform(hn) - need < 0) {  // read too early
        if (!wait_lds(&sh.hand_n, need, sh, ctl)) return false;
        fetch_hands(s);
      }
    }
    mem_order();
    read_rec<kAxis>(ring + SweepShared<kAxis>::kStep, lane, y);
    gather(in0);
    step(s, x);
    mem_order();
    lds_put(&sh.used, 2 * group + 1);  // the first half's records are read, in order
    read_rec<kAxis>(ring + 2 * SweepShared<kAxis>::kStep, lane, x);
    gather(in1);
    fetch_hands(s + 2);
    step(s + 1, y);
    mem_order();
    read_rec<kAxis>(ring + 3 * SweepShared<kAxis>::kStep, lane, y);
    group++;
    const int av = lds_get(&sh.avail[group & 1]);
    gather(in0);
    step(s + 2, x);
    mem_order();
    lds_put(&sh.used, 2 * group);  // all of the group's records
    if (uniform(av) - (group + 1) < 0 && q + 1 < bd.groups &&
        !wait_lds(&sh.avail[group & 1], group + 1, sh, ctl))
      return false;
    mem_order();
    read_rec<kAxis>(sh.ring[(group & 1) * kGroup], lane, x);  // (after the last group: not used)
    gather(in1);
    fetch_next_hands(s + 4);
    step(s + 3, y);
    if (!FWD && (q & 1) != 0) {
      // at most 16 memory operations (two to four a step) are not complete:
      // all but the last eight steps are
      mem_order();
      __builtin_amdgcn_s_waitcnt(0x4F70);  // vmcnt(16)
      mem_order();
      if (lane == 0) st_agent(st.prog + kProgStride * bd.w, ((long long)k << 32) | (s + kGroup - 8));
    }
  }
  hseq += n_in;
  return true;
}

// The sweep wavefront's loop.
template <bool kAxis>
__device__ __forceinline__ void sweeper(const Dev &d, const SyntheticState &st, SweepShared<kAxis> &sh, const Band &bd) {
  int group = 0, hseq = 0;
  __builtin_amdgcn_s_setprio(3);  // before the workgroup's other wavefront on this SIMD
  for (int k = st.k0;; k++) {
    if (k > st.k0 && !wait_lds(&sh.clr, k - 1, sh, st.ctl)) break;
    if (!sweep_pass<true, kAxis>(d, st, sh, bd, k, group, hseq)) break;
    vm_wait();
    lds_put(&sh.fwd_done, k);
    if (!wait_lds(&sh.bgo, k, sh, st.ctl)) break;
    if (!sweep_pass<false, kAxis>(d, st, sh, bd, k, group, hseq)) break;
    vm_wait();
    if ((threadIdx.x & 63) == 0) st_agent(st.prog + kProgStride * bd.w, ((long long)k << 32) | bd.n);
    lds_put(&sh.bwd_done, k);
    if (!next_iteration(k, sh, st.ctl)) break;
  }
  lds_put(&sh.quit, 1);
}

// A loader wavefront (id = 0 .. kLoaders-1): fetches the records of every
// kLoaders-th group of plane steps into registers, forms what a step needs
// besides the recurrence (the Euler fluxes of U), and hands them on through
// LDS when the sweep has read what was there.  The loads in flight are held in this wavefront's registers (kGroup
// steps of 7 KiB in each of kLoaders wavefronts), so two groups of LDS do.  A
// forward sweep follows the flux workgroups tile by tile: the records of plane
// p exist when the tiles of the levels up to (p-6)/kTI in the band's rows are
// done.
template <bool kAxis>
__device__ __forceinline__ void loader(const Dev &d, const SyntheticState &st, SweepShared<kAxis> &sh, const Band &bd,
                                       int id) {
  const int lane = threadIdx.x & 63, nw = st.nw;
  const double g1 = d.gamma - 1.0;
  constexpr int kGeo = kAxis ? 2 : 6;
  const __amdgpu_buffer_rsrc_t rr = rec_rsrc(st);
  const __amdgpu_buffer_rsrc_t rd = rsrc_of(st.dstar, padded_blocks(st) * kBlk4);
  const __amdgpu_buffer_rsrc_t rg = rsrc_of(st.geo, nblocks(st) * kGeo * 128);
  const unsigned v = (unsigned)lane * 16u;
  int gbase = 0;  // groups of the sweeps before this one
  for (int k = st.k0;; k++) {
    for (int dir = 0; dir < 2; dir++) {
      const bool fwd = dir == 0;
      int level = kLev * kBandTiles * bd.w;  // the tiles of lower levels are done
      // whether the tiles of group gr are done, as far as one look at each further level says
      auto look = [&](int gr) -> bool {
        const int top = min((bd.first + min((gr + 1) * kGroup, bd.n) - 1 - 6) / kTI,
                            st.ntx - 1 + kLev * (kBandTiles * (bd.w + 1) - 1));
        for (; level <= top; level++) {
          const int b = kBandTiles * bd.w + lane, a = level - kLev * b;
          const bool mine = lane < kBandTiles && b < st.nty && a >= 0 && a < st.ntx;
          if (__any(mine && ld_agent(st.ready + (mine ? b * st.ntx + a : 0)) < k)) return false;
        }
        mem_order();
        return true;
      };
      if (!fwd && !wait_lds(&sh.fwd_done, k, sh, st.ctl)) return;  // dU* is at memory
      for (int gr = id; gr < bd.groups; gr += kLoaders) {
        const int s0 = gr * kGroup;
        if (fwd) {
          Patience pt(st.ctl);
          while (!look(gr)) {
            if (uniform(lds_get(&sh.quit))) return;
            if (pt.over(true)) {
              lds_put(&sh.quit, 1);
              return;
            }
          }
        }
        double2 q[kGroup][9];
#pragma unroll
        for (int t = 0; t < kGroup; t++) {
          const int s = min(s0 + t, bd.n - 1), p = fwd ? bd.first + s : bd.last - s;
          const int blk = (p - 6) * nw + bd.w;
          const __amdgpu_buffer_rsrc_t r0 = fwd ? rr : rd;
          const int o0 = fwd ? blk * (kBlk * 8) : (blk + kPad * nw) * (kBlk4 * 8);
          q[t][0] = ld_pair(r0, v, o0);
          q[t][1] = ld_pair(r0, v + 1024u, o0);
          for (int m = 2; m < 6; m++) q[t][m] = ld_pair(rr, v + m * 1024u, blk * (kBlk * 8));
          const int og = blk * (kGeo * 1024);
          q[t][6] = ld_pair(rg, v + (fwd ? 0u : 1024u), og);
          if (!kAxis) {
            q[t][7] = ld_pair(rg, v + (fwd ? 2048u : 4096u), og);
            q[t][8] = ld_pair(rg, v + (fwd ? 3072u : 5120u), og);
          }
        }
        // while the loads are under way: the tiles of this wavefront's next group
        if (fwd && gr + kLoaders < bd.groups) (void)look(gr + kLoaders);
        double f[kGroup][5];
#pragma unroll
        for (int t = 0; t < kGroup; t++) {
          double2 *y = q[t];
          if (s0 + t >= bd.n) {  // past the last plane: a step without cells
            y[0] = y[1] = y[3] = y[4] = y[5] = y[6] = {0.0, 0.0};
            y[2] = {1.0, 0.0};
            y[5].y = 1.0;
          }
          if (fwd) {  // Res to Res/alfa
            y[0] = {y[0].x * y[4].x, y[0].y * y[4].x};
            y[1] = {y[1].x * y[4].x, y[1].y * y[4].x};
          } else {
            y[6] = {-y[6].x, -y[6].y};
          }
          const double u[4] = {y[2].x, y[2].y, y[3].x, y[3].y};
          const Euler w(u, y[5].y, g1);  // 1/rho of the record's state from the record
          f[t][0] = fma(u[1], w.vx, w.p);
          f[t][1] = u[2] * w.vx;
          f[t][2] = w.e * w.vx;
          f[t][3] = fma(u[2], w.vy, w.p);
          f[t][4] = w.e * w.vy;
        }
        const int gn = gbase + gr, slot = gn & 1;
#pragma unroll
        for (int t = 0; t < kGroup; t++) {
          // the place of a half group is free when that half of group gn - 2 has been read
          if (t % 2 == 0 && !wait_lds(&sh.used, 2 * (gn - kGroups) + t / 2 + 1, sh, st.ctl)) return;
          const double2 *y = q[t];
          double2 *o = reinterpret_cast<double2 *>(sh.ring[slot * kGroup + t]) + lane;
          o[0] = y[0];
          o[64] = y[1];
          o[128] = y[2];
          o[192] = y[3];
          o[256] = y[4];
          o[320] = {y[5].x, y[6].x};
          o[384] = {y[6].y, f[t][0]};
          o[448] = {f[t][1], f[t][2]};
          o[512] = {f[t][3], f[t][4]};
          if (!kAxis) {
            o[576] = y[7];
            o[640] = y[8];
          }
        }
        mem_order();
        lds_put(&sh.avail[slot], gn + 1);  // after the records: LDS performs a wavefront's operations in order
      }
      gbase += bd.groups;
    }
    if (!next_iteration(k, sh, st.ctl)) return;
  }
}

// The receiver wavefront: brings the neighbouring band's values from memory
// to LDS, up to 64 at a time, in order.
template <bool kAxis>
__device__ __forceinline__ void receiver(const Dev &d, const SyntheticState &st, SweepShared<kAxis> &sh, const Band &bd) {
  const int lane = threadIdx.x & 63, nw = st.nw;
  if (nw == 1) return;
  int hseq = 0, gbase = 0;
  for (int k = st.k0;; k++) {
    for (int dir = 0; dir < 2; dir++, gbase += bd.groups) {
      const bool fwd = dir == 0;
      if (fwd ? bd.w == 0 : bd.w == nw - 1) continue;
      const __amdgpu_buffer_rsrc_t rh =
          rsrc_of(hand_of(d, st, fwd, fwd ? bd.w - 1 : bd.w + 1), (size_t)hand_len(d.nx) * 4);
      Patience pt(st.ctl);
      for (int have = 0; have < bd.links;) {
        const int at = have + lane;
        const unsigned v = at < bd.links ? (unsigned)at * 32u : kOff;
        const double2 a = ld_pair(rh, v, 0), b = ld_pair(rh, v + 16u, 0);
        auto there = [](double x) { return (unsigned)((unsigned long long)__double_as_longlong(x) >> 32) != kEmptyHi; };
        const unsigned long long m =
            __ballot(at < bd.links && there(a.x) && there(a.y) && there(b.x) && there(b.y));
        int cnt = m == ~0ull ? 64 : __builtin_ctzll(~m);
        // the sweep has read the values of the steps before kGroup (used / 2 - gbase)
        cnt = min(cnt, kGroup * ((uniform(lds_get(&sh.used)) >> 1) - gbase) + kHand - have);
        if (cnt > 0) {
          if (lane < cnt) {
            double2 *o = reinterpret_cast<double2 *>(sh.hand[at & (kHand - 1)]);
            o[0] = a;
            o[1] = b;
          }
          mem_order();
          have += cnt;
          lds_put(&sh.hand_n, hseq + have);
          pt.n = 0;
        } else {
          if (uniform(lds_get(&sh.quit))) return;
          __builtin_amdgcn_s_sleep(1);
          if (pt.over(true)) {
            lds_put(&sh.quit, 1);
            return;
          }
        }
      }
      hseq += bd.links;
    }
    if (!next_iteration(k, sh, st.ctl)) return;
  }
}

// The loop's end word: results for the host, then no further iteration.
__device__ __forceinline__ void end_loop(const SyntheticState &st, int it, int bad, int stopped, int last, double res) {
  if ((threadIdx.x & 63) != 0) return;
  st.iters[0] = it;
  st.iters[1] = bad;
  st.iters[2] = stopped;
  reinterpret_cast<double *>(st.iters + 4)[0] = res;  // max |Res_4| of the launch's last iteration
  st_agent(st.ctl + kCtlLast, last);
  if (bad) st_agent(st.ctl + kCtlStop, 1);
}

// A band's fourth helper: empties the hand-off slots that its sweep has read
// (each direction's during the other direction's sweep, before the band's own
// sweep of that direction can end, so before they are written again).  In
// the last band, where the forward sweep ends last and the backward sweep
// begins, it also decides: a T<0.1 stop before U changes, and whether another
// iteration runs (src/Hybrid_Sub.f90:99-104).
template <bool kAxis>
__device__ __forceinline__ void keeper(const Dev &d, const SyntheticState &st, SweepShared<kAxis> &sh, const Band &bd) {
  const int lane = threadIdx.x & 63, nw = st.nw;
  const bool top = bd.w == nw - 1;
  auto clear = [&](bool fwd) {
    const int from = fwd ? bd.w - 1 : bd.w + 1;
    if (from < 0 || from >= nw) return;
    const __amdgpu_buffer_rsrc_t rh = rsrc_of(hand_of(d, st, fwd, from), (size_t)hand_len(d.nx) * 4);
    const double e = __longlong_as_double((long long)kEmpty);
    for (int q = lane; q < 2 * bd.links; q += 64) st_pair(rh, (unsigned)q * 16u, 0, e, e);
  };
  for (int k = st.k0;; k++) {
    if (!wait_lds(&sh.fwd_done, k, sh, st.ctl)) return;
    clear(true);
    const int bad = top ? uniform(ld_agent(st.ctl + kCtlBad)) : 0;
    vm_wait();
    if (!bad) lds_put(&sh.bgo, k);
    if (top) {
      double res = 0.0;
      for (int t = lane; t < st.ntx * st.nty; t += 64) res = fmax(res, ld_agent(st.tres + t));
      for (int off = 32; off > 0; off >>= 1) res = fmax(res, __shfl_xor(res, off, 64));
      bool more = !bad && res > st.tol && k < st.maxit;
      const bool stopped = more && k >= st.kstop;  // the launch ends here; a later one continues at k + 1
      if (stopped) more = false;
      if (!more) {
        end_loop(st, k, bad, stopped ? 1 : 0, bad ? k - 1 : k, res);
        vm_wait();
      }
      if (lane == 0) st_agent(st.ctl + kCtlGo, more ? k + 1 : -1);
      if (bad) {
        lds_put(&sh.quit, 1);
        return;
      }
    }
    if (!wait_lds(&sh.bwd_done, k, sh, st.ctl)) return;
    clear(false);
    vm_wait();
    lds_put(&sh.clr, k);
    if (!next_iteration(k, sh, st.ctl)) return;
  }
}

// A copy of x with every 32-bit word read once and made wavefront-uniform
// (scalar registers): the fields of a job in memory would otherwise be
// reloaded after every store.
template <typename T>
__device__ __forceinline__ T uniform_copy(const T &x) {
  static_assert(sizeof(T) % 4 == 0, "word copy");
  T y;
  const int *src = reinterpret_cast<const int *>(&x);
  int *dst = reinterpret_cast<int *>(&y);
#pragma unroll
  for (int k = 0; k < (int)(sizeof(T) / 4); k++) dst[k] = __builtin_amdgcn_readfirstlane(src[k]);
  return y;
}

template <bool kAxis>
__device__ __forceinline__ void sweep_role(const Dev &d, const SyntheticState &st, SweepShared<kAxis> &sh, int band) {
  for (int t = threadIdx.x; t < (kHand + 2) * 4; t += kThreads) sh.hand[t / 4][t % 4] = 0.0;
  if (threadIdx.x == 0) {
    for (int q = 0; q < kGroups; q++) sh.avail[q] = 0;
    sh.used = sh.hand_n = sh.quit = 0;
    sh.fwd_done = sh.bwd_done = sh.bgo = sh.clr = st.k0 - 1;
  }
  __syncthreads();
  if (ld_agent(st.ctl + kCtlGo) != st.k0) return;
  const Band bd(d, uniform(band));
  const int wave = uniform((int)(threadIdx.x >> 6));
  // wavefront 4 shares the SIMD of the sweep (0): the one with the least to do
  if (wave == 0) sweeper<kAxis>(d, st, sh, bd);
  else if (wave <= kLoaders) loader<kAxis>(d, st, sh, bd, wave - 1);
  else if (wave == 4) receiver<kAxis>(d, st, sh, bd);
  else keeper<kAxis>(d, st, sh, bd);
}

// A flux workgroup (of st.nflux): the fluxes of its tiles, iteration after
// iteration.  A tile of iteration k+1 is computed as soon as the backward
// sweep of iteration k has passed every cell that it reads, so the fluxes run
// beside the sweep, from the last planes to the first; at the end only the
// first tile's are left, and the forward sweep begins behind them.  When the
// loop ends the workgroup writes its tiles' U to the mesh array.
__device__ __forceinline__ void flux_role(const Dev &d, const SyntheticState &st, FluxShared &sh, int wg) {
  const int tid = threadIdx.x, nx = d.nx, ny = d.ny;
  const int ntiles = st.ntx * st.nty;
  int *ctl = st.ctl;
  // thread 0: waits until the backward sweep of iteration k has passed the
  // cells from (ilo, jlo) on in the rows up to jhi
  auto passed = [&](int k, int ilo, int jlo, int jhi) -> bool {
    for (int w = (jlo - 3) / kBand; w <= (jhi - 3) / kBand; w++) {
      const Band bd(d, w);
      const long long want = ((long long)k << 32) | (bd.last - (ilo + max(jlo, bd.j0)) + 1);
      Patience pt(ctl);
      while (ld_agent(st.prog + kProgStride * w) < want) {
        __builtin_amdgcn_s_sleep(8);
        if (pt.over(false)) return false;
      }
    }
    return true;
  };
  for (int k = st.k0;; k++) {
    if (tid == 0) {
      Patience pt(ctl);
      int go;
      while ((go = ld_agent(ctl + kCtlGo)) != k && go >= 0) {
        __builtin_amdgcn_s_sleep(32);
        if (pt.over(false)) { go = -2; break; }
      }
      sh.word = go;
    }
    __syncthreads();
    const int go = sh.word;
    __syncthreads();
    if (go != k) {
      if (go != -1) return;
      break;
    }
    for (int q = ntiles - 1 - wg; q >= 0; q -= st.nflux) {
      const int tile = uniform(st.order[q]);
      TileGeo tg;
      tile_geo(d, st, tile, tg);
      if (k > st.k0) {
        if (tid == 0)
          sh.word = passed(k - 1, max(3, tg.i0 - 2), max(3, tg.j0 - 2), min(ny - 3, tg.j0 + kTJ + 1)) ? 1 : 0;
        __syncthreads();
        const int ok = sh.word;
        __syncthreads();
        if (!ok) return;
      }
      double rmax = 0.0;
      int bad = 0;
      flux_tile(d, st, sh, tg, k == st.k0, rmax, bad);
      // the tile's max |Res_4| and T<0.1 flag, then its iteration number once
      // every store of the workgroup is complete
      for (int off = 32; off > 0; off >>= 1) rmax = fmax(rmax, __shfl_down(rmax, off, 64));
      if ((tid & 63) == 0) sh.red[tid >> 6] = rmax;
      bad = __syncthreads_or(bad);
      if (tid == 0) {
        double m = sh.red[0];
        for (int e = 1; e < kThreads / 64; e++) m = fmax(m, sh.red[e]);
        st_agent(st.tres + tile, m);
        if (bad) st_agent(ctl + kCtlBad, 1);
      }
      vm_wait();
      __syncthreads();
      if (tid == 0) st_agent(st.ready + tile, k);
    }
  }
  // U of the last complete iteration to the mesh array
  const int last = uniform(ld_agent(ctl + kCtlLast));
  if (last < st.k0) return;
  const __amdgpu_buffer_rsrc_t ru = ub_rsrc(st);
  for (int q = ntiles - 1 - wg; q >= 0; q -= st.nflux) {
    const int tile = uniform(st.order[q]);
    const int i0 = 3 + (tile % st.ntx) * kTI, j0 = 3 + (tile / st.ntx) * kTJ;
    if (tid == 0) sh.word = passed(last, i0, j0, min(ny - 3, j0 + kTJ - 1)) ? 1 : 0;
    __syncthreads();
    const int ok = sh.word;
    __syncthreads();
    if (!ok) return;
    for (int t = tid; t < kTI * kTJ; t += kThreads) {
      const int b = t % kTJ, i = i0 + ((t / kTJ - b) & (kTI - 1)), j = j0 + b;
      if (i > nx - 3 || j > ny - 3) continue;
      const unsigned o = (unsigned)pblk_of(i, j, st.nw) * (kBlk4 * 8u) + 16u * ((j - 3) & 63);
      const double2 u01 = ld_pair(ru, o, 0), u23 = ld_pair(ru, o + 1024u, 0);
      const int c = cidx(d, i, j), N = d.ncell;
      d.U[c] = u01.x;
      d.U[N + c] = u01.y;
      d.U[2 * N + c] = u23.x;
      d.U[3 * N + c] = u23.y;
    }
  }
}

// LDS of a workgroup of either role
template <bool kAxis>
struct LoopShared {
  static constexpr size_t kBytes =
      sizeof(SweepShared<kAxis>) > sizeof(FluxShared) ? sizeof(SweepShared<kAxis>) : sizeof(FluxShared);
};

// Workgroup b of an instance's `blocks`: bands sit at multiples of st.stride,
// the flux workgroups in between.  With stride 8 the bands of one instance
// are on one XCD (workgroups go to the eight XCDs in turn), where a hand-off
// through memory takes 0.30 us one way; between XCDs 0.36-0.49 us.
template <bool kAxis>
__device__ __forceinline__ void ns_workgroup(const Dev &d, const SyntheticState &st, int b, char *lds) {
  const int before = min(st.nw, (b + st.stride - 1) / st.stride);  // bands at workgroups below b
  if (b % st.stride == 0 && b / st.stride < st.nw)
    sweep_role<kAxis>(d, st, *reinterpret_cast<SweepShared<kAxis> *>(lds), b / st.stride);
  else if (b - before < st.nflux)
    flux_role(d, st, *reinterpret_cast<FluxShared *>(lds), b - before);
}

// The inner loop (src/Hybrid_Sub.f90:99-104) of one instance, launched
// cooperatively (all workgroups resident).
template <bool kAxis>
__global__ void __launch_bounds__(kThreads) k_ns_loop(Dev d, SyntheticState st) {
  __shared__ __align__(16) char lds[LoopShared<kAxis>::kBytes];
  ns_workgroup<kAxis>(d, st, blockIdx.x, lds);
}

// The inner loops of a batch of instances in one launch: job J has the
// workgroups J.wg0 .. J.wg0 + J.blocks - 1, a gang.  The workgroups of a gang
// wait for each other, so all of them have to be resident.  Workgroups go to the
// eight XCDs in turn and each XCD starts its share in order, so of the first gang
// that is not complete a missing workgroup waits only for lower-numbered ones of
// its XCD: those of earlier gangs, which are complete and end, and its own
// gang's, which leave room (synthetic_batch_layout: at most half of the device's
// workgroups).  The launch has no such launch beside it (NsTurn).  A gang
// starts once its last workgroup has arrived; that wait alone takes as long as
// gangs before it do, and is bounded by the time in which none of them goes on.
__global__ void __launch_bounds__(kThreads) k_ns_batch(const NsJob *__restrict__ jobs, int njobs) {
  __shared__ __align__(16) char lds[LoopShared<false>::kBytes];
  int lo = 0, hi = njobs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) / 2;
    if (jobs[mid].wg0 <= (int)blockIdx.x) lo = mid;
    else hi = mid - 1;
  }
  const NsJob &J = jobs[lo];
  int *word = reinterpret_cast<int *>(lds);
  if (threadIdx.x < 64) {
    int *ctl = J.st.ctl;
    if (threadIdx.x == 0) __hip_atomic_fetch_add(ctl + kCtlArrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    StallLimit limit(kStartTicks);
    bool ok = true;
    for (int n = 1; ok && uniform(ld_agent(ctl + kCtlArrived)) < J.blocks; n++) {
      __builtin_amdgcn_s_sleep(32);
      if ((n & 63) != 0) continue;
      // the earlier gangs' iterations
      long long sum = 0;
      for (int q = threadIdx.x; q < lo; q += 64) sum += ld_agent(jobs[q].st.ctl + kCtlGo);
      for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
      if (uniform(ld_agent(ctl + kCtlErr)) != 0) {
        ok = false;
      } else if (limit.over(sum, wall_clock64())) {
        st_agent(ctl + kCtlErr, 1);
        ok = false;
      }
    }
    if (threadIdx.x == 0) *word = ok ? 1 : 0;
  }
  __syncthreads();
  const int ok = *word;
  __syncthreads();
  if (!ok) return;
  const int b = (int)blockIdx.x - J.wg0;
  const Dev d = uniform_copy(J.d);
  const SyntheticState st = uniform_copy(J.st);
  if (st.axis) ns_workgroup<true>(d, st, b, lds);
  else ns_workgroup<false>(d, st, b, lds);
}

// U0 <- U and the synthetic correction of S on cells 3..n-3 (src/Hybrid_Sub.f90:108-153)
__global__ void k_ns_feedback(Dev d, SyntheticState st) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int nci = (d.nx - 5) * (d.ny - 5);
  if (t >= nci) return;
  const int i = t % (d.nx - 5) + 3, j = t / (d.nx - 5) + 3;
  const int N = d.ncell, c = cidx(d, i, j);
  const double sq = sqrt(2.0 / d.gamma), cv = d.cv;
  for (int m = 0; m < 4; m++) d.U0[m * N + c] = d.U[m * N + c];
  const double *U = d.U, *U2 = d.U2;
  const double rns = U[c], uns = U[N + c] / U[c], vns = U[2 * N + c] / U[c];
  const double tns = (U[3 * N + c] - 0.5 * U[c] * (uns * uns + vns * vns)) / (cv * U[c]);
  const double rk = U2[c], uk = U2[N + c] / U2[c], vk = U2[2 * N + c] / U2[c];
  const double tk = (U2[3 * N + c] - 0.5 * U2[c] * (uk * uk + vk * vk)) / (cv * U2[c]);
  double s0[4];
  s0[0] = rns - rk;
  s0[1] = (uns - uk) * d.ma / sq;
  s0[2] = (vns - vk) * d.ma / sq;
  s0[3] = tns - tk;
  for (int k = 0; k < 4; k++) {
    d.S[k * N + c] = d.S[k * N + c] + s0[k];
    d.S0[k * N + c] = s0[k] + st.s00[k * N + c];
  }
}

// the next launch of the inner loop continues at iteration k0
__global__ void k_ns_resume(Dev d, SyntheticState st, int k0) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t == 0) {
    st.ctl[kCtlGo] = k0;
    st.ctl[kCtlBad] = 0;
    st.ctl[kCtlStop] = 0;
    st.iters[1] = 0;
    st.iters[2] = 0;
  }
  clear_hands(d, st, t, (size_t)gridDim.x * blockDim.x);
}

// Launches whose workgroups wait for each other (k_ns_loop, k_ns_batch) take turns
// on a device, whatever streams and threads they come from: two that gather at
// the same time could each hold workgroup slots that the other needs, until the
// waits run out.  A launch's stream waits for the launch before it; nothing waits
// on the host.  Other kernels run beside them.
namespace {
constexpr int kMaxDevices = 64;
struct {
  std::mutex mu;
  hipEvent_t last = nullptr;  // recorded behind the device's last such launch
} g_turn[kMaxDevices];
}  // namespace
hipError_t NsTurn::begin(hipStream_t stream) {
  const hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  s = stream;
  lock = std::unique_lock<std::mutex>(g_turn[dev].mu);
  hipEvent_t &last = g_turn[dev].last;
  return last ? hipStreamWaitEvent(s, last, 0) : hipEventCreateWithFlags(&last, hipEventDisableTiming);
}
hipError_t NsTurn::end() { return hipEventRecord(g_turn[dev].last, s); }

// the degenerate loop of a mesh without swept cells: max |Res_4| over no
// cells is 0, so the reference runs one iteration that changes nothing
__global__ void k_ns_empty(SyntheticState st) {
  if (threadIdx.x == 0 && blockIdx.x == 0) st.iters[0] = st.ctl[kCtlGo] == 1 ? 1 : 0;
}

static const void *ns_loop_kernel(const SyntheticState &st) {
  return st.axis ? reinterpret_cast<const void *>(k_ns_loop<true>) : reinterpret_cast<const void *>(k_ns_loop<false>);
}
// workgroups of an instance: its bands at multiples of the stride, its flux workgroups between and after them
static int ns_blocks(const SyntheticState &st) {
  return std::max(st.stride * (st.nw - 1) + 1, st.nw + st.nflux);
}

// whether every swept cell (3..nx-3, 3..ny-3) has the face normals ni = (1,0)
// and nj = (0,1) exactly (a zero of either sign), in the caller's Fortran
// (nx, ny) arrays
static bool axis_aligned(const gsis_params &p, int nx, int ny) {
  for (int j = 3; j <= ny - 3; j++)
    for (int i = 3; i <= nx - 3; i++) {
      const size_t g = (size_t)(i - 1) + (size_t)nx * (j - 1);
      if (!(p.ni1[g] == 1.0 && p.ni2[g] == 0.0 && p.nj1[g] == 0.0 && p.nj2[g] == 1.0)) return false;
    }
  return true;
}

int synthetic_init(Dev &d, const gsis_params &p, SyntheticState &st) {
  const size_t N = d.ncell;
  st.rs = d.ny - 5 > 0 && d.nx - 5 > 0 ? d.ny - 5 : 0;
  st.np = st.rs > 0 ? d.nx + d.ny - 11 : 0;
  if (st.rs > kMaxBands * kBand) {
    g_syn_err = "synthetic solve: at most " + std::to_string(kMaxBands * kBand + 5) + " nodes in j";
    return GSIS_EUNSUPPORTED;
  }
  st.ntx = st.rs > 0 ? (d.nx - 5 + kTI - 1) / kTI : 0;
  st.nty = st.rs > 0 ? (st.rs + kTJ - 1) / kTJ : 0;
  const int ntiles = st.ntx * st.nty;
  st.axis = st.rs > 0 && axis_aligned(p, d.nx, d.ny);
  st.nw = (st.rs + kBand - 1) / kBand;
  st.stride = 8;
  if (ntiles > 0) {
    int dev = 0, ncu = 0, per = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, ns_loop_kernel(st), kThreads, 0);
    if (e != hipSuccess || per < 1) {
      g_syn_err = std::string("synthetic solve: occupancy query: ") + hipGetErrorString(e) + ", " +
                  std::to_string(per) + " workgroups of " + std::to_string(kThreads) + " threads per CU";
      return GSIS_EHIP;
    }
    // one workgroup per CU: the fluxes run beside the sweeps, so more of them
    // at a time would only share the sweeps' CUs
    st.nflux = std::min(ntiles, ncu - st.nw);
    if (ns_blocks(st) > ncu * per) st.stride = 1;  // (a device of few CUs: bands next to each other)
    if (st.nflux < 1 || ns_blocks(st) > ncu * per) {
      g_syn_err = "synthetic solve: the inner-loop launch does not fit the device";
      return GSIS_EUNSUPPORTED;
    }
  }
  const size_t nq = (size_t)st.np * st.nw * 64;  // cells of the blocked sweep layout
  // 32-bit buffer offsets of the blocked arrays and of U; the largest blocked ones
  // are the records and, with normals, the geometry (the padded ones have 4
  // doubles a cell and kPad planes more at either end)
  const size_t npad = (size_t)(st.np + 2 * kPad) * st.nw * 64;
  if (std::max({kNRec * nq, 2 * geo_pairs(st.axis) * nq, 4 * npad}) * sizeof(double) >= ((size_t)1 << 31) ||
      (size_t)4 * N * sizeof(double) >= ((size_t)1 << 31)) {
    g_syn_err = "synthetic solve: the mesh is too large for the sweep's buffers (2 GiB)";
    return GSIS_EUNSUPPORTED;
  }
  const size_t n_geo = (size_t)2 * geo_pairs(st.axis) * nq;
  const size_t n_hand = st.nw > 0 ? (size_t)2 * st.nw * hand_len(d.nx) * 4 : 0;
  const size_t n_dbl = 4 * N + (size_t)kNRec * nq + 8 * npad + n_geo + n_hand + (size_t)ntiles +
                       (size_t)kProgStride * std::max(st.nw, 1);
  const size_t bytes = n_dbl * 8 + 128 + 8 * (size_t)ntiles + 64;
  void *mem = nullptr;
  if (hipMalloc(&mem, bytes) != hipSuccess || hipMemset(mem, 0, bytes) != hipSuccess) {
    g_syn_err = "synthetic solve: device allocation failed";
    return GSIS_EHIP;
  }
  double *b = reinterpret_cast<double *>(mem);  // every array with pairs starts at a multiple of 16 bytes
  st.rec = b; b += kNRec * nq;
  st.dstar = b; b += 4 * npad;
  st.ub = b; b += 4 * npad;
  st.geo = b; b += n_geo;
  st.hand = b; b += n_hand;
  st.s00 = b; b += 4 * N;
  st.prog = reinterpret_cast<long long *>(b); b += (size_t)kProgStride * std::max(st.nw, 1);
  st.tres = b; b += ntiles;
  st.ctl = reinterpret_cast<int *>(b);
  st.iters = st.ctl + 16;
  st.ready = st.ctl + 32;
  st.order = st.ready + ntiles;
  st.mem = mem;
  auto bail = [&](const char *msg) {
    (void)hipFree(mem);
    st.mem = nullptr;
    g_syn_err = msg;
    return GSIS_EHIP;
  };
  if (ntiles > 0) {  // tiles by level, as the sweeps pass them
    std::vector<int> order(ntiles);
    for (int t = 0; t < ntiles; t++) order[t] = t;
    std::stable_sort(order.begin(), order.end(),
                     [&](int x, int y) { return x % st.ntx + kLev * (x / st.ntx) < y % st.ntx + kLev * (y / st.ntx); });
    if (hipMemcpy(st.order, order.data(), sizeof(int) * ntiles, hipMemcpyHostToDevice) != hipSuccess)
      return bail("synthetic solve: tile order upload failed");
  }
  if (nq > 0) {
    hipLaunchKernelGGL(k_rec_init, dim3((unsigned)((nq + 255) / 256)), dim3(256), 0, 0, d, st);
    if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess)
      return bail("synthetic solve: record initialisation failed");
  }
  st.tol = p.ns_tol;
  st.maxit = p.ns_maxit > 0 ? p.ns_maxit : 100000;
  st.local_dt = p.local_dt;
  st.if_viscous = p.if_viscous;
  st.cfl = p.cfl;
  st.dtmax = p.dtmax;
  st.dtmin = p.dtmin;
  st.on = true;
  return 0;
}

int synthetic_begin(const Dev &d, SyntheticState &st, hipStream_t s) {
  if (!st.on) {
    g_syn_err = "synthetic solve not initialised";
    return GSIS_EARG;
  }
  const int nc = (d.nx - 1) * (d.ny - 1);
  hipLaunchKernelGGL(k_ns_prepare, dim3((std::max(nc, st.ntx * st.nty) + 255) / 256), dim3(256), 0, s, d, st);
  return 0;
}

int synthetic_run(const Dev &d, SyntheticState &st, int k0, int kstop, hipStream_t s) {
  if (!st.on || k0 < 1 || kstop < k0) {
    g_syn_err = "synthetic solve: not initialised, or an empty range of inner iterations";
    return GSIS_EARG;
  }
  if (k0 > 1) hipLaunchKernelGGL(k_ns_resume, dim3(32), dim3(256), 0, s, d, st, k0);
  if (st.nflux > 0) {
    Dev dd = d;
    SyntheticState ss = st;
    ss.k0 = k0;
    ss.kstop = kstop;
    void *args[] = {&dd, &ss};
    NsTurn turn;
    hipError_t e = turn.begin(s);
    if (e == hipSuccess)
      e = hipLaunchCooperativeKernel(ns_loop_kernel(st), dim3(ns_blocks(st)), dim3(kThreads), args, 0, s);
    if (e == hipSuccess) e = turn.end();
    if (e != hipSuccess) {
      g_syn_err = std::string("synthetic solve: cooperative launch failed: ") + hipGetErrorString(e);
      return GSIS_EHIP;
    }
  } else if (k0 == 1) {
    hipLaunchKernelGGL(k_ns_empty, dim3(1), dim3(64), 0, s, st);
  }
  return 0;
}

bool synthetic_batchable(const SyntheticState &st) { return st.on && st.rs <= 4 * kBand; }

// Flux workgroups per instance: the fewest tiles each with which the whole batch
// is resident at once, but at most kBatchTiles (a tile takes about 4 us, a sweep
// that its fluxes run beside 50-200 us); beyond that the last gangs start when
// earlier ones have ended.  A gang has at most half of the device's workgroups,
// however many tiles its mesh has: it has to be resident as a whole, and what
// other streams run beside it has to find room on every XCD while it gathers.
int synthetic_batch_layout(std::vector<NsJob> &jobs) {
  constexpr int kBatchTiles = 16;
  int dev = 0, ncu = 0, per = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, reinterpret_cast<const void *>(k_ns_batch), kThreads, 0) !=
          hipSuccess ||
      per < 1) {
    g_syn_err = "synthetic solve: occupancy query of the batched launch failed";
    return -1;
  }
  const int most = ncu * per / 2;  // workgroups of a gang
  for (int tiles = 1;; tiles++) {
    int at = 0;
    for (NsJob &j : jobs) {
      const int nt = j.st.ntx * j.st.nty;
      j.st.nflux = std::max(1, std::min((nt + tiles - 1) / tiles, most - j.st.nw));
      j.st.stride = 8 * (j.st.nw - 1) + 1 <= j.st.nw + j.st.nflux ? 8 : 1;
      j.wg0 = at;
      j.blocks = ns_blocks(j.st);
      at += j.blocks;
    }
    if (at <= ncu * per || tiles >= kBatchTiles) return at;
  }
}

void launch_ns_batch(const NsJob *djobs, int n, int blocks, hipStream_t s) {
  if (n > 0) hipLaunchKernelGGL(k_ns_batch, dim3(blocks), dim3(kThreads), 0, s, djobs, n);
}

void synthetic_finish(const Dev &d, SyntheticState &st, hipStream_t s) {
  const int nci = (d.nx - 5) * (d.ny - 5);
  if (nci > 0) hipLaunchKernelGGL(k_ns_feedback, dim3((nci + 255) / 256), dim3(256), 0, s, d, st);
}

int synthetic_step(const Dev &d, SyntheticState &st, hipStream_t s) {
  int rc = synthetic_begin(d, st, s);
  if (!rc) rc = synthetic_run(d, st, 1, 0x7fffffff, s);
  if (!rc) synthetic_finish(d, st, s);
  return rc;
}

int synthetic_state(SyntheticState &st, hipStream_t s, bool *unfinished, int *iters, bool *bad_t, double *res) {
  int h[6] = {0, 0, 0, 0, 0, 0};
  if (hipMemcpyAsync(h, st.iters, sizeof(h), hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess) {
    g_syn_err = "synthetic solve: reading the loop state failed";
    return GSIS_EHIP;
  }
  *unfinished = h[2] != 0 && h[1] == 0;
  *iters = h[0];
  *bad_t = h[1] != 0;
  double r;
  memcpy(&r, h + 4, sizeof(r));
  *res = r;
  return 0;
}

int synthetic_read_iters(SyntheticState &st, hipStream_t s, int *iters, int *bad_t) {
  int h[2] = {0, 0}, c[4] = {0, 0, 0, 0};
  if (!st.on) {
    if (iters) *iters = 0;
    if (bad_t) *bad_t = 0;
    return 0;
  }
  if (hipMemcpyAsync(h, st.iters, sizeof(h), hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipMemcpyAsync(c, st.ctl, sizeof(c), hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess) {
    g_syn_err = "synthetic solve: reading the iteration counter failed";
    return GSIS_EHIP;
  }
  if (iters) *iters = h[0];
  if (bad_t) *bad_t = h[1];
  if (c[kCtlErr]) {
    g_syn_err = "synthetic solve: a wait between the inner loop's workgroups timed out";
    return GSIS_EHIP;
  }
  return 0;
}

void synthetic_free(SyntheticState &st) {
  if (st.mem) (void)hipFree(st.mem);
  st.mem = nullptr;
  st.on = false;
}

}  // namespace gsis
