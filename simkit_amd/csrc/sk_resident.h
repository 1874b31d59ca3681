// Resident PCG: the whole PCG run of one system (block-Jacobi or two-level) in a
// single launch whose workgroups (at most one per CU) keep their rows' matrix blocks
// on chip - registers first, then LDS, the rest streamed from L2 - and meet
// once per iteration through self-tagged words in global memory instead of
// at launch boundaries. Described at resident_pcg_kernel.
#pragma once

#include "sk_coarse.h"
#include "sk_internal.h"

#include <memory>

namespace sk {

constexpr int kResMaxParts = 256;     // workgroups at most (the CUs of an MI355X)
constexpr int kResLds = 160 * 1024;   // LDS a workgroup may use
constexpr int kResStaticLds = 2048;   // bound on the kernel's static LDS
// Threads per workgroup and blocks per thread held in registers, by precision.
constexpr int kResNT64 = 512, kResKR64 = 8, kResShort64 = 5;
constexpr int kResNT32 = 512, kResKR32 = 12, kResShort32 = 6;
constexpr int kResMaxTier = 4;        // blocks per thread in LDS, and streamed from L2, at most (each)
// With the coarse correction: its values in flight leave fewer registers for blocks.
constexpr int kResTwoKR64 = 5, kResTwoKR32 = 9, kResTwoTier = 6;
constexpr int kResMaxPieces = 8;      // aggregates a workgroup's rows reach into, at most (one wave serves them)
constexpr double kResWait = 2.0;      // seconds a workgroup waits for another before the run is given up
constexpr uint32_t kResMaxEpoch = 0x70000000u;  // exchanges are numbered anew from a run that starts past this one

// Cut of a mesh's rows into contiguous ranges, one per workgroup, with the
// index data the kernel reads (built once per mesh and cut on the host).
struct ResidentPlan {
  std::vector<int32_t> parts;      // [G + 1] the cut (the cache key, with fp32)
  bool fp32 = false;
  int two_ld = 0, two_need = 0, two_agg = 0;  // what LDS holds of the coarse space (part of the key)
  int G = 0, K = 0, KR = 0, KL = 0, KS = 0;  // blocks per thread: K = registers (up to KR) + LDS (KL) + streamed (KS)
  int max_rows = 0, max_local = 0, max_halo = 0, n_exp = 0;
  size_t lds = 0;                  // dynamic LDS bytes
  DevBuf<int32_t> row0;            // [G + 1]
  DevBuf<uint16_t> lcol;           // [nblk] LDS byte offset of the block's column
  DevBuf<uint32_t> tflag;          // [G NT] which of a thread's blocks end a row
  DevBuf<uint16_t> trow;           // [G NT] local row of each thread's first block (rows: none)
  // The halo of a part: the vertices of other parts that its rows couple to (hvert, ascending; halo_ptr[G + 1]),
  // and their places among all exported vertices (ResidentArgs::halo, exp0, exslot).
  DevBuf<int32_t> halo_ptr, hvert, halo, exp0;
  DevBuf<uint16_t> exslot;
};

// What the kernel reports to the host (pinned).
struct ResidentResult {
  int iter, done, refines, aborted;
  uint32_t epoch;
};

// The coarse space of the two-level preconditioner as the cut sees it. A piece
// is the part of an aggregate that one workgroup's rows hold (pieces are
// numbered in row order); a workgroup owns the aggregates that begin in it.
struct ResidentTwo {
  int n_piece = 0, max_need = 0;
  DevBuf<int32_t> piece0;          // [G + 1] first piece of each workgroup
  DevBuf<int32_t> pagg;            // [n_piece] aggregate of each piece
  DevBuf<int32_t> apiece;          // [n_agg + 1] first piece of each aggregate
  DevBuf<int32_t> own0;            // [G + 1] first aggregate owned by each workgroup
  // the aggregates of the workgroup's rows and halo, and where each vertex's stands in that list
  DevBuf<int32_t> need0, need;     // [G + 1], ids
  DevBuf<uint16_t> lrow, lhalo;    // [nv], [all halos]
  DevBuf<uint64_t> cwords, uwords; // [2][n_piece][8] (of A p, of a residual), [n_agg][8] exchanged words
};

// A simulator's side of the resident solver: its plan and exchange buffers.
struct ResidentState {
  std::vector<int32_t> parts;            // the caller's cut; empty: the default one
  std::shared_ptr<ResidentPlan> plan;    // null: not built or not eligible
  std::unique_ptr<ResidentTwo> two;      // with a coarse space
  bool tried = false;                    // plan has been looked for
  bool off = false;                      // a run gave up waiting: launches only from now on
  int64_t runs = 0, launch_solves = 0, gave_up = 0;  // solves by this kernel and by launches; runs given up
  bool give_up = false;                  // runs count as given up (test hook)
  DevBuf<uint64_t> slots, zx, xx;
  DevBuf<char> stream;
  DevBuf<int> abort_flag;
  ResidentResult* host = nullptr;        // pinned
  uint32_t epoch = 0;
  ~ResidentState();
};

// Workgroups for a mesh of nv vertices and nblk blocks; 0: not eligible.
int resident_parts(int64_t nv, int64_t nblk, bool fp32);

// The CUs of the current device that one resident run of `parts` workgroups
// needs, held until the run has ended: runs of one process that overlap on one
// GPU never ask for more workgroups together than can be resident at once, on
// any XCD. (Other processes are not seen. Where one holds CUs for long, a run
// waits out kResWait, is solved by launches, and so are its simulator's later
// ones.)
class ResidentPermit {
 public:
  ResidentPermit() = default;
  ~ResidentPermit() { release(); }
  ResidentPermit(const ResidentPermit&) = delete;
  ResidentPermit& operator=(const ResidentPermit&) = delete;
  // False when the device has fewer CUs than that, or the stream's CU mask leaves out some.
  bool acquire(int parts, hipStream_t st);
  void release();

 private:
  int dev_ = -1, held_ = 0;
  hipStream_t st_ = nullptr;
};

struct ResidentSolve {
  const void* vals;   // SELL values (T)
  const void* binv;   // block-Jacobi inverses (T)
  const uint8_t* fixed;
  const double* g;    // right-hand side is -g on the free DOFs
  double* dx;
  double rtol, inner_rtol;
  int max_iter, max_refine;
  bool fp32;          // FP32 matrix with FP64 residual replacement
  const CoarseSpace* coarse;  // non-null: two-level preconditioner (built)
};

// Looks for (or builds) the plan of a simulator on mesh m and allocates the
// exchange buffers, once; R.plan stays null when the mesh is not eligible or
// memory runs out.
void resident_prepare(ResidentState& R, sk_mesh* m, bool fp32, const CoarseSpace* coarse);
// Enqueues the run (without waiting); the result is in R.host once the stream
// has been synchronized.
int resident_launch(ResidentState& R, sk_mesh* m, const ResidentSolve& s, hipStream_t st);
// Has the next run number its exchanges from `epoch` on, with all words cleared.
int resident_set_epoch(ResidentState& R, uint32_t epoch);
// Number of neighbour vertices (itself included) of every vertex.
void vertex_degrees(const int32_t* T, int64_t nv, int64_t nt, std::vector<int32_t>& deg);
// The vertices by descending degree, ties in index order (sk_sell_order).
void degree_order(const std::vector<int32_t>& deg, int32_t* order);

}  // namespace sk
