// Resident PCG (see sk_resident.h) and the vertex numbering it likes.
#include "sk_resident.h"

#include <algorithm>
#include <cmath>
#include <condition_variable>
#include <mutex>
#include <numeric>

namespace sk {
namespace {

// ---------------------------------------------------------------------------
// Exchange through self-tagged words: every 64-bit word carries 32 bits of
// payload and the 32-bit number (epoch) of the exchange it belongs to, written
// by one relaxed agent-scope store (which goes through to the memory all XCDs
// share). A reader polls the words it needs until all carry the epoch, so data
// and signal arrive in one trip: no flag, fence or cache invalidation.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void put_word(uint64_t* p, uint32_t epoch, uint32_t v) {
  __hip_atomic_store(p, ((uint64_t)epoch << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t get_word(const uint64_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool tagged(uint64_t w, uint32_t epoch) { return (uint32_t)(w >> 32) == epoch; }

// Words of a vertex's three components: used, and the stride between vertices
// (a power of two, so that a vertex's words share one or half a 64-byte chunk).
template <typename V>
constexpr int kVertWords = 3 * (int)sizeof(V) / 4;
template <typename V>
constexpr int kVertStride = sizeof(V) == 8 ? 8 : 4;

// Reduction slots: eight words (four FP64 sums) of one workgroup in a 64-byte
// chunk, written by eight neighbouring threads and read by all threads
// together in memory order. How the words lie decides what a meeting costs:
// 256 workgroups exchanging ten words each took 4.0 us with one array per
// word (every word of a workgroup on a line of its own) and 2.1 us this way.
// The slots are written to kResCopies places, 128 KB apart, each read by a
// quarter of the workgroups.
constexpr int kSlotWords = 8;
constexpr int kResCopies = 4;
constexpr int kResCopyWords = 16384;
static_assert(2 * kSlotWords * kResMaxParts <= kResCopyWords, "a copy holds both parities");

template <typename T>
struct ResidentArgs {
  int G, K, KL, KS;
  const int32_t* row0;
  const int32_t* bptr;
  const uint16_t* lcol;       // [nblk] LDS byte offset of the block's column in a T vector
  const uint32_t* tflag;      // [G NT] bit k: the thread's k-th block is the last of its row
  const uint16_t* trow;
  const int32_t* sell_pos;
  const T* vals;
  const T* binv;
  const uint8_t* fixed;
  const double* g;
  double* x;
  const int32_t* halo_ptr;
  const int32_t* hvert;       // halo vertices
  const int32_t* halo;        // place of each halo vertex among all exported vertices
  const int32_t* exp0;        // [G + 1] exported vertices of the workgroups before this one
  const uint16_t* exslot;     // partial slot of each exported vertex's row (see product)
  uint64_t* slots;  // [kResCopies] x [2][G][kSlotWords]: parity, workgroup, word
  uint64_t* zx;     // [2][exported vertices][kVertStride<T>]: A p (or a replaced residual), by the meeting's parity
  uint32_t zx_half; // words of one of the two
  uint64_t* xx;     // [exported vertices][8]: FP64 correction (kMixed)
  T* stream;        // [G][KS][9][NT] streamed blocks
  int* abort_flag;
  ResidentResult* host;
  uint32_t epoch;   // last epoch used so far
  int max_rows, max_local, max_halo;
  double rtol2, inner_rtol2;
  int max_iter, max_refine;
  // two-level preconditioner (ResidentTwo, CoarseSpace)
  int ld, n_agg, max_need;
  double shift;
  const int32_t *piece0, *pagg, *apiece, *own0, *need0, *need;
  const uint16_t *lrow, *lhalo;
  const int32_t *agg_ptr, *agg_col;
  const double *tm, *dsc, *dv;
  const _Float16* einv;
  uint64_t *cwords, *rwords, *uwords;
};

// Dynamic LDS (bytes): everything but the matrix tiers and the coarse space, one tier block per thread, and where
// the coarse space starts behind both. It holds 16-byte words.
__host__ __device__ constexpr size_t base_lds(bool fp32, int max_rows, int max_local, int max_halo) {
  const size_t NT = fp32 ? kResNT32 : kResNT64, v = fp32 ? 12 : 24;
  return 24 * (max_rows + NT + 1) + (fp32 ? 24 * (size_t)max_local + 12 * (size_t)max_rows : 0) + 2 * v * max_local +
         v * max_halo + 4 * (size_t)max_halo + 2 * NT + 64;
}
__host__ __device__ constexpr size_t tier_lds(bool fp32) { return (fp32 ? kResNT32 * 36 : kResNT64 * 72); }
__host__ __device__ constexpr size_t two_start(bool fp32, int max_rows, int max_local, int max_halo, int KL) {
  return (base_lds(fp32, max_rows, max_local, max_halo) + KL * tier_lds(fp32) + 15) / 16 * 16;
}
// LDS of the coarse space: offsets in doubles from its start.
struct TwoLds {
  int c, uw, raw, tm, dsc, s, col, agg, end;
};
__host__ __device__ constexpr TwoLds two_lds(int ld, int max_need, int n_agg) {
  TwoLds o{};
  o.c = 0;                                // [ld] scaled restricted residual
  o.uw = o.c + ld;                        // [max_need][6] rigid motions
  o.raw = o.uw + 6 * max_need;            // [pieces][8 waves][6] of the restriction, then [unknowns][8 waves] of the
                                          // coarse product: wave sums
  o.tm = o.raw + kResMaxPieces * 8 * 6;   // [pieces][36]
  o.dsc = o.tm + kResMaxPieces * 36;      // [pieces][6]
  o.s = o.dsc + kResMaxPieces * 6;        // [pieces][6] staging
  o.col = o.s + kResMaxPieces * 6;        // [pieces] first unknown, count, first and last wave (four ints)
  o.agg = o.col + 2 * kResMaxPieces;      // [n_agg + 1] first piece and unknown of each aggregate (16 bits each)
  o.end = o.agg + (n_agg + 2) / 2;
  return o;
}
// and behind it the list's aggregates (four bytes each) and two bytes per local vertex: place of its aggregate in the workgroup's list << 3 | fixed DOFs.

constexpr bool two_lds_aligned() {
  for (int n = 0; n < 32; ++n) {
    const int rows = 100 + n % 2, local = 200 + n / 2 % 2, halo = 300 + n / 4 % 2, KL = n / 8 % 2;
    if (two_start(n & 16, rows, local, halo, KL) % 16 || two_lds(8, 1 + n % 2, 1 + n / 2 % 2).col % 2) return false;
  }
  return true;
}
static_assert(two_lds_aligned(), "the pieces' int4 lie on 16 bytes whatever the sizes");

// The restricted residual c follows r by c -= alpha W^T A p. What rounding leaves between them stays at the size that
// c had, while r goes on to shrink, and a preconditioner that is applied to two different residuals ends in
// directions that p.Ap does not bound: FP64 solves to 1e-16 and below ran to the iteration limit and returned them.
// So c is formed from r again once r has shrunk by a million since the last time (FP64, once in a solve to 1e-8; by a
// thousand where r is rounded to FP32), and every 4,096 iterations at the latest, long before the 16-bit tags of its
// words come round.
template <bool kMixed>
constexpr double kRenew = kMixed ? 1e-6 : 1e-12;  // of r.r
constexpr int kRenewAfter = 4096;

constexpr int kAggWords = 8;
// Six doubles as eight words of 48 payload bits under a 16-bit tag (half a
// line): word m of half h from its three doubles, and back.
__device__ __forceinline__ uint64_t pack48(int m, uint64_t d0, uint64_t d1, uint64_t d2) {
  constexpr uint64_t k48 = (1ull << 48) - 1;
  return m == 0 ? d0 & k48 : m == 1 ? (d0 >> 48 | d1 << 16) & k48 : m == 2 ? (d1 >> 32 | d2 << 32) & k48 : d2 >> 16;
}
__device__ __forceinline__ void put_word48(uint64_t* p, uint32_t epoch, uint64_t v) {
  __hip_atomic_store(p, ((uint64_t)(epoch & 0xffffu) << 48) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool tagged48(uint64_t w, uint32_t epoch) { return (uint32_t)(w >> 48) == (epoch & 0xffffu); }

// Ends a poll that has lasted kPollTicks (kResWait seconds of the 100 MHz
// clock) or that another workgroup has ended: every wait is bounded, and the
// host then solves by launches.
constexpr long long kPollTicks = (long long)(kResWait * 1e8);
struct Poll {
  int n = 0;
  long long t0 = 0;
  __device__ __forceinline__ bool give_up(const int* abort_flag) {
    if ((++n & 255) != 0) return false;
    const long long now = wall_clock64();
    if (t0 == 0) t0 = now;
    return now - t0 > kPollTicks || __hip_atomic_load(abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
  }
};

// x + x of the lane 16 (32) away, in both.
__device__ __forceinline__ double add_row_pair(double v) {
  const uint64_t u = (uint64_t)__double_as_longlong(v);
  const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)u, (uint32_t)u, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)(u >> 32), (uint32_t)(u >> 32), false, false);
  return __longlong_as_double((long long)(((uint64_t)hi[0] << 32) | lo[0])) +
         __longlong_as_double((long long)(((uint64_t)hi[1] << 32) | lo[1]));
}
__device__ __forceinline__ double add_half_pair(double v) {
  const uint64_t u = (uint64_t)__double_as_longlong(v);
  const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)u, (uint32_t)u, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((uint32_t)(u >> 32), (uint32_t)(u >> 32), false, false);
  return __longlong_as_double((long long)(((uint64_t)hi[0] << 32) | lo[0])) +
         __longlong_as_double((long long)(((uint64_t)hi[1] << 32) | lo[1]));
}

// One workgroup's view of the exchange.
template <int NT>
struct Meet {
  static constexpr int nw = NT / kWave;
  double* red;   // [4 nw] wave sums
  double* tot;   // [4 nw] per-wave sums over the workgroups
  int* bad;
  uint64_t* slots;
  int G;
  int parity;
  const int* abort_flag;
  const int32_t* halo;  // [H] in LDS
  int H;

  // Wave sums of this thread's NV values into red (a barrier must follow before publish).
  template <int NV>
  __device__ __forceinline__ void wave_sums(const double (&v)[NV]) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const double s = wave_sum_last(v[k]);
      if (threadIdx.x % kWave == kWave - 1) red[k * nw + threadIdx.x / kWave] = s;
    }
  }
  __device__ __forceinline__ double local(int k) const {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < nw; ++w) s += red[k * nw + w];
    return s;
  }
  // The workgroup's NV <= 4 sums, one word per thread.
  template <int NV>
  __device__ __forceinline__ void publish(uint32_t epoch) {
    parity ^= 1;
    const int w = threadIdx.x % kSlotWords, c = threadIdx.x / kSlotWords;
    if (G > 1 && c < kResCopies && w < 2 * NV) {
      const uint64_t u = (uint64_t)__double_as_longlong(local(w >> 1));
      put_word(slots + (size_t)c * kResCopyWords + (parity * G + (int)blockIdx.x) * kSlotWords + w, epoch,
               (w & 1) ? (uint32_t)(u >> 32) : (uint32_t)u);
    }
  }
  // Waits for every workgroup's NV sums and (V not void) the words of the
  // workgroup's halo vertices in `words`, which go to dest (3 V per vertex, in
  // LDS). Each thread reads words NT apart; what has arrived is not read again.
  // The sums' wave sums go to tot.
  template <int NV, typename V>
  __device__ __forceinline__ void collect(uint32_t epoch, const uint64_t* words, uint32_t* dest) {
    constexpr int NS = NV > 0 ? kSlotWords * kResMaxParts / NT : 0;  // slot words per thread
    constexpr int VS = kVertStride<V>, VW = kVertWords<V>;
    constexpr int NH = sizeof(V) == 8 ? 8 : 5;                       // halo words per thread in flight
    const int t = opaque(threadIdx.x), sw = t % kSlotWords, hw = t % VS;
    const uint64_t* s = slots + (size_t)(blockIdx.x % kResCopies) * kResCopyWords + parity * G * kSlotWords + t;
    const bool halos = words != nullptr;
    uint32_t need = 0, sum[NS > 0 ? NS : 1];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      sum[k] = 0;
      if (G > 1 && sw < 2 * NV && (t + k * NT) / kSlotWords < G) need |= 1u << k;
    }
#pragma unroll
    for (int k = 0; k < NH; ++k) {
      if (halos && hw < VW && (t + k * NT) / VS < H) need |= 1u << (NS + k);
    }
    Poll poll;
    while (need) {
      uint64_t a[NS > 0 ? NS : 1], b[NH];
#pragma unroll
      for (int k = 0; k < NS; ++k)
        if (need >> k & 1) a[k] = get_word(s + k * NT);
#pragma unroll
      for (int k = 0; k < NH; ++k)
        if (need >> (NS + k) & 1) b[k] = get_word(words + (uint32_t)(halo[(t + k * NT) / VS] * VS + hw));
#pragma unroll
      for (int k = 0; k < NS; ++k)
        if ((need >> k & 1) && tagged(a[k], epoch)) {
          sum[k] = (uint32_t)a[k];
          need &= ~(1u << k);
        }
#pragma unroll
      for (int k = 0; k < NH; ++k)
        if ((need >> (NS + k) & 1) && tagged(b[k], epoch)) {
          dest[(t + k * NT) / VS * VW + hw] = (uint32_t)b[k];
          need &= ~(1u << (NS + k));
        }
      if (need && poll.give_up(abort_flag)) {
        *bad = 1;
        break;
      }
    }
    if (halos) {  // halos larger than NH words per thread
      for (int j = t + NH * NT; j < H * VS; j += NT) {
        if (hw >= VW) break;
        const uint64_t* p = words + (size_t)halo[j / VS] * VS + hw;
        uint64_t w = get_word(p);
        while (!tagged(w, epoch)) {
          if (poll.give_up(abort_flag)) {
            *bad = 1;
            break;
          }
          w = get_word(p);
        }
        dest[j / VS * VW + hw] = (uint32_t)w;
      }
    }
    if constexpr (NV > 0) {
      if (G == 1) {
        if ((int)threadIdx.x < nw * NV)
          tot[threadIdx.x] = threadIdx.x % nw == 0 ? local(threadIdx.x / nw) : 0.0;
      } else {
        double d = 0.0;  // both threads of a pair add the pair's double of every slot they read
#pragma unroll
        for (int k = 0; k < NS; ++k) {
          const uint32_t other = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)sum[k], 0xB1, 0xf, 0xf, true);
          const uint32_t lo = (t & 1) ? other : sum[k], hi = (t & 1) ? sum[k] : other;
          d += __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
        }
        d = dpp_add<0x128, 0xf>(d);  // row_ror 8: the other slot of the row of 16 lanes
        d = add_half_pair(add_row_pair(d));
        const int lane = threadIdx.x % kWave;
        if (lane < 2 * NV && lane % 2 == 0) tot[lane / 2 * nw + threadIdx.x / kWave] = d;
      }
    }
  }
  // Totals over all workgroups (after the barrier that follows collect): lane
  // 8 k + w takes wave w's sum of value k.
  template <int NV>
  __device__ __forceinline__ void totals(double (&v)[NV]) const {
    static_assert(nw == 8, "eight waves");
    const int lane = threadIdx.x % kWave;
    double s = tot[lane < NV * nw ? lane : 0];
    s = dpp_add<0xB1, 0xf>(s);   // quad_perm [1, 0, 3, 2]
    s = dpp_add<0x4E, 0xf>(s);   // quad_perm [2, 3, 0, 1]
    s = dpp_add<0x141, 0xf>(s);  // row_half_mirror: the other half of the eight lanes
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const uint64_t u = (uint64_t)__double_as_longlong(s);
      const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, k * nw);
      const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), k * nw);
      v[k] = __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
    }
  }
};

// Block-Jacobi PCG on H dx = -g (free DOFs), x0 = 0, of one whole run:
// kMixed = false in T = double to ||r|| <= rtol ||b||; kMixed in T = float with
// FP64 residual replacement each time the FP32 residual has dropped by
// inner_rtol, to ||b - A dx|| <= rtol ||b|| in FP64 (the scheme of
// run_mixed_solve).
//
// A workgroup owns a contiguous range of rows; workgroups of one XCD own
// neighbouring ranges. The rows' matrix blocks, in row order, are dealt K
// consecutive ones to a thread, which holds the first KR in registers, the
// next KL in LDS and the last KS in a private global array that L2 serves. The
// product leaves one partial per (row, thread) pair in LDS at slot row + thread
// (consecutive for a row, since both only grow along the block list), which
// the row's thread then sums in order. r and p of the rows and of their halo
// (the vertices of other workgroups they couple to) live in LDS.
//
// One meeting per iteration: after the product every workgroup publishes its
// exported rows' A p and its shares of
//   p.Ap, Ap.B^-1 Ap, r.z, r.r   (z = B^-1 r),
// so that everybody knows alpha = r.z / p.Ap, beta by the next r.z =
// alpha^2 Ap.B^-1 Ap - r.z (with z.Ap = p.Ap), and the stopping test on r.r,
// and then updates r, z and p of its own rows and of its halo alike (the same
// operations on the same values, so that the copies of p never differ). r.z in
// alpha and r.r are direct sums of the current residual: the expansion enters
// beta only. Iteration counts at 48^3 equal the two-launch form's (2,731 and
// 2,837 over a step in FP64 and mixed precision).
// On hard systems FP64 counts stay too (nu = 0.499, stiffness of 1e3 and 1e9 in
// layers or anything between at random: within 0.5%), while FP32 ones move either
// way: from the direct sum to this, at random 658 -> 778 (12^3) and 1,189 -> 1,483
// (20^3), in layers 27,874 -> 3,581. With z.Ap in the exchange as a fifth sum (rz
// - 2 alpha z.Ap + alpha^2 Ap.B^-1 Ap) they are the direct sum's again, 708, 1,188
// and 32,915.
// Slots and exported vertices' words exist twice and take turns by meeting: a
// workgroup writes a buffer again only after a meeting that every workgroup
// joined after its last read of it. (The FP64 correction's words are used once
// between two meetings.)
// All workgroups sum the same words in the same order and take the same
// decisions; results are bit-reproducible for a fixed cut.
//
// kTwo adds the coarse correction W E^-1 W^T r of the two-level preconditioner
// (sk_coarse.h), and with it a second meeting per iteration. In the first,
// workgroups also publish the restriction of their rows' A p to each aggregate
// they reach into (a piece: six doubles in one 64-byte chunk); everybody then
// holds the whole restricted residual c, and multiplies the rows of the coarse
// inverse of the aggregates that begin in it, read from L2. In the second they
// publish r.r, r.z with their share of c.y, and their aggregates' rigid motions,
// which the workgroups whose rows or halo lie in these add to z. Measured over a
// step, launches then this kernel: 48^3 FP64 25.5 -> 17.5 ms, mixed 19.8 -> 13.2;
// 32^3 13.0 -> 8.2 and 12.3 -> 8.1; 10^3 5.7 -> 3.7 and 6.3 -> 3.9. An iteration
// at 48^3 (31.4 and 24.7 us) is bound by its chain of phases: product 8 (FP64, five
// of a thread's blocks from L2) or 2 to 5, pieces of all 512 aggregates 4,
// rows of the inverse 3.5 to 4.5, second meeting 3 to 5, update 3, the rest around
// 1 each. With more blocks in registers the values in flight spill (152 registers
// at eight FP64 blocks: product 16 us).
//
// Why: the two-launch form reads 107 MB (FP64) of values per iteration and
// pays two launch boundaries; 256 CUs hold 128 MB in registers and 40 MB in
// LDS, so nothing but the halo has to move. Measured per iteration over a
// whole step, launches then this kernel: 48^3 FP64 30.8 -> 10.7 us, mixed 20.9
// -> 8.2; 32^3 mixed 12.6 -> 5.6; 10^3 FP64 11.9 -> 5.4 us. What bounds it is
// the meeting (about 2.2 us at 256 workgroups, 1.5 us at 8) and the latency of
// the phases between barriers; in FP64 at 48^3 also the product (2.9 us, two of
// a thread's twelve blocks streamed from L2). Exchanging B^-1 A p instead of
// A p, so that the halo needs neither r nor B^-1, was slower: the owner's x and
// r then leave LDS (FP64 10.7 -> 12.7 us, mixed equal).
template <typename T, int NT, int KR, bool kMixed, bool kTwo>
__global__ __launch_bounds__(NT, NT / 256) void resident_pcg_kernel(ResidentArgs<T> a) {
  extern __shared__ __align__(16) double dyn[];
  __shared__ double s_red[4 * (NT / kWave)];
  __shared__ double s_tot[4 * (NT / kWave)];
  __shared__ int s_bad;
  using PV = std::conditional_t<kMixed, double, T>;  // partials
  constexpr int kTier = kTwo ? kResTwoTier : kResMaxTier;
  const int t = threadIdx.x;
  // workgroup b runs on XCD b % 8: neighbouring parts there, so that most halo words stay in its L2
  const int me = a.G % 8 == 0 ? (blockIdx.x % 8) * (a.G / 8) + blockIdx.x / 8 : blockIdx.x;
  const int v0 = a.row0[me], R = a.row0[me + 1] - v0;
  const int b0 = a.bptr[v0], nb = a.bptr[v0 + R] - b0;
  const int h0 = a.halo_ptr[me], H = a.halo_ptr[me + 1] - h0;
  const int x0 = a.exp0[me], E = a.exp0[me + 1] - x0;
  const int K = a.K;
  T* P = reinterpret_cast<T*>(dyn);                                   // [max_local][3], at a constant address
  T* RL = P + 3 * a.max_local;                                        // [max_local][3] r
  T* HA = RL + 3 * a.max_local;                                       // [max_halo][3] what the halo's owners sent
  T* XL = HA + 3 * a.max_halo;                                        // [max_rows][3] x (kMixed; else in a.x)
  PV* part = reinterpret_cast<PV*>(XL + (kMixed ? 3 * a.max_rows + (a.max_halo + a.max_rows) % 2 : 0));
  double* P64 = reinterpret_cast<double*>(part + 3 * (a.max_rows + NT + 1));  // [max_local][3] (kMixed)
  T* L = reinterpret_cast<T*>(P64 + (kMixed ? 3 * a.max_local : 0));  // [KL][9][NT]
  int32_t* HX = reinterpret_cast<int32_t*>(L + (size_t)9 * NT * a.KL);  // [max_halo] places of the halo vertices
  uint16_t* EX = reinterpret_cast<uint16_t*>(HX + a.max_halo);        // [NT] partial slots of the exported rows
  const TwoLds tl = two_lds(a.ld, a.max_need, a.n_agg);
  double* W2 = dyn + two_start(sizeof(T) == 4, a.max_rows, a.max_local, a.max_halo, a.KL) / 8;  // coarse space (kTwo)
  double *C2 = W2 + tl.c, *UW = W2 + tl.uw, *RAW = W2 + tl.raw, *YS = RAW, *TM = W2 + tl.tm, *DS = W2 + tl.dsc, *SD = W2 + tl.s;
  int4* PC = reinterpret_cast<int4*>(W2 + tl.col);
  ushort2* AG = reinterpret_cast<ushort2*>(W2 + tl.agg);
  int32_t* NE = reinterpret_cast<int32_t*>(W2 + tl.end);               // [max_need] the list's aggregates
  uint16_t* LN = reinterpret_cast<uint16_t*>(NE + a.max_need);         // [max_local]
  T* S = a.stream + (size_t)me * a.KS * 9 * NT;
  if (t == 0) s_bad = 0;

  // the thread's blocks, their columns' byte offsets and which of them end a row
  T A[KR][9];
  uint32_t meta[(KR + 2 * kTier + 1) / 2];
#pragma unroll
  for (int k = 0; k < (KR + 2 * kTier + 1) / 2; ++k) meta[k] = 0;
  const int tb0 = t * K;
  auto load_block = [&](int k, T (&B)[9]) -> uint32_t {
#pragma unroll
    for (int m = 0; m < 9; ++m) B[m] = T(0);
    if (k >= K || tb0 + k >= nb) return 0;
    const int b = b0 + tb0 + k;
    const int64_t q = a.sell_pos[b];
#pragma unroll
    for (int m = 0; m < 9; ++m) B[m] = a.vals[slot_index<kSellC, 1>(q, m)];
    return a.lcol[b];
  };
  auto word = [&](int k) { return (meta[k / 2] >> (16 * (k & 1))) & 0xffffu; };
#pragma unroll
  for (int k = 0; k < KR; ++k) meta[k / 2] |= load_block(k, A[k]) << (16 * (k & 1));
#pragma unroll
  for (int k = 0; k < kTier; ++k)
    if (k < a.KL) {
      T B[9];
      meta[(KR + k) / 2] |= load_block(KR + k, B) << (16 * ((KR + k) & 1));
#pragma unroll
      for (int m = 0; m < 9; ++m) L[(k * 9 + m) * NT + t] = B[m];
    }
#pragma unroll
  for (int k = 0; k < kTier; ++k)
    if (k < a.KS) {
      T B[9];
      constexpr int k0 = KR + kTier;
      meta[(k0 + k) / 2] |= load_block(KR + a.KL + k, B) << (16 * ((k0 + k) & 1));
#pragma unroll
      for (int m = 0; m < 9; ++m) S[(k * 9 + m) * NT + t] = B[m];
    }
  const uint32_t flags = a.tflag[me * NT + t];
  const int slot0 = (int)a.trow[me * NT + t] + t;

  // y = A src for the workgroup's rows, as partials. The source entries of the
  // next U blocks are read before the current U are multiplied: the partials'
  // stores would otherwise keep every block's LDS reads behind the last block's.
  auto product = [&](const auto* __restrict__ src) {
    using V = std::remove_cv_t<std::remove_reference_t<decltype(src[0])>>;
    constexpr int U = sizeof(V) == 8 ? 2 : 4;
#pragma unroll
    for (int k = 0; k < (KR + 2 * kTier + 1) / 2; ++k) meta[k] = (uint32_t)opaque((int)meta[k]);
    const int tt = opaque(t);
    V y0 = 0, y1 = 0, y2 = 0;
    PV* o = part + 3 * slot0;
    const uint32_t fl = (uint32_t)opaque((int)flags);
    auto read = [&](uint32_t off, V (&p)[3]) {  // offsets are those of T vectors
      const V* q = reinterpret_cast<const V*>(reinterpret_cast<const char*>(src) + off * (sizeof(V) / sizeof(T)));
      p[0] = q[0];
      p[1] = q[1];
      p[2] = q[2];
    };
    auto add = [&](const T (&B)[9], const V (&p)[3], uint32_t last) {
      y0 = fma((V)B[2], p[2], fma((V)B[1], p[1], fma((V)B[0], p[0], y0)));
      y1 = fma((V)B[5], p[2], fma((V)B[4], p[1], fma((V)B[3], p[0], y1)));
      y2 = fma((V)B[8], p[2], fma((V)B[7], p[1], fma((V)B[6], p[0], y2)));
      if (last) {
        o[0] = (PV)y0;
        o[1] = (PV)y1;
        o[2] = (PV)y2;
        o += 3;
        y0 = y1 = y2 = V(0);
      }
    };
    T B0[9];  // the first streamed block, on its way during the others
    if (a.KS > 0) {
#pragma unroll
      for (int m = 0; m < 9; ++m) B0[m] = S[m * NT + tt];
    }
    V p[2][U][3];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (u < KR) read(word(u), p[0][u]);
#pragma unroll
    for (int k = 0; k < KR; k += U) {
      if (k < K) {
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (k + U + u < KR) read(word(k + U + u), p[(k / U + 1) & 1][u]);
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (k + u < KR) add(A[k + u], p[(k / U) & 1][u], fl & (1u << (k + u)));
      }
    }
#pragma unroll
    for (int k = 0; k < kTier; ++k)
      if (k < a.KL) {
        T B[9];
        V q[3];
        read(word(KR + k), q);
#pragma unroll
        for (int m = 0; m < 9; ++m) B[m] = L[(k * 9 + m) * NT + tt];
        add(B, q, fl & (1u << (KR + k)));
      }
    if (a.KS > 0) {
      V q[3];
      read(word(KR + kTier), q);
      add(B0, q, fl & (1u << (KR + kTier)));
    }
#pragma unroll
    for (int k = 1; k < kTier; ++k)
      if (k < a.KS) {
        T B[9];
        V q[3];
        read(word(KR + kTier + k), q);
#pragma unroll
        for (int m = 0; m < 9; ++m) B[m] = S[(k * 9 + m) * NT + tt];
        add(B, q, fl & (1u << (KR + kTier + k)));
      }
    o[0] = (PV)y0;  // the open row's partial (or a slot that no row reads)
    o[1] = (PV)y1;
    o[2] = (PV)y2;
  };

  // the thread's row
  const bool row = t < R;
  const int v = v0 + t;
  int s0 = 0, s1 = -1, fx = 7;
  if (row) {
    const int o0 = a.bptr[v] - b0, o1 = a.bptr[v + 1] - b0;
    s0 = t + o0 / K;
    s1 = t + (o1 - 1) / K;
    fx = 0;
    if (a.fixed) fx = (a.fixed[3 * v] ? 1 : 0) | (a.fixed[3 * v + 1] ? 2 : 0) | (a.fixed[3 * v + 2] ? 4 : 0);
  }
  auto rhs = [&](int q) { return (!row || ((fx >> q) & 1)) ? 0.0 : -a.g[3 * (int64_t)v + q]; };
  auto row_sum = [&](PV (&y)[3]) {
    // a row rarely spans more than kSpan threads: that many reads at once, then the rest
    constexpr int kSpan = 5;
    PV w[kSpan][3];
#pragma unroll
    for (int k = 0; k < kSpan; ++k)
#pragma unroll
      for (int q = 0; q < 3; ++q) w[k][q] = part[3 * (s0 + k < s1 ? s0 + k : s1) + q];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      y[q] = w[0][q];
#pragma unroll
      for (int k = 1; k < kSpan; ++k) y[q] += s0 + k <= s1 ? w[k][q] : PV(0);
    }
    for (int s = s0 + kSpan; s <= s1; ++s) {
#pragma unroll
      for (int q = 0; q < 3; ++q) y[q] += part[3 * s + q];
    }
#pragma unroll
    for (int q = 0; q < 3; ++q)
      if ((fx >> q) & 1) y[q] = PV(0);
  };
  // B^-1 of a vertex: read again each iteration rather than kept (the product needs the registers)
  auto load_binv = [&](int64_t vertex, T (&B)[kBinv]) {
#pragma unroll
    for (int k = 0; k < kBinv; ++k) B[k] = a.binv[kBinv * vertex + k];
  };
  // z = B^-1 r and p = z + beta p, in one order of operations for owners and halos
  auto precondition = [&](const T (&B)[kBinv], const T (&r)[3], T (&z)[3]) {
    z[0] = fma(B[2], r[2], fma(B[1], r[1], B[0] * r[0]));
    z[1] = fma(B[4], r[2], fma(B[3], r[1], B[1] * r[0]));
    z[2] = fma(B[5], r[2], fma(B[4], r[1], B[2] * r[0]));
  };
  auto direction = [&](int l, const T (&B)[kBinv], const T (&r)[3], T beta) {
    T z[3];
    precondition(B, r, z);
#pragma unroll
    for (int q = 0; q < 3; ++q) P[3 * l + q] = fma(beta, P[3 * l + q], z[q]);
  };
  // The exported rows' three values, staged in the rows' own partial slots, by all threads in word order
  // (after a barrier).
  auto put_exports = [&](auto tag, uint64_t* words, uint32_t epoch) {
    using V = decltype(tag);
    constexpr int VS = kVertStride<V>, VW = kVertWords<V>;
    constexpr int U = sizeof(V) == 8 ? 2 : 4;
    for (int j0 = t; j0 < E * VS; j0 += U * NT) {  // U words' LDS reads under way together
      const int w = j0 % VS < VW ? j0 % VS : 0;
      uint32_t u[U];
      int e[U];
#pragma unroll
      for (int k = 0; k < U; ++k) e[k] = EX[j0 + k * NT < E * VS ? (j0 + k * NT) / VS : 0];
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const PV* src = part + 3 * e[k];
        if constexpr (sizeof(V) == 8) u[k] = reinterpret_cast<const uint32_t*>(src)[w];
        else u[k] = __float_as_uint((float)src[w]);
      }
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (j0 % VS < VW && j0 + k * NT < E * VS) put_word(words + (size_t)x0 * VS + j0 + k * NT, epoch, u[k]);
    }
  };
  for (int j = t; j < H; j += NT) HX[j] = a.halo[h0 + j];
  for (int j = t; j < E; j += NT) EX[j] = a.exslot[x0 + j];
  const int hv = t < H ? a.hvert[h0 + t] : 0;

  // ---- coarse space
  const int p0 = kTwo ? a.piece0[me] : 0, np = kTwo ? a.piece0[me + 1] - p0 : 0;
  const int a0 = kTwo ? a.own0[me] : 0, nown = kTwo ? a.own0[me + 1] - a0 : 0;
  const int n0 = kTwo ? a.need0[me] : 0, nneed = kTwo ? a.need0[me + 1] - n0 : 0;
  const int wid = t / kWave;
  int my_piece = -1, pf = 0, pl = -1;  // of the thread's row; of the wave's rows
  if constexpr (kTwo) {
    for (int j = t; j < R; j += NT) {
      const int64_t k = 3 * (int64_t)(v0 + j);
      const int f = a.fixed ? (a.fixed[k] ? 1 : 0) | (a.fixed[k + 1] ? 2 : 0) | (a.fixed[k + 2] ? 4 : 0) : 0;
      LN[j] = (uint16_t)(a.lrow[v0 + j] << 3 | f);
    }
    for (int j = t; j < H; j += NT) {
      const int64_t k = 3 * (int64_t)a.hvert[h0 + j];
      const int f = a.fixed ? (a.fixed[k] ? 1 : 0) | (a.fixed[k + 1] ? 2 : 0) | (a.fixed[k + 2] ? 4 : 0) : 0;
      LN[R + j] = (uint16_t)(a.lhalo[h0 + j] << 3 | f);
    }
    for (int j = t; j < nneed; j += NT) NE[j] = a.need[n0 + j];
    for (int j = t; j < np * 36; j += NT) TM[j] = a.tm[36 * (int64_t)a.pagg[p0 + j / 36] + j % 36];
    for (int j = t; j < np * 6; j += NT) {
      const int c = a.agg_col[a.pagg[p0 + j / 6]] + j % 6;
      DS[j] = c < a.agg_col[a.pagg[p0 + j / 6] + 1] ? a.dsc[c] : 0.0;
    }
    for (int j = t; j <= a.n_agg; j += NT) AG[j] = make_ushort2((uint16_t)a.apiece[j], (uint16_t)a.agg_col[j]);
    for (int j = t; j < np; j += NT) {
      const int c = a.agg_col[a.pagg[p0 + j]];
      const int r0 = max(0, a.agg_ptr[a.pagg[p0 + j]] - v0), r1 = min(R, a.agg_ptr[a.pagg[p0 + j] + 1] - v0);
      PC[j] = make_int4(c, a.agg_col[a.pagg[p0 + j] + 1] - c, r0 / kWave, (r1 - 1) / kWave);
    }
    for (int j = t; j < a.ld; j += NT) C2[j] = 0.0;
    auto piece_of = [&](int r) {
      // pieces of one workgroup are aggregates pagg[p0], pagg[p0] + 1, ...
      int j = 0;
      while (j + 1 < np && v0 + r >= a.agg_ptr[a.pagg[p0 + j + 1]]) ++j;
      return j;
    };
    if (row) my_piece = piece_of(t);
    if (wid * kWave < R) {
      pf = piece_of(wid * kWave);
      pl = piece_of(min(wid * kWave + kWave - 1, R - 1));
    }
  }
  // The wave's shares of W^T q over the thread's rows, by piece (every thread).
  auto restrict_rows = [&](double q0, double q1, double q2) {
    const int t = opaque((int)threadIdx.x);
    double d[3] = {0.0, 0.0, 0.0};
    if (row) {
#pragma unroll
      for (int q = 0; q < 3; ++q) d[q] = a.dv[3 * (int64_t)(v0 + t) + q];
    }
    const double m[6] = {q0, q1, q2, d[1] * q2 - d[2] * q1, d[2] * q0 - d[0] * q2, d[0] * q1 - d[1] * q0};
    for (int j = pf; j <= pl; ++j) {
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        const double w = wave_sum_last(j == my_piece ? m[q] : 0.0);
        if (t % kWave == kWave - 1) RAW[(j * (NT / kWave) + t / kWave) * 6 + q] = w;
      }
    }
  };
  // The pieces' scaled restrictions (wave 0, after a barrier) as `words`: of A p in cwords, of a residual in rwords.
  auto put_pieces = [&](uint32_t epoch, uint64_t* words) {
    const int t = opaque((int)threadIdx.x);
    if (t >= kWave) return;
    const int j = t / 6, q = t % 6;
    if (t < np * 6) {
      const int w0 = PC[j].z, w1 = PC[j].w;
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < NT / kWave; ++w)
        if (w >= w0 && w <= w1) s += RAW[(j * (NT / kWave) + w) * 6 + q];
      SD[t] = s;
    }
    wave_lds_fence();
    double d = 0.0;
    if (t < np * 6) {
#pragma unroll
      for (int m = 0; m < 6; ++m) d += TM[36 * j + 6 * m + q] * SD[6 * j + m];
      d *= DS[t];
    }
    wave_lds_fence();
    if (t < np * 6) SD[t] = d;
    wave_lds_fence();
    if (t < np * kAggWords) {
      const uint64_t* d3 = reinterpret_cast<const uint64_t*>(SD + 3 * (t / 4));
      put_word48(words + (size_t)p0 * kAggWords + t, epoch, pack48(t % 4, d3[0], d3[1], d3[2]));
    }
  };
  // c = keep c + f (sum over an aggregate's pieces). Slot n is word n % 8 of aggregate n / 8: neighbouring lanes
  // read neighbouring words, and lanes 0 to 2 of a quad make a double each of their own word and the next one.
  // The thread's first kSlots sums stay in registers until f is known, further ones are read again.
  constexpr int kSlots = 8;
  auto three_of_four = [&](uint64_t w) {
    constexpr uint64_t k48 = (1ull << 48) - 1;
    const int m = threadIdx.x % 4;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)w, 0xF9, 0xf, 0xf, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(w >> 32), 0xF9, 0xf, 0xf, true);
    const uint64_t next = ((uint64_t)hi << 32) | lo;  // quad_perm [1, 2, 3, 3]
    return __longlong_as_double((long long)((w & k48) >> (16 * m) | next << (48 - 16 * m)));
  };
  // sums of the slots t + (i0 + i) NT
  auto get_slots = [&](int i0, uint32_t epoch, const uint64_t* words, auto& d) {
    constexpr int N = sizeof(d) / sizeof(double);
    const int t = opaque((int)threadIdx.x) + i0 * NT;
    Poll poll;
    int most = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int I = (t + i * NT) / kAggWords;
      d[i] = 0.0;
      if (I < a.n_agg) most = max(most, AG[I + 1].x - AG[I].x);
    }
    for (int k = 0; k < most; ++k) {  // the k-th pieces of all slots together
      uint64_t u[N];
      uint32_t need = 0;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int I = (t + i * NT) / kAggWords;
        u[i] = 0;
        if (I < a.n_agg && k < AG[I + 1].x - AG[I].x) need |= 1u << i;
      }
      const uint32_t mine = need;
      while (need) {
#pragma unroll
        for (int i = 0; i < N; ++i)
          if (need >> i & 1) u[i] = get_word(words + (uint32_t)((AG[(t + i * NT) / kAggWords].x + k) * kAggWords + t % kAggWords));
#pragma unroll
        for (int i = 0; i < N; ++i)
          if ((need >> i & 1) && tagged48(u[i], epoch)) need &= ~(1u << i);
        if (need && poll.give_up(a.abort_flag)) {
          s_bad = 1;
          break;
        }
      }
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const double x = three_of_four(u[i]);
        if (mine >> i & 1) d[i] += x;
      }
    }
  };
  auto add_slots = [&](int i0, const auto& d, double keep, double f) {
    constexpr int N = sizeof(d) / sizeof(double);
    const int t = opaque((int)threadIdx.x) + i0 * NT, m = t % kAggWords, q = m % 4 + m / 4 * 3;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int I = (t + i * NT) / kAggWords;
      if (I < a.n_agg && m % 4 < 3 && AG[I].y + q < AG[I + 1].y) {
        double* c = C2 + AG[I].y + q;
        *c = fma(f, d[i], keep * *c);
      }
    }
  };
  auto add_all = [&](uint32_t epoch, const double (&dh)[kSlots], double f) {
    add_slots(0, dh, 1.0, f);
    for (int i0 = kSlots; i0 * NT < a.n_agg * kAggWords; ++i0) {
      double d[1];
      get_slots(i0, epoch, a.cwords, d);
      add_slots(i0, d, 1.0, f);
    }
  };
  // c = the residual's restriction, a slot per thread at a time: this is rare, and eight at once, inlined here too,
  // take registers that the product needs (FP64 14.55 ms a step at 48^3 against 14.14; mixed, where the replaced
  // residual is read this way as well, 16.5 against 15.5).
  auto take_residual = [&](uint32_t epoch) {
    for (int i0 = 0; i0 * NT < a.n_agg * kAggWords; ++i0) {
      double d[1];
      get_slots(i0, epoch, a.rwords, d);
      add_slots(i0, d, 0.0, 1.0);
    }
  };
  // y = (S16 + shift) c for the unknowns of the aggregates that begin here, as wave shares (after a barrier).
  auto coarse_product = [&]() {
    const uint4* E8 = reinterpret_cast<const uint4*>(a.einv);
    const int t = opaque((int)threadIdx.x), ld8 = a.ld >> 3;
    double c[8];
#pragma unroll
    for (int h = 0; h < 8; ++h) c[h] = t < ld8 ? C2[8 * t + h] : 0.0;
    for (int i = 0; i < nown; ++i) {
      const int4 pc = PC[i + np - nown];
      uint4 e[6];
#pragma unroll
      for (int q = 0; q < 6; ++q)
        e[q] = q < pc.y && t < ld8 ? E8[(uint32_t)((pc.x + q) * ld8 + t)] : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        const uint32_t wd[4] = {e[q].x, e[q].y, e[q].z, e[q].w};
        double y = 0.0;
#pragma unroll
        for (int h = 0; h < 4; ++h)
          y += (double)half_lo(wd[h]) * c[2 * h] + (double)half_hi(wd[h]) * c[2 * h + 1];
        y = wave_sum_last(y);
        if (t % kWave == kWave - 1) YS[(6 * i + q) * (NT / kWave) + t / kWave] = y;
      }
    }
  };
  // From the wave shares (after a barrier; wave 0): the aggregates' rigid motions; c.y is added to s_red[0].
  auto put_motions = [&](uint32_t epoch) {
    const int t = opaque((int)threadIdx.x);
    if (t >= kWave) return;
    const int i = t / 6, q = t % 6, j = i + np - nown;  // piece of owned aggregate i
    double cy = 0.0;
    if (t < nown * 6) {
      const int4 pc = PC[j];
      double y = 0.0;
      if (q < pc.y) {
#pragma unroll
        for (int w = 0; w < NT / kWave; ++w) y += YS[t * (NT / kWave) + w];
        const double c = C2[pc.x + q];
        y += a.shift * c;
        cy = c * y;
        y *= DS[6 * j + q];
      }
      SD[t] = y;
    }
    cy = wave_sum_last(cy);
    if (t == kWave - 1) s_red[0] += cy;
    wave_lds_fence();
    double u = 0.0;
    if (t < nown * 6) {
#pragma unroll
      for (int m = 0; m < 6; ++m) u += TM[36 * j + 6 * q + m] * SD[6 * i + m];
    }
    wave_lds_fence();
    if (t < nown * 6) SD[t] = u;
    wave_lds_fence();
    if (t < nown * kAggWords) {
      const uint64_t* d3 = reinterpret_cast<const uint64_t*>(SD + 3 * (t / 4));
      put_word48(a.uwords + (size_t)a0 * kAggWords + t, epoch, pack48(t % 4, d3[0], d3[1], d3[2]));
    }
  };
  // The rigid motions of the workgroup's list, into UW.
  auto get_motions = [&](uint32_t epoch) {
    Poll poll;
    for (int j = opaque((int)threadIdx.x); j < nneed * kAggWords; j += NT) {
      const uint64_t* p = a.uwords + (uint32_t)(NE[j / kAggWords] * kAggWords + j % kAggWords);
      uint64_t w = get_word(p);
      while (!tagged48(w, epoch)) {
        if (poll.give_up(a.abort_flag)) {
          s_bad = 1;
          break;
        }
        w = get_word(p);
      }
      uint16_t* o = reinterpret_cast<uint16_t*>(UW) + 3 * j;
      o[0] = (uint16_t)w;
      o[1] = (uint16_t)(w >> 16);
      o[2] = (uint16_t)(w >> 32);
    }
  };
  // z += the rigid motion of local vertex l (mesh vertex w) on its free DOFs
  auto prolong = [&](int l, const double (&d)[3], T (&z)[3]) {
    const int n = LN[l];
    const double* u = UW + 6 * (n >> 3);
    const double c[3] = {u[0] + u[4] * d[2] - u[5] * d[1], u[1] + u[5] * d[0] - u[3] * d[2],
                         u[2] + u[3] * d[1] - u[4] * d[0]};
#pragma unroll
    for (int q = 0; q < 3; ++q)
      if (!((n >> q) & 1)) z[q] = (T)((double)z[q] + c[q]);
  };

  // start: r = b, x = 0, p = z
  double acc0[1] = {0.0};
  if (row) {
    T B[kBinv], r[3];
    load_binv(v, B);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const double b = rhs(q);
      acc0[0] += b * b;
      r[q] = (T)b;
      RL[3 * t + q] = r[q];
      if (kMixed) XL[3 * t + q] = T(0);
      else a.x[3 * (int64_t)v + q] = 0.0;
      P[3 * t + q] = T(0);
    }
    direction(t, B, r, T(0));
  }
  for (int j = t; j < H; j += NT) {
    const int64_t w = a.hvert[h0 + j];
    T B[kBinv], r[3];
    load_binv(w, B);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      r[q] = (a.fixed && a.fixed[3 * w + q]) ? T(0) : (T)-a.g[3 * w + q];
      RL[3 * (R + j) + q] = r[q];
      P[3 * (R + j) + q] = T(0);
    }
    direction(R + j, B, r, T(0));
  }

  Meet<NT> meet{s_red, s_tot, &s_bad, a.slots, a.G, 0, a.abort_flag, HX, H};
  uint32_t epoch = a.epoch;
  int iter = 0, done = 0, refines = 0;
  double tol2 = 0.0, target = 0.0;
  bool fresh = true;  // the tolerance starts from this residual
  __syncthreads();
  if constexpr (kTwo) {
    double acc1[1] = {acc0[0]};
    double dh[kSlots];
    // what `directions` reads from memory: offsets of the row and of the first halo vertex, B^-1 of the latter
    T BH[kBinv];
    double dr[3], dq[3];
    auto prefetch_directions = [&]() {
      const int64_t w = row ? opaque(v) : 0, u = opaque(hv);
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        dr[q] = a.dv[3 * w + q];
        dq[q] = a.dv[3 * u + q];
      }
      load_binv(u, BH);
    };
    // Second meeting of an iteration (c complete, after a barrier): totals of r.z and r.r
    auto second = [&](double rzb, double rrl, double& rz_out, double& rr_out) -> bool {
      coarse_product();
      double vb[2] = {rzb, rrl};
      meet.template wave_sums<2>(vb);
      lds_barrier();
      ++epoch;
      put_motions(epoch);
      meet.template publish<2>(epoch);
      meet.template collect<2, T>(epoch, nullptr, nullptr);
      prefetch_directions();
      get_motions(epoch);
      lds_barrier();
      if (s_bad) return false;
      meet.template totals<2>(vb);
      rz_out = vb[0];
      rr_out = vb[1];
      return true;
    };
    // p = z + beta p, z = B^-1 r + coarse part (zb: the row's B^-1 r)
    auto directions = [&](T beta, const T (&zb)[3]) {
      const int l = opaque(t);
      if (row) {
        T z[3] = {zb[0], zb[1], zb[2]};
        prolong(l, dr, z);
#pragma unroll
        for (int q = 0; q < 3; ++q) P[3 * l + q] = fma(beta, P[3 * l + q], z[q]);
      }
      for (int j = l; j < H; j += NT) {
        if (j != l) {
          const int64_t w = a.hvert[h0 + j];
#pragma unroll
          for (int q = 0; q < 3; ++q) dq[q] = a.dv[3 * w + q];
          load_binv(w, BH);
        }
        T z[3];
        const T rh[3] = {RL[3 * (R + j)], RL[3 * (R + j) + 1], RL[3 * (R + j) + 2]};
        precondition(BH, rh, z);
        prolong(R + j, dq, z);
#pragma unroll
        for (int q = 0; q < 3; ++q) P[3 * (R + j) + q] = fma(beta, P[3 * (R + j) + q], z[q]);
      }
      lds_barrier();
    };
    T z[3] = {T(0), T(0), T(0)};  // the row's B^-1 r
    double rz = 0.0, rr = 0.0;
    bool go = true;
    {  // the first residual
      T B[kBinv], r[3] = {T(0), T(0), T(0)};
      double v2[2] = {0.0, 0.0};
      if (row) {
        load_binv(v, B);
#pragma unroll
        for (int q = 0; q < 3; ++q) r[q] = RL[3 * t + q];
        precondition(B, r, z);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          v2[0] += (double)r[q] * (double)z[q];
          v2[1] += (double)r[q] * (double)r[q];
        }
      }
      restrict_rows((double)r[0], (double)r[1], (double)r[2]);
      meet.template wave_sums<1>(acc1);
      lds_barrier();
      meet.template publish<1>(++epoch);
      put_pieces(epoch, a.rwords);
      meet.template collect<1, T>(epoch, nullptr, nullptr);
      take_residual(epoch);
      lds_barrier();
      go = !s_bad;
      if (go) {
        meet.template totals<1>(acc1);
        target = a.rtol2 * acc1[0];
        go = second(v2[0], v2[1], rz, rr);
      }
      if (go) {
        tol2 = (kMixed ? a.inner_rtol2 : a.rtol2) * rr;
        if (!(isfinite(acc1[0]) && isfinite(rr) && isfinite(rz))) done = 3;
        else if (!(rr > tol2)) done = 1;
        go = done == 0;
        if (go) directions(T(0), z);
      }
    }
    double rr_hi = rr;  // largest r.r since c was last formed from r, and the iterations since
    int since = 0;
    while (go) {
      if (!kMixed && iter >= a.max_iter) break;
      product(P);
      T B[kBinv], r[3] = {T(0), T(0), T(0)}, ap[3] = {T(0), T(0), T(0)};
      lds_barrier();
      double va[1] = {0.0};
      if (row) {
        const int l = opaque(t);
        PV y[3];
        row_sum(y);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          ap[q] = (T)y[q];
          part[3 * s0 + q] = (PV)ap[q];
          va[0] += (double)P[3 * l + q] * (double)ap[q];
        }
      }
      restrict_rows((double)ap[0], (double)ap[1], (double)ap[2]);
      meet.template wave_sums<1>(va);
      lds_barrier();
      meet.template publish<1>(++epoch);
      uint64_t* zx = a.zx + meet.parity * a.zx_half;
      put_exports(T(0), zx, epoch);
      put_pieces(epoch, a.cwords);
      get_slots(0, epoch, a.cwords, dh);
      meet.template collect<1, T>(epoch, zx, reinterpret_cast<uint32_t*>(HA));
      load_binv(row ? opaque(v) : 0, B);
      double xg[3];
      if (!kMixed && row) {
#pragma unroll
        for (int q = 0; q < 3; ++q) xg[q] = a.x[3 * (int64_t)opaque(v) + q];
      }
      lds_barrier();
      if (s_bad) break;
      meet.template totals<1>(va);
      const double pAp = va[0];
      if (!(pAp > 0.0)) {
        done = isfinite(pAp) ? 2 : 3;
        break;
      }
      const T alpha = (T)(rz / pAp);
      ++iter;
      const bool renew = rr < kRenew<kMixed> * rr_hi || ++since == kRenewAfter;
      if (!renew) add_all(epoch, dh, -(double)alpha);
      const int l = opaque(t);
      double v2[2] = {0.0, 0.0};
      if (row) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          if (kMixed) XL[3 * l + q] = fma(alpha, P[3 * l + q], XL[3 * l + q]);
          else a.x[3 * (int64_t)(v0 + l) + q] = fma((double)alpha, (double)P[3 * l + q], xg[q]);
          r[q] = fma(-alpha, ap[q], RL[3 * l + q]);
          RL[3 * l + q] = r[q];
        }
        precondition(B, r, z);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          v2[0] += (double)r[q] * (double)z[q];
          v2[1] += (double)r[q] * (double)r[q];
        }
      }
      for (int j = l; j < H; j += NT) {
#pragma unroll
        for (int q = 0; q < 3; ++q) RL[3 * (R + j) + q] = fma(-alpha, HA[3 * j + q], RL[3 * (R + j) + q]);
      }
      if (renew) {
        restrict_rows((double)r[0], (double)r[1], (double)r[2]);
        lds_barrier();
        put_pieces(++epoch, a.rwords);
        take_residual(epoch);
        rr_hi = 0.0;
        since = 0;
      }
      lds_barrier();
      double rz_next;
      if (!second(v2[0], v2[1], rz_next, rr)) break;
      if (!isfinite(rr)) {
        done = 3;
        break;
      }
      rr_hi = rr > rr_hi ? rr : rr_hi;
      const bool conv = !(rr > tol2), limit = iter >= a.max_iter;
      if constexpr (!kMixed) {
        if (conv) {
          done = 1;
          break;
        }
      } else if (conv || limit) {
        // residual replacement: dx += x and r = b - A dx in FP64; the search direction is kept
        ++epoch;
        ++refines;
        if (row) {
          double x64[3];
#pragma unroll
          for (int q = 0; q < 3; ++q) {
            double& dx = a.x[3 * (int64_t)v + q];
            x64[q] = refines == 1 ? (double)XL[3 * t + q] : dx + (double)XL[3 * t + q];
            dx = x64[q];
            XL[3 * t + q] = T(0);
            P64[3 * t + q] = x64[q];
            part[3 * s0 + q] = x64[q];
          }
        }
        lds_barrier();
        put_exports(double(0), a.xx, epoch);
        meet.template collect<0, double>(epoch, a.xx, reinterpret_cast<uint32_t*>(P64 + 3 * R));
        lds_barrier();
        if (s_bad) break;
        product(P64);
        lds_barrier();
        double vb[1] = {0.0};
        v2[0] = v2[1] = 0.0;
        if (row) {
          PV y[3];
          row_sum(y);
          load_binv(v, B);
#pragma unroll
          for (int q = 0; q < 3; ++q) {
            const double rq = ((fx >> q) & 1) ? 0.0 : rhs(q) - (double)y[q];
            vb[0] += rq * rq;
            r[q] = (T)rq;
            part[3 * s0 + q] = (PV)r[q];
            RL[3 * t + q] = r[q];
          }
          precondition(B, r, z);
#pragma unroll
          for (int q = 0; q < 3; ++q) {
            v2[0] += (double)r[q] * (double)z[q];
            v2[1] += (double)r[q] * (double)r[q];
          }
        }
        restrict_rows((double)r[0], (double)r[1], (double)r[2]);
        meet.template wave_sums<1>(vb);
        lds_barrier();
        meet.template publish<1>(++epoch);
        zx = a.zx + meet.parity * a.zx_half;
        put_exports(T(0), zx, epoch);
        put_pieces(epoch, a.rwords);
        meet.template collect<1, T>(epoch, zx, reinterpret_cast<uint32_t*>(HA));
        take_residual(epoch);
        lds_barrier();
        if (s_bad) break;
        meet.template totals<1>(vb);
        if (!(vb[0] > target) || refines >= a.max_refine || limit) {
          done = vb[0] <= target ? 1 : isfinite(vb[0]) ? 0 : 3;
          break;
        }
        for (int j = t; j < H; j += NT) {
#pragma unroll
          for (int q = 0; q < 3; ++q) RL[3 * (R + j) + q] = HA[3 * j + q];
        }
        if (!second(v2[0], v2[1], rz_next, rr)) break;
        tol2 = a.inner_rtol2 * rr;
        rr_hi = rr;
        since = 0;
      }
      const T beta = (T)(rz_next / rz);
      rz = rz_next;
      directions(beta, z);
    }
  } else {
  if (kMixed) {  // ||b||^2 in FP64
    meet.template wave_sums<1>(acc0);
    lds_barrier();
    meet.template publish<1>(++epoch);
    meet.template collect<1, T>(epoch, nullptr, nullptr);
    lds_barrier();
    meet.template totals<1>(acc0);
    target = a.rtol2 * acc0[0];
  }
  const bool start = !kMixed || acc0[0] > 0.0;
  if (!start) done = acc0[0] == 0.0 ? 1 : 3;
  for (bool go = start && !s_bad; go;) {
    product(P);
    T B[kBinv], r[3], ap[3];
    load_binv(row ? opaque(v) : 0, B);
    lds_barrier();
    double va[4] = {0.0, 0.0, 0.0, 0.0};
    ++epoch;
    if (row) {
      const int l = opaque(t);
      PV y[3];
      row_sum(y);
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        ap[q] = (T)y[q];
        part[3 * s0 + q] = (PV)ap[q];  // staged for put_exports in the row's own slot
        r[q] = RL[3 * l + q];
      }
      T z[3], u[3];
      precondition(B, r, z);
      precondition(B, ap, u);
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        va[0] += (double)P[3 * l + q] * (double)ap[q];
        va[1] += (double)u[q] * (double)ap[q];
        va[2] += (double)r[q] * (double)z[q];
        va[3] += (double)r[q] * (double)r[q];
      }
    }
    meet.template wave_sums<4>(va);
    lds_barrier();
    meet.template publish<4>(epoch);
    uint64_t* zx = a.zx + meet.parity * a.zx_half;
    put_exports(T(0), zx, epoch);
    meet.template collect<4, T>(epoch, zx, reinterpret_cast<uint32_t*>(HA));
    T BH[kBinv];
    load_binv(row ? opaque(v) : 0, B);
    load_binv(opaque(hv), BH);
    double xg[3];
    if (!kMixed && row) {
#pragma unroll
      for (int q = 0; q < 3; ++q) xg[q] = a.x[3 * (int64_t)opaque(v) + q];
    }
    lds_barrier();
    if (s_bad) break;
    meet.template totals<4>(va);
    const double pAp = va[0], rz = va[2], rr = va[3];
    if (fresh) tol2 = (kMixed ? a.inner_rtol2 : a.rtol2) * rr;
    fresh = false;
    if (!(isfinite(rr) && isfinite(rz))) {
      done = 3;
      break;
    }
    const bool conv = !(rr > tol2), limit = iter >= a.max_iter;
    if (conv || limit) {
      if constexpr (!kMixed) {
        done = conv ? 1 : 0;
        break;
      } else {
        // residual replacement: dx += x and r = b - A dx in FP64. p was formed from the old r; with the new
        // one, z + beta p_before is z + (r.z / old r.z) (p - old z).
        ++epoch;
        ++refines;
        if (row) {
          double x64[3];
#pragma unroll
          for (int q = 0; q < 3; ++q) {
            double& dx = a.x[3 * (int64_t)v + q];
            x64[q] = refines == 1 ? (double)XL[3 * t + q] : dx + (double)XL[3 * t + q];
            dx = x64[q];
            XL[3 * t + q] = T(0);
            P64[3 * t + q] = x64[q];
            part[3 * s0 + q] = x64[q];
          }
        }
        lds_barrier();
        put_exports(double(0), a.xx, epoch);
        meet.template collect<0, double>(epoch, a.xx, reinterpret_cast<uint32_t*>(P64 + 3 * R));
        lds_barrier();
        if (s_bad) break;
        product(P64);
        lds_barrier();
        double vb[2] = {0.0, 0.0};
        ++epoch;
        if (row) {
          PV y[3];
          row_sum(y);
          T z[3];
          load_binv(v, B);
#pragma unroll
          for (int q = 0; q < 3; ++q) {
            const double rq = ((fx >> q) & 1) ? 0.0 : rhs(q) - (double)y[q];
            vb[0] += rq * rq;
            r[q] = (T)rq;
            part[3 * s0 + q] = (PV)r[q];
          }
          precondition(B, r, z);
#pragma unroll
          for (int q = 0; q < 3; ++q) vb[1] += (double)r[q] * (double)z[q];
        }
        meet.template wave_sums<2>(vb);
        lds_barrier();
        meet.template publish<2>(epoch);
        zx = a.zx + meet.parity * a.zx_half;
        put_exports(T(0), zx, epoch);
        meet.template collect<2, T>(epoch, zx, reinterpret_cast<uint32_t*>(HA));
        lds_barrier();
        if (s_bad) break;
        meet.template totals<2>(vb);
        if (!(vb[0] > target) || refines >= a.max_refine || limit) {
          done = vb[0] <= target ? 1 : isfinite(vb[0]) ? 0 : 3;
          break;
        }
        const T ratio = (T)(vb[1] / rz);
        auto replace = [&](int l, const T (&Bl)[kBinv], const T (&rn)[3]) {
          T ro[3], zo[3], zn[3];
#pragma unroll
          for (int q = 0; q < 3; ++q) ro[q] = RL[3 * l + q];
          precondition(Bl, ro, zo);
          precondition(Bl, rn, zn);
#pragma unroll
          for (int q = 0; q < 3; ++q) {
            P[3 * l + q] = fma(ratio, P[3 * l + q] - zo[q], zn[q]);
            RL[3 * l + q] = rn[q];
          }
        };
        if (row) replace(t, B, r);
        for (int j = t; j < H; j += NT) {
          const T hr[3] = {HA[3 * j], HA[3 * j + 1], HA[3 * j + 2]};
          load_binv(a.hvert[h0 + j], BH);
          replace(R + j, BH, hr);
        }
        fresh = true;
        lds_barrier();
        continue;
      }
    }
    if (!(pAp > 0.0)) {
      done = isfinite(pAp) ? 2 : 3;
      break;
    }
    const double inv_pAp = 1.0 / pAp, inv_rz = 1.0 / rz;  // side by side
    const T alpha = (T)(rz * inv_pAp);
    // with alpha as rounded for the update: r.z of the residual that it leaves
    const double al = (double)alpha, rz_next = al * al * va[1] - rz;
    const T beta = (T)(rz_next > 0.0 ? rz_next * inv_rz : 0.0);
    ++iter;
    const int l = opaque(t);
    if (row) {
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        if (kMixed) XL[3 * l + q] = fma(alpha, P[3 * l + q], XL[3 * l + q]);
        else a.x[3 * (int64_t)(v0 + l) + q] = fma((double)alpha, (double)P[3 * l + q], xg[q]);
        r[q] = fma(-alpha, ap[q], RL[3 * l + q]);
        RL[3 * l + q] = r[q];
      }
      direction(l, B, r, beta);
    }
    for (int j = l; j < H; j += NT) {
      if (j != l) load_binv(a.hvert[h0 + j], BH);
      T rh[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        rh[q] = fma(-alpha, HA[3 * j + q], RL[3 * (R + j) + q]);
        RL[3 * (R + j) + q] = rh[q];
      }
      direction(R + j, BH, rh, beta);
    }
    lds_barrier();
  }
  }
  __syncthreads();
  if (s_bad) {
    if (t == 0) {
      __hip_atomic_store(a.abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      a.host->aborted = 1;
    }
    return;
  }
  if (kMixed && row && refines == 0) {
#pragma unroll
    for (int q = 0; q < 3; ++q) a.x[3 * (int64_t)v + q] = 0.0;
  }
  if (blockIdx.x == 0 && t == 0) {
    a.host->iter = iter;
    a.host->done = done;
    a.host->refines = refines;
    a.host->epoch = epoch;
  }
}

__global__ void resident_fill_kernel(int64_t n, uint64_t* p, uint64_t word) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = word;
}

int fill_words(DevBuf<uint64_t>& b, uint64_t word, hipStream_t st) {
  if (b.n) resident_fill_kernel<<<grid_for((int64_t)b.n), kBlock, 0, st>>>((int64_t)b.n, b.p, word);
  SK_HIP_CHECK(hipGetLastError());
  return SK_OK;
}

size_t two_lds_bytes(int ld, int max_need, int n_agg, int max_local) {
  return 8 * (size_t)two_lds(ld, max_need, n_agg).end + 4 * (size_t)max_need + 2 * (size_t)max_local + 16;  // 16: its start is rounded up
}
struct Permits {
  std::mutex mu;
  std::condition_variable cv;
  int used = 0, cus = -1;
};
Permits g_permits[64];

}  // namespace

ResidentState::~ResidentState() {
  if (host) (void)hipHostFree(host);
}

bool ResidentPermit::acquire(int parts, hipStream_t st) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return false;
  // Workgroups are dealt to the XCDs in turn, so one XCD takes up to an eighth, rounded up: charged for that on every
  // XCD, the runs that hold a permit fit each of them, not only the chip as a whole.
  const int need = (parts + 7) / 8 * 8;
  uint32_t mask[16] = {};
  int allowed = -1;
  if (hipExtStreamGetCUMask(st, 16, mask) == hipSuccess) {
    allowed = 0;
    for (uint32_t w : mask) allowed += __builtin_popcount(w);
  } else {
    (void)hipGetLastError();
  }
  Permits& P = g_permits[dev];
  std::unique_lock<std::mutex> lock(P.mu);
  if (P.cus < 0) {
    int n = 0;
    P.cus = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess ? n : 0;
  }
  // A stream restricted to some CUs: what it leaves on each XCD, and which other streams share it, is not known here.
  if (need > P.cus || (allowed >= 0 && allowed < P.cus)) return false;
  P.cv.wait(lock, [&] { return P.used + need <= P.cus; });
  P.used += need;
  dev_ = dev;
  held_ = need;
  st_ = st;
  return true;
}

void ResidentPermit::release() {
  if (!held_) return;
  // a step that ends early (an error) may not have waited for the run yet
  if (hipStreamQuery(st_) != hipSuccess) {
    (void)hipGetLastError();
    (void)hipStreamSynchronize(st_);
  }
  Permits& P = g_permits[dev_];
  {
    std::lock_guard<std::mutex> lock(P.mu);
    P.used -= held_;
  }
  P.cv.notify_all();
  held_ = 0;
}

int resident_parts(int64_t nv, int64_t nblk, bool fp32) {
  const int NT = fp32 ? kResNT32 : kResNT64;
  // at least enough workgroups that a row has a thread (with 10% for an uneven cut)
  const int64_t need = (11 * nv + 10 * NT - 1) / (10 * (int64_t)NT);
  int64_t G = nv <= NT ? 1 : need;
  // and about one block per thread: the product's latency costs more than the meeting of more workgroups
  // (per iteration, at 4 / 2 / 1 blocks per thread: 10^3 FP64 5.8 / 5.7 / 5.4 us, a 29 x 13 x 21 box 7.5 /
  // 7.1 / 6.9, 32^3 mixed 5.9 / 5.6 / 5.6)
  const int64_t target = NT;
  G = std::max(G, (nblk + target - 1) / target);
  if (G > 8) G = (G + 7) / 8 * 8;  // the same number of workgroups on every XCD
  if (G > kResMaxParts) G = kResMaxParts;
  if (nv > (int64_t)G * NT) return 0;
  return (int)std::max<int64_t>(G, 1);
}

// Blocks per thread in registers: the short variant where all of a thread's
// blocks fit it (no register spilled: 10^3 FP64 5.8 us an iteration against
// 6.5 us with the long one), else the long one.
static int resident_kr(bool fp32, bool two, int K) {
  if (fp32) return K <= kResShort32 ? kResShort32 : two ? kResTwoKR32 : kResKR32;
  return K <= kResShort64 ? kResShort64 : two ? kResTwoKR64 : kResKR64;
}

static std::shared_ptr<ResidentPlan> build_plan(sk_mesh* m, const std::vector<int32_t>& parts, bool fp32, int two_ld,
                                                int two_need, int two_agg, int* status) {
  *status = SK_OK;
  const int NT = fp32 ? kResNT32 : kResNT64;
  const int G = (int)parts.size() - 1;
  const int32_t *bptr = m->h_bptr.data(), *bcol = m->h_bcol.data();
  auto p = std::make_shared<ResidentPlan>();
  p->parts = parts;
  p->fp32 = fp32;
  p->two_ld = two_ld;
  p->two_need = two_need;
  p->two_agg = two_agg;
  p->G = G;
  int max_nb = 0;
  for (int g = 0; g < G; ++g) {
    p->max_rows = std::max(p->max_rows, parts[g + 1] - parts[g]);
    max_nb = std::max(max_nb, bptr[parts[g + 1]] - bptr[parts[g]]);
  }
  if (p->max_rows > NT) return nullptr;
  p->K = std::max(1, (max_nb + NT - 1) / NT);
  p->KR = resident_kr(fp32, two_ld > 0, p->K);
  const int tier = two_ld ? kResTwoTier : kResMaxTier;
  const int KR = p->KR;
  std::vector<int32_t> loc(m->nv, -1), halo_ptr(1, 0), halo;
  std::vector<int16_t> place(m->nv, -1);
  std::vector<int32_t> owner(m->nv), exp0(1, 0);
  for (int g = 0; g < G; ++g)
    for (int32_t r = parts[g]; r < parts[g + 1]; ++r) owner[r] = g;
  std::vector<uint16_t> lcol(m->nblk), trow((size_t)G * NT);
  std::vector<int32_t> tlast;
  tlast.reserve(m->nv);
  std::vector<int32_t> mine;
  for (int g = 0; g < G; ++g) {
    const int32_t r0 = parts[g], r1 = parts[g + 1];
    mine.clear();
    for (int32_t b = bptr[r0]; b < bptr[r1]; ++b) {
      const int32_t w = bcol[b];
      if ((w < r0 || w >= r1) && loc[w] < 0) {
        loc[w] = 0;
        mine.push_back(w);
      }
    }
    std::sort(mine.begin(), mine.end());
    const int rows = r1 - r0, local = rows + (int)mine.size();
    p->max_local = std::max(p->max_local, local);
    p->max_halo = std::max(p->max_halo, (int)mine.size());
    if (local * (fp32 ? 12 : 24) > 65535) return nullptr;
    for (size_t i = 0; i < mine.size(); ++i) {
      loc[mine[i]] = rows + (int)i;
      place[mine[i]] = 0;
    }
    int tk = 0;  // next thread whose first row is to be noted
    for (int32_t r = r0; r < r1; ++r) {
      for (int32_t b = bptr[r]; b < bptr[r + 1]; ++b) {
        const int32_t w = bcol[b];
        const int c = w >= r0 && w < r1 ? w - r0 : loc[w];
        lcol[b] = (uint16_t)(c * (fp32 ? 12 : 24));
      }
      tlast.push_back(bptr[r + 1] - 1 - bptr[r0]);  // the row's last block in the workgroup's list
      for (; tk < NT && tk * p->K < bptr[r + 1] - bptr[r0]; ++tk) trow[(size_t)g * NT + tk] = (uint16_t)(r - r0);
    }
    for (; tk < NT; ++tk) trow[(size_t)g * NT + tk] = (uint16_t)rows;
    for (int32_t w : mine) loc[w] = -1;
    halo.insert(halo.end(), mine.begin(), mine.end());
    halo_ptr.push_back((int32_t)halo.size());
  }
  // the exported vertices' places in their owners' lists, and the halos by them
  for (int g = 0; g < G; ++g) {
    int16_t e = 0;
    for (int32_t r = parts[g]; r < parts[g + 1]; ++r)
      if (place[r] >= 0) place[r] = e++;
    exp0.push_back(exp0.back() + e);
  }
  p->n_exp = exp0.back();
  std::vector<int32_t> where(std::max<size_t>(1, halo.size()), 0);
  for (size_t i = 0; i < halo.size(); ++i) where[i] = exp0[owner[halo[i]]] + place[halo[i]];
  std::vector<uint16_t> exslot(std::max(1, p->n_exp), 0);
  for (int64_t v = 0; v < m->nv; ++v)
    if (place[v] >= 0) {
      const int32_t r0 = parts[owner[v]];
      exslot[exp0[owner[v]] + place[v]] = (uint16_t)(v - r0 + (bptr[v] - bptr[r0]) / p->K);
    }
  const size_t base = base_lds(fp32, p->max_rows, p->max_local, p->max_halo) +
                      (two_ld ? two_lds_bytes(two_ld, two_need, two_agg, p->max_local) : 0) + kResStaticLds;
  if (base > (size_t)kResLds) return nullptr;
  const int rest = std::max(0, p->K - KR);
  p->KL = (int)std::min<size_t>(std::min(rest, tier), (kResLds - base) / tier_lds(fp32));
  p->KS = rest - p->KL;
  if (p->KS > tier) return nullptr;
  // the threads' row-end bits: registers, the LDS tier (`tier` bits), the streamed tier
  static_assert(kResKR32 + 2 * kResMaxTier <= 32 && kResTwoKR32 + 2 * kResTwoTier <= 32, "one bit per block");
  std::vector<uint32_t> tflag((size_t)G * NT, 0);
  for (int g = 0; g < G; ++g)
    for (int32_t r = parts[g]; r < parts[g + 1]; ++r) {
      const int th = tlast[r] / p->K, k = tlast[r] % p->K;
      tflag[(size_t)g * NT + th] |= 1u << (k < KR + p->KL ? k : KR + tier + (k - KR - p->KL));
    }
  p->lds = base - kResStaticLds + p->KL * tier_lds(fp32);
  // more than half of a CU's LDS: one workgroup per CU, so the runs spread over the chip
  p->lds = std::max<size_t>(p->lds, kResLds / 2 + 1024);
  std::vector<int32_t> row0(parts);
  auto up = [&]() -> int {
    SK_TRY(p->row0.upload(row0));
    SK_TRY(p->lcol.upload(lcol));
    SK_TRY(p->tflag.upload(tflag));
    SK_TRY(p->trow.upload(trow));
    SK_TRY(p->halo_ptr.upload(halo_ptr));
    SK_TRY(p->halo.upload(where));
    SK_TRY(p->hvert.upload(halo));
    SK_TRY(p->exp0.upload(exp0));
    SK_TRY(p->exslot.upload(exslot));
    return SK_OK;
  };
  *status = up();
  return *status == SK_OK ? p : nullptr;
}

// The coarse space seen by a cut; null when a workgroup would reach into more
// than kResMaxPieces aggregates.
static std::unique_ptr<ResidentTwo> build_two(const sk_mesh* m, const std::vector<int32_t>& parts, const CoarseSpace& C,
                                              int* status) {
  *status = SK_OK;
  const int G = (int)parts.size() - 1, n_agg = C.n_agg;
  std::vector<int32_t> ap(n_agg + 1), vagg(m->nv);
  if (hipMemcpy(ap.data(), C.agg_ptr.p, ap.size() * sizeof(int32_t), hipMemcpyDeviceToHost) != hipSuccess) {
    set_error("resident PCG: the aggregates could not be read");
    *status = SK_ERR_HIP;
    return nullptr;
  }
  for (int I = 0; I < n_agg; ++I)
    for (int32_t v = ap[I]; v < ap[I + 1]; ++v) vagg[v] = I;
  auto two = std::make_unique<ResidentTwo>();
  std::vector<int32_t> piece0(1, 0), pagg, apiece(n_agg + 1, -1), own0(G + 1), need0(1, 0), need, mine, ids;
  std::vector<uint16_t> lrow(m->nv), lhalo;
  std::vector<int32_t> seen(m->nv, -1), place(n_agg, -1);
  for (int g = 0; g < G; ++g) {
    const int32_t r0 = parts[g], r1 = parts[g + 1];
    own0[g] = (int32_t)(std::lower_bound(ap.begin(), ap.end() - 1, r0) - ap.begin());
    for (int I = vagg[r0]; I <= vagg[r1 - 1]; ++I) {
      if (apiece[I] < 0) apiece[I] = (int32_t)pagg.size();
      pagg.push_back(I);
    }
    if (vagg[r1 - 1] - vagg[r0] >= kResMaxPieces) return nullptr;
    piece0.push_back((int32_t)pagg.size());
    // the halo in the plan's order (ascending) and the aggregates of rows and halo
    mine.clear();
    for (int32_t b = m->h_bptr[r0]; b < m->h_bptr[r1]; ++b) {
      const int32_t w = m->h_bcol[b];
      if ((w < r0 || w >= r1) && seen[w] != g) {
        seen[w] = g;
        mine.push_back(w);
      }
    }
    std::sort(mine.begin(), mine.end());
    ids.clear();
    auto list = [&](int32_t w) {
      const int I = vagg[w];
      if (place[I] < 0) {
        place[I] = (int32_t)ids.size();
        ids.push_back(I);
      }
      return (uint16_t)place[I];
    };
    for (int32_t r = r0; r < r1; ++r) lrow[r] = list(r);
    for (int32_t w : mine) lhalo.push_back(list(w));
    for (int32_t I : ids) place[I] = -1;
    if (ids.size() >= (1u << 13)) return nullptr;
    need.insert(need.end(), ids.begin(), ids.end());
    need0.push_back((int32_t)need.size());
    two->max_need = std::max(two->max_need, (int)ids.size());
  }
  own0[G] = n_agg;
  apiece[n_agg] = (int32_t)pagg.size();
  two->n_piece = (int)pagg.size();
  if (two->n_piece > 65535) return nullptr;  // 16-bit numbers in LDS
  if (lhalo.empty()) lhalo.push_back(0);
  auto up = [&]() -> int {
    SK_TRY(two->piece0.upload(piece0));
    SK_TRY(two->pagg.upload(pagg));
    SK_TRY(two->apiece.upload(apiece));
    SK_TRY(two->own0.upload(own0));
    SK_TRY(two->need0.upload(need0));
    SK_TRY(two->need.upload(need));
    SK_TRY(two->lrow.upload(lrow));
    SK_TRY(two->lhalo.upload(lhalo));
    SK_TRY(two->cwords.alloc((size_t)two->n_piece * 16));
    SK_TRY(two->uwords.alloc((size_t)n_agg * 8));
    SK_HIP_CHECK(hipMemset(two->cwords.p, 0, two->cwords.n * 8));
    SK_HIP_CHECK(hipMemset(two->uwords.p, 0, two->uwords.n * 8));
    return SK_OK;
  };
  *status = up();
  return *status == SK_OK ? std::move(two) : nullptr;
}

static int prepare(ResidentState& R, sk_mesh* m, bool fp32, const CoarseSpace* coarse) {
  std::vector<int32_t> parts = R.parts;
  if (parts.empty()) {
    const int G = resident_parts(m->nv, m->nblk, fp32);
    if (G == 0) return SK_OK;
    std::vector<int32_t> ap;
    int most = 0;
    if (coarse) {
      ap.resize(coarse->n_agg + 1);
      SK_HIP_CHECK(hipMemcpy(ap.data(), coarse->agg_ptr.p, ap.size() * sizeof(int32_t), hipMemcpyDeviceToHost));
      for (int I = 0; I < coarse->n_agg; ++I) most = std::max(most, ap[I + 1] - ap[I]);
    }
    // With a coarse space and workgroups enough for one per aggregate, a whole number of workgroups for each, as few
    // as let the average one's blocks fit the short variant: pieces of an aggregate are read one after the other.
    // (A step, at 1 / 2 / 4 workgroups per aggregate and with equal cuts: 10^3 FP64 3.7 / 3.9 / 4.3 / 5.0 ms, 24^3 8.2
    // / 8.0 / 9.0 / 10.0, an 8 x 60 x 8 box 10.9 / 9.5 / 10.3 / 14.7.)
    const int64_t NT = fp32 ? kResNT32 : kResNT64, fill = NT * (fp32 ? kResShort32 : kResShort64);
    const int split = !coarse ? 0 : (int)std::max((most + NT - 1) / NT, (m->nblk + coarse->n_agg * fill - 1) / (coarse->n_agg * fill));
    if (coarse && G >= coarse->n_agg && split * coarse->n_agg <= kResMaxParts) {
      parts.push_back(0);
      for (int I = 0; I < coarse->n_agg; ++I)
        for (int k = 1; k <= split; ++k) {
          const int32_t end = ap[I] + (int32_t)((int64_t)(ap[I + 1] - ap[I]) * k / split);
          if (end > parts.back()) parts.push_back(end);
        }
    } else {
      for (int g = 0; g <= G; ++g) parts.push_back((int32_t)(m->nv * g / G));
    }
  }
  std::unique_ptr<ResidentTwo> two;
  if (coarse) {
    int s = SK_OK;
    two = build_two(m, parts, *coarse, &s);
    if (s != SK_OK) return s;
    if (!two) return SK_OK;
  }
  const int two_ld = coarse ? coarse->ld : 0, two_need = coarse ? two->max_need : 0,
            two_agg = coarse ? coarse->n_agg : 0;
  std::shared_ptr<ResidentPlan> plan;
  {
    std::lock_guard<std::mutex> lock(m->plan_mu);
    for (auto& p : m->plans)
      if (p->fp32 == fp32 && p->two_ld == two_ld && p->two_need == two_need &&
          p->two_agg == two_agg && p->parts == parts) plan = p;
    if (!plan) {
      int s = SK_OK;
      plan = build_plan(m, parts, fp32, two_ld, two_need, two_agg, &s);
      if (s != SK_OK) return s;
      if (plan) {
        if (m->plans.size() >= 4) m->plans.erase(m->plans.begin());
        m->plans.push_back(plan);
      }
    }
  }
  if (!plan) return SK_OK;
  const int NT = fp32 ? kResNT32 : kResNT64;
  SK_TRY(R.slots.alloc((size_t)kResCopies * kResCopyWords));
  const size_t nx = std::max(1, plan->n_exp);
  SK_TRY(R.zx.alloc(2 * nx * (fp32 ? kVertStride<float> : kVertStride<double>)));
  if (fp32) SK_TRY(R.xx.alloc(nx * kVertStride<double>));
  SK_TRY(R.stream.alloc(std::max<size_t>(16, (size_t)plan->G * plan->KS * 9 * NT * (fp32 ? 4 : 8))));
  SK_TRY(R.abort_flag.alloc(1));
  SK_HIP_CHECK(hipMemset(R.slots.p, 0, R.slots.n * 8));
  SK_HIP_CHECK(hipMemset(R.zx.p, 0, R.zx.n * 8));
  if (fp32) SK_HIP_CHECK(hipMemset(R.xx.p, 0, R.xx.n * 8));
  SK_HIP_CHECK(hipMemset(R.abort_flag.p, 0, sizeof(int)));
  SK_HIP_CHECK(hipDeviceSynchronize());
  if (!R.host) SK_HIP_CHECK(hipHostMalloc((void**)&R.host, sizeof(ResidentResult), hipHostMallocCoherent));
  *R.host = ResidentResult{};
  R.epoch = 0;
  R.plan = plan;
  R.two = std::move(two);
  return SK_OK;
}

void resident_prepare(ResidentState& R, sk_mesh* m, bool fp32, const CoarseSpace* coarse) {
  if (R.tried) return;
  R.tried = true;
  R.plan.reset();
  R.two.reset();
  if (no_throw([&] { return prepare(R, m, fp32, coarse); }) == SK_OK) return;
  // no memory for it: the launches need none of this
  (void)hipGetLastError();
  R.plan.reset();
  R.two.reset();
  for (DevBuf<uint64_t>* b : {&R.slots, &R.zx, &R.xx}) b->release();
  R.stream.release();
  R.abort_flag.release();
}

template <typename T, int NT, int KR, bool kMixed, bool kTwo>
static int launch(ResidentState& R, sk_mesh* m, const ResidentSolve& s, hipStream_t st) {
  const ResidentPlan& p = *R.plan;
  ResidentArgs<T> a{p.G, p.K, p.KL, p.KS, p.row0.p, m->bptr.p, p.lcol.p, p.tflag.p, p.trow.p, m->sell_pos.p, (const T*)s.vals,
                    (const T*)s.binv, s.fixed, s.g, s.dx, p.halo_ptr.p, p.hvert.p, p.halo.p, p.exp0.p, p.exslot.p, R.slots.p, R.zx.p,
                    (uint32_t)(R.zx.n / 2),
                    R.xx.p, reinterpret_cast<T*>(R.stream.p), R.abort_flag.p, R.host, R.epoch, p.max_rows,
                    p.max_local, p.max_halo, s.rtol * s.rtol, s.inner_rtol * s.inner_rtol, s.max_iter, s.max_refine};
  if (kTwo) {
    const CoarseSpace& C = *s.coarse;
    const ResidentTwo& w = *R.two;
    a.ld = C.ld;
    a.n_agg = C.n_agg;
    a.max_need = w.max_need;
    a.shift = C.shift;
    a.piece0 = w.piece0.p;
    a.pagg = w.pagg.p;
    a.apiece = w.apiece.p;
    a.own0 = w.own0.p;
    a.need0 = w.need0.p;
    a.need = w.need.p;
    a.lrow = w.lrow.p;
    a.lhalo = w.lhalo.p;
    a.agg_ptr = C.agg_ptr.p;
    a.agg_col = C.agg_col.p;
    a.tm = C.tm.p;
    a.dsc = C.dsc.p;
    a.dv = C.dv64.p;
    a.einv = C.einv.p;
    a.cwords = w.cwords.p;
    a.rwords = w.cwords.p + w.cwords.n / 2;
    a.uwords = w.uwords.p;
  }
  resident_pcg_kernel<T, NT, KR, kMixed, kTwo><<<p.G, NT, p.lds, st>>>(a);
  SK_HIP_CHECK(hipGetLastError());
  return SK_OK;
}

// Every word tagged with `epoch`, so that none belongs to a later exchange.
static int clear_all_words(ResidentState& R, uint32_t epoch, hipStream_t st) {
  for (DevBuf<uint64_t>* b : {&R.slots, &R.zx, &R.xx}) SK_TRY(fill_words(*b, (uint64_t)epoch << 32, st));
  if (R.two)
    for (DevBuf<uint64_t>* b : {&R.two->cwords, &R.two->uwords}) SK_TRY(fill_words(*b, (uint64_t)epoch << 48, st));
  return SK_OK;
}

int resident_set_epoch(ResidentState& R, uint32_t epoch) {
  SK_TRY(clear_all_words(R, epoch, nullptr));
  SK_HIP_CHECK(hipDeviceSynchronize());
  R.epoch = epoch;
  *R.host = ResidentResult{0, 0, 0, 0, epoch};
  return SK_OK;
}

int resident_launch(ResidentState& R, sk_mesh* m, const ResidentSolve& s, hipStream_t st) {
  if (R.host->epoch > R.epoch) R.epoch = R.host->epoch;
  if (R.epoch > kResMaxEpoch) {  // tags start over long before they wrap
    SK_TRY(clear_all_words(R, 0, st));
    R.epoch = 0;
  }
  *R.host = ResidentResult{0, 0, 0, 0, R.epoch};
  auto run = [&](auto two) {
    constexpr bool kTwo = decltype(two)::value;
    constexpr int kLong32 = kTwo ? kResTwoKR32 : kResKR32, kLong64 = kTwo ? kResTwoKR64 : kResKR64;
    if (s.fp32)
      return R.plan->KR == kResShort32 ? launch<float, kResNT32, kResShort32, true, kTwo>(R, m, s, st)
                                       : launch<float, kResNT32, kLong32, true, kTwo>(R, m, s, st);
    return R.plan->KR == kResShort64 ? launch<double, kResNT64, kResShort64, false, kTwo>(R, m, s, st)
                                     : launch<double, kResNT64, kLong64, false, kTwo>(R, m, s, st);
  };
  return s.coarse ? run(std::true_type{}) : run(std::false_type{});
}


}  // namespace sk

using namespace sk;

extern "C" {

// Recursive coordinate bisection: vertices [lo, hi) of idx into parts [g0, g1).
static void bisect(const double* X, const std::vector<float>& w, std::vector<int32_t>& idx, int64_t lo, int64_t hi,
                   int g0, int g1, int32_t* ptr) {
  if (g1 - g0 == 1) {
    ptr[g0] = (int32_t)lo;
    return;
  }
  double mn[3], mx[3];
  for (int c = 0; c < 3; ++c) mn[c] = 1e300, mx[c] = -1e300;
  double total = 0.0;
  for (int64_t i = lo; i < hi; ++i) {
    const double* x = X + 3 * (int64_t)idx[i];
    total += w[idx[i]];
    for (int c = 0; c < 3; ++c) {
      mn[c] = std::min(mn[c], x[c]);
      mx[c] = std::max(mx[c], x[c]);
    }
  }
  int ax = 0;
  for (int c = 1; c < 3; ++c)
    if (mx[c] - mn[c] > mx[ax] - mn[ax]) ax = c;
  const int a1 = (ax + 1) % 3, a2 = (ax + 2) % 3;
  auto less = [&](int32_t p, int32_t q) {
    const double *x = X + 3 * (int64_t)p, *y = X + 3 * (int64_t)q;
    if (x[ax] != y[ax]) return x[ax] < y[ax];
    if (x[a1] != y[a1]) return x[a1] < y[a1];
    if (x[a2] != y[a2]) return x[a2] < y[a2];
    return p < q;
  };
  const int gm = g0 + (g1 - g0) / 2;
  // weighted selection of the cut; each side keeps at least one vertex per part
  const double want = total * (gm - g0) / (g1 - g0);
  int64_t a = lo + (gm - g0), b = hi - (g1 - gm);
  int64_t l = lo, h = hi;
  double acc = 0.0;
  while (h - l > 1) {
    const int64_t mid = (l + h) / 2;
    std::nth_element(idx.begin() + l, idx.begin() + mid, idx.begin() + h, less);
    double s = 0.0;
    for (int64_t i = l; i < mid; ++i) s += w[idx[i]];
    if (acc + s >= want) h = mid;
    else acc += s, l = mid;
  }
  const int64_t cut = std::min(std::max(h, a), b);
  std::nth_element(idx.begin() + lo, idx.begin() + cut, idx.begin() + hi, less);
  bisect(X, w, idx, lo, cut, g0, gm, ptr);
  bisect(X, w, idx, cut, hi, gm, g1, ptr);
}

static int part_order(const double* X, const int32_t* T, int64_t nv, int64_t nt, int precision, int32_t* order,
                      int* n_parts, int32_t* part_ptr) {
  SK_REQUIRE(X && T && order && n_parts && part_ptr, "sk_part_order: null argument");
  SK_REQUIRE(precision == SK_PREC_FP64 || precision == SK_PREC_MIXED, "sk_part_order: bad precision");
  SK_REQUIRE(nv > 0 && nt > 0, "sk_part_order: empty mesh");
  for (int64_t k = 0; k < 4 * nt; ++k) SK_REQUIRE(T[k] >= 0 && T[k] < nv, "sk_part_order: tet index out of range");
  *n_parts = 0;
  std::vector<int32_t> deg;
  vertex_degrees(T, nv, nt, deg);
  int64_t nblk = 0;
  for (int32_t d : deg) nblk += d;
  const int G = resident_parts(nv, nblk, precision == SK_PREC_MIXED);
  if (G == 0) {
    degree_order(deg, order);
    return SK_OK;
  }
  std::vector<float> w(nv);
  const float mean = (float)nblk / (float)nv;
  for (int64_t v = 0; v < nv; ++v) w[v] = (float)deg[v] + mean;
  std::vector<int32_t> idx(nv);
  std::iota(idx.begin(), idx.end(), 0);
  bisect(X, w, idx, 0, nv, 0, G, part_ptr);
  part_ptr[G] = (int32_t)nv;
  const bool fp32 = precision == SK_PREC_MIXED;
  const int NT = fp32 ? kResNT32 : kResNT64;
  for (int g = 0; g < G; ++g) {  // a part that build_plan will refuse: the launches' order then
    int64_t nb = 0;
    for (int32_t i = part_ptr[g]; i < part_ptr[g + 1]; ++i) nb += deg[idx[i]];
    const int K = (int)((nb + NT - 1) / NT);
    if (part_ptr[g + 1] - part_ptr[g] > NT || K > resident_kr(fp32, false, K) + 2 * kResMaxTier) {
      degree_order(deg, order);
      return SK_OK;
    }
  }
  for (int g = 0; g < G; ++g)
    std::sort(idx.begin() + part_ptr[g], idx.begin() + part_ptr[g + 1], [&](int32_t p, int32_t q) {
      return deg[p] != deg[q] ? deg[p] > deg[q] : p < q;
    });
  std::copy(idx.begin(), idx.end(), order);
  *n_parts = G;
  return SK_OK;
}

int sk_part_order(const double* X, const int32_t* T, int64_t nv, int64_t nt, int precision, int32_t* order,
                  int* n_parts, int32_t* part_ptr) {
  return no_throw([&] { return part_order(X, T, nv, nt, precision, order, n_parts, part_ptr); });
}

}  // extern "C"
