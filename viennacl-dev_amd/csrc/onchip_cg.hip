// onchip_cg.hip -- all CG iterations of a DIA system in one launch, the vectors held on chip.
//
// A kernel per step reads and writes every vector through the memory side of the chip in every
// iteration (seven passes in the update, two in the product) and pays a kernel boundary per step.
// The register files (512 KB a CU, 128 MB in all) hold the whole solve instead: a workgroup of 1024
// lanes per CU owns a contiguous range of rows (the owners of cg_sums.hpp) with x, r and A p in
// registers and p in LDS, and runs every iteration on them.  Between CUs travel
//   * the inner products: a workgroup publishes its three sums in one 64-byte line, each double as
//     two 8-byte words that carry the iteration number, and every workgroup reads all lines until
//     the numbers are right.  Data and flag are one word, so no order between stores is needed, and
//     the lines alternate between two sets, so that none is overwritten before everyone has read it;
//   * the rows of p that the stencil reaches outside a workgroup's own range.  Two forms:
//     ghost: the workgroup keeps r and p of those rows as well (r in registers, p in LDS) and
//       updates them itself from its neighbours' A p, which they stored before they published their
//       sums: one exchange per iteration.  Up to two rows a lane (n <= 2^19);
//     halo:  p of the own rows is stored after the update, neighbours are told by a flag, and the
//       reached rows are read from memory: a second, neighbours-only wait per iteration (about 1 us),
//       for as many workgroups on each side as own reached rows (oc_reach), but no ghost state.  With more than two rows a lane the ghosts' registers spill (100^3: 24 us
//       an iteration as ghost, 11 as halo; Jacobi on 97 x 83 x 71: 30 and 20).
// From 128 workgroups on, the first of each XCD adds up its XCD's sums and all others read those eight:
// 256 workgroups that poll 256 lines hold each other up (exchange at 64^3 3.5 us, 2.4 in two steps;
// CG on 128^3 9.5 -> 7.5 ms; with 128 workgroups both take 2.3 us, and 64 take 1.7 in one step).
// Data that another workgroup reads is stored and loaded at agent scope, which the XCDs' L2s keep
// coherent, and a wave waits for its stores before its workgroup publishes.  Workgroups of one XCD own
// neighbouring rows, so that most of that stays in its L2: storing p of 128^3 takes 2.1 us an
// iteration, and 6.3 with neighbours on different XCDs.
// The operator's values stay in registers (small systems), or as one bit per entry where every
// diagonal has one value (the constant-coefficient Laplacians), as packed 4-bit codes into value
// tables in LDS, or as stored: as many diagonals as fit in LDS, the others read again in every iteration
// (Jacobi-CG on 97 x 83 x 71, whose 32 MB of values come to just the L2s' size: 20 us an iteration with
// all of them read, 12 with six of seven diagonals in LDS, 9.5 since the sums meet per XCD first).
//
// What bounds it: 256^2 runs 3.9 us an iteration, of which the exchange of the sums takes 1.7 and the
// workgroup's own sums 0.6 (7.4 us with one launch per iteration); 128^3 runs 14 us (47 us with three):
// 6 for the product, whose far rows come from L2, 2 for storing p, 3 waiting for the workgroups at the
// XCDs' edges, whose far rows come from further away.
//
// The mixed solver runs its FP32 inner iterations between two FP64 corrections the same way, up to 16
// rows a lane: 160^3 variable coefficients 29 us an iteration (51 us with three launches), of which the
// FP32 values, 115 MB read from the Infinity Cache, are the larger part (19 us at 6 TB/s).
//
// Every sum is formed in the order of the kernel-per-step modes (cg_sums.hpp), so the results are
// theirs bit for bit.
//
// All workgroups must run at once.  The grids of the on-chip solves of a device together are at most one
// workgroup per CU (solves take turns, OcTurn); every wait is bounded by the wall clock, and a workgroup
// that gives up raises a flag that ends all the others' waits.
#include <algorithm>
#include <condition_variable>
#include <cstdlib>
#include <mutex>

#include "cg_sums.hpp"
#include "internal.hpp"
#include "onchip_cg.hpp"

namespace vclhip {

// Hooks of the tests (onchip_cg_wait_limit, onchip_cg_off, onchip_cg_last and onchip_cg_plan, not part of
// the API), per thread: the wait limit in microseconds (below zero: the usual ones), whether solves leave
// this mode out, and whether the last CG solve ran here (1), gave up (2) or neither (0).
static thread_local double t_wait_us = -1;
static thread_local bool t_off = false;
static thread_local int t_on_chip = 0;

namespace {

constexpr int kOcThreads = 1024;
constexpr int kOcBlocks = kOcThreads / kBlock;  // 256-lane groups of a workgroup, one chunk at a time each
constexpr uint32_t kOcDiags = 7;                // diagonals at most
constexpr uint32_t kOcChunks = 8;               // chunks of a workgroup at most
constexpr int kOcSums = 3;
constexpr uint32_t kOcLine = 8;                 // 8-byte words of a workgroup's line
constexpr uint32_t kXcds = 8;
constexpr uint32_t kOcLines = kOwners + kXcds;  // lines of a set: the workgroups' and the XCDs'
constexpr size_t kOcLds = 160 * 1024 - 2048;    // dynamic LDS at most (the static part stays below 2 KB)
constexpr uint64_t kOcClock = 100;              // wall clock ticks per microsecond
constexpr uint32_t kOcSlice = 4096;             // iterations of a launch at most: it then lets other work in
static_assert(kOcSlice % 2 == 0, "a launch ends with A p in ex1");

// Where the operator's values are: in registers; as 4-bit codes in registers, the tables in LDS; as one
// bit per entry in registers, one value per diagonal; or as stored, read in every iteration, but for
// the first half of the diagonals or all but the last, which LDS holds.
enum OcVal { kValRegs = 0, kValCodes = 1, kValStream = 2, kValOne = 3, kValHalf = 4, kValMost = 5 };
constexpr bool val_stored(OcVal v) { return v == kValStream || v == kValHalf || v == kValMost; }
constexpr uint32_t val_held(OcVal v, uint32_t nd) { return v == kValMost ? nd - 1 : (v == kValHalf ? nd / 2 : 0); }

// Relaxed accesses at agent scope: single-location coherence between the XCDs.
template <typename U>
__device__ __forceinline__ U ld_agent(const U* p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename U>
__device__ __forceinline__ void st_agent(U* p, U v)
{
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A device array as a buffer resource: 32-bit byte offsets instead of 64-bit addresses, loads past
// its end give 0 and stores past it do nothing.  Agent: at agent scope, as above.
template <typename T>
struct OcBuf {
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ __forceinline__ OcBuf(const T* p, size_t count)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(p), 0, static_cast<int>(count * sizeof(T)), 0x00027000))
  {
  }
  template <bool Agent = false>
  __device__ __forceinline__ T load(uint32_t i) const
  {
    constexpr int aux = Agent ? 16 : 0;
    if constexpr (sizeof(T) == 8)
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(rsrc, i * sizeof(T), 0, aux));
    else if constexpr (sizeof(T) == 4)
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(rsrc, i * sizeof(T), 0, aux));
    else
      return __builtin_amdgcn_raw_buffer_load_b8(rsrc, i, 0, aux);
  }
  template <bool Agent = false>
  __device__ __forceinline__ void store(uint32_t i, T v) const
  {
    constexpr int aux = Agent ? 16 : 0;
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    if constexpr (sizeof(T) == 8)
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), rsrc, i * sizeof(T), 0, aux);
    else
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), rsrc, i * sizeof(T), 0, aux);
  }
};
constexpr uint32_t kOcNowhere = 0x1ffffff0u;  // an index past the end of every buffer

// The rows that a workgroup of `rows` rows reaches along its diagonals, as disjoint segments in LDS
// one after the other: its row l (counted from its first) is entry own + l, and that row's neighbour
// on diagonal i entry delta[i] + l.  Rows outside the system have entries too (they stay zero), so
// that no access needs a check.  Diagonals of `far` are left out.  Offsets ascending.
struct OcSegments {
  uint32_t count, ext, own;
  int32_t start[kOcDiags + 1];  // first row of the segment, from the workgroup's first row
  uint32_t base[kOcDiags + 1];  // its entry
  uint32_t delta[kOcDiags];
};

__host__ __device__ inline void oc_segments(uint32_t rows, uint32_t nd, const int32_t* off, uint32_t far, OcSegments& g)
{
  g.count = 0;
  g.ext = 0;
  g.own = 0;
  int32_t end = 0;
  bool own_done = false;
  for (uint32_t i = 0; i <= nd; ++i) {
    for (int pass = 0; pass < 2; ++pass) {
      // pass 0: the own rows, in front of the first diagonal at or above 0; pass 1: diagonal i
      if (pass == 0 ? own_done || (i < nd && off[i] < 0) : i == nd || (far >> i & 1u) != 0) continue;
      const int32_t s = pass == 0 ? 0 : off[i], e = s + static_cast<int32_t>(rows);
      own_done = own_done || pass == 0;
      if (g.count == 0 || s > end) {
        g.start[g.count] = s;
        g.base[g.count] = g.ext;
        ++g.count;
        end = s;
      }
      g.ext += static_cast<uint32_t>(e - end);
      end = e;
      const uint32_t at = g.base[g.count - 1] + static_cast<uint32_t>(s - g.start[g.count - 1]);
      if (pass == 0)
        g.own = at;
      else
        g.delta[i] = at;
    }
  }
}

// Workgroup w's owners, product chunks and tiles.
struct OcPart {
  uint32_t o0, o1, p0, p1, t0, t1;
};

__host__ __device__ inline OcPart oc_part(uint32_t n, uint32_t gp, uint32_t m, uint32_t w)
{
  OcPart q;
  const uint32_t tiles = cg_tiles(n), owners = gp < kOwners ? gp : kOwners;
  q.o0 = w * m;
  q.o1 = q.o0 + m < owners ? q.o0 + m : owners;
  uint32_t unused;
  owner_range(gp, q.o0, q.p0, unused);
  owner_range(gp, q.o1 - 1, unused, q.p1);
  part_range(tiles, q.p0, gp, q.t0, unused);
  part_range(tiles, q.p1, gp, q.t1, unused);
  return q;
}

// For how many workgroups on each side one has to wait in the halo form: the farthest owner of a row
// that its own rows reach along the diagonals (offsets ascending; the rows past the system's end count
// as well, as they are loaded).  Walked over the workgroups themselves (at most 256): where the product
// chunks are no multiple of the owners these hold unequal numbers of rows, and a bound from one of
// their sizes is too short for others.
inline uint32_t oc_reach(uint32_t n, uint32_t gp, uint32_t m, uint32_t nwg, uint32_t nd, const int32_t* off)
{
  uint32_t first[kOwners + 1] = {0};
  for (uint32_t w = 0; w < nwg; ++w) {
    const OcPart q = oc_part(n, gp, m, w);
    first[w] = q.t0 * kBlock;
    first[w + 1] = q.t1 * kBlock;
  }
  auto owner = [&](int64_t row) {
    const int64_t r = std::min<int64_t>(std::max<int64_t>(row, 0), static_cast<int64_t>(n) - 1);
    return static_cast<uint32_t>(std::upper_bound(first, first + nwg, static_cast<uint32_t>(r)) - first) - 1;
  };
  uint32_t reach = 0;
  for (uint32_t w = 0; w < nwg; ++w) {
    const uint32_t lo = owner(static_cast<int64_t>(first[w]) + off[0]);
    const uint32_t hi = owner(static_cast<int64_t>(first[w + 1]) - 1 + off[nd - 1]);
    if (lo < w) reach = std::max(reach, w - lo);
    if (hi > w) reach = std::max(reach, hi - w);
  }
  return reach;
}

template <typename T>
struct OcArgs {
  uint32_t n, nd, gp, m, nwg;
  uint32_t mixed;   // the mixed solver's inner iteration: its end test
  uint32_t far;     // halo form: mask of the diagonals read from memory (the first and the last)
  uint32_t ext;     // LDS entries for p
  uint32_t per_xcd; // workgroups that add up their sums before all others see them; 0: none do
  uint32_t reach;   // halo form: workgroups on each side that own reached rows
  int32_t off[kOcDiags];
  const T* val;
  const uint8_t* code;
  const T* table;
  T* x;
  T* r;
  T* p;
  const T* d;
  T* ex0;  // ghost form: A p of even iterations; halo form: p
  T* ex1;  // ghost form: A p of odd iterations; both: A p at the start and the end of a launch
  KState* st;
  unsigned long long* lines;  // two sets of one line per workgroup
  uint32_t* flags;            // halo form: one 64-byte line per workgroup
  uint32_t* abort;
  uint64_t wait_first;        // wall clock ticks that a wait of the launch's first iteration may take
  uint64_t wait;              // and one of a later iteration, when all workgroups are known to run
};

// One poll more after a failed one?  Looks at the abort flag and the clock now and then (always
// when the limit is zero, which is how a test makes a wait give up).
struct OcWait {
  uint64_t t0 = 0;  // read at the first look
  uint32_t polls = 0;
  __device__ __forceinline__ bool again(uint32_t* abort, uint64_t limit)
  {
    if ((++polls & 63u) != 0 && limit != 0) return true;
    const uint64_t now = wall_clock64();
    if (t0 == 0) t0 = now;
    if (ld_agent(abort) == 0 && now - t0 < limit) return true;
    st_agent(abort, 1u);
    return false;
  }
};

// A uniform value, formed again from here on (comparisons with it are not hoisted out of a loop, where
// each takes two scalar registers and is spilled).
__device__ __forceinline__ uint32_t again(uint32_t v)
{
  v = __builtin_amdgcn_readfirstlane(v);
  asm volatile("" : "+s"(v));
  return v;
}
// Tells the compiler that a value is the same in all lanes.
__device__ __forceinline__ bool uniform(bool b) { return __builtin_amdgcn_readfirstlane(b ? 1u : 0u) != 0; }
__device__ __forceinline__ double uniform(double v)
{
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const uint32_t l = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(u));
  const uint32_t h = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(u >> 32));
  return __builtin_bit_cast(double, static_cast<unsigned long long>(h) << 32 | l);
}

// v, or +0 where mask is zero (it is that or all bits): without a branch, which the compiler makes of a
// selected product.
template <typename T>
__device__ __forceinline__ T masked(T v, uint32_t mask)
{
  if constexpr (sizeof(T) == 8) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const uint32_t l = static_cast<uint32_t>(u) & mask, h = static_cast<uint32_t>(u >> 32) & mask;
    return __builtin_bit_cast(T, static_cast<unsigned long long>(h) << 32 | l);
  } else {
    return __builtin_bit_cast(T, __builtin_bit_cast(uint32_t, v) & mask);
  }
}

// The wavefront sums of three values (wave_sum's, bit for bit) in the lanes of rows 0, 1 and 2: each
// step folds what is left of two values into one register, so that the last four steps run once
// (23 instructions for 66).
__device__ __forceinline__ double wave_sums3(double v0, double v1, double v2)
{
  swap_rows<32>(v0, v2);
  v0 += v2;  // half 0: the first value's, half 1: the third's
  double u = v1;
  swap_rows<32>(v1, u);
  v1 += u;
  swap_rows<16>(v0, v1);
  return row_sum(v0 + v1);
}

// Slot of ND holds a diagonal of the operator, in offset order with the last one in the last slot, or
// nothing (a zero entry): the slots are a compile-time number, so that a row's loads and sums have no
// branches.
template <uint32_t ND>
__host__ __device__ inline uint32_t slot_diagonal(uint32_t slot, uint32_t nd)
{
  return slot + 1 < nd ? slot : (slot == ND - 1 ? nd - 1 : ND);
}

// ND: slots for diagonals.  W: the width of the vector kernels' packs.  CPV: chunks of a 256-lane group at most, TPC:
// tiles of a chunk at most (CPV * TPC rows a lane).  Ghosts: ghost rows a lane at most, 0 for the
// halo form.
template <typename T, uint32_t ND, bool Jac, int W, int CPV, int TPC, OcVal Val, int Ghosts>
__global__ __launch_bounds__(kOcThreads) void onchip_cg_kernel(OcArgs<T> a)
{
  constexpr int S = CPV * TPC;
  extern __shared__ __align__(16) unsigned char oc_lds[];
  __shared__ double red[kOcSums][kOcChunks][kWavesPerBlock];
  __shared__ double tot[kOcSums][kWavesPerBlock];
  __shared__ OcSegments seg;
  __shared__ uint32_t ok;

  KState* const st = a.st;
  const uint32_t iter0 = st->iter;
  // workgroups of one XCD take neighbouring rows: what they exchange then stays in its L2
  const uint32_t w = gridDim.x % 8 == 0 ? xcd_logical_block() : blockIdx.x;
  const uint32_t tid = threadIdx.x, n = a.n, nd = a.nd;
  constexpr uint32_t kAbsent = ND;
  const uint32_t vb = __builtin_amdgcn_readfirstlane(tid / kBlock), t = tid % kBlock;
  const uint32_t wave = __builtin_amdgcn_readfirstlane((tid / kWave) % kWavesPerBlock), lane = tid % kWave;
  const OcPart q = oc_part(n, a.gp, a.m, w);
  const uint32_t lo = q.t0 * kBlock, rows = (q.t1 - q.t0) * kBlock;  // rows past the system's end are held as zeros
  const uint32_t mv = a.gp <= kOwners ? 1u : cg_vec_per_owner(n);
  const uint32_t v0 = a.gp <= kOwners ? q.o0 : q.o0 * mv;
  const uint32_t nvec = (q.o1 - q.o0) * mv;

  T* const stab = reinterpret_cast<T*>(oc_lds);
  T* const lp = stab + (Val == kValCodes ? kOcDiags * kDiaCodes : 0u);
  T* const lsq = lp + a.ext;
  T* const lv = lsq + rows;  // [slot][row] of the values held
  constexpr uint32_t kHeld = val_held(Val, ND);

  // Nothing to do, or others have given up before this workgroup started: one lane looks and all waves
  // go by what it saw.  The abort word may be raised at any time, and waves that looked for themselves
  // could part, some leaving and the rest going on without the sums and the waits of those.
  if (tid == 0) {
    ok = (st->flags & (kFlagDone | kFlagPause)) == 0 && ld_agent(a.abort) == 0 ? 1u : 0u;
    oc_segments(rows, nd, a.off, a.far, seg);
  }
  if constexpr (Val == kValCodes)
    for (uint32_t i = tid; i < ND * kDiaCodes; i += kOcThreads) {  // by slot
      const uint32_t d = slot_diagonal<ND>(i / kDiaCodes, nd);
      stab[i] = d != kAbsent ? a.table[d * kDiaCodes + i % kDiaCodes] : T(0);
    }
  for (uint32_t i = tid; i < a.ext; i += kOcThreads) lp[i] = T(0);
  __syncthreads();
  if (!uniform(ok != 0)) return;
  const uint32_t own = __builtin_amdgcn_readfirstlane(seg.own);
  const uint32_t all_ghosts = __builtin_amdgcn_readfirstlane(seg.ext) - rows;
  uint32_t delta[ND], dia[ND];  // by slot
#pragma unroll
  for (uint32_t i = 0; i < ND; ++i) {
    dia[i] = slot_diagonal<ND>(i, nd);
    delta[i] = dia[i] != kAbsent && !(a.far >> dia[i] & 1u) ? __builtin_amdgcn_readfirstlane(seg.delta[dia[i]]) : own;
  }

  const OcBuf<T> bval(a.val, static_cast<size_t>(nd) * n), bx(a.x, n), br(a.r, n), bp(a.p, n), bd(Jac ? a.d : a.r, n);
  const OcBuf<T> bex0(a.ex0, n), bex1(a.ex1, n);
  const OcBuf<uint8_t> bcode(a.code, a.code ? static_cast<size_t>(nd) * n : 0);

  // the lane's rows: tile j of chunk c is the workgroup's row first[c] + j * kBlock, for j < tiles_of[c]
  uint32_t first[CPV], tiles_of[CPV];
#pragma unroll
  for (int c = 0; c < CPV; ++c) {
    const uint32_t pc = q.p0 + vb + static_cast<uint32_t>(c) * kOcBlocks;
    uint32_t b = q.t0, e = q.t0;
    if (pc < q.p1) part_range(cg_tiles(n), pc, a.gp, b, e);
    first[c] = (b - q.t0) * kBlock + t;
    tiles_of[c] = __builtin_amdgcn_readfirstlane(e - b);
  }
  // the vector chunks, as rows of the workgroup
  uint32_t vc0[CPV], vc1[CPV];
#pragma unroll
  for (int c = 0; c < CPV; ++c) {
    const uint32_t vc = vb + static_cast<uint32_t>(c) * kOcBlocks;
    uint32_t b = lo, e = lo;
    if (vc < nvec) cg_vec_rows(n, v0 + vc, b, e);
    vc0[c] = __builtin_amdgcn_readfirstlane(b - lo);
    vc1[c] = __builtin_amdgcn_readfirstlane(e - lo);
  }

  uint32_t all_most = 0;  // tiles of the longest chunk
#pragma unroll
  for (int c = 0; c < CPV; ++c) all_most = tiles_of[c] > all_most ? tiles_of[c] : all_most;

  // Rows a lane does not have (tiles past tiles_of) go through the loads and the arithmetic as well, with
  // zeros or whatever LDS holds: without branches per row the loads of all rows are in flight together.
  // They are kept out of the sums and the stores.
  T x[S], r[S], ap[S];
  T v[Val == kValRegs ? S : 1][ND];
  T one[ND];
  constexpr int NC = Val == kValCodes ? S : (S + 3) / 4;
  uint32_t codes[NC];
#pragma unroll
  for (int s = 0; s < NC; ++s) codes[s] = 0;
#pragma unroll
  for (uint32_t i = 0; i < ND; ++i) {
    one[i] = Val == kValOne && dia[i] != kAbsent ? a.table[dia[i] * kDiaCodes + 1] : T(0);
    if (!(one[i] > 0 || one[i] < 0)) one[i] = T(0);  // zero and NaN are not there
  }
#pragma unroll
  for (int c = 0; c < CPV; ++c)
#pragma unroll
    for (int j = 0; j < TPC; ++j) {
      const int s = c * TPC + j;
      x[s] = r[s] = ap[s] = T(0);
      if constexpr (Val == kValRegs)
#pragma unroll
        for (uint32_t i = 0; i < ND; ++i) v[s][i] = T(0);
      if (static_cast<uint32_t>(j) < tiles_of[c]) {
        const uint32_t l = first[c] + j * kBlock, row = lo + l;
        x[s] = bx.load(row);
        r[s] = br.load(row);
        ap[s] = bex1.load(row);
        lp[own + l] = bp.load(row);
#pragma unroll
        for (uint32_t i = 0; i < kHeld; ++i) lv[i * rows + l] = T(0);
#pragma unroll
        for (uint32_t i = 0; i < ND; ++i)
          if (dia[i] != kAbsent && row < n) {
            const uint32_t at = dia[i] * n + row;
            if constexpr (kHeld > 0)
              if (i < kHeld) lv[i * rows + l] = bval.load(at);
            if constexpr (Val == kValRegs) v[s][i] = a.code ? a.table[dia[i] * kDiaCodes + bcode.load(at)] : bval.load(at);
            if constexpr (Val == kValCodes) codes[s] |= static_cast<uint32_t>(bcode.load(at)) << (4 * i);
            if constexpr (Val == kValOne)
              codes[s / 4] |= (one[i] != T(0) ? static_cast<uint32_t>(bcode.load(at)) : 0u) << (8 * (s % 4) + i);
          }
      }
    }

  // the lane's ghost rows: LDS entries tid, tid + 1024, ... of the entries beside the own rows
  constexpr int NG = Ghosts > 0 ? Ghosts : 1;
  uint32_t grow[NG];
  T gr[NG];
  auto ghost_at = [&](uint32_t g) { return g < own ? g : g + rows; };
  auto ghost_row = [&](uint32_t e) {  // kOcNowhere outside the system
    uint32_t k = 0;
    while (k + 1 < seg.count && e >= seg.base[k + 1]) ++k;
    const uint32_t row = lo + static_cast<uint32_t>(seg.start[k]) + (e - seg.base[k]);
    return row < n ? row : kOcNowhere;
  };
  if constexpr (Ghosts > 0) {
#pragma unroll
    for (int k = 0; k < NG; ++k) {
      const uint32_t g = tid + static_cast<uint32_t>(k) * kOcThreads;
      grow[k] = kOcNowhere;
      gr[k] = T(0);
      if (g < all_ghosts) {
        const uint32_t e = ghost_at(g);
        grow[k] = ghost_row(e);
        gr[k] = br.load(grow[k]);
        lp[e] = bp.load(grow[k]);
      }
    }
  }

  // wave 0 reduces the chunk partials: lane 8 q + ch holds chunk ch of sum q, lane 8 q + o owner o
  const uint32_t rq = lane >> 3, rc = lane & 7u;
  uint32_t own_b = 0, own_e = 0;
  if (rc < q.o1 - q.o0) {
    if (rq == 0) {
      own_b = rc * mv;
      own_e = own_b + mv;
    } else {
      owner_range(a.gp, q.o0 + rc, own_b, own_e);
      own_b -= q.p0;
      own_e -= q.p0;
    }
  }

  const double rr_stop = static_cast<double>(st->inner_tol) * st->rr_ref;
  const double nrs = st->nrs, tol2 = st->tol * st->tol, atol2 = st->abs_tol * st->abs_tol;
  const uint32_t max_iters = st->max_iters;
  double alpha = st->alpha, beta = st->beta;
  const __amdgpu_buffer_rsrc_t line_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(a.lines, 0, 2 * kOcLines * kOcLine * 8, 0x00027000);

  bool more = false;
  for (uint32_t k = 0;; ++k) {
    // nothing derived from a lane's rows is kept across iterations: it is cheaper to form again than
    // to spill
#pragma unroll
    for (int c = 0; c < CPV; ++c) keep_here(first[c]);
#pragma unroll
    for (int s = 0; s < NC; ++s)
      if constexpr (Val == kValCodes || Val == kValOne) keep_here(codes[s]);
#pragma unroll
    for (int s = 0; s < S; ++s) {
      if constexpr (Val == kValRegs)
#pragma unroll
        for (uint32_t i = 0; i < ND; ++i) keep_here(v[s][i]);
    }
    uint32_t gid = tid;  // this lane's first ghost
    keep_here(gid);
    const uint32_t ghosts = again(all_ghosts), most = again(all_most);
    uint32_t cnt[CPV];
#pragma unroll
    for (int c = 0; c < CPV; ++c) cnt[c] = again(tiles_of[c]);
    const uint32_t iter = iter0 + k + 1;  // this iteration's number, the tag of its words
    const uint64_t limit = k == 0 ? a.wait_first : a.wait;
    // ---- update: x, r, p of the own rows (and r, p of the ghosts from the neighbours' A p)
    const T ta = static_cast<T>(alpha), tb = static_cast<T>(beta);
    const OcBuf<T>& ex_in = Ghosts > 0 && !(k & 1u) ? bex1 : bex0;
    const OcBuf<T>& ex_out = Ghosts > 0 && (k & 1u) ? bex1 : bex0;
    T ga[NG], gd[NG];
    if constexpr (Ghosts > 0) {
#pragma unroll
      for (int i = 0; i < NG; ++i) {
        if (static_cast<uint32_t>(i) * kOcThreads < ghosts) {
          ga[i] = ex_in.template load<true>(grow[i]);
          if constexpr (Jac) gd[i] = bd.load(grow[i]);
        }
      }
    }
    T dg[Jac ? S : 1];
    if constexpr (Jac)
#pragma unroll
      for (int c = 0; c < CPV; ++c)
#pragma unroll
        for (int j = 0; j < TPC; ++j)
          dg[c * TPC + j] = bd.load(static_cast<uint32_t>(j) < cnt[c] ? lo + first[c] + j * kBlock : kOcNowhere);
#pragma unroll
    for (int j = 0; j < TPC; ++j)
      if (static_cast<uint32_t>(j) < most) {
        T pv[CPV], sq[CPV];
#pragma unroll
        for (int c = 0; c < CPV; ++c) pv[c] = lp[own + first[c] + j * kBlock];
#pragma unroll
        for (int c = 0; c < CPV; ++c) {
          const int s = c * TPC + j;
          x[s] += ta * pv[c];
          r[s] -= ta * ap[s];
          T z = r[s];
          if constexpr (Jac) z = lo + first[c] + j * kBlock < n ? r[s] / dg[s] : T(0);
          pv[c] = z + tb * pv[c];
          sq[c] = r[s] * z;
        }
#pragma unroll
        for (int c = 0; c < CPV; ++c)
          if (static_cast<uint32_t>(j) < cnt[c]) {
            const uint32_t l = first[c] + j * kBlock;
            lp[own + l] = pv[c];
            lsq[l] = sq[c];
            if constexpr (Ghosts == 0) ex_out.template store<true>(lo + l, pv[c]);
          }
      }
    if constexpr (Ghosts > 0) {
#pragma unroll
      for (int i = 0; i < NG; ++i) {
        const uint32_t g = gid + static_cast<uint32_t>(i) * kOcThreads;
        if (g < ghosts) {
          const uint32_t e = ghost_at(g);
          gr[i] -= ta * ga[i];
          T z = gr[i];
          if constexpr (Jac) z = gr[i] / gd[i];
          lp[e] = z + tb * lp[e];
        }
      }
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // p is where the neighbours read it
    }
    __syncthreads();
    if constexpr (Ghosts == 0) {
      if (tid == 0) st_agent(a.flags + w * 16, iter);
    }

    // the first tiles' values, on their way during the waits
    T vv[val_stored(Val) ? CPV : 1][ND - kHeld];
    auto load_values = [&](int c, int j) {
      const uint32_t row = lo + first[c] + j * kBlock;
      const bool here = static_cast<uint32_t>(j) < cnt[c] && row < n;
#pragma unroll
      for (uint32_t i = kHeld; i < ND; ++i)
        vv[c][i - kHeld] = bval.load(here && dia[i] != kAbsent ? dia[i] * n + row : kOcNowhere);
    };
    if constexpr (val_stored(Val))
#pragma unroll
      for (int c = 0; c < CPV; ++c) load_values(c, 0);

    // ---- partial sums of <r,z> per vector chunk, in the packs' order
    double acc_v[CPV];
#pragma unroll
    for (int c = 0; c < CPV; ++c) {
      acc_v[c] = 0;
      const uint32_t packed_end = vc0[c] + ((vc1[c] - vc0[c]) / W) * W;
      for (uint32_t i = vc0[c] + W * t; i < packed_end; i += W * kBlock)
#pragma unroll
        for (int e = 0; e < W; ++e) acc_v[c] += static_cast<double>(lsq[i + e]);
      if (W > 1)
        for (uint32_t i = packed_end + t; i < vc1[c]; i += kBlock) acc_v[c] += static_cast<double>(lsq[i]);
    }

    // ---- halo form: wait for the neighbours' p, then read what the stencil reaches
    constexpr int kAhead = TPC < 2 ? TPC : 2;  // tiles of a chunk whose reached rows are on their way at a time
    T far0[CPV][kAhead], far1[CPV][kAhead];
    auto load_far = [&](int c, int j) {
      const uint32_t row = lo + first[c] + j * kBlock;
      const uint32_t c0 = row + static_cast<uint32_t>(a.off[0]), c1 = row + static_cast<uint32_t>(a.off[nd - 1]);
      const bool here = static_cast<uint32_t>(j) < cnt[c];
      far0[c][j % kAhead] = ex_in.template load<true>(here && c0 < n ? c0 : kOcNowhere);
      far1[c][j % kAhead] = ex_in.template load<true>(here && c1 < n ? c1 : kOcNowhere);
    };
    if constexpr (Ghosts == 0) {
      if (tid >= kOcThreads - 2 * kWave) {
        const uint32_t i = tid - (kOcThreads - 2 * kWave);
        if (i <= 2 * a.reach && w + i >= a.reach && w + i - a.reach < a.nwg) {
          OcWait wait;
          while (ld_agent(a.flags + (w + i - a.reach) * 16) < iter)
            if (!wait.again(a.abort, limit)) {
              ok = 0;
              break;
            }
        }
      }
      __syncthreads();
      if (!uniform(ok != 0)) return;
#pragma unroll
      for (int j = 0; j < kAhead; ++j)
#pragma unroll
        for (int c = 0; c < CPV; ++c) load_far(c, j);
      for (uint32_t g = gid; g < ghosts; g += kOcThreads) {
        const uint32_t e = ghost_at(g);
        lp[e] = ex_in.template load<true>(ghost_row(e));
      }
      __syncthreads();
    }

    // ---- product: A p of the own rows (dia_kernel's sum), <Ap,Ap> and <p,Ap> per product chunk
    double acc_a[CPV], acc_p[CPV];
#pragma unroll
    for (int c = 0; c < CPV; ++c) acc_a[c] = acc_p[c] = 0;
#pragma unroll
    for (int j = 0; j < TPC; ++j)
      if (static_cast<uint32_t>(j) < most) {
#pragma unroll
        for (int c = 0; c < CPV; ++c) {
          const int s = c * TPC + j;
          const uint32_t l = first[c] + j * kBlock, row = lo + l;
          const bool here = static_cast<uint32_t>(j) < cnt[c];
          T sum = 0;
#pragma unroll
          for (uint32_t i = 0; i < ND; ++i) {
            T xv;
            if constexpr (Ghosts == 0) {
              if (i == 0)
                xv = far0[c][j % kAhead];
              else if (i == ND - 1)
                xv = far1[c][j % kAhead];
              else
                xv = lp[delta[i] + l];
            } else {
              xv = lp[delta[i] + l];
            }
            T val;
            uint32_t there;  // all bits where the entry is there
            if constexpr (Val == kValOne) {
              val = one[i];
              there = static_cast<uint32_t>(static_cast<int32_t>(codes[s / 4] << (31 - (8 * (s % 4) + i))) >> 31);
            } else {
              if constexpr (Val == kValRegs) val = v[s][i];
              if constexpr (Val == kValCodes) val = stab[i * kDiaCodes + (codes[s] >> (4 * i) & 15u)];
              if constexpr (val_stored(Val)) {
                if (i < kHeld)
                  val = lv[i * rows + l];
                else
                  val = vv[c][i - kHeld];
              }
              there = __builtin_islessgreater(val, T(0)) ? ~0u : 0u;  // not zero, not NaN
            }
            sum += masked(xv * val, there);  // an absent entry adds a zero, whatever xv is
          }
          // the next tiles', while this one's sums go on
          if constexpr (val_stored(Val))
            if (j + 1 < TPC) load_values(c, j + 1);
          if constexpr (Ghosts == 0)
            if (j + kAhead < TPC) load_far(c, j + kAhead);
          ap[s] = sum;
          if constexpr (Ghosts > 0) ex_out.template store<true>(here ? row : kOcNowhere, sum);
          if constexpr (Jac)
            acc_a[c] += here && row < n ? static_cast<double>(sum * (sum / dg[s])) : 0.0;
          else
            acc_a[c] += here ? static_cast<double>(sum * sum) : 0.0;
          acc_p[c] += here ? static_cast<double>(lp[own + l] * sum) : 0.0;
        }
      }

    // ---- the workgroup's three sums
#pragma unroll
    for (int c = 0; c < CPV; ++c) {
      const uint32_t at = vb + static_cast<uint32_t>(c) * kOcBlocks;
      const double sum = wave_sums3(acc_v[c], acc_a[c], acc_p[c]);
      if ((lane & 15u) == 0 && lane < 16 * kOcSums) red[lane / 16][at][wave] = sum;
    }
    if constexpr (Ghosts > 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // A p is where the neighbours read it
    __syncthreads();
    const uint32_t set = (iter & 1u) * kOcLines;
    if (tid < kWave) {
      double sum = 0;
#pragma unroll
      for (uint32_t i = 0; i < CPV * kOcBlocks; ++i) {
        const double* const w4 = red[rq < kOcSums ? rq : 0][(own_b + i) & 7u];
        double part = w4[0];
#pragma unroll
        for (int j = 1; j < kWavesPerBlock; ++j) part += w4[j];
        if (own_b + i < own_e) sum += part;
      }
      if (a.m >= 2) sum += dpp_move<kDppXor1>(sum);
      if (a.m >= 4) sum += dpp_move<kDppXor2>(sum);
      if (rc == 0 && rq < kOcSums) {
        const unsigned long long bits = __builtin_bit_cast(unsigned long long, sum);
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        __builtin_amdgcn_raw_buffer_store_b128(u32x4{static_cast<uint32_t>(bits), iter, static_cast<uint32_t>(bits >> 32), iter},
                                               line_rsrc, (set + w) * kOcLine * 8 + 16 * rq, 0, 16);
      }
    }
    // ---- everyone's sums, then the binary tree over them
    auto read_line = [&](uint32_t line, double (&s3)[kOcSums]) {
      OcWait wait;
      uint32_t word[4 * kOcSums];
      for (;;) {
        bool all = true;
#pragma unroll
        for (int i = 0; i < kOcSums; ++i) {
          typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
          const u32x4 b = __builtin_amdgcn_raw_buffer_load_b128(line_rsrc, (set + line) * kOcLine * 8 + 16 * i, 0, 16);
          word[4 * i] = b.x;
          word[4 * i + 1] = b.y;
          word[4 * i + 2] = b.z;
          word[4 * i + 3] = b.w;
        }
        asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < 2 * kOcSums; ++i) all = all && word[2 * i + 1] == iter;
        if (all) break;
        if (!wait.again(a.abort, limit)) {
          ok = 0;
          break;
        }
      }
#pragma unroll
      for (int i = 0; i < kOcSums; ++i)
        s3[i] = __longlong_as_double(static_cast<long long>(static_cast<unsigned long long>(word[4 * i + 2]) << 32 | word[4 * i]));
    };
    if (a.per_xcd != 0) {
      // the subtree of an XCD's workgroups first, by the first of them; then the XCDs' sums
      if (tid < kWave) {
        double s3[kOcSums] = {0, 0, 0};
        if (w % a.per_xcd == 0) {
          if (lane < a.per_xcd) read_line(w + lane, s3);
#pragma unroll
          for (int i = 0; i < kOcSums; ++i) s3[i] = wave_tree(s3[i]);
          if (lane < kOcSums) {
            const double v = lane == 0 ? s3[0] : (lane == 1 ? s3[1] : s3[2]);
            const unsigned long long bits = __builtin_bit_cast(unsigned long long, v);
            typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
            __builtin_amdgcn_raw_buffer_store_b128(u32x4{static_cast<uint32_t>(bits), iter, static_cast<uint32_t>(bits >> 32), iter},
                                                   line_rsrc, (set + kOwners + w / a.per_xcd) * kOcLine * 8 + 16 * lane, 0, 16);
          }
#pragma unroll
          for (int i = 0; i < kOcSums; ++i) s3[i] = 0;
        }
        if (lane < kXcds) read_line(kOwners + lane, s3);
#pragma unroll
        for (int i = 0; i < kOcSums; ++i) {
          s3[i] += dpp_move<kDppXor1>(s3[i]);
          s3[i] += dpp_move<kDppXor2>(s3[i]);
          s3[i] += dpp_move<kDppHalfMirror>(s3[i]);
        }
        if (lane < kOcSums) {
          tot[lane][0] = lane == 0 ? s3[0] : (lane == 1 ? s3[1] : s3[2]);
#pragma unroll
          for (int i = 1; i < kWavesPerBlock; ++i) tot[lane][i] = 0;
        }
      }
    } else if (tid < kOwners) {
      double s3[kOcSums] = {0, 0, 0};
      if (tid < a.nwg) read_line(tid, s3);
#pragma unroll
      for (int i = 0; i < kOcSums; ++i) {
        s3[i] = wave_tree(s3[i]);
        if (lane == 0) tot[i][wave] = s3[i];
      }
    }
    __syncthreads();
    if (!uniform(ok != 0)) return;
    const double rr = (tot[0][0] + tot[0][1]) + (tot[0][2] + tot[0][3]);
    const double ApAp = (tot[1][0] + tot[1][1]) + (tot[1][2] + tot[1][3]);
    const double pAp = (tot[2][0] + tot[2][1]) + (tot[2][2] + tot[2][3]);

    // ---- cg_iter_kernel's step (cg.hpp:170-180)
    // mixed1_iter_kernel's end test asks for an FP64 correction
    const bool conv = uniform(a.mixed ? rr < rr_stop || rr / nrs < tol2 : fabs(rr / nrs) < tol2 || fabs(rr) < atol2);
    const bool done = conv || iter >= max_iters;
    alpha = uniform(rr / pAp);
    beta = uniform((alpha * alpha * ApAp - rr) / rr);
    // the vectors are needed again: by the next launch, or by the correction
    more = done ? a.mixed != 0 : k + 1 == kOcSlice;
    if (w == 0 && tid == 0) {
      record_history(st, iter, rr);
      if (done || more) {
        st->iter = iter;
        st->rr = rr;
        st->rr2 = rr;
        st->alpha = alpha;
        st->beta = beta;
        if (done && a.mixed) {
          st->flags = (st->flags | kFlagPause) & ~kFlagNoPause;
        } else {
          st->converged = conv ? 1u : 0u;
          if (done) st->flags |= kFlagDone;
        }
      }
    }
    if (done || more) break;
  }

#pragma unroll
  for (int c = 0; c < CPV; ++c)
#pragma unroll
    for (int j = 0; j < TPC; ++j)
      if (static_cast<uint32_t>(j) < tiles_of[c]) {
        const int s = c * TPC + j;
        const uint32_t l = first[c] + j * kBlock, row = lo + l;
        bx.store(row, x[s]);
        if (more) {  // p (halo form) and A p (ghost form, kOcSlice being even) are there already
          br.store(row, r[s]);
          if constexpr (Ghosts > 0)
            bp.store(row, lp[own + l]);
          else
            bex1.store(row, ap[s]);
        }
      }
}

// ------------------------------------------------------------------ host side

// The solves that run on a device, for those of other host threads.
struct OcDevice {
  std::mutex mu;
  std::condition_variable cv;
  uint32_t used = 0;               // CUs of the on-chip launches that run
  uint32_t launched = 0;           // solves that run by launches of their own (LaunchedSolve)
  uint64_t tickets = 0, turn = 0;  // of the on-chip launches: given out, and whose turn it is
};
constexpr int kOcDevices = 64;
OcDevice* oc_device(int dev)
{
  static OcDevice* const d = new OcDevice[kOcDevices];  // never freed: threads may still wait when the process ends
  return dev >= 0 && dev < kOcDevices ? d + dev : nullptr;
}

// A solve's share of its device's CUs while a launch of its runs.  Solves of several host threads whose
// workgroups fit the device together run together; the others wait, in the order in which they came, and
// a solve of more than one launch queues again between them.  A solve that took the launched modes
// instead would get what the others' launches leave it, which is next to nothing: of two threads with
// Jacobi-CG on 97 x 83 x 71 one got 2.5 solves a second and the other 130 (41.6 each if both are launched).
class OcTurn {
 public:
  OcTurn(OcDevice* d, uint32_t cus, uint32_t want) : d_(*d), cus_(cus), want_(want) {}
  ~OcTurn() { give(); }
  OcTurn(const OcTurn&) = delete;
  OcTurn& operator=(const OcTurn&) = delete;
  // Whether a first launch should be left out: it would take most of the device from a solve that another
  // thread runs by launches (BiCGStab on 70 x 66 x 61 beside Jacobi-CG on 97 x 83 x 71 got 20 solves a second,
  // and 157 with both launched; a quarter of the CUs leaves it 144).
  bool in_the_way() const
  {
    std::lock_guard<std::mutex> lock(d_.mu);
    return d_.launched > 0 && want_ > cus_ / 4;
  }
  void take()
  {
    std::unique_lock<std::mutex> lock(d_.mu);
    const uint64_t ticket = d_.tickets++;
    d_.cv.wait(lock, [&] { return d_.turn == ticket && d_.used + want_ <= cus_; });
    ++d_.turn;
    d_.used += want_;
    held_ = true;
    d_.cv.notify_all();  // the next one may fit as well
  }
  void give()
  {
    if (!held_) return;
    std::lock_guard<std::mutex> lock(d_.mu);
    d_.used -= want_;
    held_ = false;
    d_.cv.notify_all();
  }

 private:
  OcDevice& d_;
  const uint32_t cus_, want_;
  bool held_ = false;
};

// Workgroups that start together do so within microseconds: after 2 ms other work holds the CUs, and
// the kernel-per-step modes, which share them, take over.  Once all run, only a process switch stops them.
uint64_t wait_ticks(bool first)
{
  return t_wait_us < 0 ? (first ? 2000 : 500000) * kOcClock : static_cast<uint64_t>(t_wait_us * kOcClock);
}

// The shape of an on-chip solve and the kernel that runs it.
template <typename T>
struct OcPlan {
  void (*kernel)(OcArgs<T>) = nullptr;
  uint32_t m = 0, nwg = 0, ext = 0, far = 0, reach = 0;
  bool ghost = false;
  size_t lds = 0;
};

template <typename T, uint32_t ND, bool Jac, int W, int TPC, int Ghosts>
void (*oc_value_kernel(OcVal how))(OcArgs<T>)
{
  if (how == kValOne) return onchip_cg_kernel<T, ND, Jac, W, 2, TPC, kValOne, Ghosts>;
  if (how == kValCodes) return onchip_cg_kernel<T, ND, Jac, W, 2, TPC, kValCodes, Ghosts>;
  if constexpr (TPC == 2) {  // more rows than that leave LDS no room
    if (how == kValMost) return onchip_cg_kernel<T, ND, Jac, W, 2, TPC, kValMost, Ghosts>;
    if (how == kValHalf) return onchip_cg_kernel<T, ND, Jac, W, 2, TPC, kValHalf, Ghosts>;
  }
  return onchip_cg_kernel<T, ND, Jac, W, 2, TPC, kValStream, Ghosts>;
}

template <typename T, uint32_t ND, bool Jac, int W>
void (*oc_kernel(bool ghost, int cpv, int tpc, uint32_t ghosts, OcVal how))(OcArgs<T>)
{
  constexpr uint32_t g1 = kOcThreads;
  if (ghost) {
    // up to two rows a lane: the values in registers
    if (cpv == 1 && tpc == 1 && ghosts <= 6 * g1) return onchip_cg_kernel<T, ND, Jac, W, 1, 1, kValRegs, 6>;
    if (cpv <= 2 && tpc == 1 && ghosts <= 6 * g1) return onchip_cg_kernel<T, ND, Jac, W, 2, 1, kValRegs, 6>;
    return nullptr;
  }
  if (cpv <= 2 && tpc <= 2) return oc_value_kernel<T, ND, Jac, W, 2, 0>(how);
  if (cpv <= 2 && tpc <= 4) return oc_value_kernel<T, ND, Jac, W, 4, 0>(how);
  if constexpr (sizeof(T) == 4)
    if (cpv <= 2 && tpc <= 8) return oc_value_kernel<T, ND, Jac, W, 8, 0>(how);
  return nullptr;
}

template <typename T>
bool oc_plan(const OnchipCg<T>& c, uint32_t cus, OcPlan<T>& pl)
{
  const uint32_t n = c.n, nd = c.dia.nd;
  if (nd == 0 || nd > kOcDiags || n >= (1u << 24)) return false;  // 32-bit byte offsets
  const uint32_t gp = cg_prod_chunks(n), tiles = cg_tiles(n);
  const uint32_t owners = gp < kOwners ? gp : kOwners;
  // fewer workgroups exchange faster (1.7 us for 64, 2.3 for 128, 2.4 for 256), so small systems put
  // several owners, one chunk or two each, on a workgroup's four 256-lane groups
  pl.m = gp <= kOwners ? 4u : (gp <= 2 * kOwners ? 2u : 1u);
  pl.nwg = (owners + pl.m - 1) / pl.m;
  if (pl.nwg > cus) return false;
  const uint32_t chunks = pl.m * ((gp + kOwners - 1) / kOwners);  // of a workgroup, at most
  const uint32_t vecs = pl.m * (gp <= kOwners ? 1u : cg_vec_per_owner(n));
  const int cpv = static_cast<int>((std::max(chunks, vecs) + kOcBlocks - 1) / kOcBlocks);
  const int tpc = static_cast<int>((tiles + gp - 1) / gp);
  const uint32_t rows = static_cast<uint32_t>((static_cast<uint64_t>(tiles) * chunks + gp - 1) / gp) * kBlock;  // at most
  const size_t tab = c.dia.code && c.dia.distinct != 1 ? kOcDiags * kDiaCodes * sizeof(T) : 0;
  const uint32_t slots = nd <= 5 ? 5 : 7;
  const uint32_t spare = (tpc <= 1 ? 1u : tpc <= 2 ? 2u : tpc <= 4 ? 4u : 8u) * kBlock;  // that lanes without a row read past the end
  // the LDS entries of a full workgroup: no workgroup has more
  auto segments = [&](uint32_t far) {
    OcSegments g;
    oc_segments(rows, nd, c.dia.first_off, far, g);
    return g.ext;
  };
  auto pick = [&](bool ghost, uint32_t far) {
    const uint32_t ext = segments(far);
    auto lds_bytes = [&](OcVal how) {
      return tab + (static_cast<size_t>(ext) + rows * (1 + val_held(how, slots)) + spare) * sizeof(T);
    };
    OcVal how = !c.dia.code ? kValStream : (c.dia.distinct == 1 ? kValOne : kValCodes);
    if (how == kValStream && !ghost && tpc <= 2)
      how = lds_bytes(kValMost) <= kOcLds ? kValMost : (lds_bytes(kValHalf) <= kOcLds ? kValHalf : kValStream);
    const size_t bytes = lds_bytes(how);
    if (bytes > kOcLds) return false;
    if (!c.wide) return false;
    const uint32_t g = ext - rows;
    auto choose = [&](auto slots) {
      constexpr uint32_t ND = decltype(slots)::value;
      return c.jacobi ? oc_kernel<T, ND, true, kVecW<T> >(ghost, cpv, tpc, g, how)
                      : oc_kernel<T, ND, false, kVecW<T> >(ghost, cpv, tpc, g, how);
    };
    void (*k)(OcArgs<T>) = slots == 5 ? choose(std::integral_constant<uint32_t, 5>()) : choose(std::integral_constant<uint32_t, 7>());
    if (!k) return false;
    pl.kernel = k;
    pl.ghost = ghost;
    pl.far = far;
    pl.ext = ext;
    pl.lds = bytes;
    return true;
  };
  if (pick(true, 0)) return true;
  // the far diagonals, all of them the first or the last
  if (nd < 2) return false;
  for (uint32_t i = 1; i + 1 < nd; ++i)
    if (static_cast<uint32_t>(std::abs(c.dia.first_off[i])) >= rows) return false;
  const uint32_t far = 1u | 1u << (nd - 1);
  pl.reach = oc_reach(n, gp, pl.m, pl.nwg, nd, c.dia.first_off);
  if (2 * pl.reach + 1 > 2 * kWave) return false;
  return pick(false, far);
}

}  // namespace

LaunchedSolve::LaunchedSolve()
{
  if (hipGetDevice(&dev_) != hipSuccess || !oc_device(dev_)) {
    dev_ = -1;
    return;
  }
  std::lock_guard<std::mutex> lock(oc_device(dev_)->mu);
  ++oc_device(dev_)->launched;
}

LaunchedSolve::~LaunchedSolve()
{
  if (dev_ < 0) return;
  std::lock_guard<std::mutex> lock(oc_device(dev_)->mu);
  --oc_device(dev_)->launched;
}

template <typename T>
int onchip_cg(const OnchipCg<T>& c, Workspace& ws, hipStream_t s, KState* fin, Onchip* outcome)
{
  *outcome = Onchip::kNo;
  t_on_chip = 0;
  OcPlan<T> pl;
  const uint32_t cus = static_cast<uint32_t>(device_cu_count());
  if (t_off || !oc_plan(c, cus, pl)) return VCLHIP_SUCCESS;
  int dev = 0;
  VCLHIP_HIP(hipGetDevice(&dev));
  OcDevice* const device = oc_device(dev);
  if (!device) return VCLHIP_SUCCESS;
  OcTurn turn(device, cus, pl.nwg);
  if (turn.in_the_way()) {
    *outcome = Onchip::kDeferred;
    return VCLHIP_SUCCESS;
  }
  VCLHIP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(pl.kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                 static_cast<int>(pl.lds)));
  int per_cu = 0;
  VCLHIP_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(pl.kernel), kOcThreads,
                                                          pl.lds));
  if (per_cu < 1) return VCLHIP_SUCCESS;
  // the exchange lines and the flags, cleared before the first launch
  struct Shared {
    unsigned long long lines[2 * kOcLines * kOcLine];
    uint32_t flags[kOwners * 16];
  };
  Shared* sh;
  T* ap2 = nullptr;
  if (!ws.try_alloc(&sh, 1) || (pl.ghost && !ws.try_alloc(&ap2, c.n))) return VCLHIP_SUCCESS;
  VCLHIP_TRY(vclhip_fill_zero(sh, sizeof(Shared), s));
  OcArgs<T> a{};
  a.n = c.n;
  a.mixed = c.after ? 1u : 0u;
  a.nd = c.dia.nd;
  a.gp = cg_prod_chunks(c.n);
  a.m = pl.m;
  a.nwg = pl.nwg;
  a.per_xcd = pl.nwg >= 128 && pl.nwg % kXcds == 0 ? pl.nwg / kXcds : 0;
  a.far = pl.far;
  a.ext = pl.ext;
  a.reach = pl.reach;
  for (uint32_t i = 0; i < c.dia.nd; ++i) a.off[i] = c.dia.first_off[i];
  a.val = c.dia.val;
  a.code = c.dia.code;
  a.table = c.dia.table;
  a.x = c.x;
  a.r = c.r;
  a.p = c.p;
  a.d = c.d;
  a.ex0 = pl.ghost ? ap2 : c.p;
  a.ex1 = c.Ap;
  a.st = c.st;
  a.lines = sh->lines;
  a.flags = sh->flags;
  a.abort = &c.st->breakdown;
  a.wait_first = wait_ticks(true);
  a.wait = wait_ticks(false);
  // (what is still to run in front of the launch is the setup's few kernels: start() waited for the stream)
  do {
    turn.take();
    hipLaunchKernelGGL(pl.kernel, dim3(pl.nwg), dim3(kOcThreads), pl.lds, s, a);
    VCLHIP_TRY(check_launch("onchip_cg_kernel"));
    if (c.after) VCLHIP_TRY(c.after());
    VCLHIP_HIP(hipMemcpyAsync(fin, c.st, sizeof(KState), hipMemcpyDeviceToHost, s));
    VCLHIP_HIP(hipStreamSynchronize(s));
    turn.give();
    a.wait_first = a.wait;
  } while (!fin->breakdown && !(fin->flags & kFlagDone));
  *outcome = fin->breakdown ? Onchip::kAborted : Onchip::kDone;
  t_on_chip = fin->breakdown ? 2 : 1;
  return VCLHIP_SUCCESS;
}

namespace {

template <typename T>
int oc_plan_of(OnchipCg<T> c, uint32_t cus, const int32_t* off, uint32_t distinct, uint32_t* reach, uint32_t* rows)
{
  static const uint8_t coded = 0;
  c.dia.distinct = distinct;
  c.dia.code = distinct ? &coded : nullptr;
  std::copy(off, off + std::min(c.dia.nd, kDiaGroup), c.dia.first_off);
  OcPlan<T> pl;
  if (!oc_plan(c, cus, pl)) return 0;
  const uint32_t gp = cg_prod_chunks(c.n);
  for (uint32_t w = 0; w < pl.nwg; ++w) {
    const OcPart q = oc_part(c.n, gp, pl.m, w);
    rows[w] = q.t0 * kBlock;
    rows[w + 1] = q.t1 * kBlock;
  }
  *reach = pl.ghost ? 0 : pl.reach;
  return static_cast<int>(pl.nwg);
}

}  // namespace

template int onchip_cg<double>(const OnchipCg<double>&, Workspace&, hipStream_t, KState*, Onchip*);
template int onchip_cg<float>(const OnchipCg<float>&, Workspace&, hipStream_t, KState*, Onchip*);

}  // namespace vclhip

extern "C" {

int onchip_cg_wait_limit(double microseconds)
{
  vclhip::t_wait_us = microseconds;
  return VCLHIP_SUCCESS;
}

int onchip_cg_off(int off)
{
  vclhip::t_off = off != 0;
  return VCLHIP_SUCCESS;
}

int onchip_cg_last(void)
{
  const int v = vclhip::t_on_chip;
  vclhip::t_on_chip = 0;
  return v;
}

// The plan of an n-row system of nd diagonals (ascending offsets; `distinct` values on a diagonal, 0: as
// stored) on a device of `cus` compute units, without one: the number of workgroups (0: not on chip),
// the first row of each and the end of the last in rows[0 .. 256], and in *reach for how many workgroups
// on each side it waits (0: the ghost form).
int onchip_cg_plan(int single, int jacobi, uint32_t n, uint32_t nd, const int32_t* off, uint32_t distinct, uint32_t cus,
                   uint32_t* reach, uint32_t* rows)
{
  if (single) {
    vclhip::OnchipCg<float> c{};
    c.n = n, c.dia.nd = nd, c.jacobi = jacobi != 0, c.wide = true;
    return vclhip::oc_plan_of(c, cus, off, distinct, reach, rows);
  }
  vclhip::OnchipCg<double> c{};
  c.n = n, c.dia.nd = nd, c.jacobi = jacobi != 0, c.wide = true;
  return vclhip::oc_plan_of(c, cus, off, distinct, reach, rows);
}

}  // extern "C"
