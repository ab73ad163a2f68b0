// cg_sums.hpp -- how CG's inner products are grouped: 256 owners, the same in every launch mode.
//
// The rows of a system are cut into 256-row tiles and the tiles into product chunks (one partial sum
// of <Ap,Ap> and <p,Ap> each, the grid of the product kernel).  Owner o of 256 takes a contiguous
// range of the product chunks, and the vector chunks (one partial sum of <r,z> each, the grid of
// the update kernel) are cut inside an owner's rows.  An inner product is the sum of an owner's
// partial sums in order and then a binary tree over the owners.  Both kinds of chunks and the
// owners thus nest: a workgroup that holds an owner's rows forms everything the owner adds, which
// is what lets one launch run all the iterations with a single value per owner and inner product
// exchanged (onchip_cg.hip), with the sums of the kernel-per-step modes bit for bit.
#pragma once

#include "device.hpp"

namespace vclhip {

constexpr uint32_t kOwners = 256;
constexpr uint32_t kCgProdMax = 2048;      // product chunks at most (the product kernels' grid)
constexpr uint32_t kCgVecRows = 1u << 18;  // rows of all owners' vector chunks of 1024 rows, one each
constexpr uint32_t kCgVecPerOwner = 8;     // vector chunks per owner at most
static_assert(kCgProdMax <= kMaxPartials && kOwners * kCgVecPerOwner <= kMaxPartials && kMaxPartials <= 4096, "partial sums");

// [begin, end) of part i of `parts` (at most kCgProdMax) near-equal contiguous parts of `total` items.
constexpr uint32_t kPartShort = 1u << 20;
static_assert(static_cast<uint64_t>(kPartShort) * kCgProdMax < 1ull << 32 && kOwners <= kCgProdMax, "products of 32 bits");
__host__ __device__ inline void part_range(uint32_t total, uint32_t i, uint32_t parts, uint32_t& begin, uint32_t& end)
{
  if (total <= kPartShort) {  // 32 bits hold the product, and its division is the shorter one
    begin = total * i / parts;
    end = total * (i + 1) / parts;
  } else {
    begin = static_cast<uint32_t>((static_cast<uint64_t>(total) * i) / parts);
    end = static_cast<uint32_t>((static_cast<uint64_t>(total) * (i + 1)) / parts);
  }
}

// Owner o's part of `count` chunks: one each while there are at most kOwners.
__host__ __device__ inline void owner_range(uint32_t count, uint32_t o, uint32_t& begin, uint32_t& end)
{
  if (count <= kOwners) {
    begin = o < count ? o : count;
    end = o < count ? o + 1 : count;
  } else {
    part_range(count, o, kOwners, begin, end);
  }
}

__host__ __device__ inline uint32_t cg_tiles(uint32_t n) { return (n + kBlock - 1) / kBlock; }

// Product chunks of an n-row system on the tile formats (chunk_grid's rule).
__host__ __device__ inline uint32_t cg_prod_chunks(uint32_t n)
{
  uint32_t g = cg_tiles(n);
  if (g > kCgProdMax) g = kCgProdMax;
  g = (g + 7u) & ~7u;
  return g < 8u ? 8u : g;
}

// Vector chunks per owner (chunks of at most 1280 rows up to 2.4 M rows); with at most kOwners
// product chunks the vector chunks are those.
__host__ __device__ inline uint32_t cg_vec_per_owner(uint32_t n)
{
  const uint32_t m = n / kCgVecRows + (n % kCgVecRows > kCgVecRows / 4 ? 1u : 0u);
  return m < 1u ? 1u : (m > kCgVecPerOwner ? kCgVecPerOwner : m);
}

// Grid of CG's vector kernels.
__host__ __device__ inline uint32_t cg_vec_chunks(uint32_t n)
{
  const uint32_t gp = cg_prod_chunks(n);
  return gp <= kOwners ? gp : kOwners * cg_vec_per_owner(n);
}

// Rows [begin, end) of vector chunk c (begin a multiple of kBlock).
__host__ __device__ inline void cg_vec_rows(uint32_t n, uint32_t c, uint32_t& begin, uint32_t& end)
{
  const uint32_t tiles = cg_tiles(n), gp = cg_prod_chunks(n);
  uint32_t t0, t1;
  if (gp <= kOwners) {
    part_range(tiles, c, gp, t0, t1);
  } else {
    const uint32_t m = cg_vec_per_owner(n);
    uint32_t p0, p1, o0, o1, unused;
    owner_range(gp, c / m, p0, p1);
    part_range(tiles, p0, gp, o0, unused);
    part_range(tiles, p1, gp, o1, unused);
    part_range(o1 - o0, c % m, m, t0, t1);
    t0 += o0;
    t1 += o0;
  }
  begin = t0 * kBlock;
  end = t1 * kBlock < n ? t1 * kBlock : n;
  if (begin > end) begin = end;
}

// The binary tree over a wavefront's lanes (xor 1, 2, 4, ..., 32), returned to every lane.  The mirrors
// read lane ^ 4 and lane ^ 8 because the values before them repeat within 4 and 8 lanes.
constexpr int kDppHalfMirror = 0x141;
constexpr int kDppMirror = 0x140;
template <typename A>
__device__ __forceinline__ A wave_tree(A v)
{
  v += dpp_move<kDppXor1>(v);
  v += dpp_move<kDppXor2>(v);
  v += dpp_move<kDppHalfMirror>(v);
  v += dpp_move<kDppMirror>(v);
  A u = v;
  swap_rows<16>(v, u);
  v += u;
  u = v;
  swap_rows<32>(v, u);
  return v + u;
}

// The tree over the 256 owner sums of K inner products (lane o holds owner o's), returned to every lane.
template <int K, typename A>
__device__ __forceinline__ void owner_tree_k(A (&s)[K], A (&out)[K])
{
  __shared__ A red[K][kWavesPerBlock];
  const int wave = threadIdx.x / kWave;
#pragma unroll
  for (int q = 0; q < K; ++q) {
    s[q] = wave_tree(s[q]);
    if ((threadIdx.x & (kWave - 1)) == 0) red[q][wave] = s[q];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < K; ++q) out[q] = (red[q][0] + red[q][1]) + (red[q][2] + red[q][3]);
  __syncthreads();
}

// The sums of K partial-sum arrays by one 256-lane workgroup (lane o is owner o), returned to every
// lane: owner sums in chunk order, the loads of up to eight chunks and all K arrays in flight
// together, then the binary tree over the lanes.
template <int K, typename A>
__device__ __forceinline__ void owner_sums_k(const A* const (&p)[K], const uint32_t (&count)[K], A (&out)[K])
{
  uint32_t b[K], e[K], most = 0;  // most: the longest owner range, the same for every lane
#pragma unroll
  for (int q = 0; q < K; ++q) {
    owner_range(count[q], threadIdx.x, b[q], e[q]);
    const uint32_t m = (count[q] + kOwners - 1) / kOwners;
    most = m > most ? m : most;
  }
  A s[K];
#pragma unroll
  for (int q = 0; q < K; ++q) s[q] = 0;
  constexpr uint32_t B = 8;
  for (uint32_t i0 = 0; i0 < most; i0 += B) {
    A v[B][K];
#pragma unroll
    for (uint32_t i = 0; i < B; ++i)
      if (i0 + i < most)
#pragma unroll
        for (int q = 0; q < K; ++q) v[i][q] = b[q] + i0 + i < e[q] ? p[q][b[q] + i0 + i] : A(0);
#pragma unroll
    for (uint32_t i = 0; i < B; ++i)
      if (i0 + i < most)
#pragma unroll
        for (int q = 0; q < K; ++q)
          if (b[q] + i0 + i < e[q]) s[q] += v[i][q];
  }
  owner_tree_k<K, A>(s, out);
}

template <typename A>
__device__ __forceinline__ void owner_sums3(const A* pa, uint32_t na, const A* pb, uint32_t nb, const A* pc,
                                            uint32_t nc, A& ra, A& rb, A& rc)
{
  const A* const p[3] = {pa, pb, pc};
  const uint32_t count[3] = {na, nb, nc};
  A out[3];
  owner_sums_k<3, A>(p, count, out);
  ra = out[0];
  rb = out[1];
  rc = out[2];
}

}  // namespace vclhip
