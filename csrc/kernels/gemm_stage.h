// Where the lanes of the 256 x 256 GEMM's stages read (gemm.hip): integer arithmetic alone, so that its bounds test walks
// it on the host.
#pragma once
#include <cstddef>

namespace vwa {

// A-image slot swizzle: chunk c of row r sits at slot c ^ F((r >> 1) & 7).  F makes every
// ds_read_b128 lane group ({0-3,12-15,20-27}, {4-11,16-19,28-31}, ... : two k-chunk columns g,
// 16 rows) hit 16 distinct (row parity, slot) bank groups: F maps the half-row indices
// {0,1,6,7} to the even slots and {2,3,4,5} to the odd ones, so XOR-ing the chunk index with 2
// (the other column of the group) cannot collide.  (Plain c ^ h measured 33 % bank conflicts.)
__host__ __device__ inline int swz(int h) { return (0x64753120 >> (4 * h)) & 7; }

// bf16 stages: half hs & 1 = h of a k-group is k 64 h .. 64 h + 64, a whole 128-byte line of every X row.  In the tiled
// weight's order (lane group g of substep s: k 32 g + 8 s) that is the groups g = 2 h, 2 h + 1 of all four substeps: MFMA
// sp of the half takes, in lane group g, substep 2 sp + (g >> 1) of group 2 h + (g & 1) -- k 64 h + 32 (g & 1) + 16 sp +
// 8 (g >> 1), chunk 4 (g & 1) + 2 sp + (g >> 1) of the X row's line.  (Substeps 2 h, 2 h + 1 of all groups took 32 of every
// 64 bytes of two lines per row, each line twice, 1.5 times the bytes through L1: 128^2 tile 12000 x 1280 x 1280 583 ->
// 646 TFLOP/s, 1500 x 5120 x 1280 532 -> 594.)
// A read's 16-lane groups now hold chunks c and c ^ 4 of complementary half rows {0,1,6,7}, {2,3,4,5}: swzk maps both
// halves to 0..3.
// LINES false keeps the substeps' own order, for weights whose products choose experts further on (GemmParams::keep_order):
// the same sums in another order move a product by its last bits, and a token whose scores nearly tie to another expert --
// 1 in 300 decoded rows of a 16-expert model when its prompt alone was computed in the other order.
__host__ __device__ inline int swzk(int h) { return (h & 1) | (h >> 2 << 1); }
__host__ __device__ inline int chunk_of(int g, int sp) { return 4 * (g & 1) + 2 * sp + (g >> 1); }

constexpr unsigned kPastEnd = 0xFFFFFFF0u;  // vector offset outside of every resource (they end below 2 GB): reads zeros

// Byte offset, in k-group 0, of lane l's 16-byte piece of tile row r (row m of X, ldx elements apart)
template <bool F8, bool LINES>
__host__ __device__ inline unsigned p8_x_piece(int m, int ldx, int r, int l) {
  const int h = (r >> 1) & 7, c = (l & 7) ^ (F8 || !LINES ? swz(h) : swzk(h));
  return (unsigned)(F8 ? (size_t)m * ldx + 16 * c : ((size_t)m * ldx + (LINES ? 8 * c : 32 * (c >> 1) + 8 * (c & 1))) * 2);
}
// ... of MFMA sp of the weight's 16-column tile T (WT: pre-tiled, else row-major [N, K])
template <bool F8, bool WT, bool LINES>
__host__ __device__ inline unsigned p8_w_piece(int T, int sp, int K, int l) {
  if (F8) return (unsigned)((size_t)T * (K / 128) * 2048 + sp * 1024 + l * 16);
  const int g = l >> 4;
  return (unsigned)(2 * (WT ? (size_t)T * (K / 128) * 2048 + (LINES ? (2 * sp + (l >> 5)) * 512 + (l & 31) * 8 : sp * 512 + l * 8)
                            : (size_t)(T * 16 + (l & 15)) * K + (LINES ? 8 * chunk_of(g, sp) : 32 * g + 8 * sp)));
}
// Scalar offset of stage hs (fp8: k-group hs, bf16: half hs & 1 of k-group hs / 2).  A stage past the last (in false) is
// issued on an empty resource, and at 0: whether the scalar offset takes part in a resource's range check, and how an empty
// one wraps there, then does not matter, and neither for any other piece (a piece inside by its vector offset stays inside
// with the scalar one added).
template <bool F8, bool LINES>
__host__ __device__ inline unsigned p8_x_step(int hs, bool in) {
  return !in ? 0 : F8 ? hs * 128 : 2 * ((hs >> 1) * 128 + (LINES ? 64 : 16) * (hs & 1));
}
template <bool F8, bool WT, bool LINES>
__host__ __device__ inline unsigned p8_w_step(int hs, bool in) {
  return !in ? 0 : F8 ? hs * 2048 : WT ? 2 * ((hs >> 1) * 2048 + (LINES ? 256 : 1024) * (hs & 1)) : p8_x_step<false, LINES>(hs, true);
}

}  // namespace vwa
