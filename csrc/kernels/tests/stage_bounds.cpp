// Walks every piece that the 256 x 256 GEMM's stages request and checks that it lies inside its operand however a scalar
// offset enters the range check: pieces inside the resource by their vector offset alone stay inside with the scalar one
// added; stages past the last are requested on an empty resource at scalar offset 0.  Build: g++ -D__host__= -D__device__=
#include <algorithm>
#include <cstdio>

#include "../gemm_stage.h"

using namespace vwa;

static long bad = 0, seen = 0;

static void piece(unsigned voff, unsigned soff, size_t bytes, bool in) {
  ++seen;
  if (!in) bad += soff != 0;
  else if (voff < bytes) bad += (size_t)voff + soff + 16 > bytes;
}

template <bool F8, bool WT, bool LINES>
static void walk(int M, int N, int K, int ldx, int splits) {
  const int KG = K / 128, per = (KG + splits - 1) / splits, spg = F8 ? 1 : 2, e = F8 ? 1 : 2;
  const size_t xb = ((size_t)(M - 1) * ldx + K) * e, wb = (size_t)N * K * e;
  for (int k0 = 0; k0 < KG; k0 += per) {
    const int nh = spg * (std::min(KG, k0 + per) - k0), h0 = spg * k0;
    for (int s = 0; s < nh + 2; ++s)
      for (int q = 0; q < 32; ++q)
        for (int l = 0; l < 64; ++l) {
          const int r = 8 * q + (l >> 3);
          const bool in = s < nh;
          for (int bm = 0; bm < M; bm += 256)
            piece(bm + r < M ? p8_x_piece<F8, LINES>(bm + r, ldx, r, l) : kPastEnd, p8_x_step<F8, LINES>(h0 + s, in), xb, in);
          for (int bn = 0; bn < N; bn += 256) {
            const int T = bn / 16 + q / 2;
            piece(T * 16 < N ? p8_w_piece<F8, WT, LINES>(T, q & 1, K, l) : kPastEnd, p8_w_step<F8, WT, LINES>(h0 + s, in), wb, in);
          }
        }
  }
}

int main() {
  const int shapes[][5] = {{256, 256, 128, 128, 1}, {130, 16, 128, 136, 1}, {257, 272, 384, 384, 2}, {511, 496, 1152, 1160, 4},
                           {300, 1296, 640, 256, 3} /* rows of a convolution overlap */, {1, 4096, 256, 256, 2}};
  for (const auto& s : shapes) {
    walk<false, true, true>(s[0], s[1], s[2], s[3], s[4]);
    walk<false, true, false>(s[0], s[1], s[2], s[3], s[4]);
    walk<false, false, true>(s[0], s[1], s[2], s[3], s[4]);
    if (s[3] % 16 == 0) walk<true, true, true>(s[0], s[1], s[2], s[3], s[4]);
  }
  std::printf("%ld pieces, %ld outside\n", seen, bad);
  return bad != 0;
}
