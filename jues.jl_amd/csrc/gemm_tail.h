// The last round of tiles of a GEMM launch shared by several workgroups a tile (gemm.hip, gemm16.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

namespace jues {
namespace {

constexpr int TAIL_XCD = 8, TAIL_GROUP = 8;

// Tile p2 of tiles_m x tiles_n in grouped order: TAIL_GROUP tile-rows share each sweep over tile-columns
__device__ inline void grouped_tile(int p2, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int group_size = TAIL_GROUP * tiles_n;
  const int gid = p2 / group_size;
  const int first_m = gid * TAIL_GROUP;
  const int gsz = min(tiles_m - first_m, TAIL_GROUP);
  const int r = p2 - gid * group_size;
  tm = first_m + r % gsz;
  tn = r / gsz;
}

// Tile p2 of the lower triangle of m x m tiles (tm >= tn), in bands of TAIL_GROUP tile-rows that sweep the tile-columns
// up to the diagonal
__device__ inline void lower_tile(int p2, int m, int& tm, int& tn) {
  constexpr int G = TAIL_GROUP;  // band g starts after G^2 g (g - 1) / 2 + G (G + 1) / 2 g tiles
  const auto before = [](int g) { return G * G * (g * (g - 1) / 2) + G * (G + 1) / 2 * g; };
  int g = (int)(sqrtf(2.0f * (float)p2) / (float)G);
  while (before(g) > p2) --g;
  while (before(g + 1) <= p2) ++g;
  int r = p2 - before(g);
  const int h = min(G, m - G * g);
  if (r < h * G * g) {
    tm = G * g + r % h;
    tn = r / h;
    return;
  }
  r -= h * G * g;
  int c = 0;
  while (r >= h - c) r -= h - c++;
  tm = G * g + c + r;
  tn = G * g + c;
}

// A TAIL launch of a product: `whole` workgroups have a tile each, and the other tiles' 16-deep k-slabs are shared by
// several workgroups a tile, whose parts of it gemm_tail_kernel adds.  Tiles are taken full ones first (grouped),
// then those past the edge of N, of M and of both: four runs of n[] tiles left to the tail, in s[] chunks each.
// Within a run, the parts are ordered chunk by chunk: neighbours read the same k-slabs.
// 256 compute units leave much of a last round of tiles idle otherwise, and split whole products write more parts
// (and round no better): FP64 3082^3 took 980 us in two chunks, 890 this way, 6460^3 8.6 and 7.6 ms (73 TFLOP/s would be
// 7.4), 276 x 9045 x 9045 902 and 792 us, 8640 x 768 x 8640 1790 and 1660; FP32 3082^3 507 and 478.
struct TailMap {
  int whole = 0, wgs = 0, nk = 0, full_m = 0, full_n = 0;
  int n[4] = {}, s[4] = {};
  bool lower = false;  // a square result of which only the tiles tm >= tn are formed

  __device__ void coords(int p2, int& tm, int& tn) const {
    const int full = lower ? full_m * (full_m + 1) / 2 : full_m * full_n;
    if (p2 < full && lower) lower_tile(p2, full_m, tm, tn);
    else if (p2 < full) grouped_tile(p2, full_m, full_n, tm, tn);
    else if ((p2 -= full) < n[1]) tm = p2, tn = full_n;
    else if ((p2 -= n[1]) < n[2]) tm = full_m, tn = p2;
    else tm = full_m, tn = full_n;
  }
  // tile of the tail, chunk of it (of `chunks`) and place of its part, of workgroup x.  The runs past an edge come
  // first (their few long chunks end last otherwise), and each run is dealt to the XCDs in equal contiguous shares.
  __device__ void part(int x, int& tile, int& chunk, int& chunks, int& place) const {
    int at = 0;
#pragma unroll
    for (int k = 1; k <= 4; ++k) {
      const int q = k & 3, count = n[q] * s[q];
      if (x < count) {
        const int per = count / TAIL_XCD, more = count % TAIL_XCD, xcd = x % TAIL_XCD;
        const int y = xcd * per + min(xcd, more) + x / TAIL_XCD;
        chunk = y / n[q];
        tile = first_tile(q) + y - chunk * n[q];
        chunks = s[q];
        place = at + y;
        return;
      }
      x -= count;
      at += count;
    }
  }
  __device__ int first_tile(int q) const { return (q > 0 ? n[0] : 0) + (q > 1 ? n[1] : 0) + (q > 2 ? n[2] : 0); }
};

// Tiles of bm x bn over wm x wn wavefronts, a slice of slab_k deep; share: the least part of a full tile's time that a
// tile past an edge takes (its slabs are staged all the same); least_slabs: of a chunk.
struct TailShape {
  int bm, bn, wm, wn, slab_k;
  double share;
  int least_slabs;
};

// The TAIL launch of an M x N x K product with `whole` full tiles to themselves and the others in `chunks` chunks,
// those past an edge in fewer by the cost of their slabs; wgs = 0 in the result if it is not of use (fewer full tiles,
// chunks under least_slabs, parts over 256 MiB).
// lower: the lower triangle of tiles of a square result.
inline TailMap tail_map(const TailShape& g, long M, long N, long K, long whole, int chunks, bool lower = false) {
  const auto cdiv = [](long a, long b) { return (a + b - 1) / b; };
  TailMap t;
  const long fm = M / g.bm, fn = N / g.bn, nk = cdiv(K, g.slab_k);
  const int em = (int)cdiv(M % g.bm, 16), en = (int)cdiv(N % g.bn, 16);  // 16-row and 16-column blocks past the edge
  const long full = lower ? fm * (fm + 1) / 2 : fm * fn;
  const long rest = (lower ? full + (em ? fm + 1 : 0) : cdiv(M, g.bm) * cdiv(N, g.bn)) - whole;
  if (full < whole || rest < 1 || rest > 2048 || (chunks > 1 && nk < (long)g.least_slabs * chunks)) return t;
  t.lower = lower;
  t.whole = (int)whole;
  t.nk = (int)nk;
  t.full_m = (int)fm;
  t.full_n = (int)fn;
  // parts of a full tile's time: the 16-row (16-column) blocks that a wavefront has, of those of a full tile
  const double um = (double)cdiv(em, g.wm) * g.wm * 16 / g.bm, un = (double)cdiv(en, g.wn) * g.wn * 16 / g.bn;
  const int n[4] = {(int)(full - whole), en && !lower ? (int)fm : 0, em ? (int)fn : 0, em && en ? 1 : 0};
  const double w[4] = {1.0, std::max(g.share, un), std::max(g.share, um), std::max(g.share, um * un)};
  long wgs = 0;
  for (int q = 0; q < 4; ++q) {
    t.n[q] = n[q];
    t.s[q] = std::max(1, (int)(chunks * w[q] + 0.5));
    wgs += (long)t.n[q] * t.s[q];
  }
  if (wgs <= 2048) t.wgs = (int)wgs;
  return t;
}

// The longest sum over k in one accumulator of a TAIL launch, slab_k of it a slab
inline long tail_chain(const TailMap& t, long slab_k) {
  int least = t.whole ? 1 : 1 << 30;
  for (int q = 0; q < 4; ++q)
    if (t.n[q]) least = std::min(least, t.s[q]);
  return (t.nk + least - 1) / least * slab_k;
}

}  // namespace
}  // namespace jues
