#include "tiled_layout.h"

#include <algorithm>
#include <cstring>

#include "hip_util.h"

namespace kvx {
namespace {

constexpr int kMaxTiles = 4;
constexpr int64_t kU32Limit = int64_t{1} << 32;
constexpr int64_t kDivLimit = int64_t{1} << 31;  // FastDivU32 divisors

bool MulOk(int64_t a, int64_t b, int64_t* out) { return !__builtin_mul_overflow(a, b, out); }

int64_t CeilDiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// One dimension of a shape while the tiles are applied: the logical
// dimension it indexes (-1: a padded leading 1), the divisions / modulos
// applied to that index so far, and its size.
struct WorkDim {
  int src = -1;
  std::vector<std::pair<bool, int64_t>> ops;  // (is_mod, divisor)
  int64_t size = 1;
};

// The physical-order shape the tiles apply to (tiling_utils.cc:911-921):
// rank 1 becomes (1, d0); higher ranks are permuted major-to-minor.
std::vector<WorkDim> PhysicalOrder(const TiledLayout& l) {
  const int r = static_cast<int>(l.dims.size());
  std::vector<WorkDim> cur;
  if (r == 1) {
    cur.push_back(WorkDim{});
    WorkDim d;
    d.src = 0;
    d.size = l.dims[0];
    cur.push_back(d);
  } else {
    for (int i = r - 1; i >= 0; --i) {
      WorkDim d;
      d.src = l.minor_to_major[i];
      d.size = l.dims[d.src];
      cur.push_back(d);
    }
  }
  return cur;
}

// Applies every tile (tiling_utils.cc:923-950): a tile of rank k splits the
// k minor-most dimensions into (ceil(d / t)) and (t) parts; a tile of larger
// rank than the shape first pads it with leading 1s.
std::vector<WorkDim> ApplyTiles(const TiledLayout& l) {
  std::vector<WorkDim> cur = PhysicalOrder(l);
  for (const std::vector<int64_t>& tile : l.tiles) {
    const size_t k = tile.size();
    if (k > cur.size()) cur.insert(cur.begin(), k - cur.size(), WorkDim{});
    const size_t start = cur.size() - k;
    std::vector<WorkDim> next(cur.begin(), cur.begin() + start);
    for (size_t i = 0; i < k; ++i) {
      WorkDim d = cur[start + i];
      d.ops.push_back({false, tile[i]});
      d.size = CeilDiv(d.size, tile[i]);
      next.push_back(d);
    }
    for (size_t i = 0; i < k; ++i) {
      WorkDim d = cur[start + i];
      d.ops.push_back({true, tile[i]});
      d.size = tile[i];
      next.push_back(d);
    }
    cur.swap(next);
  }
  return cur;
}

// Standard-form units run in tiled order when tiling (each workgroup writes
// one contiguous span of the tiled buffer, padding included) and in linear
// order when detiling (each workgroup writes whole rows of the linear
// image). On the Llama-3-8B set in T(8,128)(2,1), one process, one launch
// each: tiling 79.2 % of HBM peak in tiled order against 78.2 % in linear
// order, detiling 77.0 % in linear order against 75.4 %.

int WidestVector(uint64_t acc, int cap) {
  for (int v = cap; v > 1; v /= 2) {
    if ((acc & static_cast<uint64_t>(v - 1)) == 0) return v;
  }
  return 1;
}

// Vector width of a standard form's units: the widest that divides a row of a
// tile (so that a vector never straddles two tiles) and that a row of the
// matrix holds. The rows themselves may start at any address and end inside a
// vector: a bf16 [4096, 32003] tiled into T(8,128)(2,1) takes 8-byte vectors
// in 99 us a call (floor 78 at 6.7 TB/s), element by element with a clearing
// pass 2066.
int UnitVector(uint64_t W, uint64_t tW, uint64_t s) {
  int v = WidestVector(tW * s, 16);
  while (v > 1 && static_cast<uint64_t>(v) > W * s) v /= 2;
  return v;
}

}  // namespace

Status ValidateTiledLayout(const TiledLayout& l) {
  if (l.itemsize != 1 && l.itemsize != 2 && l.itemsize != 4 && l.itemsize != 8) {
    return InvalidArgumentError("tiled layout: itemsize must be 1, 2, 4 or 8");
  }
  const size_t r = l.dims.size();
  if (r > static_cast<size_t>(kTiledMaxRank)) {
    return InvalidArgumentError("tiled layout: at most 8 dimensions");
  }
  if (l.minor_to_major.size() != r) {
    return InvalidArgumentError("tiled layout: minor_to_major needs one entry per dimension");
  }
  std::vector<bool> seen(r, false);
  for (int m : l.minor_to_major) {
    if (m < 0 || static_cast<size_t>(m) >= r || seen[m]) {
      return InvalidArgumentError("tiled layout: minor_to_major is not a permutation");
    }
    seen[m] = true;
  }
  for (int64_t d : l.dims) {
    if (d < 0) return InvalidArgumentError("tiled layout: negative dimension");
  }
  if (l.tiles.size() > static_cast<size_t>(kMaxTiles)) {
    return InvalidArgumentError("tiled layout: at most 4 tiles");
  }
  for (const std::vector<int64_t>& t : l.tiles) {
    if (t.empty() || t.size() > static_cast<size_t>(kTiledMaxRank)) {
      return InvalidArgumentError("tiled layout: a tile has 1 to 8 dimensions");
    }
    for (int64_t d : t) {
      if (d < 1) {
        return InvalidArgumentError(
            "tiled layout: tile dimensions must be >= 1 (combined dimensions are not supported)");
      }
    }
  }
  return OkStatus();
}

int64_t LogicalElements(const TiledLayout& l) {
  int64_t n = 1;
  for (int64_t d : l.dims) {
    if (!MulOk(n, d, &n)) return -1;
  }
  return n;
}

StatusOr<int64_t> TiledBufferElements(const TiledLayout& l) {
  KVX_RETURN_IF_ERROR(ValidateTiledLayout(l));
  if (l.dims.empty()) return int64_t{1};
  int64_t n = 1;
  for (const WorkDim& d : ApplyTiles(l)) {
    if (!MulOk(n, d.size, &n)) return InvalidArgumentError("tiled layout: size overflows");
  }
  return n;
}

int64_t TiledPlan::CutAtOrBelow(int64_t x) const {
  if (x <= 0) return 0;
  if (x >= logical_bytes) return logical_bytes;
  const int64_t s = layout.itemsize;
  if (!tiled) return x;
  if (!standard && !column) return x / s * s;
  const int64_t row_bytes = static_cast<int64_t>(W) * s;
  const int64_t row = x / row_bytes;
  const int64_t b = row / static_cast<int64_t>(H);
  const int64_t h = row % static_cast<int64_t>(H);
  const int64_t rows = static_cast<int64_t>(CutRows());
  return (b * static_cast<int64_t>(H) + h / rows * rows) * row_bytes;
}

// Regions of one matrix along its rows and across them (transposed form);
// tiling covers the padding too.
static uint64_t ColumnRegionsAlong(const TiledPlan& p) {
  const uint64_t per = kColBytes / static_cast<uint64_t>(p.layout.itemsize);
  return (p.nT0 * p.tH + per - 1) / per;
}
static uint64_t ColumnRegionsAcross(uint64_t rows) { return (rows + kColRows - 1) / kColRows; }

// Whether the transposed form takes the layout: rows hold a vector (the kernel
// steps their last one back to the row's end), tiled vectors of 16 bytes stay
// in one row group of one tile, and the matrices fill at least a sixteenth of
// their regions, where the two forms meet: bf16 batches of [32, 32], a
// sixteenth full, detile / tile in 23.5 / 38.1 us against 52.1 / 63.5 element
// by element, [16, 32], half of that, in 42.2 / 69.6 against 52.0 / 66.7 and
// [16, 16] in 41.3 / 67.4 against 34.1 / 45.5.
static bool ColumnFits(const TiledPlan& p) {
  const uint64_t s = static_cast<uint64_t>(p.layout.itemsize);
  if (p.tW * p.P * s % 16 != 0 || p.W * s < 16) return false;
  const uint64_t along = ColumnRegionsAlong(p);
  const uint64_t across = ColumnRegionsAcross(p.nT1 * p.tW);
  uint64_t regions = 0;
  if (__builtin_mul_overflow(along, across, &regions) ||
      __builtin_mul_overflow(regions, p.B, &regions) ||
      regions >= static_cast<uint64_t>(kDivLimit)) {
    return false;
  }
  return regions * (kColRows * kColBytes / 16) <= static_cast<uint64_t>(p.logical_bytes);
}

// Whether the standard form's units at vector width v stay within the
// kernels' 32-bit unit indices and FastDivU32 divisors: linear order counts
// B * ceil(H / P) * ceil(W * s / v) units, tiled order tiled_bytes / (P * v).
static bool StdUnitsFit(const TiledPlan& p, int v, bool tile) {
  if (v <= 0) return false;
  const uint64_t s = static_cast<uint64_t>(p.layout.itemsize);
  const uint64_t ng = (p.H + p.P - 1) / p.P;
  const uint64_t ncv = (p.W * s + static_cast<uint64_t>(v) - 1) / static_cast<uint64_t>(v);
  uint64_t units = 0;
  if (ncv >= static_cast<uint64_t>(kDivLimit) || ng >= static_cast<uint64_t>(kDivLimit) ||
      __builtin_mul_overflow(p.B * ng, ncv, &units) ||
      units >= static_cast<uint64_t>(kU32Limit)) {
    return false;
  }
  if (tile) {
    const uint64_t ncvt = p.tW * s / static_cast<uint64_t>(v);
    const uint64_t tunits = static_cast<uint64_t>(p.tiled_bytes) / (p.P * static_cast<uint64_t>(v));
    if (ncvt >= static_cast<uint64_t>(kDivLimit) || tunits >= static_cast<uint64_t>(kU32Limit)) {
      return false;
    }
  }
  return true;
}

StatusOr<TiledPlan> PlanTiled(const TiledLayout& l) {
  KVX_RETURN_IF_ERROR(ValidateTiledLayout(l));
  TiledPlan p;
  p.layout = l;
  const int64_t s = l.itemsize;
  const int64_t logical = LogicalElements(l);
  if (logical < 0 || !MulOk(logical, s, &p.logical_bytes)) {
    return InvalidArgumentError("tiled layout: size overflows");
  }
  KVX_ASSIGN_OR_RETURN(int64_t phys, TiledBufferElements(l));
  const int r = static_cast<int>(l.dims.size());
  p.tiled = !l.tiles.empty() && r > 0;
  if (!p.tiled) {
    p.tiled_bytes = p.logical_bytes;
    return p;
  }
  if (!MulOk(phys, s, &p.tiled_bytes)) return InvalidArgumentError("tiled layout: size overflows");
  p.padded = phys > logical;
  p.zero_vec = WidestVector(static_cast<uint64_t>(p.tiled_bytes), 16);
  if (logical == 0) return p;

  // Standard form: the reference's IsStandardRowMajorTiled
  // (tiling_utils.cc:56-82) plus this kernel's own limits.
  bool standard = true, column = r >= 2;
  for (int i = 0; i < r; ++i) {
    standard = standard && l.minor_to_major[i] == r - 1 - i;
    // The two minor dimensions swapped, the others row-major.
    column = column && l.minor_to_major[i] == (i == 0 ? r - 2 : i == 1 ? r - 1 : r - 1 - i);
  }
  const bool rows_first = standard;
  standard = standard || column;  // the tiles are the same
  uint32_t P = 1;
  if (l.tiles.size() == 1) {
    standard = standard && l.tiles[0].size() == 2;
  } else if (l.tiles.size() == 2) {
    standard = standard && l.tiles[0].size() == 2 && l.tiles[1].size() == 2 &&
               l.tiles[1][1] == 1 && (l.tiles[1][0] == 2 || l.tiles[1][0] == 4) &&
               l.tiles[0][0] % l.tiles[1][0] == 0;
    if (standard) {
      P = static_cast<uint32_t>(l.tiles[1][0]);
      standard = P * s == 4;
    }
  } else {
    standard = false;
  }
  bool geom = false;
  if (standard) {
    const uint64_t W = static_cast<uint64_t>(l.dims[r - 1]);
    const uint64_t H = r == 1 ? 1 : static_cast<uint64_t>(l.dims[r - 2]);
    const uint64_t B = static_cast<uint64_t>(logical) / (W * H);
    const int64_t tH = l.tiles[0][0], tW = l.tiles[0][1];
    const int64_t BH = static_cast<int64_t>(B * H);
    geom = H < static_cast<uint64_t>(kDivLimit) && W < static_cast<uint64_t>(kDivLimit) &&
           tH <= kDivLimit && tW <= kDivLimit && BH < kU32Limit && tH * tW < kDivLimit;
    p.P = P;
    p.B = B;
    p.H = H;
    p.W = W;
    p.tH = static_cast<uint64_t>(tH);
    p.tW = static_cast<uint64_t>(tW);
    p.nT0 = (H + p.tH - 1) / p.tH;
    p.nT1 = (W + p.tW - 1) / p.tW;
    if (!rows_first) {
      p.nT0 = (W + p.tH - 1) / p.tH;
      p.nT1 = (H + p.tW - 1) / p.tW;
      p.column = geom && ColumnFits(p);
    }
    // Whether the layout's aligned vectors make it standard; a packed layout
    // whose rows are no whole number of 4-byte words is standard too, where
    // the general form could take it.
    p.vec = WidestVector(W * s | static_cast<uint64_t>(tW * s), 16);
    p.standard = rows_first && geom && (P == 1 || p.vec >= 4) && StdUnitsFit(p, p.vec, true);
    if (rows_first && geom && !p.standard) {
      const int v = UnitVector(W, p.tW, s);
      p.ragged = (P == 1 || v >= 4) && StdUnitsFit(p, v, true);
    }
  }

  // General form: the final shape's dimensions.
  std::vector<WorkDim> fin = ApplyTiles(l);
  bool gen_ok = logical < kU32Limit && fin.size() <= static_cast<size_t>(kTiledMaxGenDims);
  for (int64_t d : l.dims) gen_ok = gen_ok && d <= kDivLimit;
  for (const auto& t : l.tiles) {
    for (int64_t d : t) gen_ok = gen_ok && d <= kDivLimit;
  }
  if (gen_ok) {
    int64_t stride = 1;
    p.gen.resize(fin.size());
    for (int k = static_cast<int>(fin.size()) - 1; k >= 0; --k) {
      TiledGenDim g{};
      g.src = fin[k].src;
      g.nops = static_cast<uint32_t>(fin[k].ops.size());
      for (size_t o = 0; o < fin[k].ops.size(); ++o) {
        if (fin[k].ops[o].first) g.is_mod |= 1u << o;
        g.op[o] = MakeFastDivU32(static_cast<uint32_t>(fin[k].ops[o].second));
      }
      g.stride = static_cast<uint64_t>(stride);
      p.gen[k] = g;
      stride *= fin[k].size;
    }
    p.standard = p.standard || p.ragged;
  } else if (!p.standard) {
    // Also a layout that only the ragged or the transposed kernels could take:
    // chunks smaller than their cuts need the general form.
    return UnimplementedError(
        "tiled layout: general layouts need fewer than 2^32 elements, dimensions and tiles "
        "of at most 2^31 and at most 16 tiled dimensions");
  }
  return p;
}

// Jobs of the transposed form over the linear bytes [lo, hi): whole matrices
// in one job, a matrix that the range cuts in one of its own.
static void AppendColumnJobs(const TiledPlan& p, uint64_t tiled, uint64_t linear, int64_t lo,
                             int64_t hi, bool tile, std::vector<TiledJob>* jobs) {
  const uint64_t s = static_cast<uint64_t>(p.layout.itemsize);
  const uint64_t row_bytes = p.W * s;
  uint64_t row = static_cast<uint64_t>(lo) / row_bytes;
  const uint64_t end = static_cast<uint64_t>(hi) / row_bytes;
  while (row < end) {
    const uint64_t b = row / p.H, h = row % p.H;
    uint64_t nb = 1, h_hi = std::min(p.H, h + (end - row));
    if (h == 0 && end - row >= p.H) {
      nb = (end - row) / p.H;
      h_hi = p.H;
    }
    TiledJob j;
    j.dev.tiled = tiled;
    j.dev.linear = linear;
    j.dev.mode = tile ? kTileCol : kDetileCol;
    j.dev.P = p.P;
    j.dev.itemsize = static_cast<uint32_t>(s);
    j.dev.log2s = static_cast<uint32_t>(__builtin_ctz(static_cast<unsigned>(s)));
    j.dev.h32 = static_cast<uint32_t>(p.H);
    j.dev.w32 = static_cast<uint32_t>(p.W);
    j.dev.nt0 = static_cast<uint32_t>(p.nT0);
    j.dev.nt1 = static_cast<uint32_t>(p.nT1);
    j.dev.tile_elems = static_cast<uint32_t>(p.tH * p.tW);
    j.dev.th = MakeFastDivU32(static_cast<uint32_t>(p.tH));
    j.dev.tw = MakeFastDivU32(static_cast<uint32_t>(p.tW));
    j.dev.b0 = static_cast<uint32_t>(b);
    j.dev.c_lo = static_cast<uint32_t>(h);
    j.dev.c_hi = static_cast<uint32_t>(h_hi);
    const uint64_t c_end = tile && h_hi == p.H ? p.nT1 * p.tW : h_hi;
    j.dev.c_end = static_cast<uint32_t>(c_end);
    const uint64_t along = tile ? ColumnRegionsAlong(p)
                                : (row_bytes + kColBytes - 1) / kColBytes;
    const uint64_t across = ColumnRegionsAcross(c_end - h);
    j.dev.ng = MakeFastDivU32(static_cast<uint32_t>(along));
    j.dev.ncv = MakeFastDivU32(static_cast<uint32_t>(across));
    j.dev.count = nb * along * across;
    j.bytes = static_cast<int64_t>(nb * (h_hi - h) * row_bytes);
    jobs->push_back(std::move(j));
    row += nb * (h_hi - h);
  }
}

Status AppendTiledJobs(const TiledPlan& p, uint64_t tiled, uint64_t linear, int64_t lo,
                       int64_t hi, bool tile, bool zero_pass, std::vector<TiledJob>* zero,
                       std::vector<TiledJob>* jobs) {
  if (!p.tiled || lo >= hi) return OkStatus();
  if (lo < 0 || hi > p.logical_bytes || p.CutAtOrBelow(lo) != lo ||
      p.CutAtOrBelow(hi) != hi) {
    return InvalidArgumentError("tiled copy range does not start and end on a tile row");
  }
  if (tiled == 0) return InvalidArgumentError("tiled copy: null tiled buffer");
  const int64_t s = p.layout.itemsize;
  // Both forms address whole elements: a buffer that is not aligned to the
  // element size would give the vector form fewer bytes per vector than one
  // element (no element per vector at all).
  if (((tiled | linear) & static_cast<uint64_t>(s - 1)) != 0) {
    return InvalidArgumentError("tiled copy: buffers not aligned to the element size");
  }
  // Packed units: one lane per unit with units of one 16-byte tiled vector
  // (v = 16 / P), except that detiling at 16-byte rows goes two lanes per
  // unit for pairs (P = 2) and four for quads (P = 4), exchanging through
  // LDS so that each wave writes 1 KiB of one row per store. Measured on the
  // Llama-3-8B set (bf16, P = 2), one process, one launch each: tiling
  // 79.2 % of HBM peak at v = 8 against 76.7 % with two lanes per 16-byte
  // unit and 67.8 % with one lane per 16-byte unit (each 16-byte tiled store
  // of a wave then leaves 16-byte holes); detiling 77.0 % with two lanes
  // (exchanging within the lane pair) against 75.7 % at v = 8, and 79.6
  // against 78.4 % for the LDS exchange over the lane-pair one. For int8
  // (P = 4) at 16-byte rows, detiling: 71.6 % through LDS against 61.8 % for
  // one lane per 16-byte tiled vector; tiling keeps one lane per tiled
  // vector (72.3 % against 67.0 % through LDS).
  auto packed = [&](int width) {
    if (p.P == 1 || (!tile && width == 16)) return width;
    return std::min(width, 16 / static_cast<int>(p.P));
  };
  const int v = p.standard ? packed(UnitVector(p.W, p.tW, static_cast<uint64_t>(s))) : 1;
  const bool lanes = p.P > 1 && !tile && v == 16;
  // The kernels index units in 32 bits. A tensor too large for the general
  // form is taken only where its units would fit at aligned vectors of its
  // buffers as well, so that whether a call is accepted does not depend on
  // which vectors move it. What passes here without a standard form has a
  // general one (PlanTiled).
  const bool use_std = p.standard && StdUnitsFit(p, v, tile);
  const int aligned = packed(WidestVector(tiled | linear, p.vec));
  if (p.standard && p.gen.empty() &&
      (!use_std || (p.P > 1 && aligned < 4) || !StdUnitsFit(p, aligned, tile))) {
    return UnimplementedError(
        "tiled copy: this layout has more 32-bit-indexed units than one launch can address "
        "at the buffers' alignment");
  }
  // Standard-form and transposed units write the padding themselves; otherwise it is cleared
  // first.
  if (tile && zero_pass && p.padded && !use_std && !p.column) {
    const int v = WidestVector(tiled, p.zero_vec);
    TiledJob z;
    z.vec = v;
    z.dev.mode = kZero;
    z.dev.tiled = tiled;
    z.dev.lo = 0;
    z.dev.count = static_cast<uint64_t>(p.tiled_bytes / v);
    z.dev.itemsize = static_cast<uint32_t>(s);
    z.dev.P = 1;
    zero->push_back(z);
  }
  if (p.column) {
    AppendColumnJobs(p, tiled, linear, lo, hi, tile, jobs);
    return OkStatus();
  }
  TiledJob j;
  j.dev.tiled = tiled;
  j.dev.linear = linear;
  j.dev.itemsize = static_cast<uint32_t>(s);
  if (use_std) {
    const uint64_t row_bytes = p.W * s;
    const uint64_t ng = (p.H + p.P - 1) / p.P;
    const uint64_t ncv = (row_bytes + v - 1) / v;
    auto group = [&](int64_t x) -> uint64_t {
      if (x >= p.logical_bytes) return p.B * ng;
      const uint64_t row = static_cast<uint64_t>(x) / row_bytes;
      return row / p.H * ng + row % p.H / p.P;
    };
    j.vec = v;
    j.dev.mode = tile ? kTileStd : kDetileStd;
    j.dev.lanes_per_unit = lanes ? p.P : 1;
    j.dev.sliced = lanes ? 1u : 0u;
    if (tile) {
      // Whole tile rows (cuts fall on them): units of tile rows [t_lo, t_hi).
      auto tile_row = [&](int64_t x) -> uint64_t {
        if (x >= p.logical_bytes) return p.B * p.nT0;
        const uint64_t row = static_cast<uint64_t>(x) / row_bytes;
        return row / p.H * p.nT0 + row % p.H / p.tH;
      };
      const uint64_t gpt = p.tH / p.P;
      const uint64_t ncvt = p.tW * s / v;
      const uint64_t per_tile_row = p.nT1 * gpt * ncvt;
      const uint64_t t_lo = tile_row(lo), t_hi = tile_row(hi);
      j.dev.lo = t_lo * per_tile_row;
      j.dev.count = (t_hi - t_lo) * per_tile_row;
      j.dev.t_ncv = MakeFastDivU32(static_cast<uint32_t>(ncvt));
      j.dev.t_gpt = MakeFastDivU32(static_cast<uint32_t>(gpt));
      j.dev.t_nt1 = MakeFastDivU32(static_cast<uint32_t>(p.nT1));
      j.dev.t_nt0 = MakeFastDivU32(static_cast<uint32_t>(p.nT0));
    } else {
      const uint64_t g_lo = group(lo), g_hi = group(hi);
      j.dev.lo = g_lo * ncv;
      j.dev.count = (g_hi - g_lo) * ncv;
    }
    j.dev.P = p.P;
    j.dev.ncv = MakeFastDivU32(static_cast<uint32_t>(ncv));
    j.dev.ng = MakeFastDivU32(static_cast<uint32_t>(ng));
    j.dev.th = MakeFastDivU32(static_cast<uint32_t>(p.tH));
    j.dev.tw = MakeFastDivU32(static_cast<uint32_t>(p.tW));
    j.dev.h32 = static_cast<uint32_t>(p.H);
    j.dev.w32 = static_cast<uint32_t>(p.W);
    j.dev.nt0 = static_cast<uint32_t>(p.nT0);
    j.dev.nt1 = static_cast<uint32_t>(p.nT1);
    j.dev.tile_elems = static_cast<uint32_t>(p.tH * p.tW);
    j.dev.log2s = static_cast<uint32_t>(__builtin_ctz(static_cast<unsigned>(s)));
  } else {
    j.vec = 0;
    j.dev.mode = tile ? kTileGen : kDetileGen;
    j.dev.lo = static_cast<uint64_t>(lo / s);
    j.dev.count = static_cast<uint64_t>((hi - lo) / s);
    j.dev.P = 1;
    j.dev.rank = static_cast<uint32_t>(p.layout.dims.size());
    for (size_t r = 0; r < p.layout.dims.size(); ++r) {
      j.dev.dims[r] = MakeFastDivU32(static_cast<uint32_t>(p.layout.dims[r]));
    }
    j.dev.ngen = static_cast<uint32_t>(p.gen.size());
    j.gen = p.gen;
  }
  j.bytes = static_cast<int64_t>(j.dev.count) *
            (use_std ? static_cast<int64_t>(p.P) * j.vec : static_cast<int64_t>(s));
  if (j.dev.count > 0) jobs->push_back(std::move(j));
  return OkStatus();
}

Status LaunchTiledThroughRing(ArgRing& ring, const std::vector<TiledJob>& jobs,
                              hipStream_t stream, hipEvent_t kernel_start) {
  if (jobs.empty()) return OkStatus();
  // One launch per kernel (vector width, rows per unit, direction, unit
  // order; element size for the general form), in order of first
  // appearance. General jobs take any vector width.
  std::vector<TiledLaunchKey> keys;
  std::vector<TiledLaunchKey> job_key(jobs.size());
  for (size_t i = 0; i < jobs.size(); ++i) {
    job_key[i] = LaunchKeyOf(jobs[i].dev, jobs[i].vec);
    if (std::find(keys.begin(), keys.end(), job_key[i]) == keys.end()) {
      keys.push_back(job_key[i]);
    }
  }
  bool started = false;
  for (const TiledLaunchKey& key : keys) {
    std::vector<const TiledJob*> mine;
    for (size_t i = 0; i < jobs.size(); ++i) {
      if (job_key[i] == key) mine.push_back(&jobs[i]);
    }
    const uint64_t per = TiledPerWorkgroup(key);
    const int64_t head = static_cast<int64_t>(mine.size() * sizeof(TiledJobDev));
    int64_t gen_bytes = 0;
    uint64_t grid = 0;
    for (const TiledJob* j : mine) {
      gen_bytes += static_cast<int64_t>(j->gen.size() * sizeof(TiledGenDim));
      grid += (j->dev.count + per - 1) / per;
    }
    if (grid >= (uint64_t{1} << 31)) return InvalidArgumentError("tiled copy too large for one launch");
    if (mine.size() == 1 && gen_bytes == 0) {
      // One job travels in the kernel's arguments: no upload (a copy kernel and
      // a gap: a [14336, 4096] bf16 detile took 52.6 us a call, 43.3 without).
      if (kernel_start != nullptr && !started) {
        KVX_HIP_RETURN_IF_ERROR(hipEventRecord(kernel_start, stream));
      }
      started = true;
      KVX_HIP_RETURN_IF_ERROR(LaunchTiledCopy(nullptr, 0, &mine[0]->dev,
                                              static_cast<uint32_t>(grid), key, stream));
      continue;
    }
    const int64_t map_off = head + gen_bytes;
    const int64_t bytes = map_off + static_cast<int64_t>(grid) * 4;
    KVX_ASSIGN_OR_RETURN(int64_t off, ring.Alloc(bytes));
    ArgSliceGuard keep([&ring, off, bytes, stream] { return ring.Commit(off, bytes, stream); },
                       stream);
    uint8_t* img = ring.host(off);
    uint32_t* map = reinterpret_cast<uint32_t*>(img + map_off);
    int64_t gen_at = head;
    uint32_t wg = 0;
    for (size_t i = 0; i < mine.size(); ++i) {
      TiledJobDev d = mine[i]->dev;
      d.wg_begin = wg;
      if (!mine[i]->gen.empty()) {
        d.gen_offset = static_cast<uint32_t>(gen_at);
        const size_t gb = mine[i]->gen.size() * sizeof(TiledGenDim);
        std::memcpy(img + gen_at, mine[i]->gen.data(), gb);
        gen_at += static_cast<int64_t>(gb);
      }
      std::memcpy(img + i * sizeof(TiledJobDev), &d, sizeof(d));
      const uint32_t n = static_cast<uint32_t>((d.count + per - 1) / per);
      for (uint32_t k = 0; k < n; ++k) map[wg + k] = static_cast<uint32_t>(i);
      wg += n;
    }
    KVX_RETURN_IF_ERROR(ring.Upload(off, bytes, stream));
    if (kernel_start != nullptr && !started) {
      KVX_HIP_RETURN_IF_ERROR(hipEventRecord(kernel_start, stream));
    }
    started = true;
    KVX_HIP_RETURN_IF_ERROR(LaunchTiledCopy(reinterpret_cast<const void*>(ring.dev(off)),
                                            static_cast<uint32_t>(map_off), nullptr,
                                            static_cast<uint32_t>(grid), key, stream));
    KVX_RETURN_IF_ERROR(keep.Commit());
  }
  return OkStatus();
}

}  // namespace kvx
