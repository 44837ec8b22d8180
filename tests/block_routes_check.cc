// Host-side checks of the block copy's dispatch (BlockCopyRouteOf in libkvx)
// on the CPU, no device calls: which kernel a launch runs and how much LDS it
// reserves, on both sides of every line of the rule. A copy that reserves LDS
// keeps LDS-heavy kernels of other streams off its CUs, so the scatters that
// gain nothing from it (blocks above 16 KiB beside others, under 160 MiB) must
// not.
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <string>
#include <utility>
#include <vector>

#include "block_copy.h"

using kvx::BlockCopyRoute;
using kvx::CopyDir;
using kvx::CopyLaunch;

namespace {

int failures = 0;

constexpr uint32_t kLds = 160u << 10;
constexpr uint32_t kTables = 4096;  // LDS the packed path declares itself

// One launch over whole storages: (storages, block bytes) of each piece.
CopyLaunch Make(int64_t n, const std::vector<std::pair<int64_t, int64_t>>& pieces) {
  static const int64_t ids = 0;  // never read
  CopyLaunch l;
  l.ids = &ids;
  l.n = n;
  uint64_t staging = uint64_t{1} << 40;
  for (const auto& p : pieces) {
    kvx::CopyPiece& c = l.pieces[l.npieces++];
    c.storages = uint64_t{1} << 30;
    c.staging = staging;
    c.stride_w = n * p.second;
    c.stride_i = p.second;
    c.nblocks = p.first * n;
    c.block_bytes = p.second;
    c.pool_blocks = 1 << 20;
    staging += static_cast<uint64_t>(p.first * n * p.second);
  }
  return l;
}

void Expect(const char* what, const CopyLaunch& l, CopyDir dir, const char* kernel, uint32_t lds) {
  BlockCopyRoute r;
  const bool ok = kvx::BlockCopyRouteOf(l, dir, kvx::LaunchVectorBytes(l, 0), &r);
  if (!ok || std::strcmp(r.kernel, kernel) != 0 || r.lds_bytes != lds) {
    std::printf("FAIL: %s: %s, %llu workgroups, %u bytes of LDS; expected %s, %u\n", what,
                ok ? r.kernel : "refused", static_cast<unsigned long long>(ok ? r.workgroups : 0),
                ok ? r.lds_bytes : 0, kernel, lds);
    ++failures;
  }
}

}  // namespace

int main() {
  const char* general = "block_copy_kernel";
  const char* fast = "block_copy_fast_kernel";
  const char* side = "block_copy_fast_side_kernel";
  const char* sliced = "block_copy_sliced_kernel";
  const uint32_t two = kLds / 2, two_side = kLds / 2 - kTables;
  const CopyDir G = CopyDir::kGather, S = CopyDir::kScatter;

  // One block size: 512 ids of 64 storages of 32 KiB, and under 160 MiB.
  Expect("512 x 64 x 32 KiB gather", Make(512, {{64, 32768}}), G, sliced, two_side);
  Expect("512 x 64 x 32 KiB scatter", Make(512, {{64, 32768}}), S, sliced, two_side);
  Expect("80 x 64 x 32 KiB gather, 160 MiB", Make(80, {{64, 32768}}), G, sliced, two_side);
  Expect("79 x 64 x 32 KiB gather", Make(79, {{64, 32768}}), G, fast, two);
  Expect("79 x 64 x 32 KiB scatter", Make(79, {{64, 32768}}), S, fast, 0);
  // A chunk of whole storages, the first of them not storage 0; and one that
  // starts inside a storage.
  CopyLaunch chunk = Make(63, {{84, 32768}});
  chunk.pieces[0].f0 = 84 * 63;
  Expect("storages 84 to 167 of 63 ids, gather", chunk, G, sliced, two_side);
  Expect("storages 84 to 167 of 63 ids, scatter", chunk, S, sliced, two_side);
  chunk.pieces[0].f0 += 1;
  Expect("the same one id further, gather", chunk, G, fast, two);
  Expect("512 x 64 x 20000 scatter", Make(512, {{64, 20000}}), S, fast, 0);
  Expect("64 x 64 x 16 KiB scatter", Make(64, {{64, 16384}}), S, fast, 0);
  Expect("1 x 64 x 32 KiB gather", Make(1, {{64, 32768}}), G, fast, two);
  // Packed: from 2048 workgroups on, both directions.
  Expect("409 x 160 x 2 KiB scatter", Make(409, {{160, 2048}}), S, general, two_side);
  Expect("409 x 160 x 2 KiB gather", Make(409, {{160, 2048}}), G, general, two_side);
  Expect("16 x 160 x 2 KiB scatter", Make(16, {{160, 2048}}), S, general, 0);
  Expect("16 x 160 x 2 KiB gather", Make(16, {{160, 2048}}), G, general, 0);
  // A scale table beside whole blocks: scatters of at most 16 KiB ...
  Expect("64 x (64 x 16 KiB + 32) scatter", Make(64, {{64, 16384}, {32, 32}}), S, side, two_side);
  Expect("31 x (64 x 16 KiB + 32) scatter", Make(31, {{64, 16384}, {32, 32}}), S, side, 0);
  Expect("64 x (64 x 16 KiB + 32) gather", Make(64, {{64, 16384}, {32, 32}}), G, side, two_side);
  // ... or of 160 MiB and more.
  for (int64_t block : {int64_t{16385}, int64_t{17408}, int64_t{20000}, int64_t{20480},
                        int64_t{24576}, int64_t{32768}, int64_t{66000}}) {
    const int64_t n = (int64_t{150} << 20) / (64 * block);
    const std::string name = "150 MiB of " + std::to_string(block) + " + 4";
    Expect((name + " scatter").c_str(), Make(n, {{64, block}, {32, 4}}), S, side, 0);
    Expect((name + " gather").c_str(), Make(n, {{64, block}, {32, 4}}), G, side, two_side);
  }
  Expect("245 x (64 x 20000 + 4) scatter", Make(245, {{64, 20000}, {32, 4}}), S, side, two_side);
  // Several sizes of whole blocks.
  Expect("53 x (32 x 32 KiB + 32 x 16 KiB) scatter", Make(53, {{32, 32768}, {32, 16384}}), S,
         general, 0);
  Expect("200 x (32 x 32 KiB + 32 x 16 KiB) scatter", Make(200, {{32, 32768}, {32, 16384}}), S,
         general, two_side);
  Expect("53 x (32 x 32 KiB + 32 x 16 KiB) gather", Make(53, {{32, 32768}, {32, 16384}}), G,
         general, two_side);
  // No limit, another limit, and the capped grids of zero-copy copies.
  for (const auto& pieces : {std::vector<std::pair<int64_t, int64_t>>{{64, 32768}},
                             std::vector<std::pair<int64_t, int64_t>>{{64, 16384}, {32, 32}}}) {
    for (CopyDir dir : {G, S}) {
      CopyLaunch l = Make(512, pieces);
      l.gather_workgroups_per_cu = 0;
      Expect("no limit", l, dir, sliced, 0);
      l.gather_workgroups_per_cu = 4;
      Expect("4 workgroups a CU", l, dir, sliced, kLds / 4 - kTables);
    }
  }
  CopyLaunch z = Make(512, {{64, 2048}, {32, 4}});
  z.max_workgroups = 64;
  Expect("capped grid", z, S, general, 0);
  // A launch that is refused has no route.
  CopyLaunch bad = Make(4, {{2, 64}});
  bad.pieces[0].pool_blocks = 0;
  BlockCopyRoute r;
  if (kvx::BlockCopyRouteOf(bad, G, 16, &r)) {
    std::printf("FAIL: a refused launch has a route\n");
    ++failures;
  }
  if (failures == 0) std::printf("block routes: all checks passed\n");
  return failures == 0 ? 0 : 1;
}
