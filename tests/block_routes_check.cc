// Host-side checks of the block copy's dispatch (BlockCopyRouteOf in libkvx)
// on the CPU, no device calls: which kernel a launch runs and how much LDS it
// reserves, on both sides of every line of the rule. Two of its lines guard
// against losses: a scatter to ids spread over a pool keeps every storage in
// flight (storage by storage it is up to a fifth slower on some allocations), and
// scatters of whole blocks reserve no LDS (with a scale table beside them up to
// 18 % slower, and LDS-heavy kernels of other streams kept off the CUs).
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

  const uint32_t one_side = kLds - kTables;

  // One block size: 512 ids of 64 storages of 32 KiB, and under 160 MiB.
  Expect("512 x 64 x 32 KiB gather", Make(512, {{64, 32768}}), G, sliced, two_side);
  Expect("512 x 64 x 32 KiB scatter", Make(512, {{64, 32768}}), S, sliced, one_side);
  Expect("80 x 64 x 32 KiB gather, 160 MiB", Make(80, {{64, 32768}}), G, sliced, two_side);
  Expect("79 x 64 x 32 KiB gather", Make(79, {{64, 32768}}), G, fast, two);
  Expect("79 x 64 x 32 KiB scatter", Make(79, {{64, 32768}}), S, fast, 0);
  Expect("64 x 64 x 16 KiB scatter", Make(64, {{64, 16384}}), S, fast, 0);
  Expect("1 x 64 x 32 KiB gather", Make(1, {{64, 32768}}), G, fast, two);
  // A chunk of whole storages, the first of them not storage 0; and one that
  // starts inside a storage.
  CopyLaunch chunk = Make(63, {{84, 32768}});
  chunk.pieces[0].f0 = 84 * 63;
  Expect("storages 84 to 167 of 63 ids, gather", chunk, G, sliced, two_side);
  Expect("storages 84 to 167 of 63 ids, scatter", chunk, S, sliced, one_side);
  chunk.pieces[0].f0 += 1;
  Expect("the same one id further, gather", chunk, G, fast, two);

  // Scatters of 512 MiB: ids spread over the pool, unknown ids of a large pool, ids
  // that fill two fifths of their range, unknown ids of a pool that small.
  struct Size { int64_t block; const char* spread; uint32_t spread_lds; const char* dense; };
  const Size sizes[] = {{2048, sliced, two_side, sliced},   {3072, sliced, two_side, sliced},
                        {4096, sliced, one_side, sliced},   {6144, general, two_side, sliced},
                        {7000, general, two_side, general}, {7168, general, two_side, sliced},
                        {8192, sliced, one_side, sliced},   {9216, fast, 0, sliced},
                        {10000, fast, 0, general},          {12288, fast, 0, sliced},
                        {16384, sliced, one_side, sliced},  {24576, fast, 0, sliced},
                        {32768, sliced, one_side, sliced},  {33 << 10, fast, 0, sliced},
                        {20000, fast, 0, fast},             {65536, fast, 0, sliced},
                        {1 << 20, fast, 0, sliced},         {1025 << 10, fast, 0, fast}};
  for (const Size& z : sizes) {
    const int64_t W = z.block < 65536 ? 64 : 8, n = (int64_t{512} << 20) / (W * z.block);
    const std::string name = std::to_string(z.block) + "-byte blocks scattered";
    const uint32_t dense_lds = z.dense == fast ? 0 : two_side;
    CopyLaunch l = Make(n, {{W, z.block}});
    l.id_span = n * 5 / 2 + 5;
    Expect((name + " over more than 5 n / 2").c_str(), l, S, z.spread, z.spread_lds);
    l.id_span = 0;
    Expect((name + ", unknown ids").c_str(), l, S, z.spread, z.spread_lds);
    l.id_span = n * 5 / 2;
    Expect((name + " over 5 n / 2").c_str(), l, S, z.dense, dense_lds);
    l.id_span = 0;
    l.pieces[0].pool_blocks = n * 5 / 2;
    Expect((name + ", a small pool").c_str(), l, S, z.dense, dense_lds);
  }
  // Dense ids in the cache go like any others.
  for (int64_t block : {8192, 10000, 12288, 16384, 32768}) {
    CopyLaunch l = Make((int64_t{159} << 20) / (64 * block), {{64, block}});
    l.id_span = l.n;
    Expect(("159 MiB of " + std::to_string(block) + ", dense").c_str(), l, S, fast, 0);
  }

  // Packed: from 2048 workgroups on, both directions.
  Expect("409 x 160 x 2 KiB scatter", Make(409, {{160, 2048}}), S, general, two_side);
  Expect("409 x 160 x 2 KiB gather", Make(409, {{160, 2048}}), G, general, two_side);
  Expect("16 x 160 x 2 KiB scatter", Make(16, {{160, 2048}}), S, general, 0);
  Expect("16 x 160 x 2 KiB gather", Make(16, {{160, 2048}}), G, general, 0);
  // Where packed blocks end: 8 KiB scattered, 16 KiB gathered.
  Expect("100 x 64 x 8191 scatter", Make(100, {{64, 8191}}), S, general, 0);
  Expect("100 x 64 x 8192 scatter", Make(100, {{64, 8192}}), S, fast, 0);
  Expect("100 x 64 x 16383 gather", Make(100, {{64, 16383}}), G, general, two_side);
  Expect("100 x 64 x 16384 gather", Make(100, {{64, 16384}}), G, fast, two);
  // A scale table beside whole blocks: gathers from 2048 workgroups on, scatters
  // never.
  Expect("64 x (64 x 16 KiB + 32) gather", Make(64, {{64, 16384}, {32, 32}}), G, side, two_side);
  Expect("31 x (64 x 16 KiB + 32) gather", Make(31, {{64, 16384}, {32, 32}}), G, side, 0);
  for (int64_t block : {8192, 10000, 12288, 16384, 17408, 20000, 24576, 32768, 66000}) {
    const int64_t n = (int64_t{150} << 20) / (64 * block);
    const std::string name = "150 MiB of " + std::to_string(block) + " + 4 scattered";
    Expect(name.c_str(), Make(n, {{64, block}, {32, 4}}), S, side, 0);
  }
  Expect("245 x (64 x 20000 + 4) scatter", Make(245, {{64, 20000}, {32, 4}}), S, side, 0);
  Expect("512 x (64 x 16 KiB + 32) scatter", Make(512, {{64, 16384}, {32, 32}}), S, sliced,
         one_side);
  // Several sizes.
  Expect("200 x (32 x 32 KiB + 32 x 16 KiB) scatter", Make(200, {{32, 32768}, {32, 16384}}), S,
         general, 0);
  Expect("200 x (32 x 32 KiB + 32 x 16 KiB) gather", Make(200, {{32, 32768}, {32, 16384}}), G,
         general, two_side);
  Expect("400 x (64 x 4000 + 64 x 2000) scatter", Make(400, {{64, 4000}, {64, 2000}}), S, general,
         two_side);
  // No limit, another limit, and the capped grids of zero-copy copies.
  for (const auto& pieces : {std::vector<std::pair<int64_t, int64_t>>{{64, 32768}},
                             std::vector<std::pair<int64_t, int64_t>>{{64, 16384}, {32, 32}}}) {
    for (CopyDir dir : {G, S}) {
      CopyLaunch l = Make(512, pieces);
      l.gather_workgroups_per_cu = 0;
      Expect("no limit", l, dir, sliced, 0);
      l.gather_workgroups_per_cu = 4;
      // (Scatters that keep every storage in flight: half as many.)
      Expect("4 workgroups a CU", l, dir, sliced, kLds / (dir == S ? 2 : 4) - kTables);
      l.gather_workgroups_per_cu = 1;
      Expect("1 workgroup a CU", l, dir, sliced, kLds - kTables);
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
  // The benchmark's isolated launches: 512 ids of 64 storages of 16384 blocks of
  // 32 KiB, random and out of one run.
  for (const char* name : {"gather", "scatter", "scatter_contiguous", "scatter_shuffled"}) {
    CopyLaunch l = Make(512, {{64, 32768}});
    l.pieces[0].pool_blocks = 16384;
    l.id_span = std::strlen(name) > 7 ? 512 : 16000;
    if (kvx::BlockCopyRouteOf(l, name[0] == 'g' ? G : S, 16, &r)) {
      std::printf("benchmark %s: %s, %u KiB\n", name, r.kernel, r.piece_kib);
    }
  }
  if (failures == 0) std::printf("block routes: all checks passed\n");
  return failures == 0 ? 0 : 1;
}
