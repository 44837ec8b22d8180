// Host-side checks of the tiled-copy job builder (PlanTiled /
// AppendTiledJobs in libkvx) on the CPU, no device calls:
//   * buffers not aligned to the element size are rejected for every form
//     (the vector form would otherwise get fewer bytes per vector than one
//     element);
//   * the 32-bit unit limits: a tensor too large for the general form is taken
//     where its units fit both at the width that moves it (16-byte vectors at
//     any address) and at the one its buffers' alignment allows, so that an 8
//     GiB tensor at a 1-byte offset stays refused;
//   * matrices of odd widths and column-major ones: their form, vector width
//     and number of units or regions on both sides of each line.
#include <cstdint>
#include <cstdio>
#include <vector>

#include "tiled_layout.h"

using kvx::Code;
using kvx::TiledJob;
using kvx::TiledLayout;

namespace {

int failures = 0;

void expect(bool ok, const char* what) {
  if (!ok) {
    std::printf("FAIL: %s\n", what);
    ++failures;
  }
}

TiledLayout Layout(int s, std::vector<int64_t> dims, std::vector<std::vector<int64_t>> tiles,
                   std::vector<int> mtm = {}) {
  TiledLayout l;
  l.itemsize = s;
  l.dims = dims;
  if (mtm.empty()) {
    for (int i = static_cast<int>(dims.size()) - 1; i >= 0; --i) mtm.push_back(i);
  }
  l.minor_to_major = mtm;
  l.tiles = tiles;
  return l;
}

// Builds the jobs of the whole tensor in one direction; returns the status
// code and checks that every vector job's units fit 32-bit indices.
Code Jobs(const kvx::TiledPlan& p, uint64_t tiled, uint64_t linear, bool tile,
          std::vector<TiledJob>* out = nullptr) {
  std::vector<TiledJob> zero, jobs;
  kvx::Status st = kvx::AppendTiledJobs(p, tiled, linear, 0, p.logical_bytes, tile,
                                        /*zero_pass=*/true, &zero, &jobs);
  for (const TiledJob& j : jobs) {
    if (j.vec != 0) {
      expect(j.dev.lo + j.dev.count <= (uint64_t{1} << 32), "vector job units fit 32 bits");
    }
  }
  if (out != nullptr) *out = jobs;
  return st.code();
}

}  // namespace

int main() {
  const uint64_t base = uint64_t{1} << 20;
  // Element-size alignment, both directions, both buffers.
  {
    auto p = kvx::PlanTiled(Layout(2, {40, 384}, {{8, 128}, {2, 1}}));
    expect(p.ok() && p->standard, "bf16 T(8,128)(2,1) plans as standard");
    for (bool tile : {true, false}) {
      expect(Jobs(*p, base, base + 1, tile) == Code::kInvalidArgument, "bf16 linear +1 refused");
      expect(Jobs(*p, base + 1, base, tile) == Code::kInvalidArgument, "bf16 tiled +1 refused");
      expect(Jobs(*p, base, base + 2, tile) == Code::kOk, "bf16 linear +2 accepted");
      expect(Jobs(*p, base + 8, base, tile) == Code::kOk, "bf16 tiled +8 accepted");
    }
  }
  {
    auto p = kvx::PlanTiled(Layout(4, {3, 20, 200}, {{8, 128}}));
    expect(p.ok() && p->standard, "f32 T(8,128) plans as standard");
    for (bool tile : {true, false}) {
      expect(Jobs(*p, base, base + 2, tile) == Code::kInvalidArgument, "f32 linear +2 refused");
      expect(Jobs(*p, base + 6, base, tile) == Code::kInvalidArgument, "f32 tiled +6 refused");
      std::vector<TiledJob> jobs;
      expect(Jobs(*p, base + 4, base, tile, &jobs) == Code::kOk, "f32 tiled +4 accepted");
      for (const TiledJob& j : jobs) expect(j.vec == 0 || j.vec >= 4, "f32 vector >= element");
    }
  }
  {
    auto p = kvx::PlanTiled(Layout(1, {40, 384}, {{8, 128}, {4, 1}}));
    expect(p.ok() && p->standard, "int8 T(8,128)(4,1) plans as standard");
    for (bool tile : {true, false}) {
      expect(Jobs(*p, base + 1, base + 3, tile) == Code::kOk, "int8 any byte offset accepted");
    }
  }
  {
    auto p = kvx::PlanTiled(Layout(2, {6, 40, 24}, {{8, 8}}, {0, 2, 1}));
    expect(p.ok() && !p->standard, "permuted bf16 plans as general");
    expect(Jobs(*p, base, base + 1, true) == Code::kInvalidArgument, "general linear +1 refused");
    expect(Jobs(*p, base + 4, base + 2, false) == Code::kOk, "general +4/+2 accepted");
  }
  // 32-bit unit limits: 8 GiB of int8 in T(8,128) has 2^29 units of 16 bytes
  // but 2^33 of one byte, and more than 2^32 elements, so the
  // element-by-element form cannot take it either.
  {
    auto p = kvx::PlanTiled(Layout(1, {65536, 131072}, {{8, 128}}));
    expect(p.ok() && p->standard && p->gen.empty(), "8 GiB int8 plans as standard only");
    for (bool tile : {true, false}) {
      std::vector<TiledJob> jobs;
      expect(Jobs(*p, base, base, tile, &jobs) == Code::kOk, "8 GiB int8, aligned buffers");
      expect(!jobs.empty() && jobs[0].vec == 16, "8 GiB int8 moves 16-byte vectors");
      expect(Jobs(*p, base, base + 4, tile, &jobs) == Code::kOk, "8 GiB int8, 4-byte aligned");
      expect(!jobs.empty() && jobs[0].vec == 16, "8 GiB int8 at 4 bytes: 16-byte vectors");
      expect(Jobs(*p, base, base + 1, tile) == Code::kUnimplemented,
             "8 GiB int8 one byte off refused (2^33 units of 1 byte)");
      expect(Jobs(*p, base + 2, base, tile) == Code::kUnimplemented,
             "8 GiB int8 two bytes off refused (2^32 units of 2 bytes)");
    }
  }
  // Odd widths: whole vectors of the tile's rows, a row's last one partial.
  {
    auto p = kvx::PlanTiled(Layout(2, {4096, 32003}, {{8, 128}, {2, 1}}));
    expect(p.ok() && p->standard && p->ragged && !p->column, "bf16 [4096, 32003] is ragged");
    std::vector<TiledJob> jobs;
    expect(Jobs(*p, base, base + 2, true, &jobs) == Code::kOk && jobs.size() == 1, "ragged tile");
    expect(jobs[0].vec == 8 && jobs[0].dev.count == uint64_t{512} * 251 * 4 * 32,
           "ragged tile: 8-byte units of every tile");
    expect(Jobs(*p, base, base + 2, false, &jobs) == Code::kOk && jobs.size() == 1,
           "ragged detile");
    expect(jobs[0].vec == 16 && jobs[0].dev.count == uint64_t{2048} * 4001,
           "ragged detile: 16-byte units of two rows, the last of a row partial");
  }
  // Their unit limit: [1, W] of int8 in T(8,2) has 4 W + 4 units of 2 bytes.
  {
    auto p = kvx::PlanTiled(Layout(1, {1, (1 << 29) + 1}, {{8, 2}}));
    expect(p.ok() && p->ragged && p->standard, "2^31 ragged units fit");
    std::vector<TiledJob> jobs;
    expect(Jobs(*p, base, base, true, &jobs) == Code::kOk && jobs.size() == 1 &&
               jobs[0].vec == 2 && jobs[0].dev.count == (uint64_t{1} << 31) + 8,
           "2^31 ragged units in one job");
    p = kvx::PlanTiled(Layout(1, {1, (1 << 30) + 1}, {{8, 2}}));
    expect(p.ok() && !p->ragged && !p->standard && !p->gen.empty(),
           "2^32 ragged units go element by element");
    expect(Jobs(*p, base, base, true, &jobs) == Code::kOk && jobs.size() == 1 &&
               jobs[0].vec == 0 && jobs[0].dev.count == (uint64_t{1} << 30) + 1,
           "2^32 ragged units: one job of elements");
  }
  // Column-major matrices: regions of 128 rows x 256 bytes.
  {
    auto p = kvx::PlanTiled(Layout(2, {4096, 14337}, {{8, 128}, {2, 1}}, {0, 1}));
    expect(p.ok() && p->column && !p->standard && !p->gen.empty(), "column-major bf16");
    std::vector<TiledJob> jobs;
    expect(Jobs(*p, base, base, false, &jobs) == Code::kOk && jobs.size() == 1 &&
               jobs[0].dev.count == uint64_t{113} * 32,
           "column-major detile: every region with data");
    p = kvx::PlanTiled(Layout(2, {3, 130, 200}, {{8, 128}, {2, 1}}, {1, 2, 0}));
    expect(p.ok() && p->column, "column-major batch");
    expect(Jobs(*p, base, base, false, &jobs) == Code::kOk && jobs.size() == 1 &&
               jobs[0].dev.count == uint64_t{3} * 2 * 2 && jobs[0].dev.c_end == 130,
           "column-major batch: data only");
    expect(Jobs(*p, base, base, true, &jobs) == Code::kOk && jobs.size() == 1 &&
               jobs[0].dev.count == uint64_t{3} * 2 * 2 && jobs[0].dev.c_end == 256,
           "column-major batch: its padding too");
    // Rows [128, 130) of the first matrix and [0, 128) of the second.
    std::vector<TiledJob> zero;
    jobs.clear();
    const int64_t row = 400;
    expect(kvx::AppendTiledJobs(*p, base, base, 128 * row, 258 * row, true, true, &zero, &jobs)
                   .code() == Code::kOk && zero.empty() && jobs.size() == 2,
           "a cut inside two matrices is two jobs");
    expect(jobs[0].dev.b0 == 0 && jobs[0].dev.c_lo == 128 && jobs[0].dev.c_hi == 130 &&
               jobs[0].dev.c_end == 256 && jobs[0].dev.count == 2,
           "the first matrix's last rows, with its padding");
    expect(jobs[1].dev.b0 == 1 && jobs[1].dev.c_lo == 0 && jobs[1].dev.c_hi == 128 &&
               jobs[1].dev.c_end == 128 && jobs[1].dev.count == 2,
           "the second matrix's first rows");
    jobs.clear();
    expect(kvx::AppendTiledJobs(*p, base, base, 64 * row, 258 * row, true, true, &zero, &jobs)
                   .code() == Code::kInvalidArgument && jobs.empty(),
           "a cut inside a tile column refused");
    // A sixteenth of their regions filled, and less; rows below a vector.
    p = kvx::PlanTiled(Layout(2, {7, 32, 32}, {{8, 128}, {2, 1}}, {1, 2, 0}));
    expect(p.ok() && p->column, "[32, 32] batches in regions");
    p = kvx::PlanTiled(Layout(2, {7, 16, 32}, {{8, 128}, {2, 1}}, {1, 2, 0}));
    expect(p.ok() && !p->column && !p->gen.empty(), "[16, 32] batches element by element");
    p = kvx::PlanTiled(Layout(1, {4096, 15}, {{8, 128}}, {0, 1}));
    expect(p.ok() && !p->column && !p->gen.empty(), "15-byte rows element by element");
    p = kvx::PlanTiled(Layout(1, {4096, 16}, {{8, 128}}, {0, 1}));
    expect(p.ok() && p->column, "16-byte rows in regions");
  }
  if (failures == 0) std::printf("tiled jobs: all checks passed\n");
  return failures == 0 ? 0 : 1;
}
