"""The rules that choose a launch's shape (tessera_amd/csrc/launch_rules.hpp): host logic without HIP, run here as a small
C++ program over the sizes the ids take."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HEAD = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "launch_rules.hpp"
using namespace qmm;
#define CHECK(x, ...) do { if (!(x)) { std::printf("line %d: %s (", __LINE__, #x); std::printf(__VA_ARGS__); std::printf(")\n"); std::exit(1); } } while (0)
"""


def run_program(tmp_path, body):
    if shutil.which("g++") is None:
        pytest.skip("g++ not found")
    src, exe = tmp_path / "rules.cpp", tmp_path / "rules"
    src.write_text(HEAD + "int main() {\n" + body + "\n}\n")
    subprocess.run(["g++", "-std=c++20", "-O1", "-Wall", "-Wextra", "-I" + os.path.join(ROOT, "tessera_amd", "csrc"), "-o", str(exe),
                    str(src)], check=True, timeout=120)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout
    return out.stdout


def test_shared_mxfp4_tiles_cover_every_step_once(tmp_path):
    """Every (tile, step) unit has one owner, its bounds say so, and the pieces of cut tiles have blocks of their own."""
    run_program(tmp_path, r"""
  const uint64_t ms[] = {17, 64, 65, 128, 129, 256, 257, 300, 453, 640, 1000, 1300, 2048};
  const uint64_t ns[] = {1, 256, 257, 1000, 2306, 5120, 6144, 17408, 40000};
  const uint64_t ks[] = {8, 16, 17, 31, 32, 40, 53, 136};
  int shared = 0;
  for (uint64_t cus : {8, 60, 256}) for (uint64_t m : ms) for (uint64_t n : ns) for (uint64_t k : ks) {
    const SharedTiles plan = shared_tiles(m, n, k, cus);
    if (plan.groups == 0) { CHECK(shared_tiles_bytes(plan) == 0, "not shared"); continue; }
    ++shared;
    const uint32_t steps = static_cast<uint32_t>(k);
    const uint64_t units = uint64_t{plan.tiles} * steps;
    CHECK(plan.tiles == (m + plan.rows - 1) / plan.rows * ((n + 255) / 256), "%u rows", plan.rows);
    CHECK(units >= uint64_t{4} * plan.groups, "%u groups", plan.groups);
    const size_t blocks = shared_tiles_bytes(plan) / (size_t{plan.rows} * 1024);
    std::vector<bool> taken(blocks, false);
    CHECK(unit_bound(0, plan.groups, plan.tiles, steps) == 0 && unit_bound(plan.groups, plan.groups, plan.tiles, steps) == units, "ends");
    for (uint32_t g = 0; g < plan.groups; ++g) {
      const uint64_t from = unit_bound(g, plan.groups, plan.tiles, steps), to = unit_bound(g + 1, plan.groups, plan.tiles, steps);
      CHECK(from < to, "group %u", g);
      for (uint64_t v : {from, (from + to) / 2, to - 1}) CHECK(unit_owner(v, plan, steps) == g, "unit %zu", static_cast<size_t>(v));
      for (uint64_t t = from / steps; t <= (to - 1) / steps; ++t) {
        if (t * steps >= from && (t + 1) * steps <= to) continue;      // the whole tile
        CHECK(g + t < blocks && !taken[g + t], "group %u tile %zu", g, static_cast<size_t>(t));
        taken[g + t] = true;
      }
    }
  }
  CHECK(shared > 300, "%d", shared);
""")


def test_shared_f16_tiles_cover_every_super_block_once(tmp_path):
    """As above for the K-quants' 128 x 128 tiles: at least two units a workgroup, and less than 40 MB of pieces."""
    run_program(tmp_path, r"""
  const uint64_t ms[] = {17, 32, 33, 64, 100, 128, 129, 300, 512, 1000, 2048};
  const uint64_t ns[] = {1, 64, 65, 128, 129, 1000, 2306, 5120, 6144, 20000};
  const uint64_t ks[] = {4, 8, 9, 11, 12, 16, 20, 21, 32, 68, 300};
  int shared = 0;
  for (uint64_t cus : {60, 256}) for (bool q4k : {false, true}) for (uint64_t m : ms) for (uint64_t n : ns) for (uint64_t k : ks) {
    const SharedTiles plan = shared_f16_tiles(m, n, k, cus, q4k);
    if (plan.groups == 0) { CHECK(shared_tiles_bytes(plan) == 0, "not shared"); continue; }
    ++shared;
    const uint32_t steps = static_cast<uint32_t>(k);
    const uint64_t units = uint64_t{plan.tiles} * steps;
    CHECK(plan.rows == 128 && plan.columns == 128 && plan.tiles == (m + 127) / 128 * ((n + 127) / 128), "%u tiles", plan.tiles);
    CHECK(units >= uint64_t{2} * plan.groups && plan.groups <= cus, "%u groups", plan.groups);
    CHECK(shared_tiles_bytes(plan) <= (size_t{40} << 20), "%zu bytes", shared_tiles_bytes(plan));
    std::vector<bool> taken(shared_tiles_bytes(plan) / 65536, false);
    CHECK(unit_bound(0, plan.groups, plan.tiles, steps) == 0 && unit_bound(plan.groups, plan.groups, plan.tiles, steps) == units, "ends");
    for (uint32_t g = 0; g < plan.groups; ++g) {
      const uint64_t from = unit_bound(g, plan.groups, plan.tiles, steps), to = unit_bound(g + 1, plan.groups, plan.tiles, steps);
      CHECK(from < to, "group %u", g);
      for (uint64_t v : {from, (from + to) / 2, to - 1}) CHECK(unit_owner(v, plan, steps) == g, "unit %zu", static_cast<size_t>(v));
      for (uint64_t t = from / steps; t <= (to - 1) / steps; ++t) {
        if (t * steps >= from && (t + 1) * steps <= to) continue;      // the whole tile
        CHECK(g + t < taken.size() && !taken[g + t], "group %u tile %zu", g, static_cast<size_t>(t));
        taken[g + t] = true;
      }
    }
  }
  CHECK(shared > 300, "%d", shared);
""")


def test_shared_f16_test_cases_are_shared(tmp_path):
    import test_gpu_shared_f16_tiles as cases
    checks = [f"  CHECK(shared_f16_tiles({m}, {n}, {k // 256}, 256, {q}).groups != 0, \"{m} x {n} x {k}\");"
              for m, n, k in cases.SHARED for q in ("true", "false")]
    checks += [f"  CHECK(shared_f16_tiles({m}, {n}, {k // 256}, 256, {str(kind == 'q4k').lower()}).groups != 0, \"{m} x {n} x {k}\");"
               for kind, few in cases.SHARED_FEW.items() for m, n, k in few]
    run_program(tmp_path, "\n".join(checks))


def test_q4k_tiles_stay_whole_where_sharing_takes_longer(tmp_path):
    """Both sides of the measured lines (beside the rule)."""
    run_program(tmp_path, r"""
  struct { uint64_t m, n, k; bool shared; } rows[] = {
    {17, 512, 2048, false}, {32, 4096, 2048, false}, {17, 6144, 3072, false}, {32, 4096, 3072, true}, {17, 7168, 4096, false},
    {17, 17408, 5120, false}, {32, 24576, 5120, false}, {17, 8192, 5120, true}, {17, 5120, 17408, true}, {32, 20480, 17408, false},
    {33, 4096, 2048, true}, {64, 7168, 3072, false}, {64, 14336, 4096, false}, {33, 40960, 5120, false}, {64, 17408, 5120, false},
    {64, 8192, 5120, true}, {64, 1024, 17408, true}, {100, 4096, 2304, false}, {100, 4096, 2048, true}, {100, 6912, 3072, false},
    {100, 8192, 3072, true}, {128, 13888, 4352, false}, {500, 1728, 3072, true}, {1000, 1728, 4096, true}, {500, 7168, 6144, false}, {1000, 3584, 5120, false}, {500, 8704, 6144, true},
    {512, 6144, 5120, true}, {512, 5120, 6144, true}, {512, 1024, 5120, true}, {256, 14336, 6144, true}};
  for (const auto& r : rows) CHECK((shared_f16_tiles(r.m, r.n, r.k / 256, 256, true).groups != 0) == r.shared, "%zu x %zu x %zu", size_t(r.m), size_t(r.n), size_t(r.k));
""")


def test_mxfp4_test_cases_are_shared(tmp_path):
    import test_gpu_mxfp4_shared_tiles as cases
    checks = "\n".join(f"  CHECK((shared_tiles({m}, {n}, {k // 128}, 256).groups != 0) == {wanted}, \"{m} x {n} x {k}\");"
                       for group, wanted in ((cases.WHOLE, "false"), (cases.SHARED, "true")) for m, n, k in group)
    run_program(tmp_path, checks)


def test_mxfp4_small_tiles_that_fill_the_chip_stay_whole(tmp_path):
    """Few steps of K and a round of small tiles: sharing cost a third more (measured beside the rule)."""
    run_program(tmp_path, r"""
  for (uint64_t m : {129, 192, 256, 385, 512, 1024, 2048}) CHECK(shared_tiles(m, 1024, 16, 256).groups == 0, "%zu", static_cast<size_t>(m));
  for (uint64_t m : {129, 256, 400, 512, 1024}) CHECK(shared_tiles(m, 2048, 16, 256).groups == 0, "%zu", static_cast<size_t>(m));
  for (uint64_t m : {65, 128, 200, 256, 512}) CHECK(shared_tiles(m, 8192, 16, 256).groups == 0, "%zu", static_cast<size_t>(m));
  CHECK(shared_tiles(512, 4096, 32, 256).groups == 0, "a full round of small tiles");
  CHECK(shared_tiles(256, 4096, 32, 256).groups != 0, "half a round");
  CHECK(shared_tiles(453, 17408, 40, 256).groups == 256 && shared_tiles(17, 6144, 40, 256).groups != 0, "sharing leads");
""")


def test_gate_up_rows_that_would_be_padding_take_small_tiles(tmp_path):
    """65 to 128 rows leave half of a 256-row tile empty, 257 to 384 half of the second."""
    run_program(tmp_path, r"""
  for (uint32_t n : {3072u, 8192u, 16384u, 17408u, 24576u, 40000u}) {
    for (uint32_t m : {65u, 100u, 128u}) CHECK(gate_up_large_tiles(m, n, 256) == 0, "%u x %u", m, n);
  }
  for (uint32_t n : {3072u, 8192u, 10240u, 17408u, 24576u}) for (uint32_t m : {257u, 300u, 384u}) CHECK(gate_up_large_tiles(m, n, 256) == 0, "%u x %u", m, n);
  CHECK(gate_up_large_tiles(300, 12288, 256) == 96, "three quarters of a round");
  CHECK(gate_up_large_tiles(129, 17408, 256) == 136 && gate_up_large_tiles(512, 17408, 256) == 128, "full rows");
  CHECK(gate_up_large_tiles(2048, 17408, 256) == 128 && gate_up_large_tiles(700, 17408, 256) == 136, "whole rounds");
  for (uint32_t m = 65; m < 3000; m += 7) for (uint32_t n : {1u, 100u, 5000u, 17408u, 60000u}) {
    CHECK(gate_up_large_tiles(m, n, 256) <= (n + 127) / 128, "%u x %u", m, n);
  }
""")


def test_decoded_weights_rows_that_would_be_padding_take_small_tiles(tmp_path):
    """64 rows and fewer, and up to 128 with a short K, stay off 256-row tiles; the tiles cover the columns."""
    run_program(tmp_path, r"""
  for (uint32_t n : {16500u, 20000u, 24576u, 32000u}) for (uint32_t k : {256u, 1024u, 2048u, 5120u}) {
    for (uint32_t m : {17u, 64u}) CHECK(f16w_tiles(m, n, k, 256).large == 0, "%u x %u x %u", m, n, k);
    CHECK((f16w_tiles(128, n, k, 256).large == 0) == (k < 4096), "128 x %u x %u", n, k);
    CHECK(f16w_tiles(256, n, k, 256).large != 0, "256 x %u x %u", n, k);
  }
  for (uint32_t m = 17; m < 3000; m += 5) for (uint32_t n : {1u, 100u, 5000u, 17408u, 60000u}) {
    const F16wTiles t = f16w_tiles(m, n, 5120, 256);
    CHECK(t.large <= (n + t.columns - 1) / t.columns && (t.columns == 256 || t.large == (n + t.columns - 1) / t.columns), "%u x %u", m, n);
  }
  CHECK(f16w_tiles(2048, 5120, 17408, 256).columns == 192 && f16w_tiles(2048, 5120, 17408, 256).large == 27, "one round of 192");
""")


def test_rope_of_one_head_shares_nothing(tmp_path):
    run_program(tmp_path, r"""
  CHECK(rope_heads_a_thread(1u << 20, 1, 128) == 1 && rope_heads_a_thread(512, 2, 128) == 8 && rope_heads_a_thread(1, 24, 128) == 1, "heads");
""")


def test_quantized_rows_are_covered(tmp_path):
    """Every thread of a row has work, sixteen workgroups at most; rows of up to 6144 columns stay with 256 threads."""
    run_program(tmp_path, r"""
  for (uint64_t rows : {1, 4, 64, 200, 255, 256, 5000}) for (uint64_t cols : {4, 1024, 1028, 5120, 6144, 6148, 8192, 17408, 1 << 20}) {
    const PackShape s = pack_shape(rows, cols);
    CHECK(s.per_row >= 1 && s.per_row <= 16 && (s.per_row == 1 || (s.per_row - 1) * s.threads * 4 < cols), "%zu x %zu", static_cast<size_t>(rows), static_cast<size_t>(cols));
    CHECK(cols > 6144 || s.threads == 256, "%zu x %zu", static_cast<size_t>(rows), static_cast<size_t>(cols));
    CHECK(rows < 256 || (s.per_row == 1 && s.threads == 256), "%zu rows", static_cast<size_t>(rows));
  }
  CHECK(pack_shape(4, 17408).threads == 256 && pack_shape(4, 17408).per_row == 16 && pack_shape(64, 17408).threads == 1024, "long rows");
""")


def test_combine_stays_within_a_launch(tmp_path):
    """Rows that four wavefronts each have threads for (2^32 of them) are never given sixteen; a lane's parts are few."""
    run_program(tmp_path, r"""
  for (uint64_t parts = 1; parts <= 100; ++parts) for (uint64_t d : {1, 64, 65, 256}) for (uint64_t rows : {1, 24, 256, 257, 1024, 1 << 22, (1 << 24) - 1}) {
    const uint32_t waves = combine_waves(rows, d, parts);
    CHECK(waves == 1 || waves == 4 || waves == 16, "%u", waves);
    CHECK(rows * waves * 64 < (uint64_t{1} << 32), "%zu rows", static_cast<size_t>(rows));
    CHECK(waves > 1 || parts <= 4, "%zu parts", static_cast<size_t>(parts));
  }
  CHECK(combine_waves(24, 256, 64) == 16 && combine_waves(24, 256, 4) == 4 && combine_waves(12288, 256, 2) == 1, "waves");
""")


def attention_call(m, n, heads, kv_heads, head_dim, q_base, window, quantized):
    keys = min(n, q_base + m)
    keys = min(keys, window) if window else keys
    padded = 64 if head_dim <= 64 else 128 if head_dim <= 128 else 256
    return f"attention_rule(AttentionCall{{{m}, {keys}, {heads}, {kv_heads}, {head_dim}, {padded}, {quantized}}}, 256, 64, 16u << 20)"


def test_attention_test_cases_take_the_kernel_they_are_for(tmp_path):
    import test_gpu_attention_tiles as cases
    special = [(m, n, heads, kv_heads, head_dim, n - m, 0) for m, n, heads, kv_heads, head_dim in cases.SPECIAL]
    run_program(tmp_path, "\n".join(
        f"  CHECK({attention_call(*case, quantized)} {wanted}, \"{case}\");"
        for group, wanted in ((cases.FEW, "== 0"), (cases.ONE_PART, "== 1"), (cases.PARTS, "> 1"), (special, "!= 0"))
        for case in group for quantized in ("false", "true")))


def test_attention_with_too_little_work_stays_with_the_rows_kernel(tmp_path):
    """Calls that lost by a half or more in the other kernel (measured; us in the rows' kernel / in the other)."""
    calls = [(64, 564, 24, 4, 256, 500, 0),      # 21 / 34
             (100, 600, 12, 2, 256, 500, 0),     # 21 / 34
             (128, 1128, 16, 2, 128, 1000, 0),   # 18 / 27
             (64, 64, 8, 8, 128, 0, 0),          # 7 / 10
             (512, 512, 2, 1, 64, 0, 0)]         # 10 / 14
    leads = [(512, 2512, 24, 4, 256, 2000, 0), (17, 8017, 24, 4, 256, 8000, 0), (200, 200, 24, 4, 256, 0, 0), (512, 512, 16, 4, 64, 0, 0)]
    run_program(tmp_path, "\n".join(f"  CHECK({attention_call(*c, 'false')} {want}, \"{c}\");" for group, want in ((calls, "== 0"), (leads, "!= 0")) for c in group))
