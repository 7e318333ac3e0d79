"""The launch shapes of the step kernels (openlb_amd/csrc/launch_shape.hpp),
compiled for the host with g++."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HEAD = r"""
#include <cstdio>
#include <set>
#include <utility>
#include "launch_shape.hpp"
using namespace lbmh;
static int bad = 0;
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); ++bad; } } while (0)
"""

TUNING = HEAD + r"""
int main() {
  const std::vector<int> groups{0, 2, 4, 8, 16, 32}, lds{0, 24576, 40960};
  // shapes in use and default in and out of the grid, passes below and above their windows
  for (uint32_t chunks : {1u, 7u, 8u, 31u, 32u, 255u, 256u, 432u, 511u, 512u, 65536u})
    for (lbmh_launch_config use : {lbmh_launch_config{0, 54}, {40960, 4}, {12288, 3}, {65536, 64}, {0, 0}, {0, 1}})
      for (lbmh_launch_config std_ : {lbmh_launch_config{0, 54}, {24576, 32}, {49152, 16}}) {
        const auto all = tuning_shapes(use, std_, groups, lds, chunks);
        CHECK(same_shape(all[0], use, chunks));
        int standard = 0;
        std::set<std::pair<int, uint32_t>> seen;
        for (const auto& c : all) {
          CHECK(c.lds_bytes >= 0 && c.lds_bytes <= 65536 && c.xcd_group >= 0 && c.xcd_group <= 64);
          CHECK(seen.insert({c.lds_bytes, effective_group(c.xcd_group, chunks)}).second);
          standard += same_shape(c, std_, chunks);
        }
        CHECK(standard == 1);
        for (int l : lds)
          for (int g : groups) CHECK(seen.count({l, effective_group(g, chunks)}));
      }
  // a group larger than the pass runs in dispatch order, as the grid's smallest does
  CHECK(tuning_shapes({24576, 32}, {24576, 32}, {4, 8}, {0, 24576}, 10)[0].xcd_group == 4);

  const auto all = tuning_shapes({0, 54}, {0, 54}, groups, lds, 432);
  lbmh_launch_config best{};
  // one lucky reading does not displace the shape in use
  int calls = 0;
  CHECK(fastest_shape(all, [&](const lbmh_launch_config&, float* ms) { *ms = ++calls == 6 ? 7.0f : 7.5f; return LBMH_OK; }, best) == LBMH_OK);
  CHECK(best.lds_bytes == 0 && best.xcd_group == 54);
  // a shape that is faster each time does
  auto real = [](const lbmh_launch_config& c, float* ms) { *ms = c.xcd_group == 16 && c.lds_bytes == 40960 ? 7.0f : 7.5f; return LBMH_OK; };
  CHECK(fastest_shape(all, real, best) == LBMH_OK && best.xcd_group == 16 && best.lds_bytes == 40960);
  // a failed trial is returned, the choice untouched
  best = lbmh_launch_config{1, 2};
  CHECK(fastest_shape(all, [](const lbmh_launch_config& c, float* ms) { *ms = 1; return c.xcd_group == 8 ? LBMH_E_DEVICE : LBMH_OK; }, best) == LBMH_E_DEVICE);
  CHECK(best.lds_bytes == 1 && best.xcd_group == 2);
  std::printf("bad %d\n", bad);
  return bad != 0;
}
"""

SPLIT = HEAD + r"""
int main() {
  const uint64_t MB = 1000000;
  // eight FP32 blocks of 60 MB fill 480 MB together, as one of 480 MB does
  CHECK(split_launch(LBMH_F32, false, 8 * 60 * MB).lds_bytes == 40960);
  CHECK(split_launch(LBMH_F64, false, 8 * 40 * MB).lds_bytes == 49152);
  CHECK(split_launch(LBMH_F32, false, 2 * 80 * MB).lds_bytes == 0);
  for (uint64_t mb : {1, 159, 255, 256, 317, 2000})
    for (int storage : {LBMH_F64, LBMH_F32, LBMH_F16})
      for (bool local : {false, true}) {
        const lbmh_launch_config c = split_launch(storage, local, mb * MB);
        CHECK(c.xcd_group == 32);
        CHECK((c.lds_bytes == 0) == (local || storage == LBMH_F16 || mb < 256));
      }
  std::printf("bad %d\n", bad);
  return bad != 0;
}
"""


def run(program, tmp_path):
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(program)
    subprocess.run(["g++", "-O1", "-std=c++17", f"-I{os.path.join(ROOT, 'include')}",
                    f"-I{os.path.join(ROOT, 'openlb_amd', 'csrc')}", str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout + out.stderr


def test_autotuners_time_the_shape_in_use_and_the_default(tmp_path):
    """Each autotuner times the shape in use and the default beside its grid, no
    mapping twice, and leaves the shape in use unless another is faster twice."""
    run(TUNING, tmp_path)


def test_split_launch_follows_what_all_blocks_hold(tmp_path):
    """Not the first block's size and boundaries: a reservation once the blocks
    together outgrow the Infinity Cache, none if any has local boundaries."""
    run(SPLIT, tmp_path)
