"""The height of the stencil's whole-column strips (imexsw_strips.h): the one a
search over every height finds, at a cost that a tall grid's procedures called
one at a time can bear.  CPU only."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "imex_sflow2d_v2_amd", "csrc")

MAIN = r"""
#include "imexsw_strips.h"
#include <cstdio>
#include <initializer_list>
using namespace imexsw;
static int all_heights(int tiles_x, int ny, long slots, int over) {
  int best = 1;
  long cost = -1;
  for (int h = 1; h <= ny; h++) {
    const long t = ((long)tiles_x * ((ny + h - 1) / h) + slots - 1) / slots * (h + over);
    if (cost < 0 || t < cost) cost = t, best = h;
  }
  return best;
}
int main(int argc, char** argv) {
  if (argc > 1) {  // 3000 calls on a grid of a million rows
    long s = 0;
    for (int i = 0; i < 3000; i++) s += column_rows(1 + i % 40, 1000000 + i, 1024, 1);
    std::printf("%s\n", s > 0 ? "ok" : "no");
    return 0;
  }
  for (long slots : {1L, 7L, 256L, 1024L, 2048L})
    for (int over : {0, 1, 3})
      for (int tx : {1, 2, 9, 17, 35, 400})
        for (int ny = 2; ny <= 5000; ny = ny < 300 ? ny + 1 : ny + 1 + ny / 7)
          if (column_rows(tx, ny, slots, over) != all_heights(tx, ny, slots, over)) {
            std::printf("tiles %d ny %d slots %ld over %d\n", tx, ny, slots, over);
            return 1;
          }
  std::printf("ok\n");
}
"""


def build(tmp_path):
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = str(tmp_path / "strips")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", CSRC, "-o", exe,
                           str(tmp_path / "main.cpp")])
    return exe


def test_same_height_as_a_full_search(tmp_path):
    r = subprocess.run([build(tmp_path)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout


def test_cost_on_a_tall_grid(tmp_path):
    # (a search over every height takes half a minute)
    r = subprocess.run([build(tmp_path), "tall"], capture_output=True, text=True, timeout=6)
    assert r.stdout == "ok\n"
