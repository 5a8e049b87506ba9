"""Launch arithmetic that needs no device (csrc/fh_plan.h), compiled with the host compiler."""

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "flash-hyperconnections_amd" / "csrc"


def _run(tmp_path, body):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    source, binary = tmp_path / "plan.cpp", tmp_path / "plan"
    source.write_text('#include <cstdio>\n#include <cstdlib>\n#include "fh_plan.h"\n'
                      "#define CHECK(x) do { if (!(x)) { std::printf(\"%d: %s\\n\", __LINE__, #x); std::exit(1); } } while (0)\n"
                      "int main() {\n" + body + "}\n")
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(source), "-o", str(binary)], check=True)
    done = subprocess.run([str(binary)], stdout=subprocess.PIPE, text=True)
    assert done.returncode == 0, done.stdout


def test_compute_units_are_kept_for_each_device_and_failures_are_not(tmp_path):
    _run(tmp_path, """
  fh::PerDevice units;
  int asked = 0;
  const auto say = [&](int value) { return [&asked, value] { ++asked; return value; }; };
  CHECK(units.get(0, say(0)) == 1);     // failed: 1 for now
  CHECK(units.get(0, say(256)) == 256); // asked again
  CHECK(units.get(1, say(64)) == 64);   // another device has its own
  CHECK(units.get(0, say(7)) == 256 && units.get(1, say(7)) == 64 && asked == 3);
  CHECK(units.get(1000, say(32)) == 32 && units.get(1000, say(33)) == 33 && units.get(-1, say(5)) == 5);
""")


def test_slices_cover_the_batch_and_start_at_their_first_token(tmp_path):
    _run(tmp_path, """
  for (int64_t batch = 1; batch <= 25; ++batch)
    for (int64_t most = 1; most <= 26; ++most) {
      int64_t next = 0;
      const int status = fh::in_slices(batch, most, [&](int64_t first, int64_t count) {
        CHECK(first == next && count >= 1 && count <= most);
        next += count;
        return 0;
      });
      CHECK(status == 0 && next == batch);
    }
  int calls = 0;  // an error ends it
  CHECK(fh::in_slices(int64_t{10}, int64_t{2}, [&](int64_t, int64_t) { return ++calls == 3 ? 9 : 0; }) == 9 && calls == 3);
  // Beyond 2^31 elements and bytes; h, x and gy by strides of their own, h transposed or broadcast.
  const int64_t first = int64_t{1} << 26, n = 3, cols = 5;
  const fh::MixBytes at = fh::mix_bytes(first, 2, n, cols, 0, 17, 40);
  CHECK(at.h == 0 && at.x == first * 34 && at.gy == first * 80);
  CHECK(at.rows == first * 30 && at.square == first * 18 && at.square_f32 == first * 36);
""")
