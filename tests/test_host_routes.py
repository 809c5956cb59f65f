"""Which way the C entries send a launch: csrc/api.hip built for the host, with launchers that say what they were given."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <cstdio>
#include "api.hip"
namespace {
int by_length;
}
namespace msgl {  // the rest of the library, as far as a tile kernel's launch asks it
int device_cus() { return 256; }
int tile_variant() { return 0; }
SharePlan share_plan(int64_t, int64_t, int64_t, int64_t, int64_t, int64_t) { return SharePlan{}; }
int launch_prefill_tile(const PrefillArgs& a, hipStream_t) {
  by_length = a.by_length;
  return MSGL_OK;
}
}  // namespace msgl
int main() {
  long long batch, rows, n_q, n_kv, longest, cross, window;
  alignas(16) static char data[16];
  int32_t* const ints = reinterpret_cast<int32_t*>(data);
  while (std::scanf("%lld %lld %lld %lld %lld %lld %lld", &batch, &rows, &n_q, &n_kv, &longest, &cross, &window) == 7) {
    by_length = -1;
    if (msgl_extend_step_workspace_bytes(batch, rows, rows, n_q, n_kv, 128, longest, (int)cross, (int)window) > 0 &&
        msgl_extend_step(data, data, data, n_kv * 128, n_kv * 128, ints, data, data, ints, ints, ints, ints, data, data, (size_t)1 << 40,
                         batch, rows, rows, n_q, n_kv, 128, 1 << 20, n_kv * 128, n_kv * 128, 0.1f, (int)longest, (int)cross,
                         (int)window, 0, nullptr) != MSGL_OK)
      return 1;
    std::printf("%d\n", by_length);
  }
}
"""
NOT, TILES, STAY = -1, 0, 1  # store and attention; rows stored by every workgroup of a small launch; by workgroups that stay


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    where = tmp_path_factory.mktemp("routes")
    src, exe = where / "routes.cpp", where / "routes"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__=1", "-I", os.path.join(ROOT, "mini-sglang-mlx_amd", "csrc"),
                    "-isystem", "/opt/rocm/include", str(src), "-Wl,--unresolved-symbols=ignore-all", "-L/opt/rocm/lib", "-lamdhip64",
                    "-Wl,-rpath,/opt/rocm/lib", "-o", str(exe)], check=True)

    def ask(ext, heads, cross=False, window=0):
        line = f"{len(ext)} {sum(ext)} {heads[0]} {heads[1]} {max(ext)} {int(cross)} {window}\n"
        return int(subprocess.run([str(exe)], input=line, check=True, capture_output=True, text=True).stdout)
    return ask


@pytest.mark.parametrize("ext,heads,want", [
    ([126] * 8, (64, 8), TILES), ([64] * 16, (64, 8), TILES), ([127] * 16, (32, 4), TILES), ([126] * 16, (32, 8), TILES),
    ([126] * 32, (16, 1), TILES), ([510] * 8, (16, 8), STAY), ([900, 1015, 800], (32, 8), STAY), ([1015], (32, 8), NOT)])
def test_prompts_of_one_round(route, ext, heads, want):
    assert route(ext, heads) == want


@pytest.mark.parametrize("ext,heads,cross,want", [
    ([267] * 22, (8, 8), False, NOT), ([310] * 23, (8, 8), False, NOT), ([511] * 16, (8, 8), False, STAY),       # 0.7, 0.87, 1.0 rounds of rows
    ([457] + [22] * 57, (8, 8), False, NOT), ([267] + [13] * 57, (16, 8), False, NOT), ([389] + [19] * 49, (32, 4), False, NOT),
    ([237, 3333, 1500, 2200, 1700, 2604], (32, 8), False, STAY), ([237, 3333, 1500, 2200, 1700, 2604], (32, 8), True, STAY),
    ([285] * 36, (64, 8), True, NOT), ([285] * 36, (64, 8), False, STAY), ([1923, 400, 476], (32, 4), True, NOT)])
def test_prompts_that_have_most_of_a_round_to_store(route, ext, heads, cross, want):
    assert route(ext, heads, cross) == want
