"""Which launches of the head_dim 128 extend kernel go to workgroups that stay (csrc/prefill_params.h): by the blocks that have
rows, not by the grid of requests that are all as long as the longest."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <cstdio>
#include "prefill_params.h"
namespace msgl { long long* clock_probe() { return nullptr; } }
int main() {
  msgl::PrefillArgs a{};
  long long batch, total_q, total_kv, n_q, n_kv, longest;
  while (std::scanf("%lld %lld %lld %lld %lld %lld", &batch, &total_q, &total_kv, &n_q, &n_kv, &longest) == 6) {
    a.batch = batch; a.total_q = total_q; a.total_kv = total_kv; a.n_q = n_q; a.n_kv = n_kv; a.max_len_extend = (int)longest;
    a.head_dim = 128; a.num_slots = 1 << 20; a.k_stride0 = a.v_stride0 = n_kv * 128; a.key_splits = 1; a.by_length = 1;
    msgl::PrefillParams p;
    int64_t blocks = 0;
    bool wide = false;
    const int rc = msgl::make_prefill_params(a, p, blocks, wide);
    std::printf("%d %d %lld\n", rc, (int)p.length_rounds, (long long)blocks);
  }
}
"""
CASES = [  # extends, tokens cached, q heads, kv heads; whether the workgroups stay
    ([4096] + [16] * 15, 0, 32, 8, True),           # 32 rounds of the grid, 2.4 of blocks
    ([1500] + [16] * 15, 0, 32, 8, False),          # 12 and 1.0
    ([88] + [2] * 63, 8000, 32, 8, False),          # 4 and 1.1
    ([380] * 30, 500, 16, 4, True),                 # 3 and 3.0
    ([200, 400, 700, 900], 100, 32, 8, False),      # 2 and 1.1
    ([771, 1500, 2710, 2000, 2200, 2393], 0, 32, 8, True),
    ([600, 100, 900], 100, 24, 3, False),           # kv heads that the XCDs cannot share out
]


@pytest.fixture(scope="module")
def rounds(tmp_path_factory):
    where = tmp_path_factory.mktemp("staying")
    src, exe = where / "staying.cpp", where / "staying"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__=1", "-I", os.path.join(ROOT, "mini-sglang-mlx_amd", "csrc"),
                    "-isystem", "/opt/rocm/include", str(src), "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib", "-o", str(exe)],
                   check=True)

    def ask(ext, cached, n_q, n_kv):
        line = f"{len(ext)} {sum(ext)} {sum(ext) + cached * len(ext)} {n_q} {n_kv} {max(ext)}\n"
        out = subprocess.run([str(exe)], input=line, check=True, capture_output=True, text=True).stdout.split()
        return [int(x) for x in out]
    return ask


@pytest.mark.parametrize("ext,cached,n_q,n_kv,stay", CASES)
def test_rounds_count_blocks_with_rows(rounds, ext, cached, n_q, n_kv, stay):
    rc, n, blocks = rounds(ext, cached, n_q, n_kv)
    assert rc == 0 and (n > 0) is stay
    if stay:  # one workgroup per compute unit, and room in its list for every block of the grid
        most = -(-max(ext) * (n_q // n_kv) // 256)
        assert blocks == 256 and n * 256 >= 8 * len(ext) * -(-most // (8 // n_kv))
