"""Which launches of the extend kernels go to workgroups that stay (csrc/prefill_params.h): by the blocks that have
rows, not by the grid of requests that are all as long as the longest; at head_dim 256 only where their lengths follow from
the rows' places, or every request's blocks fill their XCDs."""
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
  long long batch, total_q, total_kv, n_q, n_kv, longest, head_dim, window, cross, row_stride;
  static const int32_t slot = 0;
  while (std::scanf("%lld %lld %lld %lld %lld %lld %lld %lld %lld %lld", &batch, &total_q, &total_kv, &n_q, &n_kv, &longest, &head_dim, &window,
                    &cross, &row_stride) == 10) {
    a.new_tokens = msgl::NewTokens{};
    if (row_stride > 0) {  // the launch stores its rows
      a.new_tokens.out_loc = &slot; a.new_tokens.rows = total_q;
      a.new_tokens.k_stride0 = n_kv * head_dim; a.new_tokens.v_stride0 = row_stride;
    }
    a.window = window; a.is_cross = (int)cross;
    a.batch = batch; a.total_q = total_q; a.total_kv = total_kv; a.n_q = n_q; a.n_kv = n_kv; a.max_len_extend = (int)longest;
    a.head_dim = head_dim; a.num_slots = 1 << 20; a.k_stride0 = a.v_stride0 = n_kv * head_dim; a.key_splits = 1; a.by_length = 1;
    msgl::PrefillParams p;
    int64_t blocks = 0;
    bool wide = false;
    const int rc = msgl::make_prefill_params(a, p, blocks, wide, msgl::prefill_block_rows(head_dim));
    std::printf("%d %d %lld %d %d\n", rc, (int)p.length_rounds, (long long)blocks, (int)p.length_heads, (int)wide);
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

    def ask(ext, cached, n_q, n_kv, head_dim=128, window=0, cross=False, order=False, row_stride=0):
        line = f"{len(ext)} {sum(ext)} {sum(ext) + cached * len(ext)} {n_q} {n_kv} {max(ext)} {head_dim} {window} {int(cross)} {row_stride}\n"
        out = subprocess.run([str(exe)], input=line, check=True, capture_output=True, text=True).stdout.split()
        return [int(x) for x in out][:None if order else 3]
    return ask


@pytest.mark.parametrize("ext,cached,n_q,n_kv,stay", CASES)
def test_rounds_count_blocks_with_rows(rounds, ext, cached, n_q, n_kv, stay):
    rc, n, blocks = rounds(ext, cached, n_q, n_kv)
    assert rc == 0 and (n > 0) is stay
    if stay:  # one workgroup per compute unit, and room in its list for every block of the grid
        most = -(-max(ext) * (n_q // n_kv) // 256)
        assert blocks == 256 and n * 256 >= 8 * len(ext) * -(-most // (8 // n_kv))


CASES_256 = [  # extends, tokens cached (mean), q heads, kv heads, window, all keys seen; whether the workgroups stay
    ([400, 237, 100, 333] * 15, 0, 16, 4, 0, False, True),     # prompts: 4.2 rounds
    ([190] * 14 + [150], 0, 16, 4, 0, False, False),           # 1.4 of them
    ([220] * 14 + [150], 0, 16, 4, 0, False, True),            # 1.6
    ([698] * 22, 500, 8, 8, 0, False, False),                  # 6 blocks a request in an XCD
    ([87, 40, 30] * 14, 100, 32, 2, 0, False, False),
    ([698] * 22, 500, 8, 8, 300, False, True),                 # a window that most exceed
    ([698] * 22, 500, 8, 8, 2000, False, False),               # and one that they do not
    ([2048] * 4, 4000, 16, 4, 0, False, True), ([2047] * 4, 4000, 16, 4, 0, False, False),  # 32 blocks a request in an XCD
    ([2731] * 4, 4000, 24, 8, 0, False, True), ([1365] * 4, 4000, 24, 8, 0, False, False),
    ([2048] * 4, 0, 16, 4, 0, True, True), ([2048] * 4, 0, 16, 4, 300, True, False), ([2048] * 4, 0, 16, 4, 2048, True, True),
    ([2048] * 4, 10, 16, 4, 0, True, False), ([979] + [51] * 53, 0, 8, 8, 0, True, False), ([2048, 2000] * 2, 0, 16, 4, 300, False, True),
]


@pytest.mark.parametrize("ext,cached,n_q,n_kv,window,cross,stay", CASES_256)
def test_rounds_of_head_dim_256(rounds, ext, cached, n_q, n_kv, window, cross, stay):
    rc, n, blocks = rounds(ext, cached, n_q, n_kv, 256, window, cross)
    assert rc == 0 and (n > 0) is stay
    if stay:
        xcds, most = 8 // min(n_kv, 8), -(-max(ext) * (n_q // n_kv) // 128)
        assert blocks == 256 and n * 256 >= 8 * len(ext) * -(-most // xcds)


@pytest.mark.parametrize("batch,length,n_q,n_kv,ordered,stay", [  # at head_dim 128, 16 blocks of a request or more
    (1, 4000, 32, 8, False, False), (2, 1981, 32, 4, False, False), (2, 3963, 16, 8, False, False), (2, 2176, 16, 2, False, False),
    (1, 4100, 32, 8, True, True), (2, 2048, 32, 8, True, True), (3, 1365, 32, 8, True, True), (5, 1171, 16, 2, True, False), (2, 900, 32, 8, False, False)])
def test_prompts_of_one_length(rounds, batch, length, n_q, n_kv, ordered, stay):
    rc, n, blocks, heads, _ = rounds([length] * batch, 0, n_q, n_kv, order=True)
    assert rc == 0 and (heads > 0) is ordered and (n > 0) is stay


@pytest.mark.parametrize("ext,n_q,n_kv,row_stride,stay,wide", [  # prompts whose rows the launch stores
    ([510] * 8, 16, 8, 0, False, False), ([510] * 8, 16, 8, 1024, True, False),      # one round of blocks, no more than compute units
    ([1015], 32, 8, 1024, False, False),                                             # half a round
    ([4000], 32, 8, 0, False, False), ([4000], 32, 8, 1024, True, False),            # one request of many blocks, below two rounds
    ([4000], 32, 8, 536864, True, False), ([4000], 32, 8, 536872, True, True),       # offsets of v's rows around 4 GiB
    ([4000], 32, 8, (1 << 23) - 8, True, True), ([1015], 32, 8, 1 << 23, False, False)])
def test_prompts_whose_rows_are_stored(rounds, ext, n_q, n_kv, row_stride, stay, wide):
    rc, n, blocks, heads, offsets = rounds(ext, 0, n_q, n_kv, order=True, row_stride=row_stride)
    assert rc == 0 and (n > 0) is stay and (not stay or blocks == 256) and bool(offsets) is wide
