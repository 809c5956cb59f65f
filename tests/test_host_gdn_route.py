"""Which kernel takes a call of the gated delta rule: csrc/gdn_route.h built for the host."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <cstdio>
#include "gdn_route.h"
int main() {
  long long tokens, batch, hv, longest;
  while (std::scanf("%lld %lld %lld %lld", &tokens, &batch, &hv, &longest) == 4)
    std::printf("%d\n", (int)msgl::gdn_route(tokens, batch, hv, longest, 256));
}
"""
TOKENS, SHORT, CHUNKS = 0, 1, 2


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    where = tmp_path_factory.mktemp("gdn_route")
    src, exe = where / "route.cpp", where / "route"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "mini-sglang-mlx_amd", "csrc"), str(src), "-o", str(exe)], check=True)

    def ask(launches):  # of (lengths, hv, longest)
        lines = "".join(f"{sum(n)} {len(n)} {hv} {longest}\n" for n, hv, longest in launches)
        return [int(x) for x in subprocess.run([str(exe)], input=lines, check=True, capture_output=True, text=True).stdout.split()]
    return ask


@pytest.mark.parametrize("lengths,hv", [
    ([4000] + [40] * 47, 32), ([2000] + [8] * 31, 32), ([720] + [1] * 15, 32), ([1265] + [5] * 35, 4), ([966] + [4] * 25, 32),
    ([204] + [1] * 6, 32), ([1923] + [89] * 68, 8), ([372] + [3] * 8, 16)])
def test_one_long_request_goes_in_chunks_of_64(route, lengths, hv):
    assert route([(lengths, hv, max(lengths)), (lengths, hv, 0)]) == [CHUNKS, CHUNKS]


def test_even_launches_keep_to_one_kernel_from_9_to_48_tokens(route):
    sizes = [(n, batch, hv) for n in range(9, 49) for batch in (1, 2, 3, 5, 8, 9, 16, 17, 24, 40, 64, 100) for hv in (4, 8, 16, 32, 48, 64)]
    assert set(route([([n] * batch, hv, n) for n, batch, hv in sizes])) == {SHORT}


@pytest.mark.parametrize("n,batch,hv,want", [
    (8, 1, 32, TOKENS), (4, 2, 32, SHORT), (3, 2, 32, TOKENS), (2, 4, 32, SHORT), (1, 4, 32, TOKENS), (3, 17, 32, TOKENS), (4, 17, 32, SHORT),
    (49, 1, 32, CHUNKS), (49, 16, 32, CHUNKS), (65, 18, 32, SHORT), (66, 18, 32, CHUNKS), (127, 48, 32, SHORT), (128, 48, 32, CHUNKS)])
def test_lines(route, n, batch, hv, want):
    assert route([([n] * batch, hv, n)]) == [want]


def test_without_the_longest_chunks_of_64_take_what_they_are_faster_for_than_token_by_token(route):
    assert route([([24] * 4, 32, 0), ([14] * 4, 32, 0), ([48], 32, 0), ([20], 32, 0), ([40] * 66, 32, 0), ([14] * 16, 32, 0)]) == \
        [CHUNKS, SHORT, CHUNKS, SHORT, CHUNKS, SHORT]
