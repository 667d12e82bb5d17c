"""The index arithmetic of the W6A16 tile kernel (rwkv-infer-next_amd/csrc/w6a16_grid.h), the very header that the kernel
and its launch include, carried through on the CPU up to the largest sizes that a call may have: divisions by
multiplication against divisions, and the map from workgroups to tiles against the tiles."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rwkv-infer-next_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "w6a16_grid.h"
using namespace w6;

static uint64_t rnd() {  // xorshift
    static uint64_t s = 88172645463325252ull;
    s ^= s << 13, s ^= s >> 7, s ^= s << 17;
    return s;
}

static void check_division(uint32_t d, uint32_t last) {
    const Divisor x = divisor(d);
    auto at = [&](uint64_t n) {
        if (n <= last && quotient((uint32_t)n, x) != n / d) {
            printf("%llu / %u gives %u\n", (unsigned long long)n, d, quotient((uint32_t)n, x));
            exit(1);
        }
    };
    const uint64_t most = last / d;
    for (uint64_t k = 0; k <= most; k = k < 64 || k + 64 > most ? k + 1 : k + 1 + rnd() % (most / 16 + 1))
        for (int e = -1; e <= 1; ++e) at(k * d + e);  // (0 - 1 lies past `last`)
    for (uint64_t n = last - 100; n <= last; ++n) at(n);
}

// The tiles of a call, over its launches as the host cuts them: each (M group, column) once, and none else but past the
// last column; of large grids the edges of every M group's run, of the launches and of the grid.
static void check_grid(uint32_t tiles, uint32_t m_groups, uint32_t wg, uint32_t block) {
    TileGrid g;
    const uint64_t n = tile_grid(tiles, m_groups, wg, g), columns = (tiles + wg - 1) / wg, most = launch_limit(block);
    auto fail = [&](const char* what, uint64_t x) {
        printf("tiles %u, M groups %u, %u to a workgroup, %u threads: %s (%llu)\n", tiles, m_groups, wg, block, what,
               (unsigned long long)x);
        exit(1);
    };
    if (n % 8 || n < columns * m_groups || n >> 34) fail("workgroups", n);
    if (most < 8 || most % 8 || (uint64_t)most * block > 0xFFFFFFFFu || (uint64_t)most * 2 * block < 0x80000000u) fail("a launch", most);
    const bool all = n <= (1u << 24);
    std::vector<bool> seen(all ? columns * m_groups : 0);
    auto at = [&](uint64_t x) {
        g.first = (uint32_t)(x / most * most / 8);
        const TilePos p = tile_pos(g, (uint32_t)(x % most));
        const uint64_t u = x / 8, v = u / m_groups, per = 1u << g.unit_shift;
        if (p.mg != u % m_groups || p.column != (v / per * 8 + x % 8) * per + v % per) fail("another place", x);
        if ((uint64_t)p.column * wg > 0x7FFFFFFF) fail("a column tile past 2^31", x);
        if (all && p.column < columns) {
            if (seen[p.column * (uint64_t)m_groups + p.mg]) fail("twice", x);
            seen[p.column * (uint64_t)m_groups + p.mg] = true;
        }
    };
    if (all) {
        for (uint64_t x = 0; x < n; ++x) at(x);
        for (size_t k = 0; k < seen.size(); ++k)
            if (!seen[k]) fail("a tile without a workgroup", k);
        return;
    }
    const uint64_t step = m_groups * (n / 8 / m_groups / 100000 + 1);
    for (uint64_t u = 0; u < n / 8; u += step)
        for (int e = -1; e <= 1; ++e)
            if (u + e < n / 8) at(8 * (u + e) + rnd() % 8);
    for (uint64_t x = most; x < n; x += most)
        for (int e = -9; e <= 9; ++e)
            if (x + e < n) at(x + e);
    for (uint64_t x = n - 4096; x < n; ++x) at(x);
}

int main(int argc, char** argv) {
    if (argv[1][0] == 'd') {
        for (uint32_t d = 1; d < 3000; ++d) check_division(d, 0x7FFFFFFF);
        for (int l = 11; l < 31; ++l)
            for (int e = -2; e <= 2; ++e) check_division((1u << l) + e, 0x7FFFFFFF);
        for (int k = 0; k < 3000; ++k) check_division(1 + (uint32_t)(rnd() % 0x7FFFFFFE), 0x7FFFFFFF);
        for (uint32_t d : {6219u, 11627u, 11727u, 23831u, 47240u, 65537u, 70001u, 100003u}) check_division(d, 0x7FFFFFFF);
    } else {
        const uint32_t sizes[] = {1, 2, 3, 4, 5, 7, 8, 9, 16, 20, 31, 48, 64, 65, 100, 160, 1021, 1024, 4096};
        for (uint32_t tiles : sizes)
            for (uint32_t m : sizes)
                for (uint32_t wg : {1u, 2u, 4u, 8u}) check_grid(tiles, m, wg, 512);
        // rows past which a 31-bit reciprocal of the M groups is off by one
        for (uint32_t wg : {4u, 8u}) {
            check_grid(4096, 6219, wg, 512), check_grid(1024, 11627, wg, 512), check_grid(1024, 11727, wg, 512);
            check_grid(256, 23831, wg, 512), check_grid(64, 47240, wg, 512), check_grid(1, 3000017, wg, 512);
        }
        // 2^32 work-items and more: M = 67.2 M rows of 512 columns of A (16 columns of weights), 16 and 64 rows of N = 2^30
        // (K = 320) and of N = 2^31 - 16 (K = 64), which a call on a card of 288 GB can have
        check_grid(1, 1050001, 4, 512), check_grid(1, 1050001, 8, 512);
        for (uint32_t m : {1u, 4u, 16u}) check_grid(1u << 26, m, 4, 256), check_grid((1u << 27) - 1, m, 4, 64);
        check_grid(1u << 22, 16, 4, 256), check_grid(1u << 26, 1, 8, 1024);
    }
    printf("fine\n");
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("amdclang++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp("grid")
    (d / "grid.cpp").write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-O2", "-Wall", "-Werror", f"-I{CSRC}", "-o", str(d / "grid"), str(d / "grid.cpp")],
                   check=True)
    return str(d / "grid")


def _run(program, what):
    r = subprocess.run([program, what], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip() == "fine", r.stdout


def test_divisions_are_exact_below_2_to_the_31(program):
    _run(program, "divisions")


def test_every_tile_has_one_workgroup(program):
    _run(program, "grids")
