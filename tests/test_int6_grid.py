"""The host arithmetic of the W6A16 kernels (rwkv-infer-next_amd/csrc/w6a16_grid.h and w6a16_plan.h, the very headers that
they include), carried through on the CPU up to the largest sizes that a call may have: divisions by multiplication
against divisions, the map from workgroups to tiles against the tiles, and every call's plan against what its kernel
assumes."""
import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC, INCLUDE = os.path.join(REPO, "rwkv-infer-next_amd", "csrc"), os.path.join(REPO, "include")

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


PLANS = r"""
#include <cstdio>
#include <cstdlib>
#include "w6a16_plan.h"
using namespace w6;

static int wide_calls, far_calls, split_calls;

static void check(int B, int M, int N, int K, int g, int split, int64_t stride, int64_t cus) {
    TilePlan plan[2];
    bool wide[2], big[2];
    for (int packed = 0; packed < 2; ++packed) {
        w6a16_args a{};
        a.B = B, a.M = M, a.N = N, a.K = K, a.group_k = g, a.split_k = split, a.a_row_stride = stride;
        a.format = packed ? W6A16_FORMAT_PACKED : W6A16_FORMAT_PLANES;
        const Layout l = layout(&a, cus);
        auto fail = [&](const char* what) {
            printf("B %d M %d N %d K %d g %d split %d stride %lld packed %d: %s\n", B, M, N, K, g, split, (long long)stride, packed, what);
            exit(1);
        };
        if (split > 1 && l.tiles * 4 > kCounterRegion) return;  // refused
        big[packed] = l.big, wide[packed] = wide_call(&a, l, cus);
        if (l.big) continue;
        if (wide[packed]) {  // row sums in their place, ranges that 32-bit offsets reach
            ++wide_calls;
            if (l.total_bytes != kCounterRegion + l.partial_bytes + (size_t)B * l.nchains * l.m_groups * 64 * 4) fail("row sums");
            if ((int64_t)K / 2 * N >= 0x7FFFFFFF || (int64_t)K / g * N * 2 >= 0x7FFFFFFF) fail("2 GB");
            if ((int64_t)K / 64 * kPackBytes >= 0x7FFFFFFF || (int64_t)l.nchains * l.m_groups * 64 * 4 >= 0x7FFFFFFF) fail("2 GB");
        }
        const TilePlan t = plan[packed] = tile_plan(&a, l, packed, cus);
        const int chunks = K / 64;
        if (t.mt < 1 || t.mt > 4 || t.cw < 1 || t.cw > 2 || (t.cw == 2 && t.mt < 3)) fail("rows");
        if (packed ? t.nt != 1 && t.nt != 2 && t.nt != 4 : t.nt != 4 && t.nt != 8) fail("columns");
        if (t.nt != 4 && t.mt > (packed ? 2 : 1)) fail("columns of these rows");
        if (t.parts < 1 || t.parts > chunks || (t.ks != 1 && t.ks != 2 && t.ks != 4) || t.parts % t.ks) fail("parts");
        if (t.ks > 1 && t.parts % 4) fail("quarters");
        const int waves = t.cw * t.parts / t.ks;
        const int most = t.far ? 16 : t.mt == 1 ? (t.nt == 8 ? 8 : 16) : t.mt == 2 && t.nt == 1 ? 16 : 8;
        if (waves > most) fail("wavefronts");
        if (64 * waves < 16 * t.nt * t.cw) fail("fewer threads than columns");
        if (t.far && (t.mt != 1 || t.nt != 4 || t.cw != 1)) fail("far");
        if (!t.far && ((M > 1 ? stride : K) >= (1 << 24) || (!packed && N >= (1 << 26)))) fail("not far");
        far_calls += t.far, split_calls += t.ks > 1;
        if (t.ks > 1) {  // counters and partial tiles inside the workspace
            const int64_t tiles = (int64_t)B * ((M + 16 * t.mt - 1) / (16 * t.mt)) * ((N / 16 + t.nt * t.cw - 1) / (t.nt * t.cw));
            if (tiles * 4 > (int64_t)kCounterRegion) fail("counters");
            if ((size_t)tiles * t.ks * 16 * t.mt * 16 * t.nt * t.cw * 4 > l.partial_bytes) fail("partial tiles");
        }
    }
    if (big[1]) return;  // (the planes have no such kernel)
    if (wide[0] != wide[1] || plan[0].parts != plan[1].parts) {
        printf("B %d M %d N %d K %d split %d: planes and packed differ\n", B, M, N, K, split);
        exit(1);
    }
}

int main() {
    const int Ms[] = {1, 2, 8, 9, 15, 16, 17, 31, 32, 33, 40, 48, 49, 64, 65, 96, 97, 128, 129, 144, 145, 160, 192, 193, 203, 256, 257, 300, 1000, 4097, 100000};
    const int Ns[] = {16, 32, 64, 80, 128, 144, 256, 768, 1024, 1088, 2048, 2560, 2752, 4096, 4112, 5120, 8192, 10240, 16336, 16384, 16400, 22528, 32768,
                      32784, 65536, 1 << 22, (1 << 26) - 16, 1 << 26, (1 << 30) + 80, 2147483632};
    const int Ks[] = {64, 128, 192, 256, 320, 512, 576, 768, 1024, 1088, 2048, 2560, 3072, 4096, 8192, 8256, 10240, 16320, 16384, 65536, 1 << 24};
    const int splits[] = {1, 2, 3, 4, 8, 9, 16, 32, 64, 256};
    for (int M : Ms)
        for (int N : Ns)
            for (int K : Ks)
                for (int split : splits)
                    for (int B : {1, 2, 7})
                        for (int g : {64, 128})
                            for (int64_t cus : {256, 304, 64}) {
                                if (K % g) continue;
                                check(B, M, N, K, g, split, K, cus);
                                if (B == 1 && g == 64 && K < (1 << 24)) check(B, M, N, K, g, split, 1 << 24, cus);
                            }
    if (!wide_calls || !far_calls || !split_calls) { printf("a form that no call took\n"); return 1; }
    printf("fine\n");
}
"""


def _compiled(tmp_path_factory, name, text):
    cxx = shutil.which("g++") or shutil.which("amdclang++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp(name)
    (d / "p.cpp").write_text(text)
    subprocess.run([cxx, "-std=c++17", "-O2", "-Wall", "-Werror", f"-I{CSRC}", f"-I{INCLUDE}", "-o", str(d / "p"), str(d / "p.cpp")],
                   check=True)
    return str(d / "p")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    return _compiled(tmp_path_factory, "grid", PROGRAM)


def _run(program, what):
    r = subprocess.run([program, what], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip() == "fine", r.stdout


def test_divisions_are_exact_below_2_to_the_31(program):
    _run(program, "divisions")


def test_every_tile_has_one_workgroup(program):
    _run(program, "grids")


def test_every_call_has_a_plan_that_its_kernel_takes(tmp_path_factory):
    _run(_compiled(tmp_path_factory, "plan", PLANS), "")
