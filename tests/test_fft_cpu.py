"""Host-side checks of the transforms' index arithmetic (no GPU)."""
import os
import subprocess

import cola_halo_amd as ch

CSRC = os.path.join(os.path.dirname(os.path.abspath(ch.__file__)), "csrc")

OFFSETS = r"""
#include "fft.h"
#include <cstdio>
int main()
{
  int b, c;
  long long stride;
  while (std::scanf("%d %lld %d", &b, &stride, &c) == 3)
    std::printf("%llu %d\n", cola::col_offset(b, stride, (1 << c) - 1), (int)cola::col_offsets_fit32(b + 1, stride, c));
}
"""


def _smooth(n):
    for p in (2, 3, 5):
        while n % p == 0:
            n //= p
    return n == 1


def test_column_offsets_of_large_grids(tmp_path):
    """The offset of a column pass's last position, for every grid up to
    3000^3 and every radix schedule, with planes of one grid (rows padded or
    not) and of three: the exact product, also beyond 2^32 (2250^3 with radix
    2 first; 2160^3, 2304^3 and 2400^3 with radix 3 or 4 first), and the rule
    that keeps such grids off the fused x pass, whose offsets are 32 bits.
    Every force transform whose four grids fit 288 GB passes that rule."""
    rows = []
    for n in range(2, 3001, 2):
        if not _smooth(n):
            continue
        radices = {r for sch in range(5) for r in ch.fft_radices(n, sch)}
        for R in radices:
            for nz in (n // 2 + 1, (n // 2 + 16) // 16 * 16, 3 * ((n // 2 + 16) // 16 * 16)):
                rows.append((n // R - 1, n * nz, 6))
    src, exe = tmp_path / "offsets.cpp", tmp_path / "offsets"
    src.write_text(OFFSETS)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", CSRC, "-I", "/opt/rocm/include", str(src),
                    "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], input="".join("%d %d %d\n" % r for r in rows), check=True, capture_output=True,
                         text=True).stdout.split()
    exact = [b * stride + (1 << c) - 1 for b, stride, c in rows]
    assert max(exact) > 2 ** 32 > min(exact)
    assert [int(v) for v in out[::2]] == exact
    assert [int(v) for v in out[1::2]] == [int(v < 2 ** 32) for v in exact]
    for n in (n for n in range(2, 3001, 2) if _smooth(n)):
        nzp = (n // 2 + 16) // 16 * 16
        for sch in range(5):
            if 32 * n * n * nzp < 288e9 and ch.fft_radices(n, sch):
                assert (n // ch.fft_radices(n, sch)[0] - 1) * n * nzp + 63 < 2 ** 32, (n, sch)


ROWS = r"""
#include "fft.h"
#include <cstdio>
int main()
{
  int n;
  while (std::scanf("%d", &n) == 1) std::printf("%d\n", cola::record_row(n, 2 * ((n / 2 + 16) / 16 * 16)));
}
"""


def test_records_of_a_line_fit_three_rows(tmp_path):
    """A line's n records of three floats in the rows of three force grids:
    all of them find a place, no row holds more than its floats, and rows
    start and end on 8 bytes, on 16 where the kernel stores 16."""
    sizes = [n for n in range(2, 4097, 2) if _smooth(n)]
    src, exe = tmp_path / "rows.cpp", tmp_path / "rows"
    src.write_text(ROWS)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", CSRC, "-I", "/opt/rocm/include", str(src),
                    "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], input="".join("%d\n" % n for n in sizes), check=True, capture_output=True,
                         text=True).stdout.split()
    for n, k in zip(sizes, map(int, out)):
        assert 3 * k >= n and 3 * k <= 2 * ((n // 2 + 16) // 16 * 16) and k % 2 == 0, (n, k)
        if n % 4 == 0 and k % 4 == 0:
            assert all((3 * min(k, max(0, n - t * k))) % 4 == 0 for t in range(3)), (n, k)
        assert all((3 * min(k, max(0, n - t * k))) % 2 == 0 for t in range(3)), (n, k)
