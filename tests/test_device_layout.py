"""Offsets and launch shapes that the host code computes for the device, from
the library's own headers, compiled here for the CPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "opt_solver_amd", "csrc")
ROCM = "/opt/rocm/include"

if not os.path.isdir(ROCM) or shutil.which("g++") is None:
    pytest.skip("no HIP headers or no g++", allow_module_level=True)


def run(tmp_path, body):
    """The output of a program around `body` with the internal headers."""
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text('#include <cstdio>\n#include "smfgpu_ldlt.hpp"\nusing namespace smfgpu;\nint main() {\n'
                   + body + "\n    return 0;\n}\n")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", CSRC, "-I", ROCM, str(src), "-o", str(exe)],
                   check=True)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout


def test_operand_planes_start_on_16_bytes(tmp_path):
    """A plane of bf16 operands holds big_work(ne) columns of f entries; the
    four planes of a front follow each other and are read 16 bytes at a
    time, so a plane's length is a multiple of 8 entries for any f and ne."""
    out = run(tmp_path, """
    int bad = 0;
    for (int ne = 1; ne <= 1200; ++ne)
        for (int f = ne; f < ne + 16; ++f) {
            const long long plane = static_cast<long long>(big_work(ne)) * f;
            if (plane % 8 != 0 || big_work(ne) < big_spec(ne) + kGroupCols || big_spec(ne) < (ne < 1024 ? ne : 1024)) ++bad;
        }
    std::printf("%d", bad);""")
    assert out == "0"


def test_panel_workspaces_start_on_even_entries(tmp_path):
    """A front's planes lie at four bf16 entries per entry of its panel
    workspace: the workspaces of a level's fronts, of any number of rows and
    columns, start on even entries."""
    out = run(tmp_path, """
    int bad = 0;
    long long at = 0;
    for (int f = 96; f < 400; f += 7)
        for (int cols = 2; cols < 40; ++cols) {
            const long long room = work_room(f, cols);
            if (room < static_cast<long long>(f) * cols || room >= static_cast<long long>(f) * cols + 8) ++bad;
            at += room;
            if (4 * at % 8 != 0) ++bad;
        }
    if (work_room(2000000, 1088) != 2176000000ll) ++bad;
    std::printf("%d", bad);""")
    assert out == "0"


def test_store_launches_stay_within_the_grid(tmp_path):
    """The store launches of a level's fronts cover every front once, each
    within the device's 65536 rows of workgroups and 2^22 workgroups."""
    out = run(tmp_path, """
    int bad = 0;
    for (int nf : {1, 2, 511, 512, 65535, 65536, 65537, 131072, 200000, 1000000})
        for (int cols : {1, 15, 128, 9000}) {
            long long done = 0;
            for (int o = 0; o < nf; o += kStoreFronts) {
                const StoreGrid g = store_grid(nf - o, cols);
                if (g.fronts < 1 || g.fronts > 65536 || g.per < 1 || g.per > cols) ++bad;
                if (static_cast<long long>(g.fronts) * g.per > (1ll << 22)) ++bad;
                done += g.fronts;
            }
            if (done != nf) ++bad;
        }
    std::printf("%d", bad);""")
    assert out == "0"


def test_row_chunks_begin_with_every_front(tmp_path):
    """A level's row chunks: each of every front once, the fronts' first
    chunks (their pivot logic) ahead of all others, so that they spread over
    the device's XCDs whatever the fronts' sizes."""
    out = run(tmp_path, """
    int bad = 0;
    for (int same = 0; same < 10; ++same) {
        std::vector<int32_t> chunks(301);
        for (int b = 0; b < 301; ++b) chunks[b] = same > 0 ? same : 1 + b * b % 37;
        std::vector<BigPart> p;
        row_parts(chunks, p);
        std::vector<int> seen(301 * 64, 0);
        size_t total = 0;
        for (int c : chunks) total += c;
        if (p.size() != total) ++bad;
        for (size_t i = 0; i < p.size(); ++i) {
            if (p[i].parts != chunks[p[i].front] || p[i].part >= p[i].parts || seen[64 * p[i].front + p[i].part]++) ++bad;
            if ((p[i].part == 0) != (i < 301)) ++bad;
        }
    }
    std::printf("%d", bad);""")
    assert out == "0"
