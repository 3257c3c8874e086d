"""Systems that iterate together in batches (ostp_krylov.h) leave what each
leaves alone, wherever a batch ends: the kernels themselves, compiled as plain
C++ and run on the CPU (tests/host), in the launch order of kr_iterate."""
import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]
HOST = ROOT / "tests" / "host"
CLANG = shutil.which("clang++", path="/opt/rocm/llvm/bin") or shutil.which("clang++") or "/opt/rocm/llvm/bin/clang++"


def build_host(src, exe, *more):
    subprocess.run([CLANG, "-O2", "-std=c++17", "-ffp-contract=off", "-mfma", "-U_FORTIFY_SOURCE", "-Wno-unknown-pragmas",
                    f"-I{HOST}", f"-I{ROOT / 'openstaple_amd' / 'csrc'}", str(src), "-o", str(exe), *more], check=True)


@pytest.fixture(scope="module")
def lines(tmp_path_factory):
    exe = tmp_path_factory.mktemp("krylov") / "krylov_batches"
    build_host(HOST / "krylov_batches.cpp", exe)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    return dict(line.split(" : ") for line in out.splitlines())


@pytest.mark.parametrize("form", ["split", "plain"])
def test_windows_do_not_depend_on_batch_ends(lines, form):
    """Two to four systems in batches that end after 8, 12, 28, ... iterations,
    one of them stopping before, at and after a batch's end and a window's end
    while another goes on: every window applied to the solutions, the
    residuals and the states are those of the system solved alone, bit for
    bit (the same operations on each number)."""
    mine = {k: v for k, v in lines.items() if k.startswith(form)}
    assert len(mine) == 39
    assert not [k for k, v in mine.items() if v != "agree"]


def test_full_window_takes_no_step(lines):
    assert lines["full"] == "agree"


def test_partial_sums_keep_their_order(tmp_path):
    """part_sum adds a thread's partials one after the other, whatever their
    number: bit for bit the plain loop."""
    src = tmp_path / "part.cpp"
    src.write_text(r"""
#include "ostp_reduce.h"
int main() {
    std::vector<double> p(40000);
    for (size_t i = 0; i < p.size(); i++) p[i] = sin(1.0 + i) * pow(10.0, (int)(i % 7) - 3);
    for (int n : {0, 1, 63, 64, 255, 256, 257, 2047, 2048, 2049, 8192, 8197, 19999})
        for (int stride : {1, 2})
            for (int t = 0; t < 256; t++) {
                double v = 0.0;
                for (int i = t; i < n; i += 256) v += p[(size_t)i * stride];
                if (ostp::part_sum<256>(p.data(), n, stride, t) != v) return 1;
            }
    return 0;
}
""")
    build_host(src, tmp_path / "part")
    subprocess.run([str(tmp_path / "part")], check=True)
