"""Buffers that are kept from one call for the next stay empty when an allocation
fails: what asks "is it there, is it large enough" must not be told yes.  A
program against the library's own headers, with every device hidden from it, so
that each device allocation fails."""
import os
import subprocess

from cfd_amd import build

PROGRAM = r"""
#include "cfd_internal.hpp"
using namespace cfd;
template <class F> static bool fails(F f) {
    try { f(); } catch (const Error&) { return true; }
    return false;
}
int main() {
    DBuf<double> b;
    if (!fails([&] { b.alloc(8); })) return 2;
    if (b.p || b.n) { std::puts("a buffer that was not allocated has a size"); return 1; }
    PcgWork w;
    for (int k = 0; k < 2; ++k)   // the second call must try again
        if (!fails([&] { w.ensure(100); })) { std::puts("a work space without its vectors"); return 1; }
    // the sizes of a work space whose first vector was there, and the next one not
    double one = 0.0;
    w.r.borrow(&one, 1);
    if (!fails([&] { w.ensure(100); })) { std::puts("a work space without all vectors"); return 1; }
    return 0;
}
"""


def test_buffers_stay_empty_when_an_allocation_fails(tmp_path):
    src, exe = tmp_path / "failed.cpp", tmp_path / "failed"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + build.CSRC, str(src), "-L" + build.PKG, "-lcfd_amd",
                    "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath," + build.PKG,
                    "-Wl,-rpath,/opt/rocm/lib", "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], env=dict(os.environ, HIP_VISIBLE_DEVICES="-1"),
                       capture_output=True, text=True)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
