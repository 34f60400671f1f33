"""The host side of the C interface in a process that has no memory left to give: the choice of a kernel and the sizes
of workspaces are worked out without an allocation."""
import os
import shutil
import subprocess

import pytest

import quadmul_amd as qm

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <dlfcn.h>
#include <new>
static bool none_left = false;
void *operator new(std::size_t n)
{
    if (none_left) throw std::bad_alloc();
    return std::malloc(n);
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }
int main(int, char **argv)
{
    void *lib = dlopen(argv[1], RTLD_NOW);
    if (!lib) { std::puts(dlerror()); return 2; }
    const auto select = (int (*)(int, int, int, int, int, int))dlsym(lib, "qm_select_config_ex");
    const auto gemm_bytes = (std::size_t (*)(int, int, int, int, int, int))dlsym(lib, "qm_gemm_workspace_bytes");
    const auto recode_bytes = (std::size_t (*)(int, int, int, int, int))dlsym(lib, "qm_gemm_recode_bytes");
    const auto linear_bytes = (std::size_t (*)(int, int, int, int, int))dlsym(lib, "qm_linear_workspace_bytes");
    const int shapes[][3] = {{1, 4096, 4096}, {16, 8192, 28672}, {48, 11008, 4096}, {300, 300, 256}, {256, 8192, 28672}, {1000, 7777, 4096}, {1531, 3307, 4100}};
    none_left = true;
    for (const auto &s : shapes) {
        std::printf("%d", select(s[0], s[1], s[2], 256, 1, 0));
        std::printf(" %zu %zu %zu\n", gemm_bytes(s[0], s[1], s[2], 256, -1, 1), recode_bytes(s[0], s[1], s[2], 256, 0), linear_bytes(s[0], s[1], s[2], 1, 256));
    }
    std::fflush(stdout);
    std::_Exit(0);
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_a_choice_allocates_nothing(tmp_path):
    source, program = tmp_path / "no_memory.cpp", tmp_path / "no_memory"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-rdynamic", str(source), "-o", str(program), "-ldl"], check=True, timeout=120)
    lib = os.path.join(os.path.dirname(qm.__file__), "lib", "libqm_hip.so")
    r = subprocess.run([str(program), lib], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.returncode, r.stdout[-500:], r.stderr[-500:])
    shapes = [(1, 4096, 4096), (16, 8192, 28672), (48, 11008, 4096), (300, 300, 256), (256, 8192, 28672), (1000, 7777, 4096), (1531, 3307, 4100)]
    want = [f"{qm.select_config(*s)} {qm.workspace_bytes(*s, scaled=True)} {qm.recode_bytes(*s)} {qm.library().qm_linear_workspace_bytes(*s, 1, 256)}" for s in shapes]
    assert r.stdout.split("\n")[:len(want)] == want
