"""A result's large columns are copied by several threads; where threads cannot
be created the copy still comes out whole. The collector's own source is built
into a small program whose pthread_create fails from a given call on."""

import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "gpudbmetalcodegen_amd" / "csrc"

PROGRAM = r"""
#include "execution/hip_result_collector.h"

#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <dlfcn.h>
#include <pthread.h>

static int left = 0;  // threads that may still be created
static int refused = 0;

extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* arg) {
    using Fn = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
    if (left-- <= 0) {
        ++refused;
        return EAGAIN;
    }
    return reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "pthread_create"))(t, a, f, arg);
}

int main(int, char** argv) {
    const size_t rows = std::strtoul(argv[1], nullptr, 10);
    std::vector<uint32_t> w32(rows);
    std::vector<int64_t> w64(rows);
    for (size_t i = 0; i < rows; ++i) {
        w32[i] = static_cast<uint32_t>(i * 2654435761u);
        w64[i] = -static_cast<int64_t>(i) * 1000003;
    }
    for (bool narrow : {true, false}) {
        left = std::atoi(argv[2]);
        gdb::codegen::ResultColumn c;
        c.raw = narrow ? static_cast<const void*>(w32.data()) : w64.data();
        c.raw32 = narrow;
        c.rawRows = rows;
        std::vector<int64_t> out(rows, 7);
        c.copyI64(out.data());
        for (size_t i = 0; i < rows; ++i)
            if (out[i] != (narrow ? static_cast<int64_t>(w32[i]) : w64[i])) return 1;
    }
    std::printf("%d\n", refused);
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("copy")
    (d / "main.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{CSRC}", f"-I{CSRC.parent.parent / 'include'}", str(d / "main.cpp"),
                    str(CSRC / "execution" / "hip_result_collector.cpp"), str(CSRC / "core" / "hip_param_binding.cpp"),
                    "-o", str(d / "main"), "-pthread", "-ldl", "-rdynamic"], check=True)
    return d / "main"


# rows: one thread's share, the first size that is split, eight shares and one row more
@pytest.mark.parametrize("rows", [(1 << 19) - 1, 1 << 19, (1 << 21) + 1])
@pytest.mark.parametrize("threads", [0, 1, 3, 100])
def test_copy_without_threads(program, rows, threads):
    r = subprocess.run([str(program), str(rows), str(threads)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    helpers = max(0, min(8, rows >> 18) - 1)
    assert int(r.stdout) == 2 * max(0, helpers - threads)
