"""The host side of results, built from the collector's own source into small
programs. A large column is copied by several threads, and still whole where
threads cannot be created (pthread_create fails from a given call on). A group
table that the device cannot order for want of memory is read and sorted here."""

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


GROUPS = r"""
#include "execution/hip_result_collector.h"

#include <cstdio>
#include <cstdlib>
#include <cstring>

int main(int, char** argv) {
    using namespace gdb::codegen;
    const uint64_t slots = std::strtoul(argv[1], nullptr, 10), groups = std::strtoul(argv[2], nullptr, 10);
    std::vector<uint64_t> table(4 * slots, 0xFFFFFFFFull);
    for (uint64_t g = 0; g < groups; ++g) {  // any slots, keys over the whole range
        uint64_t* w = &table[4 * ((g * 7 + 3) % slots)];
        w[0] = (g * 2654435761u & 0xFFFFFFFEull) | (g + 1) << 32;
        w[1] = static_cast<uint64_t>(-static_cast<int64_t>(g));
        w[2] = g;
        w[3] = ~g;
    }
    HipResultSchema schema;
    schema.kind = HipResultSchema::HASH_AGG;
    schema.hash.tableName = "t";
    schema.hash.slotsSymbol = "slots";
    schema.hash.slotWords = 4;
    const GenericResult r = HipResultCollector::collect(
        schema,
        [&](const std::string&, size_t off, void* dst, size_t bytes) {
            std::memcpy(dst, reinterpret_cast<const char*>(table.data()) + off, bytes);
        },
        [&](const std::string&) { return slots; });
    if (r.rows() != groups || r.columns.size() != 5) return 1;
    for (size_t i = 0; i < groups; ++i) {
        const int64_t g = r.columns[1].i64[i] - 1;
        if (r.columns[0].i64[i] != static_cast<int64_t>(g * 2654435761u & 0xFFFFFFFEull)) return 2;
        if (i && r.columns[0].i64[i] <= r.columns[0].i64[i - 1]) return 3;
        if (r.columns[2].i64[i] != -g || r.columns[3].i64[i] != g || r.columns[4].i64[i] != ~g) return 4;
    }
    return 0;
}
"""


def build(d: Path, source: str) -> Path:
    (d / "main.cpp").write_text(source)
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{CSRC}", f"-I{CSRC.parent.parent / 'include'}", str(d / "main.cpp"),
                    str(CSRC / "execution" / "hip_result_collector.cpp"), str(CSRC / "core" / "hip_param_binding.cpp"),
                    "-o", str(d / "main"), "-pthread", "-ldl", "-rdynamic"], check=True)
    return d / "main"


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    return build(tmp_path_factory.mktemp("copy"), PROGRAM)


# rows: one thread's share, the first size that is split, eight shares and one row more
@pytest.mark.parametrize("rows", [(1 << 19) - 1, 1 << 19, (1 << 21) + 1])
@pytest.mark.parametrize("threads", [0, 1, 3, 100])
def test_copy_without_threads(program, rows, threads):
    r = subprocess.run([str(program), str(rows), str(threads)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    helpers = max(0, min(8, rows >> 18) - 1)
    assert int(r.stdout) == 2 * max(0, helpers - threads)


def test_groups_sorted_on_the_host(tmp_path):
    program = build(tmp_path, GROUPS)
    for slots, groups in ((64, 0), (64, 1), (64, 64), (4096, 2000)):
        assert subprocess.run([str(program), str(slots), str(groups)], timeout=60).returncode == 0, (slots, groups)
