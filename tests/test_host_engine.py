"""The batch runner's host code against a C ABI of host memory that counts its
calls and refuses an allocation on demand: what a device cannot show."""
import os
import subprocess

import pytest

import chysx

ROOT = os.path.dirname(os.path.dirname(chysx.__file__))
HOST = os.path.join(ROOT, "csrc", "host")
INCLUDE = os.path.join(os.path.dirname(ROOT), "include")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#include "engine.h"

static std::map<void*, size_t> live;
static int refuse = -1, syncs = 0, copies = 0;
extern "C" {
int chx_malloc(void** p, size_t n) {
    if (refuse >= 0 && refuse-- == 0) return CHX_ERR_DEVICE;
    *p = std::calloc(1, n);
    live[*p] = n;
    return CHX_OK;
}
int chx_free(void* p) { live.erase(p); std::free(p); return CHX_OK; }
int chx_host_malloc(void** p, size_t n) { *p = std::calloc(1, n); return CHX_OK; }
int chx_host_free(void* p) { std::free(p); return CHX_OK; }
int chx_memcpy_h2d(void* d, const void* s, size_t n, uintptr_t) { ++copies; std::memcpy(d, s, n); return CHX_OK; }
int chx_memcpy_h2d_async(void* d, const void* s, size_t n, uintptr_t) { std::memcpy(d, s, n); return CHX_OK; }
int chx_memcpy_d2h(void* d, const void* s, size_t n, uintptr_t) { std::memcpy(d, s, n); return CHX_OK; }
int chx_zero(void* p, size_t n, uintptr_t) { std::memset(p, 0, n); return CHX_OK; }
int chx_device_synchronize(void) { ++syncs; return CHX_OK; }
int chx_stream_synchronize(uintptr_t) { ++syncs; return CHX_OK; }
int chx_resident_grid_limit(int* n) { *n = 256; return CHX_OK; }
int chx_batch_is_resident(const chx_cloth_batch* b, int* r) { *r = b->res_grid > 0; return CHX_OK; }
const char* chx_last_error_message(void) { return "refused"; }
int chx_event_create(void**) { return CHX_OK; }
int chx_event_destroy(void*) { return CHX_OK; }
int chx_event_record(void*, uintptr_t) { return CHX_OK; }
int chx_event_synchronize(void*) { return CHX_OK; }
int chx_profile_range_push(const char*) { return CHX_OK; }
int chx_profile_range_pop(void) { return CHX_OK; }
int chx_dihedral_rest_angle(const int*, const float*, int, float*, uintptr_t) { return CHX_OK; }
int chx_triangle_rest_shape(const int*, const float*, int, float, float, float*, float*, uintptr_t) { return CHX_OK; }
int chx_batch_check(const chx_cloth_batch*, uintptr_t) { return CHX_OK; }
int chx_batch_energy(const chx_cloth_batch*, int, double*, uintptr_t) { return CHX_OK; }
int chx_cloth_assemble(const chx_cloth_batch*, uintptr_t) { return CHX_OK; }
int chx_cloth_solve(const chx_cloth_batch*, int, uintptr_t) { return CHX_OK; }
int chx_cloth_step(const chx_cloth_batch*, uintptr_t) { return CHX_OK; }
int chx_cloth_step_graph(const chx_cloth_batch*, uintptr_t, void**) { return CHX_OK; }
int chx_graph_destroy(void*) { return CHX_OK; }
int chx_graph_launch(void*, uintptr_t) { return CHX_OK; }
}

using chysx::engine::BatchRunner;

static chx_instance cloth(int rows, int exports) {
    static unsigned plan[1];
    chx_instance d{};
    d.n_rows = rows;
    d.res_plan = plan;
    d.res_part_rows = 256;
    d.res_parts = (rows + 255) / 256;
    d.res_exports = exports;
    d.res_form = CHX_RES_FORM_SHEET;
    return d;
}
#define REQUIRE(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

int main() {
CASE
    return 0;
}
"""

CASES = {
    # a layout that cannot get its exchange area leaves none behind, and the
    # next update makes up for it
    "refused area": r"""
    for (int many = 0; many < 2; ++many) {
        BatchRunner r;
        std::vector<chx_instance> ds(many ? 3 : 1, cloth(2000, 100));
        r.bind_many(ds);
        REQUIRE(r.resident() && live.count(r.desc().xbuf));
        ds[0] = cloth(2000, 100000);
        refuse = 0;
        bool thrown = false;
        try { r.update_many(ds, 0); } catch (const std::exception&) { thrown = true; }
        refuse = -1;
        REQUIRE(thrown && !r.resident());
        REQUIRE(r.desc().xbuf == nullptr || live.count(r.desc().xbuf));
        r.update_many(ds, 0);
        REQUIRE(r.resident() && live.count(r.desc().xbuf));
        const chx_instance& d = many ? r.desc().inst[0] : r.desc().single;
        REQUIRE(d.res_exports == 100000 && live[r.desc().xbuf] >= 8 * r.desc().res_xwords);
        syncs = copies = 0;
        r.update_many(ds, 0);
        REQUIRE(syncs == 0 && copies == 0);
    }
""",
    # the same when a grid limit asks for the area
    "refused area of a grid limit": r"""
    for (int many = 0; many < 2; ++many) {
        BatchRunner r;
        r.set_grid_blocks(4);
        std::vector<chx_instance> ds(many ? 3 : 1, cloth(2000, 100));
        r.bind_many(ds);
        REQUIRE(!r.resident() && r.desc().xbuf == nullptr);
        refuse = 0;
        bool thrown = false;
        try { r.set_grid_blocks(0); } catch (const std::exception&) { thrown = true; }
        refuse = -1;
        REQUIRE(thrown && !r.resident() && r.desc().xbuf == nullptr);
        r.update_many(ds, 0);
        REQUIRE(r.resident() && live.count(r.desc().xbuf));
        const chx_instance& d = many ? r.desc().inst[0] : r.desc().single;
        REQUIRE(d.res_xbase == CHX_RES_CONTROL_WORDS);
    }
""",
    # a grid limit is a number unless the work list changes with it
    "grid limit": r"""
    for (int many = 0; many < 2; ++many) {
        BatchRunner r;
        std::vector<chx_instance> ds(many ? 3 : 1, cloth(2000, 100));
        r.bind_many(ds);
        syncs = copies = 0;
        for (int limit : {256, 64, 4, 200, 0}) {
            r.set_grid_blocks(limit);
            REQUIRE(r.resident() == (limit != 4) && r.desc().grid_blocks == limit);
            REQUIRE(!r.resident() || (r.desc().res_grid >= 8 && (limit == 0 || r.desc().res_grid <= limit)));
            REQUIRE(syncs == 0 && copies == 0);
        }
        if (!many) continue;
        r.set_grid_blocks(16);  // two workgroups a group: each cloth is a large item
        REQUIRE(r.resident() && r.desc().res_n_big == 3 && syncs >= 2 && copies >= 1);
        REQUIRE(r.desc().res_items[2] == 0 && r.desc().res_items[6] == 8);
        r.set_grid_blocks(0);
        REQUIRE(r.resident() && r.desc().res_n_big == 0 && r.desc().res_items[6] == 0);
    }
""",
}


@pytest.mark.parametrize("case", CASES)
def test_runner(case, tmp_path, objects):
    src, exe = tmp_path / "case.cpp", tmp_path / "case"
    src.write_text(PROGRAM.replace("CASE", CASES[case]))
    subprocess.run(["g++", "-std=c++17", "-O0", "-pthread", "-I", INCLUDE, "-I", HOST, str(src), *objects,
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], timeout=60, capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.fixture(scope="module")
def objects(tmp_path_factory):
    """The host files that the runner needs, compiled once."""
    folder, out, jobs = tmp_path_factory.mktemp("host"), [], []
    for name in ("engine", "resident_plan", "topology", "constraints"):
        out.append(str(folder / f"{name}.o"))
        jobs.append(subprocess.Popen(["g++", "-std=c++17", "-O0", "-I", INCLUDE, "-I", HOST, "-c",
                                      os.path.join(HOST, f"{name}.cpp"), "-o", out[-1]]))
    assert all(j.wait() == 0 for j in jobs)
    return out
