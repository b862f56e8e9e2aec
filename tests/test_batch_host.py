"""The host side of a batch (tile lists, graph, capture) on the CPU: a program
that defines the HIP runtime functions libfls.so calls, so that every list a
launch or a captured graph reads can be checked to be alive, and allocations and
copies can be made to fail."""
import pathlib
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]

PROGRAM = r"""
#include <dlfcn.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <set>
#include <vector>
#include "fls/fls.h"

struct Dim3 { uint32_t x, y, z; };
static std::set<void*> live, filled, ever;
static std::vector<void*> captured;  // lists that the captured graph reads
static bool capturing = false, user_capture = false, fail_malloc = false, fail_copy = false;
static int stale = 0, launches = 0, graph_launches = 0;
static Dim3 pushed[2];

// The runtime, as far as a batch needs it.  Nothing runs on a device.
extern "C" {
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 8; return 0; }
int hipGetLastError() { return 0; }
int hipMalloc(void** p, size_t n) {
    if (fail_malloc) return 2;      // hipErrorOutOfMemory
    if (user_capture) return 900;   // hipErrorStreamCaptureUnsupported
    *p = malloc(n);
    live.insert(*p);
    ever.insert(*p);
    return 0;
}
int hipFree(void* p) {
    if (user_capture) return 900;
    live.erase(p);  // never given back to malloc: every list keeps an address of its own
    return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int) {
    if (fail_copy) return 1;
    if (user_capture) return 900;
    memcpy(d, s, n);
    filled.insert(d);
    return 0;
}
int hipStreamCreateWithFlags(void** s, unsigned) { *s = (void*)0x77; return 0; }
int hipStreamDestroy(void*) { return 0; }
int hipStreamBeginCapture(void*, int) { capturing = true; captured.clear(); return 0; }
int hipStreamEndCapture(void*, void** g) { capturing = false; *g = (void*)0x55; return 0; }
int hipGraphInstantiate(void** e, void*, void*, char*, size_t) { *e = (void*)0x66; return 0; }
int hipGraphExecDestroy(void*) { return 0; }
int hipGraphDestroy(void*) { return 0; }
int hipGraphLaunch(void*, void*) {
    ++graph_launches;
    for (void* p : captured) stale += !live.count(p) || !filled.count(p);
    return 0;
}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t, void*) { pushed[0] = g; pushed[1] = b; return 0; }
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* n, void** s) {
    *g = pushed[0];
    *b = pushed[1];
    *n = 0;
    *s = nullptr;
    return 0;
}
int hipLaunchKernel(const void*, Dim3, Dim3, void** args, size_t, void*) {
    ++launches;
    void* p;
    memcpy(&p, args[1], sizeof p);  // the batch kernel's tile list
    if (!ever.count(p)) return 0;
    if (capturing) captured.push_back(p);
    else stale += !live.count(p) || !filled.count(p);
    return 0;
}
}

static void* lib;
template <typename F> static F* get(const char* name) {
    void* f = dlsym(lib, name);
    if (!f) { printf("no %s\n", name); exit(3); }
    return (F*)f;
}
#define NEED(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

int main(int argc, char** argv) {
    lib = dlopen(argv[1], RTLD_NOW | RTLD_GLOBAL);
    if (!lib) { printf("%s\n", dlerror()); return 3; }
    auto create = get<decltype(fls_batch_create)>("fls_batch_create");
    auto run = get<decltype(fls_batch_run)>("fls_batch_run");
    auto per_segment = get<decltype(fls_batch_run_per_segment)>("fls_batch_run_per_segment");
    auto graph = get<decltype(fls_batch_graph_launch)>("fls_batch_graph_launch");
    auto destroy = get<decltype(fls_batch_destroy)>("fls_batch_destroy");
    fls_segment seg[3] = {};
    for (int i = 0; i < 3; ++i) {
        seg[i].n_values = (i + 1) * 100000;
        seg[i].col.encoding = FLS_ENC_BITPACK;
        seg[i].col.bw = 5;
        seg[i].col.n_words = (seg[i].n_values + 1023) / 1024 * 160;
        seg[i].col.words = (const uint32_t*)0x1000;  // never read here
        seg[i].hi = 9;
    }
    uint64_t* counts = (uint64_t*)0x2000;
    fls_batch* b = nullptr;
    NEED(create(seg, 3, &b) == FLS_OK);
    const fls_tune small = {16, 256, FLS_SCHED_DYNAMIC, 0}, large = {64, 256, FLS_SCHED_DYNAMIC, 0};
    BODY
    NEED(stale == 0);
    destroy(b);
    NEED(live.empty());
    printf("OK\n");
    return 0;
}
"""

FAILED_UPLOAD = r"""
    NEED(run(b, &small, counts, nullptr) == FLS_OK);
    NEED(graph(b, &small, counts, nullptr) == FLS_OK);
    FAIL = true;
    NEED(run(b, &large, counts, nullptr) != FLS_OK);
    FAIL = false;
    const int replays = graph_launches;
    NEED(graph(b, &small, counts, nullptr) == FLS_OK && graph_launches == replays + 1 && stale == 0);
    FAIL = true;
    NEED(run(b, &large, counts, nullptr) != FLS_OK);
    NEED(graph(b, &large, counts, nullptr) != FLS_OK);
    FAIL = false;
    NEED(graph(b, &small, counts, nullptr) == FLS_OK);
    NEED(run(b, &large, counts, nullptr) == FLS_OK && stale == 0);
    NEED(graph(b, &small, counts, nullptr) == FLS_OK);
"""

# hipMalloc, hipMemcpy and hipFree fail in a capture that forbids them
CAPTURED = r"""
    NEED(run(b, &small, counts, nullptr) == FLS_OK);
    user_capture = true;
    int before = launches;
    NEED(run(b, &small, counts, nullptr) == FLS_OK);
    NEED(launches == before + 2);
    NEED(per_segment(b, &small, counts, nullptr) == FLS_OK);
    NEED(launches == before + 2 + 1 + 3);  // one clears the counters
    NEED(run(b, &small, counts, nullptr) == FLS_OK);
    user_capture = false;
"""


def run_body(tmp_path, body):
    src, exe = tmp_path / "batch_host.cpp", tmp_path / "batch_host"
    src.write_text(PROGRAM.replace("BODY", body))
    subprocess.run(["g++", "-O1", "-std=c++17", "-rdynamic", f"-I{ROOT / 'include'}", str(src), "-o", str(exe), "-ldl"],
                   check=True)
    r = subprocess.run([str(exe), str(ROOT / "fastlanesgpu_amd" / "libfls.so")], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "OK", (r.returncode, r.stdout, r.stderr[-2000:])


@pytest.mark.parametrize("fail", ["fail_malloc", "fail_copy"])
def test_after_a_failed_tile_upload_no_list_is_stale(tmp_path, fail):
    """No graph replays and no launch reads a list that was freed on the way to a
    list that could not be allocated or filled."""
    run_body(tmp_path, FAILED_UPLOAD.replace("FAIL", fail) + "    (void)per_segment;")


def test_per_segment_launches_are_captured_after_a_run(tmp_path):
    """After a run, the launches of one segment each need no allocation or copy:
    a capture takes them, as it takes another run."""
    run_body(tmp_path, CAPTURED + "    (void)graph, (void)large;")
