"""The host side of the library without a device: its C sources compiled over stand-ins for the HIP runtime, with a main() of the test's own.
A launch calls the test's on_launch() with its entry point and its argument record and then counts as finished."""
import os
import subprocess

import pytest

from qwental_amd import build

PRELUDE = r"""
#include "gpu_hip.c"
#include "qw_path.c"
static qw_ioslot io_slots[QW_IO_SLOTS];
static uint64_t device_clock = 1; // ten ticks a launch
static uint32_t io_counts[QW_IO_SLOTS * (4 + QW_FIN_BYTES) / 4];
static void on_launch(const char *fname, unsigned gx, unsigned bx, const void *args);
hipError_t hipModuleGetFunction(hipFunction_t *f, hipModule_t m, const char *name) { return (void)m, *f = (hipFunction_t)strdup(name), hipSuccess; }
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned by, unsigned bz, unsigned lds, hipStream_t st, void **params, void **extra) {
    (void)gy, (void)gz, (void)by, (void)bz, (void)lds, (void)st, (void)extra;
    on_launch((const char *)f, gx, bx, params[0]);
    const bool io = !strcmp((const char *)f, "qwk_io");
    const qwk_io_args *a = params[0];
    const size_t at = start_of((const char *)f);
    uint64_t *started = NULL;
    if (at) memcpy(&started, (const char *)params[0] + at, sizeof started);
    if (io) started = a->t_enter;
    if (started) *started = device_clock;
    device_clock += 10;
    if (io && a->t_done) *a->t_done = device_clock;
    for (int i = 0; i < QW_IO_SLOTS; i++) {
        io_slots[i].done = io_slots[i].copied = 1;
        if (!io) io_slots[i].t1[0] = device_clock;
    }
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t st) { return (void)st, hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return (void)e, "error"; }
hipError_t hipMalloc(void **p, size_t n) { return (*p = aligned_alloc(256, (n + 255) & ~(size_t)255)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned flags) { return (void)flags, hipMalloc(p, n); }
hipError_t hipFree(void *p) { return free(p), hipSuccess; }
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipMemset(void *p, int v, size_t n) { return memset(p, v, n), hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { return (void)k, memmove(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) { return (void)k, (void)st, memmove(d, s, n), hipSuccess; }
bool qw_noalloc_scratch(int dev, void **ptr, size_t *bytes, const char **err) { return (void)dev, (void)ptr, (void)bytes, (void)err, false; }
static qw_gpu *device(void) { // what qw_gpu_open sets up, without tile-major copies
    static char tabs[QW_TAB_BYTES];
    qw_gpu *g = calloc(1, sizeof *g);
    g->kernels = calloc(QW_MAX_KERNELS, sizeof *g->kernels);
    g->ncu = 256, g->tick = 1e-9, g->tabs = tabs, g->io = io_slots, g->io_count = io_counts, g->total_mem = (size_t)1 << 38;
    g->io_func = find_func(g, "qwk_io");
    read_switches(g);
    return g;
}
"""


def run(tmp_path, source, *flags, timeout=120):
    """Compile PRELUDE + source with the library's own include paths and run it; the text it printed. Fails when main() does not return 0."""
    if not os.path.exists(build.CLANG):
        pytest.skip("no clang of the ROCm tree here")
    (tmp_path / "t.c").write_text(PRELUDE + source)
    (tmp_path / "qw_kernels_gfx950.hsaco").write_bytes(b"\0")
    exe = str(tmp_path / "t")
    subprocess.run([build.CLANG, "-std=c23", "-O1", "--embed-dir=" + str(tmp_path), "-I", os.path.join(build.ROOT, "include"), "-I", build.CSRC, "-I", os.path.join(build.ROCM, "include"), *flags,
                    str(tmp_path / "t.c"), os.path.join(build.CSRC, "qw_par.c"), "-o", exe, "-Wl,--unresolved-symbols=ignore-all", "-pthread"], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True, timeout=timeout)
    assert r.returncode == 0, r.stdout
    return r.stdout
