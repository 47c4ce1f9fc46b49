"""The word a batch's last launch raises for the host, without a device: gpu_hip.c compiled over stand-ins for the few
runtime calls that a batch without dispatches makes. A launch "runs" when the test says so."""
import os
import subprocess

import pytest

from qwental_amd import build

SOURCE = r"""
#include "gpu_hip.c"
static struct { qwk_io_args a; } queue[64];
static int queued, ran;
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned by, unsigned bz, unsigned lds, hipStream_t st, void **params, void **extra) {
    (void)f, (void)gx, (void)gy, (void)gz, (void)bx, (void)by, (void)bz, (void)lds, (void)st, (void)extra;
    queue[queued++].a = *(qwk_io_args *)params[0];
    return hipSuccess;
}
static void run_all(void) {
    for (; ran < queued; ran++) {
        const qwk_io_args *a = &queue[ran].a;
        if (a->t_enter) *a->t_enter = 10;
        if (a->t_done) *a->t_done = 5;
        if (a->flag) *a->flag = a->flagval;
    }
}
hipError_t hipStreamQuery(hipStream_t st) { (void)st; return ran < queued ? hipErrorNotReady : hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t st) { (void)st; run_all(); return hipSuccess; }
bool qw_noalloc_scratch(int dev, void **ptr, size_t *bytes, const char **err) { (void)dev, (void)ptr, (void)bytes, (void)err; return false; }
static qw_ioslot slots[QW_IO_SLOTS];
static uint32_t counts[QW_IO_SLOTS];
int main(void) {
    const uint64_t at[] = {0, 1, 0x7ffffffe, 0xfffffffe, 0xffffffff, 0x1ffffffff};
    for (int i = 0; i < 6; i++) {
        qw_gpu *g = calloc(1, sizeof *g);
        g->io = slots, g->io_count = counts, g->tick = 1, g->batch_seq = at[i];
        for (int again = 0; again < 3; again++) { // the slot is taken again each time
            queued = ran = 0;
            qw_batch *b = qw_batch_begin(g, false);
            qw_batch_submit(b);
            if (qw_batch_poll(b)) return printf("batch %llx: done before its launches ran\n", (unsigned long long)b->seq), 1;
            run_all();
            if (!b->io->done || !qw_batch_poll(b)) return printf("batch %llx: not done although its launches ran\n", (unsigned long long)b->seq), 1;
            if (qw_batch_wait(b) < 0) return printf("wait failed\n"), 1;
        }
        free(g);
    }
    return 0;
}
"""


def test_a_batch_is_done_when_its_launches_have_run(tmp_path):
    """Batch numbers whose low 32 bits are zero or pass through it: the poll must not take an untouched word for a raised one."""
    if not os.path.exists(build.CLANG):
        pytest.skip("no clang of the ROCm tree here")
    (tmp_path / "t.c").write_text(SOURCE)
    (tmp_path / "qw_kernels_gfx950.hsaco").write_bytes(b"\0")
    exe = str(tmp_path / "t")
    subprocess.run([build.CLANG, "-std=c23", "-O1", "--embed-dir=" + str(tmp_path), "-I", os.path.join(build.ROOT, "include"), "-I", build.CSRC, "-I", os.path.join(build.ROCM, "include"),
                    str(tmp_path / "t.c"), "-o", exe, "-Wl,--unresolved-symbols=ignore-all", "-pthread"], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
