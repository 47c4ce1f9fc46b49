"""Threads of a workgroup: what the kernels are compiled for against what the host refuses to record otherwise."""
import os
import re
import subprocess

import pytest

import hostrt
from qwental_amd import build

SIZES = r"""
static void on_launch(const char *fname, unsigned gx, unsigned bx, const void *args) { (void)fname, (void)gx, (void)bx, (void)args; }
int main(int argc, char **argv) {
    (void)argc;
    char name[64];
    unsigned n;
    FILE *f = fopen("@names", "r");
    while (f && fscanf(f, "%63s %u", name, &n) == 2)
        if (wg_rule(name)->threads != n) return printf("%s: compiled for %u threads, the host's rule says %u\n", name, n, wg_rule(name)->threads), 1;
    if (!f) return printf("no list: %s\n", argv[0]), 1;
    qw_gpu *g = device();
    static qw_kernel k = {.name = "test"};
    qwk_qmvm_args q = {.K = 512};
    qwk_pre_args p = {.r = {.D = 1024}};
    qwk_hc_args h = {.D = 2048};
    qwk_cmb_args c = {0};
    const struct { const char *fname; const void *args; size_t size; unsigned fits; } all[] = {
        {"qwk_qmvs_x1", &q, sizeof q, 128}, {"qwk_qmvm", &q, sizeof q, 768}, {"qwk_pre_w1_s8", &p, sizeof p, 256}, {"qwk_qmvm_swiglu", &p, sizeof p, 256},
        {"qwk_hc_down_r4", &h, sizeof h, 256}, {"qwk_hc_upv", &h, sizeof h, 256}, {"qwk_cmb", &c, sizeof c, 256}, {"qwk_select", &c, sizeof c, 1024}};
    for (size_t i = 0; i < sizeof all / sizeof *all; i++)
        for (unsigned bx = 64; bx <= 1024; bx += 64) {
            qw_batch *b = qw_batch_begin(g, false);
            b->k = &k;
            const bool ok = add_launch(b, all[i].fname, 1, bx, all[i].args, all[i].size);
            if (ok != (bx == all[i].fits) || ok == b->failed || b->nl != ok) return printf("%s with %u threads: %s\n", all[i].fname, bx, ok ? "recorded" : "refused"), 1;
            batch_free(b);
        }
    return 0;
}
"""


def test_sizes_that_the_kernels_assume(tmp_path):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc here")
    src = subprocess.run([build.HIPCC, "--offload-arch=gfx950", "-std=c++17", "--cuda-device-only", "-E", "-P", "-I", os.path.join(build.CSRC, "kernels"), os.path.join(build.CSRC, "kernels", "qw_kernels.hip")],
                         stdout=subprocess.PIPE, text=True, check=True).stdout
    found = dict(re.findall(r"void\s+(qwk_\w+)\s*\(\s*\w+\s+a\s*\)\s*\{\s*__builtin_assume\(__builtin_amdgcn_workgroup_size_x\(\)\s*==\s*\(([^;]+)\)\)\s*;", src))
    assert len(found) > 60 and len(found) == src.count("__builtin_assume(__builtin_amdgcn_workgroup_size_x()")
    names = tmp_path / "names"
    names.write_text("".join("%s %d\n" % (k, eval(re.sub(r"(\d)u", r"\1", v))) for k, v in found.items()))
    hostrt.run(tmp_path, SIZES.replace("@names", str(names)))
