"""Groups of a ragged step that go out as one launch (the kernels qwk_*_j), without a device: where the kernels lie, and which launches a step
makes."""
import os
import re
import subprocess

import pytest

import hostrt
import test_gpu_joined
import qwental_amd as q
from qwental_amd import build

NAMES = r"""
static void on_launch(const char *fname, unsigned gx, unsigned bx, const void *args) { (void)fname, (void)gx, (void)bx, (void)args; }
int main(void) {
    for (size_t i = 0; i < sizeof joinable / sizeof *joinable; i++) printf("%s_j\n", joinable[i]);
    return 0;
}
"""


def entry_points(hsaco):
    with open(hsaco, "rb") as f:
        elf = f.read()
    out = subprocess.run([os.path.join(build.ROCM, "llvm", "bin", "llvm-readelf"), "-sW", "-"], input=elf[elf.index(b"\x7fELF"):], stdout=subprocess.PIPE, check=True).stdout.decode()
    return sorted(set(re.findall(r" FUNC .* (qwk_\w+)$", out, re.M)))


def test_the_joined_kernels_lie_in_a_code_object_of_their_own(tmp_path):
    if not (os.path.exists(build.HSACO) and os.path.exists(build.JOINED)):
        pytest.skip("no code objects here")
    joined = hostrt.run(tmp_path, NAMES).split()
    assert entry_points(build.JOINED) == sorted(joined)
    main = entry_points(build.HSACO)
    assert len(main) > 150 and not [n for n in main if n.endswith("_j")] and all(n[:-2] in main for n in joined)


# Ragged steps of given layers and cuts: every launch with its grid, and of a joint one the workgroups of each group
STEPS = r"""
hipError_t hipMemGetInfo(size_t *avail, size_t *total) { return *avail = *total = (size_t)1 << 38, hipSuccess; }
static bool listen;
static void on_launch(const char *fname, unsigned gx, unsigned bx, const void *args) {
    (void)bx;
    if (!listen || !strcmp(fname, "qwk_io") || !strcmp(fname, "qwk_tab_init") || !strncmp(fname, "qwk_pack", 8)) return;
    printf(" %s:%u", fname, gx);
    const size_t n = strlen(fname), size = !strncmp(fname, "qwk_pre", 7) ? sizeof(qwk_pre_args) : !strncmp(fname, "qwk_gu", 6) ? sizeof(qwk_gu_args) : !strncmp(fname, "qwk_cmb", 7) ? sizeof(qwk_cmb_args) : sizeof(qwk_dn_args);
    if (n < 2 || strcmp(fname + n - 2, "_j")) return;
    for (unsigned j = 0; j < QW_JOIN_MAX; j++) {
        unsigned g;
        memcpy(&g, (const char *)args + QW_JOIN_MAX * size + 4 * j, 4);
        printf("%c%u", j ? '+' : '=', g);
    }
}
static const struct { int gu, dn, sg, su, sd, router, D, I, E, K, before, cut[9]; } steps[] = {
@steps
};
int main(void) {
    qw_gpu *g = device();
    g->repack = true, g->copy_uses = QW_HIP_COPY_USES, g->copy_budget = (size_t)1 << 37;
    for (size_t i = 0; i < sizeof steps / sizeof *steps; i++) {
        const size_t D = (size_t)steps[i].D, I = (size_t)steps[i].I, E = (size_t)steps[i].E;
        qw_path *p = qw_path_open(g, (int)D, (int)I, (int)E, steps[i].K, 16, true);
        const int types[] = {steps[i].gu, steps[i].gu, steps[i].dn, steps[i].sg, steps[i].su, steps[i].sd, steps[i].router, steps[i].router};
        const size_t values[] = {E * I * D, E * I * D, E * D * I, I * D, I * D, D * I, E * D, D};
        qw_buf w[8], x, out;
        qw_tensor t[8];
        for (int k = 0; k < 8; k++) {
            if (!qw_hip_buf_new_device(g, values[k] * 2, &w[k])) return printf("no memory\n"), 1; // (enough for all of these types)
            t[k] = (qw_tensor){.buf = &w[k], .type = types[k]};
        }
        if (!p || !qw_buf_new(g, 64 * D * 2, &x) || !qw_buf_new(g, 64 * D * 2, &out)) return printf("no buffers\n"), 1;
        const qw_moe_layer M = {.router = t[6], .sh_gate_w = t[7], .gate = t[0], .up = t[1], .down = t[2], .sh_gate = t[3], .sh_up = t[4], .sh_down = t[5]};
        int R = 0, ng = 0;
        qw_par *par = qw_par_new();
        for (; steps[i].cut[ng]; ng++) R += steps[i].cut[ng];
        for (int b = 1; b <= 16; b++) {
            bool in = false;
            for (int k = 0; k < ng; k++) in |= steps[i].cut[k] == b;
            for (int k = 0; k < 2; k++) qw_par_observe(par, b, in ? 1e-3 : 50);
        }
        int n[64], cut[64];
        for (int r = 0; r < R; r++) n[r] = 1;
        if (qw_par_split(par, R, cut) != ng) return printf("another cut\n"), 1;
        for (int k = 0; k <= steps[i].before; k++) {
            listen = k == steps[i].before;
            qw_vstep_info info;
            qw_par *one = qw_par_new();
            for (int b = 1; b <= 16; b++)
                for (int q = 0; q < 2; q++) qw_par_observe(one, b, qw_par_group_cost(par, b));
            if (!qw_path_par_vstep(p, one, &M, n, R, &x, &out, &info)) return printf("%s\n", g->err), 1;
            if (listen) {
                printf(" |");
                for (int q = 0; q < info.ngroups; q++) printf(" %d", info.groups[q]);
                printf("\n");
            }
            qw_par_free(one);
        }
        qw_par_free(par);
        qw_path_close(p);
        qw_buf_free(&x), qw_buf_free(&out);
        for (int k = 0; k < 8; k++) qw_buf_free(&w[k]);
    }
    return 0;
}
"""


def launches(tmp_path, steps):
    """Of every step (types, router type, D, I, E, K, like steps before it, cut): [(kernel, grid, workgroups of each group or None)] and the groups."""
    rows = ["{%s, {%s}}," % (", ".join(map(str, (*s[0], *s[1:7]))), ", ".join(map(str, s[7]))) for s in steps]
    out = []
    for line in hostrt.run(tmp_path, STEPS.replace("@steps", "\n".join(rows))).splitlines():
        made, cut = line.split("|")
        found = re.findall(r"(\w+):(\d+)(?:=([\d+]+))?", made)
        out.append(([(k, int(gx), [int(v) for v in per.split("+") if v != "0"] if per else None) for k, gx, per in found], list(map(int, cut.split()))))
    assert len(out) == len(steps)
    return out


IQ3, IQ3_Q8, NL, K4, Q8 = (21, 21, 21, 21, 21), (21, 21, 8, 8, 8), (21, 20, 12, 23, 20), (12, 14, 12, 12, 14), (8, 8, 8, 8, 8)


def test_compute_units_by_the_groups_work(tmp_path):
    """A group of two rows reads a seventh of the experts that one of sixteen reads, and gets about that many of the workgroups."""
    steps = [(IQ3, 1, 512, 256, 512, 10, 1, c) for c in ([16, 2], [15, 3], [16, 16, 16, 2], [9, 9], [15, 15, 15], [16, 15, 7])] + [(NL, 1, 1024, 640, 128, 4, 1, [15, 3])]
    for (made, cut), (E, K) in zip(launches(tmp_path, steps), (s[4:6] for s in steps)):
        work = [1 + E * (1 - (1 - K / E) ** r) for r in cut]
        for kernel, gx, per in made:
            assert kernel.endswith("_j") and len(per) == len(cut)
            if not kernel.startswith(("qwk_gu_", "qwk_dnr_")):
                continue
            assert gx == sum(per) <= 256 and all(p % 8 == 0 for p in per)  # behind one another, eights for the eight XCDs
            for p, w in zip(per, work):
                assert abs(p - 256 * w / sum(work)) <= 12, (cut, kernel, per)


ROUNDS = r"""
static void on_launch(const char *fname, unsigned gx, unsigned bx, const void *args) { (void)fname, (void)gx, (void)bx, (void)args; }
int main(void) {
    for (unsigned tpe = 16; tpe <= 160; tpe += 16)
        for (unsigned U = 1; U <= 161; U++)
            for (unsigned nwg = 1; nwg <= 256; nwg++) { // (dn_range_body's loop)
                const unsigned V = U * tpe, all = (V + nwg - 1) / nwg, per = all > tpe ? QW_RANGE_PER(all, tpe) : all;
                unsigned rounds = 0, most = 0;
                for (unsigned base = 0; base < V; base += nwg * per) rounds++, most += per;
                if (per > tpe || rounds != QW_ROUNDS(all, tpe) || most >= all + rounds) return printf("%u experts of %u tiles, %u workgroups: %u rounds of %u\n", U, tpe, nwg, rounds, per), 1;
            }
    return 0;
}
"""


def test_rounds_of_down_by_ranges_are_filled_evenly(tmp_path):
    """No workgroup has more than its share and a tile a round, and none more than an expert's tiles in a round."""
    hostrt.run(tmp_path, ROUNDS)


def test_every_joined_kernel_has_a_test_that_sees_it_run(tmp_path):
    cases = next(m for m in test_gpu_joined.test_groups_that_go_out_together.pytestmark if m.name == "parametrize").args[1]
    seen = {"qwk_%s_j" % k for c in cases for k in c[8] + (c[9] or [])}
    assert seen == set(hostrt.run(tmp_path, NAMES).split())


def test_which_launches_a_step_makes(tmp_path):
    """Sets of up to four neighbouring groups of the same kernels, launch for launch; all launches of a group are joined, or none."""
    iq3, kq = (IQ3, 1, 512, 256, 64, 4, 1), (K4, 1, 512, 256, 64, 4, 1)  # (Q6_K rows of less than 64 MB: not joined)
    j3 = ["qwk_pre_w1_s121_j", "qwk_gu_f121_c2_j", "qwk_dnq_f121_c1_s121_c1_j"]
    one = ["qwk_pre_w1_s121", "qwk_gu_f121_c2", "qwk_dnc_f121_c1_s121_c1"]
    alone = [k[:-2] for k in j3]
    nl = ["qwk_pre_w1_kq_j", "qwk_gu_f121_c2_j", "qwk_dnr_f120_c10_s120_c10_j", "qwk_cmb_j"]
    steps = [((*iq3, [16]), alone), ((*iq3, [9, 9]), j3), ((*iq3, [16] * 4), j3), ((*iq3, [12] * 5), j3 + alone), ((*iq3, [8] * 6), j3 + j3), ((*iq3, [16, 16, 1]), None),
             ((*iq3[:-1], 0, [9, 9]), None), ((IQ3_Q8, *iq3[1:], [7, 7, 7]), ["qwk_pre_w1_s8_j", j3[1], "qwk_dnq_f121_c1_s8_c4_j"]), ((NL, 1, 512, 640, 64, 4, 1, [16] * 3), nl),
             ((*kq, [9, 9]), ["qwk_pre_w1_kq", "qwk_gu_f112_c2", "qwk_dnr_f14_c1_s14_c1", "qwk_cmb"] * 2)]
    for (step, want), (made, cut) in zip(steps, launches(tmp_path, [s for s, _ in steps])):
        if want is None and step[-1] == [9, 9]:  # the first step of a path: its first group also makes the path's table, and is another sequence of launches
            want = alone + alone
        elif want is None:  # a group of one row has a form of its own
            at = cut.index(1)
            want = {0: one + j3, 1: alone + one + alone, 2: j3 + one}[at]
        assert [k for k, _, _ in made] == want, (step, cut)
        for k, _, per in made:
            assert (per is not None) == k.endswith("_j")


# A device on which groups side by side take F + sum(a + r rows), one by itself F + a + r rows: steps of `rows` again and again, then the cut of each
# (three times as long from gate/up rows in GGUF order, which Q8_0 layers run until their copies are due)
PLANNED = r"""
hipError_t hipMemGetInfo(size_t *avail, size_t *total) { return *avail = *total = (size_t)1 << 38, hipSuccess; }
static double F, A, Rr;
static void on_launch(const char *fname, unsigned gx, unsigned bx, const void *args) {
    (void)gx, (void)bx;
    if (strncmp(fname, "qwk_gu", 6)) return;
    const bool joint = fname[strlen(fname) - 1] == 'j' && fname[strlen(fname) - 2] == '_';
    const qwk_gu_args *a = args;
    const unsigned *gxs = (const unsigned *)(a + QW_JOIN_MAX);
    double t = F;
    for (unsigned j = 0; j < (joint ? QW_JOIN_MAX : 1); j++) t += joint && !gxs[j] ? 0 : A + Rr * a[j].nbr;
    if (!strncmp(fname, "qwk_gu_f8_", 10)) t *= 3;
    static uint32_t noise = 1; // two per cent either way
    noise = noise * 1664525u + 1013904223u;
    device_clock += (uint64_t)(t * 1000 * (0.98 + 0.04 * (noise >> 8) / (1 << 24)));
}
int main(void) {
    qw_gpu *g = device();
    const int type = @type, D = @D, I = @I;
    g->repack = true, g->copy_uses = QW_HIP_COPY_USES, g->copy_budget = (size_t)1 << 37;
    qw_path *p = qw_path_open(g, D, I, 64, 4, 16, true);
    qw_buf w, x, out;
    if (!qw_hip_buf_new_device(g, (size_t)64 * D * I * 2, &w) || !qw_buf_new(g, (size_t)128 * D, &x) || !qw_buf_new(g, (size_t)128 * D, &out)) return printf("no buffers\n"), 1;
    const qw_tensor W = {.buf = &w, .type = type}, R = {.buf = &w, .type = 1};
    const qw_moe_layer M = {.router = R, .sh_gate_w = R, .gate = W, .up = W, .down = W, .sh_gate = W, .sh_up = W, .sh_down = W};
    const double layers[][3] = {@layers};
    const int rows[] = {@rows};
    enum { NR = sizeof rows / sizeof *rows };
    for (size_t l = 0; l < sizeof layers / sizeof *layers; l++) {
        F = layers[l][0], A = layers[l][1], Rr = layers[l][2];
        qw_par *par = qw_par_new();
        uint32_t seed = 1;
        qw_vstep_info info;
        for (int step = 0; step < 600; step++) {
            seed = seed * 1664525u + 1013904223u;
            const int n = rows[(seed >> 16) % NR], ones[64] = {[0 ... 63] = 1};
            if (!qw_path_par_vstep(p, par, &M, ones, n, &x, &out, &info)) return printf("%s\n", g->err), 1;
        }
        for (int i = 0; i < NR; i++) {
            int cut[64];
            const int ng = qw_par_split(par, rows[i], cut);
            printf("%.6g ", (qw_par_cost(par, rows[i]) - qw_par_step_cost(par)) * 1e3);
            for (int k = 0; k < ng; k++) printf("%d ", cut[k]);
            printf("\n");
        }
        qw_par_free(par);
    }
    return 0;
}
"""


def planned(tmp_path, layers, rows, type=21, D=512, I=256):
    """Per layer and step size: the estimate and the cut that the table has come to."""
    text = PLANNED.replace("@layers", ", ".join("{%g, %g, %g}" % l for l in layers)).replace("@rows", ", ".join(map(str, rows)))
    out = hostrt.run(tmp_path, text.replace("@type", str(type)).replace("@D", str(D)).replace("@I", str(I))).splitlines()
    return iter([list(map(float, line.split())) for line in out])


def test_the_cut_and_the_estimate_that_a_layers_times_ask_for(tmp_path):
    """Layers whose groups cost from next to nothing to 120 rows' worth beside their rows, in steps of one group, of one set and of several."""
    layers, rows = [(1, 2, 5), (1, 20, 2.5), (10, 4, 0.5), (1, 60, 0.5), (40, 10, 0.25)], [2, 5, 16, 18, 20, 31, 45, 64]
    made = planned(tmp_path, layers, rows)
    for F, a, r in layers:
        for R in rows:
            estimate, *cut = next(made)
            time = lambda sizes: sum(F for i in range(0, len(sizes), 4)) + sum(a + r * b for b in sizes)  # (no time depends on the order)
            assert sum(cut) == R
            # as good as the fewest groups, which is the best there is (a group's cost beside its rows is never negative)
            assert time(cut) <= 1.04 * time([16] * (R // 16) + [R % 16] * (R % 16 > 0)), (F, a, r, cut)
            # a group by itself: its own time; groups side by side: what they share is priced as in the sets that its sizes came in
            assert estimate == pytest.approx(time(cut), rel=0.03, abs=F if len(cut) > 1 else 0), (F, a, r, cut)


@pytest.mark.parametrize("rows", [28, 45])
def test_times_of_kernels_that_will_not_run_again_are_not_kept(tmp_path, rows):
    """A layer whose copies come after 32 dispatches: what was tried before has no price, and is tried with the copies there."""
    F, a, r = 10, 5, 1
    estimate, *cut = next(planned(tmp_path, [(F, a, r)], [rows], 8, 2048, 512))
    time = lambda sizes: sum(F for i in range(0, len(sizes), 4)) + sum(a + r * b for b in sizes)
    assert time(cut) <= 1.04 * time([16] * (rows // 16) + [rows % 16]), cut
    assert estimate == pytest.approx(time(cut), rel=0.05), cut


def test_times_of_sets_in_the_planners_table():
    p = q.Par()
    p.observe_set([12, 12, 8], 1e6)      # the first sample of a size is dropped, as of a group by itself
    assert [p.joint_cost(b) for b in (12, 8)] == [0, 0] and p.cost(20) == 0
    p.observe_set([12, 12, 8], 60.0)     # nothing known: half evenly, half by rows; one sample a size
    assert p.joint_cost(12) == pytest.approx(60 * (1 / 3 + 12 / 32) / 2) and p.joint_cost(8) == pytest.approx(60 * (1 / 3 + 8 / 32) / 2)
    assert 2 * p.joint_cost(12) + p.joint_cost(8) == pytest.approx(60.0)
    before = p.joint_cost(12), p.joint_cost(8)
    p.observe_set([12, 12, 8], 120.0)    # in proportion to what is known
    assert p.joint_cost(12) == pytest.approx(1.1 * before[0]) and p.joint_cost(8) == pytest.approx(1.1 * before[1])
    assert p.group_cost(12) == p.joint_cost(12)  # never by itself
    for bad in ([], [0, 4], [17, 4], [4] * 65):
        p.observe_set(bad, 10.0)
    p.observe_set([12, 8], -1.0)
    p.observe_set([12, 8], 0.0)
    assert p.joint_cost(12) == pytest.approx(1.1 * before[0]) and p.joint_cost(4) == 0
    for _ in range(2):
        p.observe_set([5], 7.0)          # a set of one is a group by itself
    assert p.group_cost(5) == 7.0 and p.joint_cost(5) == 0
    p.free()
    p = q.Par()                          # sixteen rows: one group at the price of a lone one, or several at theirs
    for b in range(1, 17):
        for _ in range(2):
            p.observe(b, 10.0 + b)
    assert p.split(16) == [16] and p.cost(16) == 26.0 and p.split(18) == [16, 2]
    for _ in range(2):
        p.observe_set([8, 8], 24.0)
    assert p.joint_cost(8) == 12.0 and p.group_cost(8) == 18.0
    assert p.split(16) == [8, 8] and p.cost(16) == 24.0 and p.split(8) == [8] and p.cost(8) == 18.0
    p.free()


FED = r"""
static void on_launch(const char *fname, unsigned gx, unsigned bx, const void *args) { (void)fname, (void)gx, (void)bx, (void)args; }
int main(void) {
    qw_gpu *g = device();
    g->repack = true;
    qw_path *p = qw_path_open(g, 512, 256, 64, 4, 16, true);
    qw_buf w, x, out;
    if (!qw_hip_buf_new_device(g, (size_t)64 * 512 * 256 * 2, &w) || !qw_buf_new(g, 64 * 1024, &x) || !qw_buf_new(g, 64 * 1024, &out)) return printf("no buffers\n"), 1;
    const qw_tensor W = {.buf = &w, .type = 21}, R = {.buf = &w, .type = 1};
    const qw_moe_layer M = {.router = R, .sh_gate_w = R, .gate = W, .up = W, .down = W, .sh_gate = W, .sh_up = W, .sh_down = W};
    qw_par *par = qw_par_new();
    for (int b = 1; b <= 16; b++)
        for (int i = 0; i < 2; i++) qw_par_observe(par, b, b == 12 ? 1e-9 : 50);
    const int ones[60] = {[0 ... 59] = 1};
    qw_vstep_info info;
    for (int step = 0; step < 400; step++)
        if (!qw_path_par_vstep(p, par, &M, ones, 60, &x, &out, &info) || info.ngroups != 5) return printf("%d groups: %s\n", info.ngroups, g->err), 1;
    printf("%.6g %.6g %.6g", qw_par_group_cost(par, 12), qw_par_joint_cost(par, 12), info.gpu_ms);
    return 0;
}
"""


def test_a_set_has_its_own_time_and_so_has_the_group_left_over(tmp_path):
    """Five groups of twelve: four of them as three launches of ten nanoseconds, the fifth as three of its own."""
    alone, beside, step = map(float, hostrt.run(tmp_path, FED).split())
    assert alone == pytest.approx(3e-5, rel=1e-3) and beside == pytest.approx(3e-5 / 4, rel=1e-3) and step == pytest.approx(6e-5, rel=1e-3)


NO_MEMORY = r"""
static unsigned joint;
static void on_launch(const char *fname, unsigned gx, unsigned bx, const void *args) { (void)gx, (void)bx, (void)args, joint += !strncmp(fname + strlen(fname) - 2, "_j", 2); }
int main(void) {
    qw_gpu *g = device();
    g->repack = true;
    qw_path *p = qw_path_open(g, 512, 256, 64, 4, 16, true);
    qw_buf w, x, out;
    if (!qw_hip_buf_new_device(g, (size_t)64 * 512 * 256 * 2, &w) || !qw_buf_new(g, 64 * 1024, &x) || !qw_buf_new(g, 64 * 1024, &out)) return printf("no buffers\n"), 1;
    const qw_tensor W = {.buf = &w, .type = 21}, R = {.buf = &w, .type = 1};
    const qw_moe_layer M = {.router = R, .sh_gate_w = R, .gate = W, .up = W, .down = W, .sh_gate = W, .sh_up = W, .sh_down = W};
    const int ones[64] = {[0 ... 63] = 1};
    for (int step = 0; step < 6; step++) {
        qw_vstep_info info;
        qw_par *par = qw_par_new();
        if (!qw_path_par_vstep(p, par, &M, ones, step ? 40 : 16, &x, &out, &info)) return printf("step %d: %s\n", step, g->err), 1;
        qw_par_free(par);
        allocations_left = step >= 3 ? -1 : 0; // none for the first steps of several groups
        if (step == 1 && allocations_refused != 1) return printf("%u refused\n", allocations_refused), 1;
    }
    return printf("%u %u", joint, allocations_refused), 0;
}
"""


def test_no_memory_for_groups_side_by_side(tmp_path):
    """One group after the other then, and the memory is asked for once and not at every step."""
    (tmp_path / "alloc.h").write_text("""#define _GNU_SOURCE
#include <stdlib.h>
static int allocations_left = -1;
static unsigned allocations_refused;
static inline void *tested_alloc(size_t a, size_t n) {
    if (allocations_left == 0) return allocations_refused++, NULL;
    return aligned_alloc(a, n);
}
#define aligned_alloc tested_alloc
""")
    assert hostrt.run(tmp_path, NO_MEMORY, "-include", str(tmp_path / "alloc.h")).split() == ["0", "1"]


SHARES = r"""
static void on_launch(const char *fname, unsigned gx, unsigned bx, const void *args) { (void)fname, (void)gx, (void)bx, (void)args; }
int main(void) {
    uint32_t seed = 7;
    for (unsigned units = 16; units <= 304; units += 16)
        for (int i = 0; i < 2000; i++) {
            const int m = 2 + i % 3;
            double work[4], all = 0;
            unsigned share[4], sum = 0;
            for (int j = 0; j < m; j++) all += work[j] = 1 + ((seed = seed * 1664525u + 1013904223u) >> 22) % (i % 7 ? 200 : 1000);
            share_units(units, work, m, share);
            for (int j = 0; j < m; j++) {
                sum += share[j];
                if (!share[j] || share[j] % 8 || (units >= 64 && share[j] + 16 < units * work[j] / all)) return printf("%u units, %d parts: %u\n", units, m, share[j]), 1;
            }
            if (units / 8 >= (unsigned)m && sum != units) return printf("%u units, %d parts: %u in all\n", units, m, sum), 1;
        }
    return 0;
}
"""


def test_every_part_gets_compute_units(tmp_path):
    """All of them are shared out, in eights, about as the work asks; and none goes without, however few there are."""
    hostrt.run(tmp_path, SHARES)
