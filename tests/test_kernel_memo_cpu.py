"""The table of kernels that a path has met: a kernel is found again, also where the table is full, and a layer takes few places of it."""
import hostrt

FULL = r"""
static void on_launch(const char *fname, unsigned gx, unsigned bx, const void *args) { (void)fname, (void)gx, (void)bx, (void)args; }
int main(void) {
    qw_path *p = calloc(1, sizeof *p);
    static qw_kernel k[4096];
    static const char *const base[] = {"one", "two", "three", "four"};
    for (int round = 0; round < 3; round++)
        for (int i = 0; i < 4096; i++) {
            const int key[QW_MEMO_KEY] = {i / 4 % 16 + 1, i / 64, round};
            bool hit;
            *kernel_memo(p, base[i % 4], key, &hit) = &k[i];
            qw_kernel **again = kernel_memo(p, base[i % 4], key, &hit);
            if (!hit || *again != &k[i]) return printf("kernel %d of round %d is not found a second time\n", i, round), 1;
        }
    return 0;
}
"""

LAYER = r"""
static void on_launch(const char *fname, unsigned gx, unsigned bx, const void *args) { (void)fname, (void)gx, (void)bx, (void)args; }
int main(void) {
    qw_gpu *g = device();
    qw_path *p = qw_path_open(g, 1024, 256, 64, 4, 16, true);
    qw_buf w, x, lg, sel, out;
    if (!qw_hip_buf_new_device(g, (size_t)64 * 1024 * 256 * 2, &w) || !qw_hip_buf_new_device(g, 16 * 2048, &x) || !qw_hip_buf_new_device(g, qw_path_logits_bytes(p, 16), &lg) ||
        !qw_hip_buf_new_device(g, qw_path_sel_bytes(p, 16), &sel) || !qw_hip_buf_new_device(g, 16 * 2048, &out)) return printf("no buffers\n"), 1;
    const qw_tensor W = {.buf = &w, .type = 8}, R = {.buf = &w, .type = 1};
    const qw_moe_layer M = {.router = R, .sh_gate_w = R, .gate = W, .up = W, .down = W, .sh_gate = W, .sh_up = W, .sh_down = W};
    for (int nb = 1; nb <= 16; nb++) {
        qw_batch *b = qw_batch_begin(g, false);
        if (!qw_path_gg_moe(p, b, &M, nb, &x, &lg, &sel, &out) || qw_batch_end(b) < 0) return printf("%d tokens: %s\n", nb, g->err), 1;
    }
    int taken = 0;
    for (int i = 0; i < QW_MEMO; i++) taken += p->memo[i].k != NULL;
    if (taken > 4 * 5 + 1) return printf("%d places\n", taken), 1; // four dispatches built for 1, 2, 4, 8 and 16 tokens, and the tables
    if (qw_path_gg_moe(p, NULL, &M, 17, &x, &lg, &sel, &out) || qw_path_gg_moe(p, NULL, &M, 0, &x, &lg, &sel, &out)) return printf("17 or 0 tokens\n"), 1;
    return 0;
}
"""


def test_a_kernel_is_found_the_second_time(tmp_path):
    hostrt.run(tmp_path, FULL)


def test_places_of_a_layer(tmp_path):
    hostrt.run(tmp_path, LAYER)
