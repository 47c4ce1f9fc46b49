"""Who writes a buffer of a batch, decided on the host before the launches go out: how long that takes, and which launches may write the shadow."""
import hostrt

# Blocks of the host code executed from the first recorded product to the last launch (-fsanitize-coverage counts each one)
STEPS = r"""
static uint64_t steps, at_launch;
void __sanitizer_cov_trace_pc(void) { steps++; }
static int products;
__attribute__((no_sanitize("coverage"))) static void on_launch(const char *fname, unsigned gx, unsigned bx, const void *args) {
    (void)gx, (void)bx;
    if (!strncmp(fname, "qwk_qmv", 7) && ((const qwk_qmvm_args *)args)->yh[0]) products++;
    at_launch = steps;
}
int main(void) {
    qw_gpu *g = device();
    qw_path *p = qw_path_open(g, 1024, 256, 64, 4, 16, true);
    uint64_t took[2][2];
    for (int again = 0; again < 2; again++) // the second time everything is known
        for (int big = 0; big < 2; big++) {
            const int n = big ? 1024 : 256;
            qw_buf w, x, y;
            if (!qw_hip_buf_new_device(g, 64 * 272, &w) || !qw_buf_new(g, 512, &x) || !qw_buf_new(g, (size_t)n * 256, &y)) return printf("no buffers\n"), 1;
            const qw_tensor W = {.buf = &w, .type = 8};
            products = 0;
            const uint64_t from = steps;
            qw_batch *b = qw_batch_begin(g, false);
            for (int i = 0; i < n; i++)
                if (!qw_path_qmv_gg(p, b, &W, 64, 256, &x, 0, &y, (size_t)i * 256, 1, true)) return printf("not recorded\n"), 1;
            if (qw_batch_end(b) < 0) return printf("failed: %s\n", g->err), 1;
            took[again][big] = at_launch - from;
            if (products != n) return printf("%d of %d products write the shadow\n", products, n), 1;
            qw_buf_free(&w), qw_buf_free(&x), qw_buf_free(&y);
        }
    printf("%llu %llu\n", (unsigned long long)took[1][0], (unsigned long long)took[1][1]);
    return 0;
}
"""


def test_work_grows_with_the_products_not_with_their_pairs(tmp_path):
    few, many = map(int, hostrt.run(tmp_path, STEPS, "-fsanitize-coverage=trace-pc").split())
    assert many < 6 * few  # four times the products: 4 and the sort's factor of 10 / 8; by pairs 16, by pairs for every launch 64


# Layers recorded by their four dispatches, with Pg, Psh and out at offsets of buffers that the layers share
LAYERS = r"""
static bool layer(qw_path *p, qw_batch *b, const qw_moe_layer *M, int nb, const qw_buf *x, const qw_buf *lg, const qw_buf *sel, const qw_buf *H, const qw_buf *psh, size_t poff, const qw_buf *pd, size_t doff,
                  const qw_buf *out, size_t ooff) {
    const uint32_t nbr = (uint32_t)nb;
    p->rbf = 1;
    qw_kernel *k[4];
    const char *const base[] = {"moe_pre_gg", "moe_gu_gg", "moe_dn_gg", "moe_cmb_gg"};
    for (int i = 0; i < 4; i++)
        if (!(k[i] = gg_kernel(p, base[i], M, nb))) return false;
    qw_batch_kernel(b, k[0]);
    bind_t(b, 0, &M->router), bind_t(b, 1, &M->sh_gate_w), qw_batch_buf(b, 2, x, 0), qw_batch_buf(b, 3, lg, 0), qw_batch_buf(b, 4, &p->cnt, 0), qw_batch_buf(b, 5, sel, 0);
    bind_t(b, 6, &M->sh_gate), bind_t(b, 7, &M->sh_up), qw_batch_buf(b, 8, H, 0), qw_batch_buf(b, 13, &p->tab, 0), qw_batch_bytes(b, 14, &nbr, 4);
    qw_batch_dispatch(b, 1, 1, 1, 256, 1, 1);
    qw_batch_kernel(b, k[1]);
    bind_t(b, 0, &M->gate), bind_t(b, 1, &M->up), bind_t(b, 2, &M->sh_down), qw_batch_buf(b, 3, psh, poff), qw_batch_buf(b, 4, x, 0), qw_batch_buf(b, 5, sel, 0), qw_batch_buf(b, 6, H, 0);
    qw_batch_buf(b, 11, &p->tab, 0), qw_batch_bytes(b, 12, &nbr, 4);
    qw_batch_dispatch(b, 1, 1, 1, 256, 1, 1);
    qw_batch_kernel(b, k[2]);
    bind_t(b, 0, &M->down), qw_batch_buf(b, 2, H, 0), qw_batch_buf(b, 3, sel, 0), qw_batch_buf(b, 7, &p->tab, 0), qw_batch_buf(b, 9, pd, doff);
    qw_batch_dispatch(b, 1, 1, 1, 128, 1, 1);
    qw_batch_kernel(b, k[3]);
    qw_batch_buf(b, 1, psh, poff), qw_batch_buf(b, 3, sel, 0), qw_batch_buf(b, 4, out, ooff), qw_batch_bytes(b, 8, &nbr, 4), qw_batch_buf(b, 9, pd, doff);
    qw_batch_dispatch(b, 1, 1, 1, 256, 1, 1);
    return true;
}
static int downs, outs, unsafe, products;
static void on_launch(const char *fname, unsigned gx, unsigned bx, const void *args) {
    (void)gx, (void)bx;
    if (!strncmp(fname, "qwk_dnc_", 8)) {
        const qwk_dn_args *a = args;
        downs++, outs += a->outh != NULL, unsafe += (a->Ph || a->Pshh) && !a->fin.flag;
    }
    if (!strncmp(fname, "qwk_qmv", 7) && strcmp(fname, "qwk_qmvm_swiglu")) products += ((const qwk_qmvm_args *)args)->yh[0] != NULL;
}
int main(void) {
    enum { D = 1024, I = 256, E = 64, K = 4 };
    qw_gpu *g = device();
    qw_path *p = qw_path_open(g, D, I, E, K, 16, true);
    qw_buf w, x, lg, sel, H, psh, pd, out, y;
    if (!qw_hip_buf_new_device(g, (size_t)E * D * I * 2, &w) || !qw_buf_new(g, 16 * D * 2, &x) || !qw_hip_buf_new_device(g, qw_path_logits_bytes(p, 16), &lg) || !qw_hip_buf_new_device(g, qw_path_sel_bytes(p, 16), &sel) ||
        !qw_hip_buf_new_device(g, 16 * (K + 1) * I * 4, &H) || !qw_buf_new(g, 2 * D * 4, &psh) || !qw_buf_new(g, 2 * K * D * 4, &pd) || !qw_buf_new(g, 2 * D * 2, &out) || !qw_buf_new(g, 64 * 4, &y))
        return printf("no buffers\n"), 1;
    const qw_tensor W = {.buf = &w, .type = 8}, R = {.buf = &w, .type = 1};
    const qw_moe_layer M = {.router = R, .sh_gate_w = R, .gate = W, .up = W, .down = W, .sh_gate = W, .sh_up = W, .sh_down = W};
    for (int last = 0; last < 2; last++) { // a dense product ends the batch, or the second layer does
        downs = outs = unsafe = products = 0;
        qw_batch *b = qw_batch_begin(g, false);
        for (int l = 0; l < 2; l++)
            if (!layer(p, b, &M, 1, &x, &lg, &sel, &H, &psh, (size_t)l * D * 4, &pd, (size_t)l * K * D * 4, &out, (size_t)l * D * 2)) return printf("not recorded\n"), 1;
        if (!last && !qw_path_qmv_gg(p, b, &W, 64, 256, &x, 0, &y, 0, 1, true)) return printf("not recorded\n"), 1;
        if (qw_batch_end(b) < 0) return printf("failed: %s\n", g->err), 1;
        if (downs != 2 || outs != 2 || products != !last) return printf("%d down + combine launches, %d with the shadow of out, %d products with theirs\n", downs, outs, products), 1;
        if (unsafe) return printf("%d launches that do not end their batch store partial results to the host in the ordinary way\n", unsafe), 1;
    }
    return 0;
}
"""


def test_only_stores_past_the_caches_are_left_to_launches_that_do_not_end_the_batch(tmp_path):
    hostrt.run(tmp_path, LAYERS)
