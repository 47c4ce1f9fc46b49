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
