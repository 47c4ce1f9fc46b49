"""What the host writes into the device's memory itself, and what it leaves to a launch, seen at the first launch of a batch: has the memory
the new bytes already? Each condition of the rule alone keeps the host from it."""
import hostrt

SOURCE = r"""
static const char *watched;
static int seen; // at the first launch since seen was -1: whether the watched byte is the new one
static void on_launch(const char *fname, unsigned gx, unsigned bx, const void *args) {
    (void)fname, (void)gx, (void)bx;
    if (seen < 0) seen = *watched == 2;
    if (!strcmp(fname, "qwk_io")) {
        const qwk_io_args *a = args;
        for (unsigned i = 0; i < a->n; i++) memcpy(a->dst[i], a->src[i], a->bytes[i]);
    }
}
static qw_gpu *g;
static qw_path *p;
static qw_tensor W;
static qw_buf y;
static bool product(qw_batch *b, const qw_buf *x) { return qw_path_qmv_gg(p, b, &W, 64, 512, x, 0, &y, 0, 1, true); }
// One batch over x, whose shadow changes from ones to twos in front of it; before: what comes in between
static int form(const char *what, size_t size, bool host, void (*before)(qw_buf *), bool (*run)(qw_batch *)) {
    qw_buf x;
    if (!qw_buf_new(g, size, &x)) return printf("no buffer\n"), 1;
    memset(x.ptr, 1, size);
    qw_batch *b = qw_batch_begin(g, false);
    if (!product(b, &x) || qw_batch_end(b) < 0) return printf("%s: %s\n", what, g->err), 1;
    if (before) before(&x);
    memset(x.ptr, 2, size);
    qw_hip_buf_mark_dirty(&x);
    watched = ((qw_hbuf *)x.handle)->dptr, seen = -1;
    size_t had, has;
    qw_hip_host_uploads(g, &had);
    b = qw_batch_begin(g, false);
    if (!product(b, &x) || !run(b)) return printf("%s: %s\n", what, g->err), 1;
    qw_hip_host_uploads(g, &has);
    if (seen != host || has - had != (host ? size : 0)) return printf("%s: the host wrote %zu bytes, the memory was %s at the first launch\n", what, has - had, seen ? "new" : "old"), 1;
    if (*watched != 2) return printf("%s: not uploaded\n", what), 1;
    qw_buf_free(&x);
    return 0;
}
static bool end(qw_batch *b) { return qw_batch_end(b) >= 0; }
static bool submit(qw_batch *b) { return qw_batch_submit(b), qw_batch_wait(b) >= 0; }
static bool flush(qw_batch *b) { return qw_batch_flush(b), qw_batch_end(b) >= 0; }
static void address(qw_buf *x) { qw_hip_buf_devptr(x); }
static void written(qw_buf *x) {
    qw_batch *b = qw_batch_begin(g, false);
    (void)(qw_path_qmv_gg(p, b, &W, 64, 512, &y, 0, x, 0, 1, true) && qw_batch_end(b) >= 0);
}
static qw_batch *other;
static void under_way(qw_buf *x) {
    other = qw_batch_begin(g, false);
    (void)product(other, x);
    qw_batch_submit(other);
}
static void elsewhere(qw_buf *x) { // on the other stream
    qw_gpu_set_stream(g, 1);
    under_way(x);
    qw_gpu_set_stream(g, 0);
}
static bool both(qw_batch *b) { return end(b) && qw_batch_wait(other) >= 0; }
static void off(qw_buf *x) { (void)x, g->sw.no_host_up = true; }
static void no_window(qw_buf *x) { (void)x, g->sw.no_host_up = false, g->host_up = false; }
int main(void) {
    g = device(), g->host_up = true;
    p = qw_path_open(g, 1024, 256, 64, 4, 16, true);
    static qw_buf w;
    if (!qw_hip_buf_new_device(g, 64 * 544, &w) || !qw_buf_new(g, 1024, &y)) return printf("no buffers\n"), 1;
    W = (qw_tensor){.buf = &w, .type = 8};
    return form("plain", 1024, true, NULL, end) || form("the limit", QW_HOST_UP_MAX, true, NULL, end) || form("more than the limit", QW_HOST_UP_MAX + 16, false, NULL, end) || form("address", 1024, false, address, end) ||
           form("written", 1024, false, written, end) || form("under way", 1024, false, under_way, both) || form("other stream", 1024, false, elsewhere, both) || form("plain again", 1024, true, NULL, end) ||
           form("submit", 1024, false, NULL, submit) || form("flush", 1024, false, NULL, flush) || form("switched off", 1024, false, off, end) || form("no window", 1024, false, no_window, end);
}
"""


def test_what_the_host_writes_itself(tmp_path):
    hostrt.run(tmp_path, SOURCE)
