/* A device for the host runtime's tests on the CPU: one in-order queue whose
 * copies, kernels and signals run only when the host waits for them, so a
 * buffer that the host reuses too early, or work that a failed call leaves
 * behind, shows.  Kernels log what they would read.  The launches that no test
 * looks at are generated as functions that return 0. */
#include <stdlib.h>
#include <string.h>

#include "mdx_device.h"

enum { OP_COPY, OP_SET, OP_ROWS, OP_POS, OP_ADVANCE, OP_FILL };
typedef struct {
    int kind, n;
    void* dst;
    const void* src;
    size_t bytes;
} op;
static op g_q[1 << 16];
static int g_head, g_tail;

/* what the tests read and set */
int fake_fail_signal = -1;                /* the signals that still succeed; -1: all do */
int fake_n_rows, fake_n_pos, fake_copied_row;
float fake_rows[1 << 20];                 /* first element of each row that a pass starts from */
int fake_pos[1 << 12];                    /* a pass's first position, as its first layer has it */
int fake_pending(void) { return g_tail - g_head; }
void fake_reset(void) { g_head = g_tail = fake_n_rows = fake_n_pos = 0; fake_fail_signal = -1; }

static int push(int kind, void* dst, const void* src, size_t bytes, int n) {
    if (g_tail == 1 << 16) abort();
    g_q[g_tail++] = (op){kind, n, dst, src, bytes};
    return 0;
}
static void run_to(int end) {
    for (; g_head < end; g_head++) {
        const op* o = &g_q[g_head];
        switch (o->kind) {
            case OP_COPY: memcpy(o->dst, o->src, o->bytes); break;
            case OP_SET: *(int*)o->dst = 1; break;
            case OP_FILL: memset(o->dst, 0, o->bytes); break;
            case OP_ROWS:
                for (int m = 0; m < o->n; m++) fake_rows[fake_n_rows++] = *(const float*)((const char*)o->src + m * o->bytes);
                break;
            case OP_POS: fake_pos[fake_n_pos++] = ((const mdx_state*)o->src)->pos; break;
            case OP_ADVANCE: ((mdx_state*)o->dst)->pos += o->n; break;
        }
    }
}

int mdxrt_device_count(void) { return 1; }
const char* mdxrt_last_error(void) { return "fake"; }
int mdxrt_clock_khz(void) { return 100000; }
int mdxrt_malloc(void** p, size_t bytes) { return (*p = aligned_alloc(256, (bytes + 255) / 256 * 256)) ? 0 : -4; }
int mdxrt_host_alloc(void** p, size_t bytes) { return mdxrt_malloc(p, bytes); }
int mdxrt_uc_acquire(void** p, size_t bytes) { return mdxrt_malloc(p, bytes); }
int mdxrt_free(void* p) { free(p); return 0; }
int mdxrt_host_free(void* p) { free(p); return 0; }
int mdxrt_h2d(void* d, const void* s, size_t n) { memcpy(d, s, n); return 0; }
int mdxrt_d2h(void* d, const void* s, size_t n) { memcpy(d, s, n); return 0; }
int mdxrt_h2d_async(void* d, const void* s, size_t n, void* st) { return push(OP_COPY, d, s, n, 0); }
int mdxrt_d2h_async(void* d, const void* s, size_t n, void* st) { return push(OP_COPY, d, s, n, 0); }
int mdxrt_copy16(void* d, const void* s, size_t n, void* st) { return push(OP_COPY, d, s, n, 0); }
int mdxrt_fill_u32(void* d, uint32_t v, size_t n, void* st) { return push(OP_FILL, d, NULL, 4 * n, 0); }
int mdxrt_stream_create(void** s) { *s = s; return 0; }
int mdxrt_stream_sync(void* s) { run_to(g_tail); return 0; }
int mdxrt_event_create(void** e) { return (*e = calloc(1, sizeof(int))) ? 0 : -4; }
int mdxrt_event_destroy(void* e) { free(e); return 0; }
int mdxrt_event_record(void* e, void* s) { *(int*)e = g_tail; return 0; }
int mdxrt_event_sync(void* e) { run_to(*(int*)e); return 0; }
int mdxrt_event_elapsed_ms(void* a, void* b, float* ms) { *ms = 1.0f; return 0; }
int fake_graphs;                          /* captures begun */
int mdxrt_graph_begin(void* s) { fake_graphs++; return 0; }
int mdxrt_graph_launch(void* e, void* s) { return 0; }
int mdxrt_signal(int* flag, unsigned long long* t, void* s) {
    if (fake_fail_signal == 0) return -4;
    if (fake_fail_signal > 0) fake_fail_signal--;
    return push(OP_SET, flag, NULL, 0, 0);
}
int mdxrt_wait(int* flag, void* s) {
    while (!*flag && g_head < g_tail) run_to(g_head + 1);
    return *flag ? 0 : -4;
}

size_t mdx_attn_decode_scratch_bytes(int nq, int nkv, int hd, int ms) { return 4096; }
size_t mdx_lmhead_scratch_bytes(void) { return 4096; }
size_t mdx_persist_xbuf_bytes(void) { return 4096; }
size_t mdx_gemm_scratch_floats(int M, int N, int K) { return 1024; }
size_t mdx_long_scratch_floats(int M, int N) { return 1024; }
size_t mdx_sample_scratch_bytes(void) { return 4096; }

int mdx_launch_rmsnorm_rows(const float* x, const float* w, float eps, int M, int d, uint16_t* x16, void* s) {
    return push(OP_ROWS, NULL, x, (size_t)d * 4, M);
}
static int log_pos(int pos) {
    mdx_state* st = (mdx_state*)calloc(1, sizeof(mdx_state));    /* lives as long as the queue */
    st->pos = pos;
    return push(OP_POS, NULL, st, 0, 0);
}
int mdx_launch_long_qkv_rope(const uint16_t* x16, int M, const mdx_wdesc* w, int pos0, const float* qn, const float* kn, float eps,
                             const float* c, const float* sn, int nq, int nkv, int hd, int style, float* q, uint16_t* kc,
                             uint16_t* vc, void* s) {
    return log_pos(pos0);
}
int mdx_launch_qk_rope_append_rows(const mdx_state* st, const float* qkv, int M, const float* qn, const float* kn, float eps,
                                   const float* c, const float* sn, int nq, int nkv, int hd, int style, float* q, uint16_t* kc,
                                   uint16_t* vc, void* s) {
    return push(OP_POS, NULL, st, 0, 0);
}
int mdx_launch_qkv_rope_append_rows(const uint16_t* x16, int M, const mdx_wdesc* w, float* scratch, const mdx_state* st,
                                    const float* qn, const float* kn, float eps, const float* c, const float* sn, int nq, int nkv,
                                    int hd, int style, float* q, uint16_t* kc, uint16_t* vc, void* s) {
    return push(OP_POS, NULL, st, 0, 0);
}
int mdx_launch_advance(mdx_state* st, int n, void* s) { return push(OP_ADVANCE, st, NULL, 0, n); }
int mdx_launch_copy_row(const float* x, int row, int d, float* dst, void* s) {
    fake_copied_row = row;
    return push(OP_COPY, dst, x + (size_t)row * d, (size_t)d * 4, 0);
}
int mdx_launch_lmhead(const float* h, const float* nw, float eps, const mdx_wdesc* w, float* logits, void* scr, mdx_state* st,
                      int* out, int adv, mdx_host_res* res, void* s) {
    return push(OP_COPY, logits, h, 4, 0);      /* logits[0]: the row's first element */
}
