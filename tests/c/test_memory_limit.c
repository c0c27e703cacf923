/*
 * CPU check of plans at the limit of device memory: the thin HIP layer is
 * replaced (this program's functions come before the library's) by one that
 * hands out addresses within a limit, launches nothing and checks that what a
 * launch would touch lies within a live allocation.
 *   - A plan that does not fit says so at every execute, launches nothing on buffers
 *     that it does not have, and runs once there is room.
 *   - A circuit without a CNOT ring needs no more device memory than one whose
 *     states stay in place (besides its phase tables).
 * Prints "ok" and exits 0 on success.
 */
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "qgtl_internal.h"

#define EXPORT __attribute__((visibility("default")))
enum { MAX_ALLOC = 4096 };
static struct { uintptr_t at; size_t len; } live[MAX_ALLOC];
static int nlive, bad, linear_passes, gate_kernels;
static size_t limit = SIZE_MAX, used, peak;
static uintptr_t next_addr = (uintptr_t)1 << 44;

static void touch(const void *p, size_t len, const char *what)
{
    const uintptr_t a = (uintptr_t)p;
    for (int i = 0; i < nlive; i++)
        if (a >= live[i].at && a + len <= live[i].at + live[i].len) return;
    if (!bad++) printf("%s touches %p + %zu: no allocation\n", what, p, len);
}

/* ---- memory */
EXPORT int qgtl_hip_init(int d) { (void)d; return 0; }
EXPORT const char *qgtl_hip_last_error(void) { return "out of memory"; }
EXPORT int qgtl_hip_malloc(void **ptr, size_t bytes)
{
    *ptr = NULL;
    if (bytes == 0) return 0;
    if (bytes > limit - used || nlive == MAX_ALLOC) return -2;
    live[nlive].at = next_addr;
    live[nlive++].len = bytes;
    *ptr = (void *)next_addr;
    next_addr += (bytes + 4095) / 4096 * 4096 + 4096;
    used += bytes;
    if (used > peak) peak = used;
    return 0;
}
EXPORT int qgtl_hip_free(void *ptr)
{
    if (!ptr) return 0;
    for (int i = 0; i < nlive; i++)
        if (live[i].at == (uintptr_t)ptr) {
            used -= live[i].len;
            live[i] = live[--nlive];
            return 0;
        }
    bad++;
    printf("freed twice: %p\n", ptr);
    return 0;
}
EXPORT int qgtl_hip_mem_free(size_t *f) { *f = limit == SIZE_MAX ? (size_t)64 << 30 : limit - used; return 0; }
EXPORT int qgtl_hip_host_alloc(void **ptr, size_t bytes) { *ptr = bytes ? calloc(1, bytes) : NULL; return bytes && !*ptr ? -2 : 0; }
EXPORT int qgtl_hip_host_free(void *ptr) { free(ptr); return 0; }
EXPORT int qgtl_hip_h2d(void *d, const void *s, size_t n) { (void)s; if (n) touch(d, n, "h2d"); return 0; }
EXPORT int qgtl_hip_d2h(void *d, const void *s, size_t n) { if (n) { touch(s, n, "d2h"); memset(d, 0, n); } return 0; }
EXPORT int qgtl_hip_d2d(void *d, const void *s, size_t n) { if (n) { touch(d, n, "d2d"); touch(s, n, "d2d"); } return 0; }
EXPORT int qgtl_hip_sync(void) { return 0; }
EXPORT int qgtl_hip_set_lane(int l) { (void)l; return 0; }
EXPORT int qgtl_hip_event_create_sync(qgtl_hip_event_t *e) { *e = (qgtl_hip_event_t)1; return 0; }
EXPORT int qgtl_hip_event_create(qgtl_hip_event_t *e) { *e = (qgtl_hip_event_t)1; return 0; }
EXPORT int qgtl_hip_event_record(qgtl_hip_event_t e) { (void)e; return 0; }
EXPORT int qgtl_hip_event_destroy(qgtl_hip_event_t e) { (void)e; return 0; }
EXPORT int qgtl_hip_lane_signal(qgtl_hip_event_t e) { (void)e; return 0; }
EXPORT int qgtl_hip_lane_wait(qgtl_hip_event_t e) { (void)e; return 0; }

/* ---- launches */
EXPORT int qgtl_hip_fill_zero_state_c64(void *psi, int n) { touch(psi, (size_t)8 << n, "fill"); return 0; }
EXPORT int qgtl_hip_fill_zero_state_c128(void *psi, int n) { touch(psi, (size_t)16 << n, "fill"); return 0; }
EXPORT int qgtl_hip_copy_f32x4(void *d, const void *s, size_t c) { touch(d, 16 * c, "copy"); touch(s, 16 * c, "copy"); return 0; }
EXPORT int qgtl_hip_c64_to_split(const void *s, void *d, int n)
{
    touch(s, (size_t)8 << n, "split");
    touch(d, (size_t)8 << n, "split");
    return 0;
}
static void states(const void *p, size_t stride, int k, int n, const char *what)
{
    touch(p, (stride * (size_t)(k - 1) + ((size_t)1 << n)) * 8, what);
}
EXPORT int qgtl_hip_pass_c64(const qgtl_pass_desc_t *p, const void *s, void *d, size_t stride, int k, int v, int split,
                             const void *tabs)
{
    (void)v, (void)split;
    states(s, stride, k, p->n, "pass");
    states(d, stride, k, p->n, "pass");
    if (tabs) touch(tabs, 2 * QGTL_PHASE_TAB * 8, "tables");
    if (p->store == QGTL_STORE_LINEAR) linear_passes++;
    if ((p->store == QGTL_STORE_LINEAR || p->store == QGTL_STORE_RING) && s == d) bad++, printf("store in place\n");
    return 0;
}
EXPORT int qgtl_hip_pass_c64_inject(const qgtl_pass_desc_t *p, const void *psi, const void *slots, void *d, size_t stride,
                                    int k, int split, int signs, const void *tabs)
{
    (void)split, (void)signs;
    states(psi, 0, 1, p->n, "inject pass");
    states(d, stride, k, p->n, "inject pass");
    touch(slots, sizeof(qgtl_inject_slot_t) * (size_t)k, "slots");
    touch(tabs, 2 * QGTL_PHASE_TAB * 8, "tables");
    if (p->store == QGTL_STORE_LINEAR) linear_passes++;
    return 0;
}
EXPORT int qgtl_hip_inject_c64(const qgtl_inject_desc_t *i, const void *psi, void *d, size_t stride, double *partials,
                               int *tiles, int split)
{
    (void)split;
    states(psi, 0, 1, i->n, "inject");
    states(d, stride, i->K, i->n, "inject");
    *tiles = 1;
    if (partials) touch(partials, (size_t)i->K * 32, "inject sums");
    return 0;
}
EXPORT int qgtl_hip_inject_sums_c64(const qgtl_inject_desc_t *i, const void *psi, double *partials, int *tiles)
{
    states(psi, 0, 1, i->n, "inject sums");
    touch(partials, (size_t)i->K * 32, "inject sums");
    *tiles = 1;
    return 0;
}
EXPORT int qgtl_hip_reduce_partials_f64(const double *p, int K, int tiles, double *out)
{
    touch(p, (size_t)K * (size_t)tiles * 32, "reduce");
    touch(out, (size_t)K * 32, "reduce");
    return 0;
}
#define GATE(name)                                                                     \
    EXPORT int name(void *b, size_t stride, int k, int n, int c, int t)                \
    {                                                                                  \
        (void)c, (void)t;                                                              \
        states(b, stride, k, n, #name);                                                \
        gate_kernels++;                                                                \
        return 0;                                                                      \
    }
GATE(qgtl_hip_cnot_c64)
GATE(qgtl_hip_swap_c64)
GATE(qgtl_hip_cz_c64)
EXPORT int qgtl_hip_gram_bf16x3(const void *D, int P, size_t N, float *part, int nchunks, int terms)
{
    (void)terms;
    touch(D, (size_t)P * N * 8, "Gram");
    touch(part, (size_t)nchunks * (size_t)qgtl_hip_gram_tiles(P) * 128 * 128 * 4, "Gram");
    return 0;
}
EXPORT int qgtl_hip_gram_reduce(const float *part, int P, int nchunks, double *C)
{
    touch(part, (size_t)nchunks * (size_t)qgtl_hip_gram_tiles(P) * 128 * 128 * 4, "Gram reduce");
    const size_t R = ((size_t)P * 2 + 127) / 128 * 128;
    touch(C, R * R * 8, "Gram reduce");
    return 0;
}
EXPORT int qgtl_hip_gram_cplx(const void *D, int P, size_t N, float *part, int nchunks, int products, int amps)
{
    (void)products, (void)amps;
    touch(D, (size_t)P * N * 8, "Gram");
    touch(part, (size_t)nchunks * qgtl_hip_gram_cplx_partial_floats(P) * 4, "Gram");
    return 0;
}
EXPORT int qgtl_hip_gram_cplx_reduce(const float *part, int P, int nchunks, double *G)
{
    touch(part, (size_t)nchunks * qgtl_hip_gram_cplx_partial_floats(P) * 4, "Gram reduce");
    const size_t R = ((size_t)P + 127) / 128 * 128;
    touch(G, R * R * 16, "Gram reduce");
    return 0;
}
static int finalize(const double *C, int P, double *Q) { touch(C, 16, "finalize"); touch(Q, (size_t)P * P * 16, "finalize"); return 0; }
EXPORT int qgtl_hip_qgt_finalize(const double *C, const double *inj, int P, double *Q, double *host)
{
    (void)host;
    touch(inj, (size_t)P * 32, "finalize");
    return finalize(C, P, Q);
}
EXPORT int qgtl_hip_qgt_finalize_psi(const double *C, int P, double *Q, double *h) { (void)h; return finalize(C, P, Q); }
EXPORT int qgtl_hip_qgt_finalize_cplx(const double *C, int P, double *Q, double *h) { (void)h; return finalize(C, P, Q); }
EXPORT int qgtl_hip_gate1q_c128(void *psi, int n, int q, const double *m) { (void)q, (void)m; touch(psi, (size_t)16 << n, "gate"); return 0; }
EXPORT int qgtl_hip_cgate_c128(void *psi, int n, int c, int t, const double *m)
{
    (void)c, (void)t, (void)m;
    touch(psi, (size_t)16 << n, "gate");
    return 0;
}
EXPORT int qgtl_hip_gram_f64(const void *D, int P, size_t N, double *part, double *G)
{
    touch(D, (size_t)P * N * 16, "Gram");
    touch(part, 8, "Gram");
    touch(G, (size_t)P * P * 16, "Gram");
    return 0;
}
EXPORT int qgtl_hip_dotc_c128(const void *D, int P, size_t N, const void *psi, double *part, double *a)
{
    touch(D, (size_t)P * N * 16, "dot");
    touch(psi, N * 16, "dot");
    touch(part, 8, "dot");
    touch(a, (size_t)P * 16, "dot");
    return 0;
}
EXPORT int qgtl_hip_qgt_finalize_plain(const double *G, const double *a, int P, double *Q)
{
    touch(a, (size_t)P * 16, "finalize");
    return finalize(G, P, Q);
}

EXPORT int qgtl_hip_fill_f32(void *d, size_t count, float v) { (void)v; touch(d, 4 * count, "fill"); return 0; }
EXPORT int qgtl_hip_pauli_apply_c64(const void *psi, void *out, int n, int nterms, const void *terms)
{
    touch(psi, (size_t)8 << n, "H psi");
    touch(out, (size_t)8 << n, "H psi");
    touch(terms, sizeof(qgtl_pauli_term_t) * (size_t)nterms, "H psi");
    return 0;
}
EXPORT int qgtl_hip_dot_states_c64(const void *D, size_t stride, int K, const void *v, int n, double *part, int *tiles,
                                   int planes)
{
    (void)planes;
    states(D, stride, K, n, "dot");
    touch(v, (size_t)8 << n, "dot");
    touch(part, (size_t)K * 32, "dot");
    *tiles = 1;
    return 0;
}
EXPORT int qgtl_hip_energy_gradient_finalize(const double *dk, const double *psi, int P, double *out)
{
    touch(dk, (size_t)P * 32, "energy");
    touch(psi, 32, "energy");
    touch(out, (size_t)(P + 1) * 8, "energy");
    return 0;
}
EXPORT int qgtl_hip_ng_assemble(const double *Q, const int *slot, int P, double lambda, const double *eg, double *A,
                                double *D, double *g)
{
    (void)lambda;
    touch(Q, (size_t)P * P * 16, "assemble");
    touch(slot, (size_t)P * 4, "assemble");
    touch(eg, (size_t)(P + 1) * 8, "assemble");
    touch(A, (size_t)P * P * 8, "assemble");
    touch(D, (size_t)P * 8, "assemble");
    touch(g, (size_t)P * 8, "assemble");
    return 0;
}
EXPORT int qgtl_hip_cholesky_solve_f64(double *A, const double *b, double *x, int P, int batch, double lambda, int *status)
{
    (void)batch, (void)lambda;
    touch(A, (size_t)P * P * 8, "solve");
    touch(b, (size_t)P * 8, "solve");
    touch(x, (size_t)P * 8, "solve");
    touch(status, 4, "solve");
    return 0;
}

/* grouped launches: the items are host structures that the copy to the device left behind */
EXPORT int qgtl_hip_cu_count(void) { return 256; }
EXPORT int qgtl_hip_event_elapsed_ms(qgtl_hip_event_t a, qgtl_hip_event_t b, float *ms) { (void)a, (void)b; *ms = 0.f; return 0; }
EXPORT int qgtl_hip_phase_tables_grouped(const qgtl_pass_desc_t *d, int n, void *tabs)
{
    touch(d, sizeof *d * (size_t)n, "phase tables");
    touch(tabs, 2 * QGTL_PHASE_TAB * 8 * (size_t)n, "phase tables");
    return 0;
}
#define GROUPED(name, item, ...)                                                       \
    EXPORT int name(const item *items, int n, uint32_t units, int grid, ##__VA_ARGS__) \
    {                                                                                  \
        (void)units, (void)grid;                                                       \
        touch(items, sizeof *items * (size_t)n, #name);                                \
        return 0;                                                                      \
    }
GROUPED(qgtl_hip_fill_grouped, qgtl_fill_item_t)
GROUPED(qgtl_hip_pass_grouped, qgtl_pass_item_t, int variant __attribute__((unused)))
GROUPED(qgtl_hip_inject_grouped, qgtl_inject_item_t)
GROUPED(qgtl_hip_gram_grouped, qgtl_gram_item_t, int terms __attribute__((unused)))
GROUPED(qgtl_hip_gram_reduce_grouped, qgtl_gram_reduce_item_t)
GROUPED(qgtl_hip_finalize_grouped, qgtl_finalize_item_t)
GROUPED(qgtl_hip_gram_cplx_grouped, qgtl_gram_item_t, int products __attribute__((unused)))
GROUPED(qgtl_hip_gram_cplx_reduce_grouped, qgtl_gram_reduce_item_t)
GROUPED(qgtl_hip_finalize_cplx_grouped, qgtl_finalize_item_t)

/* ---- circuits: L layers of RY, RZ on every qubit and a line or ring of two-qubit gates */
enum { N_QUBITS = 14, LAYERS = 4 };
static int circuit(int two, int ring, qgtl_op_t *ops)
{
    int k = 0, par = 0;
    for (int l = 0; l < LAYERS; l++) {
        for (int q = 0; q < N_QUBITS; q++) {
            ops[k++] = (qgtl_op_t){GATE_TYPE_RY, q, -1, par++, 0.3};
            ops[k++] = (qgtl_op_t){GATE_TYPE_RZ, q, -1, par++, 0.4};
        }
        for (int q = 0; q + 1 < N_QUBITS + ring; q++) ops[k++] = (qgtl_op_t){two, q, (q + 1) % N_QUBITS, -1, 0.0};
    }
    return k;
}

static int fail(const char *what) { printf("%s\n", what); return 1; }

int main(void)
{
    static qgtl_op_t ops[LAYERS * N_QUBITS * 3];
    const int P = 2 * N_QUBITS * LAYERS;
    double *Q = malloc(sizeof(double) * 2 * (size_t)P * P);
    /* graphs are not part of this */
    const qgtl_tune_t tune = {.no_graph = 1};
    const int modes[3] = {QGTL_MODE_MIXED, QGTL_MODE_MIXED, QGTL_MODE_FP64_PLAIN};

    /* 1. too little memory, at every allocation in turn: an error each time */
    for (int kind = 0; kind < 3; kind++) {
        const int k = circuit(kind == 0 ? GATE_TYPE_CZ : GATE_TYPE_CNOT, kind == 1, ops);
        limit = SIZE_MAX;
        peak = used;
        qgtl_plan_t *p = qgtl_plan_create(N_QUBITS, k, ops, modes[kind], &tune);
        if (!p || qgtl_plan_execute(p, Q, NULL)) return fail("a plan with room enough fails");
        qgtl_plan_destroy(p);
        if (used) return fail("a destroyed plan keeps memory");
        const size_t need = peak;
        p = qgtl_plan_create(N_QUBITS, k, ops, modes[kind], &tune);
        for (size_t l = 0; l < need; l += need / 200) {
            limit = l;
            const int r1 = qgtl_plan_execute(p, Q, NULL), r2 = qgtl_plan_execute(p, Q, NULL);
            if (bad) return 1;
            if (!r1 != !r2) return fail("a second execute at the same limit ends otherwise");
            if (!r1) break;                  /* optional buffers left out */
        }
        limit = SIZE_MAX;
        if (qgtl_plan_execute(p, Q, NULL) || bad) return fail("a plan that did not fit does not run with room enough");
        qgtl_plan_destroy(p);
        if (used) return fail("a destroyed plan keeps memory");
    }
    /* ... and to a Hamiltonian's, the energy's and the natural gradient's buffers */
    {
        const int k = circuit(GATE_TYPE_CNOT, 1, ops);
        qgtl_pauli_term_t terms[2 * N_QUBITS];
        const int nt = qgtl_tfim_terms(N_QUBITS, 1.0, 0.5, terms);
        const qgtl_ng_config_t cfg = {.lambda = 1e-3, .eta = 0.1, .method = QGTL_SOLVE_CHOLESKY};
        double th[LAYERS * N_QUBITS * 3] = {0.0};
        for (int grow = 0; grow < 2; grow++) {
            limit = SIZE_MAX;
            qgtl_plan_t *p = qgtl_plan_create(N_QUBITS, k, ops, QGTL_MODE_MIXED, &tune);
            if (!p || qgtl_plan_set_hamiltonian(p, 1, terms) || (grow && qgtl_plan_execute(p, Q, NULL)))
                return fail("a plan with room enough fails");
            const size_t base = used;
            int ok = 0;
            for (size_t l = 0; !ok && l < (size_t)64 << 20; l += 100000) {
                limit = base + l;
                const int r1 = qgtl_ng_step(p, th, &cfg, NULL, 0.5, NULL), r2 = qgtl_ng_step(p, th, &cfg, NULL, 0.5, NULL);
                if (bad) return 1;
                if (!r1 != !r2) return fail("a second step at the same limit ends otherwise");
                ok = !r1;
            }
            if (!ok) return fail("no step with room enough");
            /* more terms than there is room for: an error, and the step says that there are none */
            limit = used;
            if (!qgtl_plan_set_hamiltonian(p, nt, terms) || !qgtl_ng_step(p, th, &cfg, NULL, 0.5, NULL) || bad)
                return fail("a Hamiltonian that did not fit is used");
            limit = SIZE_MAX;
            if (qgtl_plan_set_hamiltonian(p, nt, terms) || qgtl_ng_step(p, th, &cfg, NULL, 0.5, NULL) || bad)
                return fail("a Hamiltonian that fits is not used");
            qgtl_plan_destroy(p);
            if (used) return fail("a destroyed plan keeps memory");
        }
    }

    /* ... and to a batch that is tuned to more than there is room for */
    {
        const int n[2] = {N_QUBITS, N_QUBITS};
        const int k = circuit(GATE_TYPE_CNOT, 1, ops), nops[2] = {k, k};
        qgtl_op_t *two = malloc(2 * sizeof(qgtl_op_t) * (size_t)k);
        memcpy(two, ops, sizeof(qgtl_op_t) * (size_t)k);
        memcpy(two + k, ops, sizeof(qgtl_op_t) * (size_t)k);
        qgtl_batch_tune_t bt = {.no_graph = 1, .gram_chunk_len = 1 << N_QUBITS};
        limit = SIZE_MAX;
        qgtl_batch_t *b = qgtl_batch_create(2, n, nops, two, &bt);
        double *Qb = malloc(sizeof(double) * 4 * (size_t)P * P);
        if (!b || qgtl_batch_execute(b, Qb, NULL) || bad) return fail("a batch with room enough fails");
        const qgtl_batch_tune_t fine = {.no_graph = 1, .gram_chunk_len = 256};
        limit = used + 1000;
        if (!qgtl_batch_set_tune(b, &fine) || !qgtl_batch_execute(b, Qb, NULL) || !qgtl_batch_execute(b, Qb, NULL) || bad)
            return fail("a tune that did not fit is used");
        limit = SIZE_MAX;
        if (qgtl_batch_set_tune(b, &fine) || qgtl_batch_execute(b, Qb, NULL) || bad) return fail("a tune that fits is not used");
        qgtl_batch_destroy(b);
        free(two);
        free(Qb);
        if (used) return fail("a destroyed batch keeps memory");
    }

    /* 2. CNOT lines within the memory that CZ lines take, whose passes stay in place */
    size_t need = 0;
    for (int kind = 0; kind < 3; kind++) {
        const int k = circuit(kind ? GATE_TYPE_CNOT : GATE_TYPE_CZ, 0, ops);
        limit = kind == 2 ? need : SIZE_MAX;
        peak = used;
        linear_passes = gate_kernels = 0;
        qgtl_plan_t *p = qgtl_plan_create(N_QUBITS, k, ops, QGTL_MODE_MIXED, &tune);
        if (!p || qgtl_plan_execute(p, Q, NULL) || bad) return fail("a circuit without a ring does not run in place");
        if (kind == 0) need = peak;
        if (kind == 1 && (!linear_passes || gate_kernels)) return fail("a CNOT line is not folded where memory allows it");
        if (kind == 2 && (linear_passes || !gate_kernels)) return fail("passes that move indices without their buffer");
        double th[LAYERS * N_QUBITS * 3] = {0.0};
        if (qgtl_plan_set_angles(p, k, th) || qgtl_plan_execute(p, Q, NULL) || bad) return fail("new angles in place");
        qgtl_plan_destroy(p);
        if (used) return fail("a destroyed plan keeps memory");
    }
    /* and within any more */
    const int k = circuit(GATE_TYPE_CNOT, 0, ops);
    for (limit = need; limit < 4 * need; limit += 20000) {
        qgtl_plan_t *p = qgtl_plan_create(N_QUBITS, k, ops, QGTL_MODE_MIXED, &tune);
        if (!p || qgtl_plan_execute(p, Q, NULL) || bad) return fail("more memory than in place, and it does not fit");
        qgtl_plan_destroy(p);
    }
    puts("ok");
    return 0;
}
