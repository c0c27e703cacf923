/*
 * CPU check (no GPU work): a plan that is given new angles holds the same pass
 * descriptors, injection operators and block matrices, bit for bit, as a plan
 * built at those angles.  Circuits: random single-qubit gates (with and without
 * parameters), the CNOT ring, other CNOT / SWAP / CZ stages and qubits without a
 * gate, below and above one tile, in both sweep forms and schedules.  Prints
 * "ok" and exits 0 on success.
 */
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "qgtl_internal.h"

static uint64_t state = 12345;
static uint32_t rnd(uint32_t n)
{
    state = state * 6364136223846793005ull + 1442695040888963407ull;
    return (uint32_t)(state >> 33) % n;
}
static double angle(void) { return rnd(1u << 30) * (6.283185307179586 / (1u << 30)); }

static int circuit(int n, qgtl_op_t *ops)
{
    static const int names[] = {GATE_TYPE_RX, GATE_TYPE_RY, GATE_TYPE_RZ, GATE_TYPE_H, GATE_TYPE_S,
                                GATE_TYPE_T, GATE_TYPE_SX, GATE_TYPE_X, GATE_TYPE_PHASE};
    int k = 0, p = 0;
    for (int b = 0; b < 4; b++) {
        for (int q = 0; q < n; q++) {
            if (rnd(5) == 0) continue;
            for (int g = 0; g < 2; g++) {
                const int type = names[rnd(9)];
                ops[k++] = (qgtl_op_t){type, q, -1, qgtl_is_param_gate(type) && rnd(4) ? p++ : -1, angle()};
            }
        }
        if (b % 2 == 0)
            for (int q = 0; q < n; q++) ops[k++] = (qgtl_op_t){GATE_TYPE_CNOT, q, (q + 1) % n, -1, 0.0};
        else if (b == 1) {
            ops[k++] = (qgtl_op_t){GATE_TYPE_SWAP, 0, n - 1, -1, 0.0};
            ops[k++] = (qgtl_op_t){GATE_TYPE_CZ, 1, n - 2, -1, 0.0};
        }
    }
    return k;
}

int main(void)
{
    static qgtl_op_t a[4000], b[4000];
    static double ang[4000];
    static const int ns[] = {4, 7, 13, 14, 17, 21, 22, 24, 30};
    int checked = 0;
    for (int v = 0; v < 4; v++)
        for (size_t i = 0; i < sizeof ns / sizeof ns[0]; i++) {
            qgtl_tune_t tune;
            memset(&tune, 0, sizeof tune);
            tune.sweep_form = v & 1;
            tune.sweep_schedule = v >> 1;
            const int k = circuit(ns[i], a);
            memcpy(b, a, sizeof a);
            for (int g = 0; g < k; g++) ang[g] = b[g].angle = angle();
            struct qgtl_plan *p = qgtl_plan_create(ns[i], k, a, QGTL_MODE_MIXED, &tune);
            struct qgtl_plan *q = qgtl_plan_create(ns[i], k, b, QGTL_MODE_MIXED, &tune);
            if (!p || !q || qgtl_plan_set_angles(p, k, ang) != 0) { printf("plan: %s\n", qgtl_last_error()); return 1; }
            if (p->nblocks != q->nblocks || p->P != q->P) { printf("shape differs\n"); return 1; }
            for (int bi = 0; bi < p->nblocks; bi++)
                if (memcmp(&p->blocks[bi], &q->blocks[bi], sizeof(qgtl_block_t))) {
                    printf("n=%d variant %d block %d differs\n", ns[i], v, bi);
                    return 1;
                }
            if (memcmp(p->params, q->params, sizeof(qgtl_param_t) * (size_t)p->P) ||
                memcmp(p->slot_param, q->slot_param, sizeof(int) * (size_t)p->P)) {
                printf("n=%d variant %d parameters differ\n", ns[i], v);
                return 1;
            }
            checked += p->nblocks;
            qgtl_plan_destroy(p);
            qgtl_plan_destroy(q);
        }
    printf("%d blocks\nok\n", checked);
    return 0;
}
