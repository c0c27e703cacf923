/*
 * CPU check (no GPU work) of M-stages folded into the passes: for random CNOT /
 * SWAP / CZ stages the index map and the sign of a pass descriptor (n > 13, the
 * tile and register parts as the kernels combine them) and of a
 * resident block (n <= 13), and the injection masks of every parameter, against
 * the gates applied one by one to every index.  Stages whose map does not fit
 * must keep their per-gate kernels.  Prints "ok" and exits 0 on success.
 */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "qgtl_internal.h"

static uint64_t state = 99;
static uint32_t rnd(uint32_t n)
{
    state = state * 6364136223846793005ull + 1442695040888963407ull;
    return (uint32_t)(state >> 33) % n;
}
static uint32_t par(uint32_t x) { return (uint32_t)__builtin_popcount(x) & 1u; }
static uint32_t bit(uint32_t x, int b) { return (x >> b) & 1u; }

/* the stage's gates on index x; *sign accumulates the CZs */
static uint32_t gates(const qgtl_op_t *ops, int k, uint32_t x, uint32_t *sign)
{
    for (int i = 0; i < k; i++) {
        const uint32_t a = bit(x, ops[i].q0), b = bit(x, ops[i].q1);
        if (ops[i].type == GATE_TYPE_CNOT) x ^= a << ops[i].q1;
        else if (ops[i].type == GATE_TYPE_SWAP) x ^= (a ^ b) * (1u << ops[i].q0 | 1u << ops[i].q1);
        else *sign ^= a & b;
    }
    return x;
}

/* kind 0: a CZ line, 1: a CNOT line, 2: random gates within bits 0..lim - 1 and CZs anywhere,
 * 3: a control below bit 4 for a high target, 4: SWAP of a low with a high qubit, 5: every pair's CZ,
 * 6: CNOTs from high to low qubits and onto high ones from bits 11, 12, and CZs */
static int stage(int kind, int n, qgtl_op_t *ops)
{
    int k = 0;
#define ADD(t, a, b) ops[k++] = (qgtl_op_t){t, a, b, -1, 0.0}
    if (kind < 2)
        for (int q = 0; q + 1 < n; q++) ADD(kind ? GATE_TYPE_CNOT : GATE_TYPE_CZ, q, q + 1);
    if (kind == 2) {
        const int lim = n < 13 ? n : 13;
        for (int i = 0; i < 20; i++) {
            const int t = (int)rnd(3), m = t == 2 ? n : lim, a = (int)rnd((uint32_t)m), b = (a + 1 + (int)rnd((uint32_t)m - 1)) % m;
            ADD(t == 0 ? GATE_TYPE_CNOT : t == 1 ? GATE_TYPE_SWAP : GATE_TYPE_CZ, a, b);
        }
    }
    if (kind == 3) ADD(GATE_TYPE_CZ, 2, 3), ADD(GATE_TYPE_CNOT, (int)rnd(4), n - 1);
    if (kind == 4) ADD(GATE_TYPE_SWAP, (int)rnd(4), n - 1), ADD(GATE_TYPE_CZ, 1, n - 1);
    if (kind == 5)
        for (int a = 0; a < 6; a++)
            for (int b = a + 1; b < 6; b++) ADD(GATE_TYPE_CZ, a * (n - 1) / 5, b * (n - 1) / 5);
    if (kind == 6)
        for (int i = 0; i < 10; i++) {
            if (n > 13) ADD(GATE_TYPE_CNOT, 13 + (int)rnd((uint32_t)n - 13), (int)rnd(11));
            ADD(GATE_TYPE_CNOT, n > 13 ? 11 + (int)rnd(2) : 0, n - 1);
            ADD(GATE_TYPE_CZ, (int)rnd((uint32_t)n - 1), n - 1);
        }
#undef ADD
    return k;
}

/* index map and sign of a descriptor as the register kernels form them, for the layout with register bits rb */
static uint32_t by_pass(const qgtl_pass_desc_t *d, const int32_t *rb, int linear, uint32_t x, uint32_t *sign)
{
    const qgtl_mstage_t *m = &d->mstage;
    const uint32_t low = (1u << 13) - 1u, r = x >> 13;
    uint32_t reg = 0, base = x & low;
    for (int i = 0; i < 5; i++) {
        reg |= bit(x, rb[i]) << i;
        base &= ~(1u << rb[i]);
    }
    uint32_t yl = 0, pre = 0, yh;
    for (int i = 0; i < 13; i++)
        if (bit(base, i)) yl ^= m->a[i];
    for (int i = 0; i < 5; i++)
        if (bit(reg, i)) yl ^= m->reg[i];
    for (int i = 0; i < 17; i++)
        if (bit(r, i)) { yl ^= m->b[i]; pre ^= m->f[i]; }
    yh = pre;
    static const int may[5] = {4, 5, 6, 11, 12};
    for (int i = 0; i < 5; i++)
        if (bit(yl, may[i])) yh ^= m->e[may[i]];
    const uint32_t full = base | r << 13;
    uint32_t acc = 0, s = 0;
    for (int i = 0; i < 30; i++)
        if (bit(full, i)) acc ^= m->sgn[i];
    s = par(acc & full) ^ bit(m->sgn_reg, (int)reg);
    for (int i = 0; i < 5; i++)
        if (bit(reg, i)) s ^= par(m->sgn_bil[i] & full);
    *sign = d->sign ? s : 0;
    return linear ? yl | yh << 13 : x;
}

static int check(int n, int kind)
{
    static qgtl_op_t ops[400], st[64];
    int k = 0, P = 0;
    const int ks = stage(kind, n, st);
    for (int q = 0; q < n; q++) ops[k++] = (qgtl_op_t){GATE_TYPE_RY, q, -1, P++, 0.1 + q};
    memcpy(ops + k, st, sizeof(qgtl_op_t) * (size_t)ks);
    k += ks;
    for (int q = 0; q < n; q++) ops[k++] = (qgtl_op_t){GATE_TYPE_RX, q, -1, P++, 0.3 + q};
    qgtl_plan_t *plan = qgtl_plan_create(n, k, ops, QGTL_MODE_MIXED, NULL);
    if (!plan || ks > QGTL_PERM_MAX || ((struct qgtl_plan *)plan)->nblocks != 2) {
        printf("n %d kind %d: %s\n", n, kind, plan ? "blocks" : qgtl_last_error());
        return 1;
    }
    const struct qgtl_plan *p = (struct qgtl_plan *)plan;
    const qgtl_block_t *b = &p->blocks[0];
    int bad = 0;
    const int fits = n > 13 && !b->mstage_kernels;
    if (n > 13 && b->mstage_kernels != (kind == 3 || kind == 4)) bad = 1;
    qgtl_res_block_t rb;
    static qgtl_c64_t tabs[2 * QGTL_RES_TAB];
    memset(&rb, 0, sizeof rb);
    if (n <= 13) qgtl_resident_block(b, n, &rb, tabs);
    for (uint32_t x = 0; x < 1u << n && !bad; x++) {
        uint32_t s = 0, s2 = 0;
        const uint32_t y = gates(st, ks, x, &s);
        if (fits) {
            const qgtl_pass_desc_t *f = &b->pass[b->npasses - 1];
            if (by_pass(f, f->ph_rbits[f->nphase - 1], f->store == QGTL_STORE_LINEAR, x, &s2) != y || s2 != s) bad = 2;
        } else if (n <= 13) {
            const uint32_t reg = x >> (n - 4), j0 = x & ((1u << (n - 4)) - 1u);
            uint32_t acc = 0, z = 0;
            for (int i = 0; i < n; i++) {
                if (bit(x, i)) z ^= rb.img[i];
                if (bit(j0, i)) acc ^= rb.sgn[i];
            }
            s2 = par(acc & j0) ^ bit(rb.sgn_reg, (int)reg);
            for (int i = 0; i < 4; i++)
                if (bit(reg, i)) s2 ^= par(rb.sgn_bil[i] & j0);
            if ((rb.has_perm ? z : x) != y || (rb.has_sign ? s2 : 0) != s) bad = 4;
        }
        /* partner, selector and sign of the first layer's injections; the constant sits in A */
        for (int q = 0; q < n && !bad; q++) {
            const qgtl_param_t *pp = &p->params[q];
            uint32_t sp = s;
            const uint32_t yp = gates(st, ks, x ^ (1u << q), (s2 = 0, &s2));
            sp ^= s2;
            if ((y ^ pp->v) != yp || par(y & pp->w) != bit(x, q)) bad = 5;
            /* a qubit of the stage holds the RY alone: A[0][1] = -1/2 before the sign */
            int used = 0;
            for (int i = 0; i < ks; i++) used |= st[i].q0 == q || st[i].q1 == q;
            const double have = (par(y & pp->z) ? -1.0 : 1.0) * pp->A.m[1].re;
            if (used ? fabs((sp ? 0.5 : -0.5) - have) > 1e-12 : pp->z != 0) bad = 6;
        }
    }
    if (bad) printf("n %d kind %d: fault %d\n", n, kind, bad);
    qgtl_plan_destroy(plan);
    return bad;
}

int main(void)
{
    static const int ns[] = {6, 9, 13, 14, 16, 17};
    int bad = 0;
    for (int i = 0; i < 6; i++)
        for (int kind = 0; kind < 7; kind++) bad |= check(ns[i], kind);
    if (!bad) printf("ok\n");
    return bad ? 1 : 0;
}
