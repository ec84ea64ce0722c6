/* SPDX-License-Identifier: Apache-2.0 */
/*
 * The HBM bank's device table (k3_bank_table) on a machine without a GPU: k3_bank.c is compiled
 * into this program against stand-ins whose "device" is host memory and which count copies and
 * waits. Exits 0 if everything holds, else with the line that does not.
 */
#include "../../kimi-k3-in-c_amd/csrc/k3_bank.c"

static int g_copies, g_waits, g_no_table;
void k3h_lock(void) {}
void k3h_unlock(void) {}
int k3h_init(void) { return 0; }
void *k3h_stream(void) { return NULL; }
void k3h_set_error(const char *fmt, const char *what) { fprintf(stderr, fmt, what); }
const char *k3k_error(void) { return "stand-in"; }
void *k3k_malloc(size_t n) { return g_no_table && n == 8 * sizeof(K3ExpertQ) ? NULL : malloc(n); }
int k3k_free(void *p) { free(p); return 0; }
int k3k_h2d(void *d, const void *h, size_t n, void *st) { (void)st; memcpy(d, h, n); g_copies++; return 0; }
int k3k_sync(void *st) { (void)st; g_waits++; return 0; }
int k3k_mx_tile(uint8_t *tp, uint8_t *ts, const uint8_t *p, const uint8_t *s, int rows, int in, void *st)
{
    (void)tp; (void)ts; (void)p; (void)s; (void)rows; (void)in; (void)st;
    return -1;
}

#define CHECK(x) do { if (!(x)) { fprintf(stderr, "line %d: %s\n", __LINE__, #x); return __LINE__ & 255 ? __LINE__ & 255 : 1; } } while (0)

static unsigned char g_bytes[32 * 32];
static int up_get(K3ExpertSrc *self, int layer, int expert, K3ExpertQ *q)
{
    (void)self;
    memset(g_bytes, 16 * layer + expert + 1, sizeof g_bytes);
    q->p1 = q->s1 = q->p3 = q->s3 = q->p2 = q->s2 = g_bytes;
    return 0;
}

/* 0 if the table of `layer` points at the bytes of its resident experts and is NULL elsewhere */
static int table_ok(K3ExpertSrc *src, const K3ExpertQ *t, int layer)
{
    for (int e = 0; e < 4; e++) {
        if (!src->resident(src, layer, e, NULL) != !t[e].p1) return 1;
        if (t[e].p1 && (*(const unsigned char *)t[e].p1 != 16 * layer + e + 1 ||
                        *(const unsigned char *)t[e].s2 != 16 * layer + e + 1)) return 1;
    }
    return 0;
}

int main(void)
{
    K3ExpertSrc up;
    K3ExpertQ q;
    const K3ExpertQ *t;
    memset(&up, 0, sizeof up);
    up.get = up_get;
    K3DevBank *b = k3_devbank_create(2, 4, 32, 32, 6, K3_BANK_ROWS, &up);       /* 6 slots for 8 experts */
    CHECK(b);
    K3ExpertSrc *src = k3_devbank_source(b);
    CHECK(!k3_bank_table(src, 0, 4, 1) && g_copies == 0);                       /* empty */
    for (int e = 0; e < 4; e++) CHECK(src->get(src, 0, e, &q) == 0);
    g_copies = g_waits = 0;
    t = k3_bank_table(src, 0, 4, 1);                                            /* all of layer 0 */
    CHECK(t && !table_ok(src, t, 0) && g_copies == 1 && g_waits == 0);
    CHECK(k3_bank_table(src, 0, 4, 1) == t && k3_bank_table(src, 0, 4, 0) == t && g_copies == 1);
    CHECK(!k3_bank_table(src, 0, 5, 0) && !k3_bank_table(src, 2, 4, 0) && !k3_bank_table(&up, 0, 4, 0));
    for (int e = 0; e < 4; e++) CHECK(src->get(src, 1, e, &q) == 0);            /* layer 1 evicts two of layer 0 */
    g_copies = g_waits = 0;
    CHECK(!k3_bank_table(src, 0, 4, 1) && g_copies == 0 && g_waits == 0);       /* nothing sent for nothing */
    t = k3_bank_table(src, 0, 4, 0);
    CHECK(t && !table_ok(src, t, 0) && g_copies == 1 && g_waits == 0);
    t = k3_bank_table(src, 1, 4, 1);
    CHECK(t && !table_ok(src, t, 1) && g_copies == 2 && g_waits == 0);
    for (int e = 0; e < 4; e++) CHECK(src->get(src, 0, e, &q) == 0);
    t = k3_bank_table(src, 0, 4, 1);
    CHECK(t && !table_ok(src, t, 0) && !k3_bank_table(src, 1, 4, 1));
    k3_devbank_destroy(b);
    g_no_table = 1;                                                             /* no memory for the table */
    b = k3_devbank_create(2, 4, 32, 32, 8, K3_BANK_ROWS, &up);
    CHECK(b);
    src = k3_devbank_source(b);
    for (int e = 0; e < 4; e++) CHECK(src->get(src, 0, e, &q) == 0);
    CHECK(!k3_bank_table(src, 0, 4, 1) && !k3_bank_table(src, 0, 4, 0));
    k3_devbank_destroy(b);
    return 0;
}
