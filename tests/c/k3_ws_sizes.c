/* SPDX-License-Identifier: Apache-2.0 */
/*
 * The workspace sizes of the device entry points, asked of their own layout functions on a
 * machine without a GPU: k3_devapi.c is compiled into this program, the other objects of the
 * library are linked to it, and k3k_cu_count is replaced (-Wl,--wrap) by the CU count given.
 *
 *   k3_ws_sizes CUS < lines of "T hidden inter experts topk prec"
 *
 * prints for each line: the least scratch k3d_moe_routed accepts, what it takes when there is
 * room, k3d_moe_ws; the same three for the router alone; and the most that either takes, with
 * the int8 or the fp64 router partials, over the batches of 1 .. T tokens (with a second argument,
 * of its multiples and T).
 */
#include "../../kimi-k3-in-c_amd/csrc/k3_devapi.c"

static int g_cus;
int __wrap_k3k_cu_count(void);
int __wrap_k3k_cu_count(void) { return g_cus; }

/* the bytes of a call with room for all it would take: its layer part before the router's (moe), and
 * the fp64 partials where `f64` (rows that are not aligned) */
static size_t takes(int T, int hidden, int inter, int n, int k, int prec, int moe, int f64)
{
    Carve c = {NULL, 0};
    MoeWs w;
    RtWs r;
    if (moe) moe_layout(&c, &w, T, hidden, inter, n, k, prec);
    (void)router_plan(&c, &r, (size_t)-1, !f64, T, hidden, n, NULL);
    return c.off;
}

int main(int argc, char **argv)
{
    int T, h, i, n, k, prec;
    if (argc < 2) return 2;
    const int step = argc > 2 ? atoi(argv[2]) : 1;
    g_cus = atoi(argv[1]);
    while (scanf("%d %d %d %d %d %d", &T, &h, &i, &n, &k, &prec) == 6) {
        size_t least[2], most[2] = {0, 0};
        Carve c = {NULL, 0};
        RtWs r;
        (void)k3dx_moe_fits(0, T, h, i, n, k, prec, &least[1]);
        (void)router_plan(&c, &r, 0, 1, T, h, n, &least[0]);
        for (int t = 1; t <= T; t = t + step < T || t == T ? t + step : T)
            for (int v = 0; v < 4; v++) {
                const size_t m = takes(t, h, i, n, k, prec, v & 1, v >> 1);
                if (m > most[v & 1]) most[v & 1] = m;
            }
        printf("%zu %zu %zu %zu %zu %zu %zu %zu\n", least[1], takes(T, h, i, n, k, prec, 1, 0), k3d_moe_ws(T, h, i, n, k, prec),
               least[0], takes(T, h, i, n, k, prec, 0, 0), k3d_router_ws(T, h, n), most[1], most[0]);
    }
    return 0;
}
