/* SPDX-License-Identifier: Apache-2.0 */
/*
 * The workspace sizes of the device entry points, asked of their own layout functions on a
 * machine without a GPU: k3_devapi.c is compiled into this program, the other objects of the
 * library are linked to it, and k3k_cu_count is replaced (-Wl,--wrap) by the CU count given.
 *
 *   k3_ws_sizes CUS < lines of "T hidden inter experts topk prec"
 *
 * prints for each line: the least scratch k3d_moe_routed accepts, what it takes when there is
 * room, k3d_moe_ws; the same three for the router alone; and the largest of each "takes" over
 * the batches of 1 .. T tokens.
 */
#include "../../kimi-k3-in-c_amd/csrc/k3_devapi.c"

static int g_cus;
int __wrap_k3k_cu_count(void);
int __wrap_k3k_cu_count(void) { return g_cus; }

static size_t moe_takes(int T, int hidden, int inter, int n, int k, int prec)
{
    Carve c = {NULL, 0};
    MoeWs w;
    RtWs r;
    moe_layout(&c, &w, T, hidden, inter, n, k, prec);
    (void)router_plan(&c, &r, (size_t)-1, T, hidden, n, NULL);
    return c.off;
}

static size_t router_takes(int T, int hidden, int n, size_t *least)
{
    Carve c = {NULL, 0};
    RtWs r;
    if (least) {
        (void)router_plan(&c, &r, 0, T, hidden, n, least);
        c.off = 0;
    }
    (void)router_plan(&c, &r, (size_t)-1, T, hidden, n, NULL);
    return c.off;
}

int main(int argc, char **argv)
{
    int T, h, i, n, k, prec;
    if (argc != 2) return 2;
    g_cus = atoi(argv[1]);
    while (scanf("%d %d %d %d %d %d", &T, &h, &i, &n, &k, &prec) == 6) {
        size_t least, rleast, mm = 0, rm = 0;
        (void)k3dx_moe_fits(0, T, h, i, n, k, prec, &least);
        const size_t rt = router_takes(T, h, n, &rleast);
        for (int t = 1; t <= T; t++) {
            const size_t m = moe_takes(t, h, i, n, k, prec), r = router_takes(t, h, n, NULL);
            if (m > mm) mm = m;
            if (r > rm) rm = r;
        }
        printf("%zu %zu %zu %zu %zu %zu %zu %zu\n", least, moe_takes(T, h, i, n, k, prec), k3d_moe_ws(T, h, i, n, k, prec),
               rleast, rt, k3d_router_ws(T, h, n), mm, rm);
    }
    return 0;
}
