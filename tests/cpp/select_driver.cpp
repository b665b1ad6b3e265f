// select_driver.cpp -- prints the kernels that run a call's routed experts
// (k3x_select.hpp), for tests/test_select.py: one call per line of stdin,
// "hidden inter experts tokens top_k split_act split_in shared scaled few rows wide".
#include "k3x_select.hpp"

#include <cstdio>

int main() {
    unsigned h, i, e, t, k, sa, si, sh, sc, few, rows, wide;
    const char* names[] = {"few", "rows", "stream", "wide", "narrow"};
    while (std::scanf("%u %u %u %u %u %u %u %u %u %u %u %u", &h, &i, &e, &t, &k, &sa, &si, &sh, &sc, &few,
                      &rows, &wide) == 12) {
        k3x_hip::RoutedCall c{};
        c.hidden = h;
        c.inter = i;
        c.experts = e;
        c.tokens = t;
        c.top_k = k;
        c.split_act = sa;
        c.split_in = si;
        c.shared = sh;
        c.scaled = sc;
        c.few = few;
        c.rows = rows;
        c.wide = wide;
        std::puts(names[k3x_hip::select_routed(c)]);
    }
    return 0;
}
