// The training shuffle's steps on the host, one element after another.  The
// links of the second step are made in ascending, descending or scattered order
// of the steps, as the GPU's lanes may make them; LIST is the sorted buffer's
// length, so that short lists reach the insertion in place.
#include <vector>

#include "../../radiancecascade_amd/csrc/rc_shuffle.hpp"

template <int LIST>
static void sort_all(int n, int *head, int *next)
{
    int buf[LIST];
    for (int p = 0; p < n; ++p) rc::shuffle_sort_list<LIST>(p, head, next, buf, 1);
}

extern "C" int shuffle_host(uint64_t state, int n, int list, int links, int *order, int *longest)
{
    std::vector<int> head(n, -1), next(n, -1), count(n, 0);
    order[0] = 0;
    for (int k = 1; k < n; ++k) {
        const int step = links == 0 ? k : links == 1 ? n - k : (int)((uint64_t)k * 7919 % (uint64_t)n);
        const int i = links == 2 && n % 7919 == 0 ? k : step;
        const int j = rc::shuffle_target(state, n, i);
        order[i] = j;
        next[i] = head[j];
        head[j] = i;
        ++count[j];
    }
    *longest = 0;
    for (int c : count) *longest = c > *longest ? c : *longest;
    switch (list) {
    case 1: sort_all<1>(n, head.data(), next.data()); break;
    case 2: sort_all<2>(n, head.data(), next.data()); break;
    case 5: sort_all<5>(n, head.data(), next.data()); break;
    case 24: sort_all<rc::kShuffleList>(n, head.data(), next.data()); break;
    default: return 1;
    }
    for (int i = 0; i < n; ++i) rc::shuffle_resolve(i, order, head.data(), next.data());
    return 0;
}
