// Host driver of qg_gram64_split.hpp: for K M N chunks triples on stdin, one line "own nch per mb nb bm bn"
// each (own: whether the FP64 Gram kernel is chosen over the library's product in `chunks` chunks).
#include <cstdio>
#include "../../qumasun_amd/csrc/qg_gram64_split.hpp"

int main() {
    long long K, chunks;
    int M, N;
    while (std::scanf("%lld %d %d %lld", &K, &M, &N, &chunks) == 4) {
        const qg::GramSplit g = qg::gram64_split(K, M, N);
        std::printf("%d %lld %lld %d %d %d %d\n", (int)qg::gram64_faster(K, M, N, chunks), (long long)g.nch,
                    (long long)g.per, g.mb, g.nb, g.bm, g.bn);
    }
}
