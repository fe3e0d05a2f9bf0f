// Counts the vectors a DenseBatch gives back: two items with five vectors, two
// of them handed over as the solve does.  No GPU work: dmed_vec_free is here.
#include <cstdio>

#include "../dmft-ed_amd/csrc/dmed_internal.h"

static int freed = 0;

extern "C" int dmed_vec_free(dmed_vec *v)
{
    if (v) ++freed;
    delete v;
    return 0;
}

int main()
{
    using namespace dmed;
    std::vector<dmed_vec *> taken;
    {
        DenseBatch b;
        for (int k = 0; k < 2; ++k) {
            DenseItem it;
            for (int q = 0; q < 2 + k; ++q) it.vecs.push_back(new dmed_vec{nullptr, DMED_FP64, 0, nullptr});
            b.items.push_back(std::move(it));
        }
        taken = std::move(b.items[0].vecs);
        b.items[0].vecs.clear();
    }
    const int by_batch = freed;
    for (dmed_vec *v : taken) dmed_vec_free(v);
    std::printf("freed %d by the batch, %d in all\n", by_batch, freed);
    return by_batch == 3 && freed == 5 ? 0 : 1;
}
