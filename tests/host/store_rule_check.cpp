// Host-side check of where quantised bytes go (dax_amd/csrc/store_rule.h), on either side of every line.  Built by
// __graft_entry__.build() with the host compiler; run by tests/test_abi_and_host.py.
#include <cstdio>
#include <initializer_list>

#include "../../dax_amd/csrc/store_rule.h"

int main() {
    using namespace daxq;
    const int64_t MB = (int64_t)1 << 20;
    long bad = 0;
    auto rows = [&](int64_t bytes, int want, int unaligned) { bad += (store_of(bytes, true) != want) + (store_of(bytes, false) != unaligned); };
    rows(1, kStoreKeep, kStoreKeep), rows(MB - 1, kStoreKeep, kStoreKeep), rows(MB, kStoreThrough, kStoreKeep), rows(8 * MB, kStoreThrough, kStoreKeep);
    rows(8 * MB + 1, kStoreKeep, kStoreKeep), rows(32 * MB - 1, kStoreKeep, kStoreKeep), rows(32 * MB, kStoreThrough, kStoreKeep);
    rows(128 * MB, kStoreThrough, kStoreKeep), rows(128 * MB + 1, kStoreThrough, kStorePast), rows(256 * MB, kStoreThrough, kStorePast);
    rows(256 * MB + 1, kStorePast, kStorePast), rows((int64_t)75600 * 13824, kStorePast, kStorePast);
    // fused producers: through the L2 as far as the Infinity Cache holds about all of it, past the caches beyond
    for (int64_t b : {(int64_t)1, MB, 9450 * (int64_t)13824, 20000 * (int64_t)13824, 280 * MB}) bad += !fused_store_through(b);
    for (int64_t b : {280 * MB + 1, 60000 * (int64_t)5120, 24000 * (int64_t)13824, 75600 * (int64_t)5120, 75600 * (int64_t)13824, (int64_t)1 << 40}) bad += fused_store_through(b);
    printf("%ld errors\n", bad);
    return bad != 0;
}
