// api_out.cpp — where the per-pair call's output arrays go (zdx_api_out.h), on
// the CPU: an array of `rows` rows is stored nowhere when it exceeds the
// caller's capacity, else in the slot when it fits there and in a device buffer
// of at least its size when it does not, and the reading side looks there too.
// Capacities and rows on both sides of the slot and of each other, for the five
// arrays (loop records, their derivatives, vertices, vertex offsets, segments).
#include "../../zedm-x_amd/csrc/zdx_api_out.h"

#include <cstdio>
#include <vector>

using namespace zdx;

template <class T>
static int check(const char* name, int per) {
    static T slot[1], dev[1];
    const int64_t fit = API_SLOT / ((int64_t)sizeof(T) * per);   // rows that just fit the slot
    const std::vector<int64_t> sizes = {0, 1, 64, fit - 1, fit, fit + 1, fit + 2, 2 * fit, 40 * fit};
    int n = 0;
    for (int64_t cap : sizes)
        for (int64_t rows : sizes) {
            ApiOut<T> o;
            o.host = slot; o.cap = cap; o.per = per;
            const int64_t made = o.dev_entries();   // as the call makes it
            if (made > 0) o.dev = dev;
            T* const at = o.at(rows);
            bool ok = (at == nullptr) == (rows > cap);
            if (at == slot) ok = ok && o.in_slot(rows) && rows * per * (int64_t)sizeof(T) <= API_SLOT;
            if (at == dev) ok = ok && !o.in_slot(rows) && rows * per <= made;
            ok = ok && (made == 0 || made == cap * per);
            if (!ok) {
                std::printf("FAIL %s: capacity %lld, rows %lld\n", name, (long long)cap, (long long)rows);
                return -1;
            }
            ++n;
        }
    ApiOut<T> unwanted;
    unwanted.cap = 8; unwanted.per = per;
    if (unwanted.at(0) || unwanted.at(4) || unwanted.dev_entries() != 0) {
        std::printf("FAIL %s: an array that is not wanted\n", name);
        return -1;
    }
    return n;
}

int main() {
    const int n[5] = {check<double>("records", 28), check<double>("derivatives", 72), check<double>("vertices", 3),
                      check<int32_t>("vertex offsets", 1), check<double>("segments", 6)};
    for (int k : n)
        if (k < 0) return 1;
    std::printf("api_out ok: %d\n", n[0] + n[1] + n[2] + n[3] + n[4]);
    return 0;
}
