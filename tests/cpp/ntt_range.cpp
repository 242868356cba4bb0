// The reduction of the transforms' signed limbs (liblightzk_amd/csrc/fr29.hpp)
// for tests/test_ntt_range_cpu.py, compiled for the host.
#include <cstdint>
namespace hzk {
struct fr_t {
    uint32_t l[8];
};
}  // namespace hzk
#define HZK_DEV inline
#include "../../liblightzk_amd/csrc/fr29.hpp"

struct limbs {
    int32_t l[9];
};

extern "C" void fr_reduce_n(const int32_t* in, int32_t* out, long n) {
    for (long i = 0; i < n; ++i) {
        limbs v;
        for (int j = 0; j < 9; ++j) v.l[j] = in[9 * i + j];
        v = hzk::fr_reduce(v);
        for (int j = 0; j < 9; ++j) out[9 * i + j] = v.l[j];
    }
}
extern "C" void fr_canonical_n(const int32_t* in, int32_t* out, long n) {
    for (long i = 0; i < n; ++i) {
        limbs v;
        for (int j = 0; j < 9; ++j) v.l[j] = in[9 * i + j];
        v = hzk::fr_canonical(v);
        for (int j = 0; j < 9; ++j) out[9 * i + j] = v.l[j];
    }
}
