// The vectors of a step that go to the device.
#include <cstdint>

extern "C" {

// out: token ids | positions | slots of the step's rows, `total` rows of n entries and `fill` rows of the scratch request (token 0 at
// position 0) in front of them or behind.
void mlr_step_rows(int n, int total, const int32_t* ids, const int32_t* counts, const int32_t* slots, const int32_t* first, int fill,
                   int fill_first, int scratch, int32_t* out) {
    const int rows = total + fill;
    int32_t *token = out, *position = out + rows, *slot = out + 2 * (int64_t)rows;
    int at = 0;
    const auto scratch_rows = [&]() {
        for (int i = 0; i < fill; ++i, ++at) {
            token[at] = position[at] = 0;
            slot[at] = scratch;
        }
    };
    if (fill_first) scratch_rows();
    for (int e = 0, k = 0; e < n; ++e)
        for (int i = 0; i < counts[e]; ++i, ++at, ++k) {
            token[at] = ids[k];
            position[at] = first[e] + i;
            slot[at] = slots[e];
        }
    if (!fill_first) scratch_rows();
}

}  // extern "C"
