// The resident decode step (resident.hip): all layers of a step of a few rows in one launch.
#pragma once
#include "kernels.h"

namespace nvllm {

constexpr int kResidentGroups = 256;   // workgroups, all of them on the chip at once, one to a CU
constexpr int kResidentRows = 8;       // rows of a step at most
constexpr int kResidentLayers = 4;     // layers of a model at least
constexpr int kResidentRest = 1024;    // steps as launches behind one that gave up, the first time
constexpr int kResidentParts = 16;     // parts of a context at most
constexpr int kResidentPart = 132;     // a part's result: 128 sums, the softmax's reference and its sum
constexpr uint32_t kResidentEmpty = 0xFFFFFFFFu;  // a place of the hand-off buffers that holds no value

struct ResidentLayer {
    const uint4 *qkv, *o, *gu, *down;  // packed weights
    const float *ln1, *ln2, *qn, *kn;
    f16_bits *k, *v;
};
// Sizes the launch takes: a hidden size of 1024, everything else multiples of 1024 up to the registers that hold a layer's weights
struct ResidentSizes {
    int NQ = 0, KO = 0, I = 0;         // features of q, k and v; of the attention's output; of the feed-forward
    int nh = 0, kv = 0, hd = 0;
};
bool resident_sizes_ok(int H, const ResidentSizes& z);
size_t resident_buffer_words(const ResidentSizes& z);

struct ResidentArgs {
    const ResidentLayer* layers = nullptr;  // device
    int L = 0, R = 0;
    ResidentSizes z;
    const uint32_t* ids = nullptr;
    const bf16_bits* embed = nullptr;
    const float* norm = nullptr;            // final norm's weights
    const DecodeRow* rows = nullptr;        // record i is row i
    const int* block_tables = nullptr;
    int max_blocks = 0;
    const float *cos = nullptr, *sin = nullptr;
    float eps = 0.f, q_scale = 0.f;
    int part_tiles = 0, parts = 1;          // a context in parts of so many 32-token tiles; parts of the longest
    uint32_t* buffer = nullptr;             // resident_buffer_words, all kResidentEmpty before the first launch
    int set = 0;                            // 0 and 1 in turn, launch by launch
    bf16_bits *xh = nullptr, *xl = nullptr; // out: the final norm's planes without 1 / rms, row-major, and the rows' sums of squares
    float* ssq = nullptr;
    int* gave_up = nullptr;                 // device and host: set when a wait ran out; the buffer is then to be emptied again
    int* host_gave_up = nullptr;
    int spins = 0;                          // a wait's turns at most
};
hipError_t launch_resident(const ResidentArgs& a, hipStream_t s);

}  // namespace nvllm
