// Per-request state moved whole: everything that the model's layers keep for a request slot is cleared, copied to another slot, or
// saved to and put back from a packed buffer in one launch.
//
// A model has a few dozen state tensors of some KB to some MB a slot.  One call of torch for each is bound by the host (10 to 20 us a
// tensor and direction), not by the bytes.  Twenty tensors, 11.9 MB a request: eight requests that fork and decode 12 tokens 7,684 us
// with a call a tensor, 5,713 so; a prompt of 2,048 tokens, whose slot is cleared and saved first, 3,969 and 3,502.  The tensors'
// addresses stand in a table on the device; the bytes of all of them are one range of chunks, a workgroup each, so that the launch
// is as wide as there is work and small tensors do not wait for each other.
#include "common.h"
#include "leone_hip.h"

namespace leone {

constexpr int kStateSlots = 64;                        // request slots a launch
constexpr int kStateThreads = 256;
constexpr int kStateChunk = kStateThreads * 4 * 16;    // bytes a workgroup: four 16-byte loads a thread

enum StateMove : int { kStateZero = 0, kStateCopy = 1, kStateSave = 2, kStateRestore = 3 };

struct StateTensor {
    long base;         // address of slot 0
    long bytes;        // of a slot, a multiple of 4
    long place;        // where it lies in a packed row, a multiple of 16
    long first_chunk;  // of the launch's chunks
};

struct StateSlotIds {
    int id[kStateSlots], to[kStateSlots];
};

template <typename T>
__device__ inline void move_bytes(const char* from, char* to, long bytes) {
    constexpr int kEach = kStateChunk / kStateThreads / sizeof(T);
    T held[kEach];
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
        const long at = (static_cast<long>(i) * kStateThreads + threadIdx.x) * sizeof(T);
        held[i] = from != nullptr && at < bytes ? *reinterpret_cast<const T*>(from + at) : T{};
    }
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
        const long at = (static_cast<long>(i) * kStateThreads + threadIdx.x) * sizeof(T);
        if (at < bytes) *reinterpret_cast<T*>(to + at) = held[i];
    }
}

__global__ void __launch_bounds__(kStateThreads)
state_slots_kernel(const StateTensor* __restrict__ table, int tensors, int move, StateSlotIds slots, char* packed, long packed_bytes) {
    const long chunk = blockIdx.x;
    int low = 0, high = tensors - 1;                   // the last tensor whose first chunk is not behind this one
    while (low < high) {
        const int mid = (low + high + 1) / 2;
        if (table[mid].first_chunk <= chunk) low = mid;
        else high = mid - 1;
    }
    const StateTensor t = table[low];
    const long at = (chunk - t.first_chunk) * kStateChunk;
    const long bytes = t.bytes - at < kStateChunk ? t.bytes - at : kStateChunk;
    const int j = blockIdx.y;
    char* slot = reinterpret_cast<char*>(t.base) + slots.id[j] * t.bytes + at;
    char* row = packed + j * packed_bytes + t.place + at;
    const char* from = move == kStateZero ? nullptr : move == kStateRestore ? row : slot;
    char* to = move == kStateCopy ? reinterpret_cast<char*>(t.base) + slots.to[j] * t.bytes + at : move == kStateSave ? row : slot;
    if ((reinterpret_cast<uintptr_t>(from) | reinterpret_cast<uintptr_t>(to) | bytes) % 16 == 0) move_bytes<uint4>(from, to, bytes);
    else move_bytes<unsigned>(from, to, bytes);                       // a slot whose size is no multiple of 16 bytes
}

}  // namespace leone

using namespace leone;

extern "C" int leone_state_chunk() { return kStateChunk; }
extern "C" int leone_state_slots_max() { return kStateSlots; }

// table: [tensors] of (address of slot 0, bytes a slot, place in a packed row, first chunk) as int64 on the device; chunks: of all tensors.
// ids and to: host arrays of `count` request slots (to: for copies alone, which read ids and write to).  move: 0 clears the slots, 1 copies
// them, 2 saves them to packed rows of packed_bytes each, 3 puts them back.  Slots of one call are different ones, and no slot is both
// read and written.
extern "C" int leone_state_slots(const void* table, int tensors, long chunks, int move, const int* ids, const int* to, int count, void* packed,
                                 long packed_bytes, hipStream_t stream) {
    LEONE_REQUIRE(table && ids && tensors > 0 && chunks > 0 && chunks < 0x7fffffff, "state_slots: %d tensors in %ld chunks", tensors, chunks);
    LEONE_REQUIRE(move >= kStateZero && move <= kStateRestore, "state_slots: unknown move %d", move);
    LEONE_REQUIRE(count > 0 && count <= kStateSlots, "state_slots: %d slots, a launch takes up to %d", count, kStateSlots);
    LEONE_REQUIRE(move != kStateCopy || to, "state_slots: a copy needs the slots it writes");
    LEONE_REQUIRE((move != kStateSave && move != kStateRestore) || (packed && packed_bytes > 0 && packed_bytes % 16 == 0 &&
                      reinterpret_cast<uintptr_t>(packed) % 16 == 0), "state_slots: the packed rows are aligned to 16 bytes");
    StateSlotIds slots = {};
    for (int i = 0; i < count; ++i) {
        LEONE_REQUIRE(ids[i] >= 0 && (move != kStateCopy || to[i] >= 0), "state_slots: negative slot");
        slots.id[i] = ids[i];
        if (move == kStateCopy) slots.to[i] = to[i];
    }
    state_slots_kernel<<<dim3(static_cast<unsigned>(chunks), count), kStateThreads, 0, stream>>>(
        static_cast<const StateTensor*>(table), tensors, move, slots, static_cast<char*>(packed), packed_bytes);
    LEONE_LAUNCH_CHECK("state_slots");
    return 0;
}
