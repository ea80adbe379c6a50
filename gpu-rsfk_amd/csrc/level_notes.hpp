// What a batch of trees tells the host while it is built: records in pinned memory that a kernel fills, their word `seq`
// last, and that the host polls.  Pinned blocks come from a pool shared with everything else that passes through pinned memory
// and keep what their last user left in them, so a record says nothing until begin() has cleared its seq, which has to happen
// before the first kernel of the batch is queued.  (Host code without HIP, so that it can be tested without a device.)
#pragma once
#include <cstddef>

namespace rsfk {

// Counts of a level.
struct LevelNote {
    int n_nodes, n_chunks, n_tail, overflow;
    int seq;
    int pad_[11];
};

class LevelNotes {
public:
    static constexpr int kNotes = 8;                 // level l writes note l % kNotes; at most two levels are queued at a time
    static constexpr std::size_t kBytes = sizeof(LevelNote) * kNotes;
    static constexpr int kReport = 1;                // seq of the batch's report

    // The block and the seq of the report, both pinned and both allocated.
    void set(void* block, int* report_seq)
    {
        notes_ = static_cast<LevelNote*>(block);
        report_seq_ = report_seq;
    }
    void* block() const { return notes_; }
    // A batch begins: nothing has arrived.  The kernels of the batch before it have ended.
    void begin()
    {
        for (int i = 0; i < kNotes; ++i) __atomic_store_n(&notes_[i].seq, 0, __ATOMIC_RELEASE);
        __atomic_store_n(report_seq_, 0, __ATOMIC_RELEASE);
    }
    LevelNote* of(int level) const { return notes_ + level % kNotes; }
    static int seq(int level) { return level + 1; }  // (never what begin() leaves)

private:
    LevelNote* notes_ = nullptr;
    int* report_seq_ = nullptr;
};

}  // namespace rsfk
