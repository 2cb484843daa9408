// The pinned words in which kernels answer the host, one yes or no a call.  Host code only, without HIP: built by itself under the sanitizers too.
#pragma once
#include <atomic>
#include <cstdint>

namespace zc {

// A word is one caller's from before the launch until the answer has been read, however many calls other threads make meanwhile.
// (Lent out in turn, a word was written again 64 calls later, under a millisecond, whether or not its first caller had been given
// the time to look: that call then failed although its product had run, or polled for as long as the others kept the stream busy.)
class AnswerWords {
public:
    static constexpr uint32_t kWords = 64;
    enum class Answer { none, yes, no };
    struct Question {
        uint32_t* slot = nullptr;   // null: every word is taken
        uint32_t answer = 0;        // the kernel stores this for yes, plus one for no
    };
    void use(uint32_t* words) { words_ = words; for (uint32_t i = 0; i < kWords; ++i) words[i] = 0; }
    uint32_t* words() const { return words_; }
    Question ask() {
        uint64_t taken = taken_.load(std::memory_order_relaxed);
        while (~taken) {
            const uint64_t bit = ~taken & (taken + 1);   // the lowest that is free
            if (!taken_.compare_exchange_weak(taken, taken | bit, std::memory_order_acquire, std::memory_order_relaxed)) continue;
            const Question q{words_ + __builtin_ctzll(bit), asked_.fetch_add(1, std::memory_order_relaxed) << 1 | 1u << 31};
            __atomic_store_n(q.slot, 0u, __ATOMIC_RELAXED);   // (an answer of 2^30 calls ago would look like this one's)
            return q;
        }
        return {};
    }
    static Answer look(const Question& q) {
        const uint32_t word = __atomic_load_n(q.slot, __ATOMIC_ACQUIRE);
        return (word & ~1u) != q.answer ? Answer::none : word & 1u ? Answer::no : Answer::yes;
    }
    // Only once the answer is there: a word whose kernel may still store to it stays taken.
    void give_back(const Question& q) { taken_.fetch_and(~(1ull << (q.slot - words_)), std::memory_order_release); }

private:
    uint32_t* words_ = nullptr;
    std::atomic<uint64_t> taken_{0};
    std::atomic<uint32_t> asked_{0};
};

}  // namespace zc
