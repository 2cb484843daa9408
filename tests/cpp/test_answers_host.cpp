// Host-only harness over the answer words of the gather's row check (zerocool_amd/csrc/zc_answers.hpp), meant to be built with
// -fsanitize=address,undefined (make asan).  A queue that runs its jobs in order stands for the stream, a job for the kernel that stores an answer.
// Every caller has to read its own answer, however long it is kept from looking and however many calls others make meanwhile.
#include "../../zerocool_amd/csrc/zc_answers.hpp"
#include <cstdio>
#include <deque>
#include <mutex>
#include <random>
#include <set>
#include <thread>
#include <vector>

using zc::AnswerWords;
using Answer = AnswerWords::Answer;
static std::atomic<int> checks{0}, failures{0};
#define CHECK(cond) do { ++checks; if (!(cond)) { ++failures; std::printf("  FAILED %s:%d: %s\n", __FILE__, __LINE__, #cond); } } while (0)

static void store(const AnswerWords::Question& q, bool no) { __atomic_store_n(q.slot, q.answer + (no ? 1u : 0u), __ATOMIC_RELEASE); }
static bool call(AnswerWords& words, bool no) {   // one whole call with nobody in between: whether it read its own answer
    const auto q = words.ask();
    if (!q.slot || AnswerWords::look(q) != Answer::none) return false;
    store(q, no);
    const bool right = AnswerWords::look(q) == (no ? Answer::no : Answer::yes);
    words.give_back(q);
    return right;
}

static void overtaken() {   // by 1, 63, 64, 65 and 1000 calls, answered before them or behind
    for (const int others : {1, 63, 64, 65, 1000})
        for (const bool no : {false, true})
            for (const bool early : {false, true}) {
                uint32_t memory[AnswerWords::kWords];
                AnswerWords words; words.use(memory);
                const auto late = words.ask();
                if (early) store(late, no);
                bool right = true;
                for (int i = 0; i < others; ++i) right = call(words, !no) && right;
                CHECK(right);
                CHECK(AnswerWords::look(late) == (!early ? Answer::none : no ? Answer::no : Answer::yes));
                if (!early) { store(late, no); CHECK(AnswerWords::look(late) == (no ? Answer::no : Answer::yes)); }
                words.give_back(late);
            }
}
static void all_taken() {
    uint32_t memory[AnswerWords::kWords];
    AnswerWords words; words.use(memory);
    std::vector<AnswerWords::Question> held;
    std::set<uint32_t*> slots;
    for (uint32_t i = 0; i < AnswerWords::kWords; ++i) { held.push_back(words.ask()); slots.insert(held.back().slot); }
    CHECK(slots.size() == AnswerWords::kWords && !slots.count(nullptr));
    for (uint32_t* s : slots) CHECK(s >= memory && s < memory + AnswerWords::kWords);
    CHECK(!words.ask().slot && !words.ask().slot);
    for (const uint32_t i : {0u, 31u, 63u}) {   // the one that comes back is the one that is lent out, with another answer
        store(held[i], true); words.give_back(held[i]);
        const auto again = words.ask();
        CHECK(again.slot == held[i].slot && again.answer != held[i].answer && AnswerWords::look(again) == Answer::none);
        CHECK(!words.ask().slot);
    }
}
static void threads(int callers, int calls) {
    uint32_t memory[AnswerWords::kWords];
    AnswerWords words; words.use(memory);
    std::mutex mutex; std::deque<std::pair<AnswerWords::Question, bool>> queue;
    std::atomic<int> running{callers}, refused{0};
    std::thread stream([&] {
        for (;;) {
            std::pair<AnswerWords::Question, bool> job;
            {
                std::lock_guard<std::mutex> lock(mutex);
                if (queue.empty()) { if (!running) return; }
                else { job = queue.front(); queue.pop_front(); }
            }
            if (job.first.slot) store(job.first, job.second); else std::this_thread::yield();
        }
    });
    std::vector<std::thread> all;
    for (int t = 0; t < callers; ++t) all.emplace_back([&, t] {
        std::mt19937 rng(t);
        for (int i = 0; i < calls; ++i) {
            const bool no = rng() % 3 == 0;
            const auto q = words.ask();
            if (!q.slot) { ++refused; std::this_thread::yield(); continue; }
            { std::lock_guard<std::mutex> lock(mutex); queue.push_back({q, no}); }
            if (rng() % 8 == 0) std::this_thread::sleep_for(std::chrono::microseconds(rng() % 300));   // kept from looking
            Answer a;
            int polls = 0;
            while ((a = AnswerWords::look(q)) == Answer::none && ++polls < 1000000) std::this_thread::yield();
            CHECK(a == (no ? Answer::no : Answer::yes));
            if (a != Answer::none) words.give_back(q);
        }
        --running;
    });
    for (auto& t : all) t.join();
    stream.join();
    if (callers <= int(AnswerWords::kWords)) CHECK(refused == 0);
}

int main() {
    overtaken();
    all_taken();
    threads(2, 2000); threads(16, 500); threads(96, 100);
    std::printf("%d checks, %d failures\n", checks.load(), failures.load());
    return failures ? 1 : 0;
}
