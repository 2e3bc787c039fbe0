// CPU check of the merge loop's heap operations by a wave (csrc/hip/choice_heap.hpp, the code the kernel
// runs): 64 lanes as coroutines that meet at every vote, against std::pop_heap / std::push_heap after every
// operation, every heap access asserted in bounds.  Prints "OK <merges>".
#undef _FORTIFY_SOURCE  // its longjmp does not go from one stack to another
#include <csetjmp>
#include <cstdio>
#include <cstdlib>
#include <algorithm>
#include <functional>
#include <random>
#include <ucontext.h>
#include <vector>

#include "../../cudacompress_amd/csrc/hip/choice_heap.hpp"

using cca::design::ChoiceHeap;
using cca::design::HeapEntry;

namespace {

constexpr int kLanes = 64;
constexpr size_t kStack = 64 * 1024;

struct Wave {
    jmp_buf at[kLanes], home;
    ucontext_t start[kLanes], main;
    std::vector<char> stacks = std::vector<char>(kLanes * kStack);
    int now = 0, left = 0;
    uint32_t value[2][kLanes];  // one vote writes here, the next there: a lane reads before it meets again
    int parity[kLanes] = {};
    const HeapEntry* heap = nullptr;
    uint32_t slots = 0;  // entries that may be read
    std::function<void(int)> body;
} W;

void lane_main() {
    const int l = W.now;
    W.body(l);
    W.left--;
    longjmp(W.home, 1);
}
// every lane up to its next meeting point, in lane order, until all have run to the end
void run(std::function<void(int)> body) {
    W.body = std::move(body);
    bool started[kLanes] = {}, ended[kLanes] = {};
    W.left = kLanes;
    for (int l = 0; l < kLanes; l++) {
        getcontext(&W.start[l]);
        W.start[l].uc_stack.ss_sp = W.stacks.data() + l * kStack;
        W.start[l].uc_stack.ss_size = kStack;
        W.start[l].uc_link = nullptr;
        makecontext(&W.start[l], lane_main, 0);
    }
    while (W.left > 0)
        for (volatile int l = 0; l < kLanes; l = l + 1) {
            if (ended[l]) { printf("FAIL lanes do not meet\n"); exit(1); }
            const int before = W.left;
            W.now = l;
            if (setjmp(W.home) == 0) {
                if (started[l]) longjmp(W.at[l], 1);
                started[l] = true;
                setcontext(&W.start[l]);
            }
            ended[l] = W.left < before;
        }
}
// the other lanes come here too before this one goes on
void meet() {
    const int l = W.now;
    if (setjmp(W.at[l]) == 0) longjmp(W.home, 1);
    W.now = l;
}

struct EmulatedLanes {
    static int lane() { return W.now; }
    // this lane's value; all lanes' once they have met
    static const uint32_t* share(uint32_t v) {
        uint32_t* const to = W.value[W.parity[W.now] ^= 1];
        to[W.now] = v;
        meet();
        return to;
    }
    static uint64_t vote(bool b) {
        const uint32_t* v = share(b);
        uint64_t m = 0;
        for (int l = 0; l < kLanes; l++) m |= (uint64_t)(v[l] & 1u) << l;
        return m;
    }
    static uint32_t read(uint32_t v, uint32_t l) { return share(v)[l]; }
    static uint32_t next(uint32_t v, uint32_t last) {
        const uint32_t* all = share(v);
        return W.now % 16 == 15 ? last : all[W.now + 1];
    }
    static HeapEntry& entry(HeapEntry* h, uint32_t c) {
        if (h != W.heap || c < 1 || c > W.slots) {
            printf("FAIL entry %u of %u\n", c, W.slots);
            exit(1);
        }
        return h[c - 1];
    }
};

bool same(const std::vector<HeapEntry>& a, const std::vector<HeapEntry>& b, int n) {
    for (int i = 0; i < n; i++)
        if (a[i].count != b[i].count || a[i].node != b[i].node) return false;
    return true;
}

}  // namespace

int main() {
    std::mt19937_64 rng(99);
    const auto less = [](const HeapEntry& a, const HeapEntry& b) { return b.count < a.count; };
    long merges = 0;
    std::vector<int> sizes{2, 3, 4, 5, 63, 64, 65, 127, 128, 129, 255, 256, 257, 1023, 1025, 2047, 2048, 4095, 4096};
    for (int t = 0; t < 8; t++) sizes.push_back(2 + (int)(rng() % 1500));
    for (size_t t = 0; t < 3 * sizes.size(); t++) {
        const int K = sizes[t % sizes.size()];
        if (K > 2048 && t >= sizes.size()) continue;
        std::vector<HeapEntry> ref(K);
        for (int i = 0; i < K; i++) {
            uint32_t c = 1;
            switch (t % 4) {
                case 0: c = 1 + (uint32_t)(rng() % 3); break;
                case 1: c = 1 + (uint32_t)(rng() % 5000); break;
                case 2: c = 1u << (rng() % 12); break;
                default: c = 1 + (uint32_t)(4000 / (1 + i)); break;
            }
            ref[i] = HeapEntry{c, (uint32_t)i};
        }
        std::make_heap(ref.begin(), ref.end(), less);
        std::vector<HeapEntry> heap = ref;
        heap.resize(K + 3, HeapEntry{7u, 0xFFFFu});  // with slack, as the workspace has after the heap
        W.heap = heap.data();
        W.slots = (uint32_t)heap.size();
        const char* fault = nullptr;
        int size = K, at_size = 0;
        // all lanes run the merge loop; lane 0 checks the heap where the others wait for it
        run([&](int lane) {
            ChoiceHeap<EmulatedLanes> c;
            HeapEntry* h = heap.data();
            c.begin(h, K);
            int n = K, next = K;
            HeapEntry top = h[0];
            auto check = [&](const char* what) {
                meet();
                if (lane == 0 && !fault && (!same(heap, ref, n) || (n > 0 && (top.count != ref[0].count || top.node != ref[0].node)))) {
                    fault = what;
                    at_size = n;
                }
                meet();
            };
            while (n > 1 && !fault) {
                HeapEntry two[2];
                for (int q = 0; q < 2; q++) {
                    two[q] = top;
                    if (lane == 0) {
                        std::pop_heap(ref.begin(), ref.end(), less);
                        ref.pop_back();
                    }
                    top = c.pop(h, n--);
                    if (n == 0) top = two[q];
                    check("pop");
                    if (n == 0) break;
                }
                const HeapEntry v{two[0].count + two[1].count, (uint32_t)next++};
                if (lane == 0) {
                    ref.push_back(v);
                    std::push_heap(ref.begin(), ref.end(), less);
                    merges++;
                }
                top = c.push(h, n++, v, top);
                check("push");
            }
            if (lane == 0) size = n;
        });
        if (fault || size != 1) {
            printf("FAIL %s K=%d size=%d\n", fault ? fault : "end", K, fault ? at_size : size);
            return 1;
        }
    }
    printf("OK %ld\n", merges);
    return 0;
}
