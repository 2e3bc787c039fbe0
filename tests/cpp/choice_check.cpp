// CPU check of the merge loop with choice bits (ChoiceEx of csrc/hip/coder.hip): the same steps, lane
// by lane, against std::pop_heap / std::push_heap after every operation, every heap access asserted
// in bounds.  Prints "OK <merges>".
#include <algorithm>
#include <cassert>
#include <cstdio>
#include <random>
#include <vector>

#include "../../cudacompress_amd/csrc/hip/huff_design.hpp"

using cca::design::HeapEntry;

namespace {

struct Lanes {
    std::vector<HeapEntry> h;  // with slack, as the workspace has after the heap
    uint32_t top[64] = {}, lo[64] = {}, hi[64] = {};
    uint64_t mall[64] = {}, mwant[64] = {};
    int sd[64] = {};

    const HeapEntry& at(int i) const { assert(i >= 0 && i < (int)h.size()); return h[i]; }

    void begin(int K) {
        for (int ln = 0; ln < 64; ln++) {
            sd[ln] = ln < 63 ? 31 - __builtin_clz(ln + 1) : 0;
            for (int d = 0; d < 6; d++) {
                const int a = ((64 | ln) >> (6 - d)) - 1;
                mall[ln] |= 1ull << a;
                mwant[ln] |= (uint64_t)(((64 | ln) >> (5 - d)) & 1) << a;
            }
            auto choice = [&](int c) {
                return ln < 63 && 2 * c < K && !(at(2 * c - 1).count < at(2 * c).count) ? 1u : 0u;
            };
            top[ln] = choice(ln + 1);
            for (int b = 0; b < 64 && 2 * (64 + b) < K; b++) {
                const uint32_t c = choice(((64 + b) << sd[ln]) + (ln + 1) - (1 << sd[ln]));
                if (b < 32) lo[ln] |= c << b;
                else hi[ln] |= c << (b - 32);
            }
        }
    }
    uint32_t walk(uint64_t m) const {
        int found = -1;
        for (int i = 0; i < 64; i++)
            if ((m & mall[i]) == mwant[i]) { assert(found < 0); found = i; }
        assert(found >= 0);
        return (uint32_t)found;
    }
    // choices on the way to 12-level node E: bit d of nb at depth d
    void update(uint32_t E, uint32_t nb, bool deep) {
        for (int ln = 0; ln < 64; ln++) {
            const uint32_t e1 = E >> 6, e2 = 64u | (E & 63u), b = e1 & 63u;
            if ((int)(e1 >> (6 - sd[ln])) == ln + 1) top[ln] = (nb >> sd[ln]) & 1u;
            if (!deep || (int)(e2 >> (6 - sd[ln])) != ln + 1) continue;
            const uint32_t bit = 1u << (b & 31u), set = (nb >> (6 + sd[ln])) & 1u ? bit : 0u;
            if (b < 32) lo[ln] = (lo[ln] & ~bit) | set;
            else hi[ln] = (hi[ln] & ~bit) | set;
        }
    }
    uint32_t node_of(uint32_t E, int ln) const { return E >> (ln < 12 ? 12 - ln : 0); }
    HeapEntry pop(int len) {
        const HeapEntry v = at(len - 1);
        if (len <= 1) return v;
        const uint32_t n = (uint32_t)len - 1;
        const bool deep = n >= 128;
        uint64_t m1 = 0, m2 = 0;
        for (int ln = 0; ln < 64; ln++) m1 |= (uint64_t)(top[ln] != 0) << ln;
        const uint32_t e1 = 64u | walk(m1);
        uint32_t E = e1 << 6;
        if (deep) {
            const uint32_t b = e1 - 64;
            for (int ln = 0; ln < 64; ln++) m2 |= (uint64_t)(((b < 32 ? lo[ln] : hi[ln]) >> (b & 31u)) & 1u) << ln;
            E |= walk(m2);
        }
        const uint32_t below_d = (uint32_t)__builtin_clz(n) - 19u;
        const uint32_t gone = (n & 1u) ? 0u : n + 1u;
        E -= (E >> below_d) == gone ? 1u << below_d : 0u;
        const uint32_t parents = n >> 1, last = parents > 1u ? parents : 1u;
        HeapEntry pn[64], moved[64];
        uint32_t sib[64] = {}, is = 0;
        bool right[64] = {};
        for (int ln = 0; ln < 64; ln++) {
            const uint32_t pk = node_of(E, ln), c = pk < last ? pk : last;
            const HeapEntry l = at((int)(2 * c) - 1), r = at((int)(2 * c));
            right[ln] = ln < 12 && ((E >> (11 - ln)) & 1u);
            pn[ln] = right[ln] ? r : l;
            sib[ln] = right[ln] ? l.count : r.count;
            const bool rise = pn[ln].count <= v.count && pk <= parents;
            assert(!rise || is == (uint32_t)ln);  // a prefix of the lanes
            is += rise;
        }
        for (uint32_t ln = 0; ln < 64; ln++) moved[ln] = ln < is ? pn[ln] : v;
        for (uint32_t ln = 0; ln <= is; ln++) {
            const uint32_t k = node_of(E, (int)ln);
            assert(k >= 1 && k <= n);
            h[k - 1] = moved[ln];
        }
        uint32_t nb = 0;
        for (uint32_t ln = 0; ln < 16; ln++) {
            const uint32_t below = ln < 15 ? moved[ln + 1].count : 0u;
            const uint32_t now = ln < is ? below : pn[ln].count;
            nb |= (uint32_t)((right[ln] ? sib[ln] : now) >= (right[ln] ? now : sib[ln])) << ln;
        }
        update(deep ? E : (e1 << 6), nb, deep);
        return moved[0];
    }
    HeapEntry push(int pos, HeapEntry v, HeapEntry top_entry) {
        const uint32_t Q = (uint32_t)pos + 1, T = 31 - (uint32_t)__builtin_clz(Q);
        HeapEntry e[64];
        uint32_t sib[64], c[64], place = T;
        for (uint32_t ln = 0; ln < 64; ln++) {
            const uint32_t cq = Q >> ((T - ln - 1u) & 31u);
            c[ln] = cq > 2u ? cq : 2u;
            e[ln] = at((int)(c[ln] >> 1) - 1);
            sib[ln] = at((int)(c[ln] ^ 1u) - 1).count;
            if (ln < T && v.count < e[ln].count && place == T) place = ln;
            assert(!(ln < T && place < ln) || v.count < e[ln].count);  // a suffix of the chain
        }
        for (uint32_t ln = place; ln < T; ln++) h[c[ln] - 1] = e[ln];
        h[(Q >> (T - place)) - 1] = v;
        uint32_t nb = 0;
        for (uint32_t ln = 0; ln < 16; ln++) {
            const uint32_t ec = ln < T ? e[ln].count : 0xFFFFFFFFu;
            const uint32_t below = ln + 1 < T && ln < 15 ? e[ln + 1].count : 0xFFFFFFFFu;
            const uint32_t now = ln >= place ? ec : std::min(v.count, below);
            const bool odd = c[ln] & 1u;
            nb |= (uint32_t)((odd ? sib[ln] : now) >= (odd ? now : sib[ln])) << ln;
        }
        update(Q << (12 - T), nb, Q >= 128);
        return place == 0 ? v : top_entry;
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
    for (int t = 0; t < 60; t++) sizes.push_back(2 + (int)(rng() % 3000));
    for (size_t t = 0; t < 3 * sizes.size(); t++) {
        const int K = sizes[t % sizes.size()];
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
        Lanes L;
        L.h = ref;
        L.h.resize(K + 3, HeapEntry{7u, 0xFFFFu});
        L.begin(K);
        int size = K, next = K;
        HeapEntry top = L.h[0];
        while (size > 1) {
            HeapEntry two[2];
            for (int q = 0; q < 2; q++) {
                two[q] = ref[0];
                if (top.count != ref[0].count || top.node != ref[0].node) { printf("FAIL top K=%d size=%d\n", K, size); return 1; }
                std::pop_heap(ref.begin(), ref.end(), less);
                ref.pop_back();
                top = L.pop(size--);
                if (!same(L.h, ref, size)) { printf("FAIL pop K=%d size=%d\n", K, size); return 1; }
            }
            const HeapEntry v{two[0].count + two[1].count, (uint32_t)next++};
            ref.push_back(v);
            std::push_heap(ref.begin(), ref.end(), less);
            top = L.push(size++, v, top);
            if (!same(L.h, ref, size)) { printf("FAIL push K=%d size=%d\n", K, size); return 1; }
            merges++;
        }
    }
    printf("OK %ld\n", merges);
    return 0;
}
