// Huffman table design and headers, src/cudaCompress/HuffmanTable.cu:117-266, :470-586 and
// src/cudaCompress/HuffmanDesign.h:13-65 (GPU dialect); src/CPU/HuffmanTableCPU.cpp:22-135
// (CPU dialect).
//
// The tree is built as by std::priority_queue over nodes compared by count only, and the leaves are
// ordered with std::sort by depth only -- what the reference's standard-library calls do (libstdc++),
// so ties resolve identically.  The GPU dialect seeds the queue as the range constructor does
// (make_heap); the CPU dialect pushes leaves one at a time.  Queue and sort hold a node's key and its
// number in one word, not a pointer to it, and the queue's top is taken without unpredictable branches:
// fetching what is compared and mispredicted branches bound a large table (65,441 symbols, pointers
// 20.6 ms, words 14.4 ms, with take_top 8.9 ms).
#include "huffman_table.hpp"

#include <algorithm>

namespace cca {

HeaderFormat header_format(int dialect, uint32_t log2) {
    if (dialect == CC_DIALECT_CPU) return HeaderFormat{CC_DIALECT_CPU, 14u, 14u};
    return HeaderFormat{CC_DIALECT_GPU, log2, log2 > 16 ? 5u : 4u};
}

namespace {

// (key, node) words, compared by key only
constexpr uint64_t word_of(uint32_t key, uint32_t node) { return (uint64_t)key << 32 | node; }
struct ByCountInverted {  // HuffmanDesign.h:47-55: "greater" so the queue top is the rarest
    bool operator()(uint64_t a, uint64_t b) const { return (uint32_t)(b >> 32) < (uint32_t)(a >> 32); }
};
struct ByDepth {  // HuffmanDesign.h:57-63
    bool operator()(uint64_t a, uint64_t b) const { return (uint32_t)(a >> 32) < (uint32_t)(b >> 32); }
};

// Takes the top off the heap h (not empty), moving what std::pop_heap moves: the hole goes down along the
// child that is less or, of equal ones, the second, and the last element comes up from where it ends.  The
// choice is computed: as a branch it is taken half of the time, at random.
uint64_t take_top(std::vector<uint64_t>& h) {
    const uint64_t top = h[0], value = h.back();
    h.pop_back();
    const size_t n = h.size();
    if (n == 0) return top;
    size_t hole = 0;
    for (size_t c = 2; c < n; c = 2 * hole + 2) {  // c, c - 1: the children
        c -= (uint32_t)(h[c - 1] >> 32) < (uint32_t)(h[c] >> 32);
        h[hole] = h[c];
        hole = c;
    }
    if (2 * hole + 2 == n) {  // an only child
        h[hole] = h[n - 1];
        hole = n - 1;
    }
    for (size_t up; hole > 0; hole = up) {
        up = (hole - 1) / 2;
        if (!ByCountInverted()(h[up], value)) break;
        h[hole] = h[up];
    }
    h[hole] = value;
    return top;
}

}  // namespace

cc_status design_table(int dialect, const uint32_t* hist, uint32_t symbol_max, EncTable& t) {
    t.count_per_length.clear();
    t.symbols.clear();
    t.symbol_max = symbol_max;
    const uint32_t nsym_space = symbol_max + 1;

    std::vector<uint64_t> leaves;  // (count, leaf), leaf k being symbol t.symbols[k]
    for (uint32_t s = 0; s < nsym_space; s++) {
        if (hist[s] == 0) continue;
        leaves.push_back(word_of(hist[s], (uint32_t)t.symbols.size()));
        t.symbols.push_back(s);
    }
    if (leaves.empty()) return CC_OK;  // empty stream: empty table
    const uint32_t k = (uint32_t)leaves.size();

    std::vector<uint64_t> q(leaves);
    if (dialect == CC_DIALECT_GPU) {
        std::make_heap(q.begin(), q.end(), ByCountInverted());
    } else {
        for (uint32_t i = 1; i <= k; i++) std::push_heap(q.begin(), q.begin() + i, ByCountInverted());
    }
    std::vector<uint32_t> parent(2 * (size_t)k, 0u);  // of the leaves, then of the inner nodes as they are made
    uint32_t nodes = k;
    while (q.size() > 1) {
        const uint64_t a = take_top(q), b = take_top(q);
        parent[(uint32_t)a] = parent[(uint32_t)b] = nodes;
        q.push_back(word_of((uint32_t)(a >> 32) + (uint32_t)(b >> 32), nodes++));
        std::push_heap(q.begin(), q.end(), ByCountInverted());
    }
    // depths from the root, the last node, down (HuffmanDesign.h:32-44)
    std::vector<uint32_t> depth(nodes, 0u);
    uint32_t deepest = 0;
    for (uint32_t i = nodes - 1; i-- > 0;) {
        depth[i] = depth[parent[i]] + 1;
        deepest = std::max(deepest, depth[i]);
    }
    for (uint32_t i = 0; i < k; i++) leaves[i] = word_of(depth[i], t.symbols[i]);
    std::sort(leaves.begin(), leaves.end(), ByDepth());
    if (deepest > 31) {
        t.symbols.clear();
        return CC_ERR_CODEWORD_TOO_LONG;
    }

    t.count_per_length.assign((size_t)deepest, 0u);
    for (uint32_t i = 0; i < k; i++) {
        const uint32_t l = (uint32_t)(leaves[i] >> 32);
        if (l > 0) t.count_per_length[l - 1]++;
        t.symbols[i] = (uint32_t)leaves[i];
    }
    return CC_OK;
}

static uint32_t header_symbol_max(const HeaderFormat& f, const EncTable& t) {
    if (f.dialect == CC_DIALECT_GPU) return t.symbol_max;
    uint32_t m = 0;  // CPU dialect: max over the table's symbols (HuffmanTableCPU.cpp:110-114)
    for (uint32_t s : t.symbols) m = std::max(m, s);
    return m;
}

void write_table(const HeaderFormat& f, const EncTable& t, BitWriter& w) {
    w.bits((uint32_t)t.count_per_length.size(), 5);
    for (uint32_t c : t.count_per_length) w.bits(c, f.count_bits);
    w.bits((uint32_t)t.symbols.size(), f.count_bits);
    const uint32_t sb = required_bits(header_symbol_max(f, t));
    w.bits(sb, f.symbits_bits);  // GPU dialect, Symbol16: 16 is written as 0 (HuffmanTable.cu:481)
    for (uint32_t s : t.symbols) w.bits(s, sb);
}

uint64_t table_bits(const HeaderFormat& f, const EncTable& t) {
    const uint32_t sb = required_bits(header_symbol_max(f, t));
    return 5ull + (uint64_t)f.count_bits * (t.count_per_length.size() + 1) + f.symbits_bits +
           (uint64_t)sb * t.symbols.size();
}

}  // namespace cca
