// The merge loop's heap operations by one wave, the descent known beforehand.
//
// Every node with two children has a choice bit (1: the pop's hole goes on to the right child, i.e. the left
// one is not strictly rarer; the other nodes' bits mean nothing), kept up to date by each pop and push, so a
// pop reads the heap once, along its path, instead of once per six levels and once more along the path.
// `top`: the choices of the top six levels, bit j local node j; lane b's lo and hi: those of the six levels
// below node 64 + b (12 levels, heaps of up to 4095 entries).  Lane i finds out whether a walk over such a
// mask ends at leaf i: its six ancestors' bits (all) then spell i (want).
//
// A merge is one wave's serial chain of instructions and sets the length of the design phase, so the forms
// below are the short ones: a lane decides by its own entry whether it moves (counts do not fall along a
// path), masks are combined on the scalar unit, and no branch depends on a lane.  Measured on MI355X: 64
// mixed bricks (largest table about 1,900 symbols) 2.6 -> 1.75 ms in the design phase, 2048 bricks 5.2 -> 4.2
// ms; a form with the bits as one mask a subtree but the old, longer selections took 2.15 ms.
//
// Written for one lane of 64 against Lanes: lane(), vote(b) (bit l: lane l's b), read(v, l) (lane l's v, the
// same l in every lane), next(v, last) (the next lane's v; at the end of a row of 16 `last`), and entry(h, c)
// (1-based).  What a lane stores before one of the first three the others see after it.
#pragma once

#include "huff_design.hpp"

namespace cca {
namespace design {

template <class Lanes>
struct ChoiceHeap {
    uint64_t top;
    uint32_t lo, hi;
    uint32_t all_lo, all_hi, want_lo, want_hi;
    uint32_t sd_up, sd_bit;  // 6 - depth of this lane's local node (lane 63: none), 1 << depth
    uint32_t up, turn;       // shift to this lane's node of a 12-level path (lane: depth), bit of its choice

    CCA_HD uint64_t subtree(uint32_t b) const { return ((uint64_t)Lanes::read(hi, b) << 32) | Lanes::read(lo, b); }
    CCA_HD void set_subtree(uint32_t b, uint64_t m) {
        lo = (uint32_t)Lanes::lane() == b ? (uint32_t)m : lo;
        hi = (uint32_t)Lanes::lane() == b ? (uint32_t)(m >> 32) : hi;
    }
    CCA_HD void begin(HeapEntry* h, int K) {
        const int ln = Lanes::lane();
        const int sd = ln < 63 ? 31 - __builtin_clz(ln + 1) : 0;
        sd_up = 6 - sd;
        sd_bit = 1u << sd;
        up = ln < 12 ? 12 - ln : 0;
        turn = ln < 12 ? 1u << (11 - ln) : 0u;
        uint64_t mall = 0, mwant = 0;
        for (int d = 0; d < 6; d++) {
            const int a = ((64 | ln) >> (6 - d)) - 1;
            mall |= 1ull << a;
            mwant |= (uint64_t)(((64 | ln) >> (5 - d)) & 1) << a;
        }
        all_lo = (uint32_t)mall;
        all_hi = (uint32_t)(mall >> 32);
        want_lo = (uint32_t)mwant;
        want_hi = (uint32_t)(mwant >> 32);
        auto choices = [&](int root) {  // of the six levels below 1-based node `root`
            const int c = (root << sd) + (ln + 1) - (1 << sd);
            return Lanes::vote(ln < 63 && 2 * c < K &&
                               !(Lanes::entry(h, 2u * (uint32_t)c).count < Lanes::entry(h, 2u * (uint32_t)c + 1u).count));
        };
        top = choices(1);
        lo = hi = 0;
        for (int b = 0; b < 64 && 2 * (64 + b) < K; b++) set_subtree(b, choices(64 + b));
    }
    // the leaf at which the walk over a subtree's choices ends
    CCA_HD uint32_t walk(uint64_t m) const {
        return (uint32_t)__builtin_ctzll(Lanes::vote(((uint32_t)m & all_lo) == want_lo) &
                                         Lanes::vote(((uint32_t)(m >> 32) & all_hi) == want_hi));
    }
    // the choices m of a subtree after those on the way to its leaf e (64 + leaf) became bits of nb
    CCA_HD uint64_t changed(uint64_t m, uint32_t e, uint32_t nb) const {
        const uint64_t on = Lanes::vote((e >> sd_up) == (uint32_t)Lanes::lane() + 1u);
        return (m & ~on) | (on & Lanes::vote((nb & sd_bit) != 0u));
    }

    // The heap's n entries left after its last one, v, was taken out.  Deep: n >= 128, so the path
    // runs through the top six levels.
    template <bool Deep>
    CCA_HD HeapEntry pop_path(HeapEntry* h, uint32_t n, HeapEntry v) {
        const uint32_t ln = (uint32_t)Lanes::lane();
        const uint32_t e1 = 64u | walk(top);
        uint64_t sub = 0;
        uint32_t E = e1 << 6;  // the path's node at depth k is E >> (12 - k), 1-based
        if (Deep) {
            sub = subtree(e1 - 64u);
            E |= walk(sub);
        }
        // the parent of a lone left child n may still point right, to n + 1
        const uint32_t below_d = (uint32_t)__builtin_clz(n) - 19u;  // 12 - depth of n
        const uint32_t gone = (n & 1u) ? 0u : n + 1u;
        E -= (E >> below_d) == gone ? 1u << below_d : 0u;
        const uint32_t pk = E >> up, parents = n >> 1;  // (nodes up to n / 2 have a child)
        const uint32_t last = parents > 1u ? parents : 1u;
        const uint32_t child = 2u * (pk < last ? pk : last);
        const HeapEntry l = Lanes::entry(h, child), r = Lanes::entry(h, child + 1u);
        const uint64_t act = Lanes::vote(pk <= parents);
        const bool right = (E & turn) != 0u;
        const HeapEntry pn{right ? r.count : l.count, right ? r.node : l.node};
        const uint32_t sib = right ? l.count : r.count;
        // the path's entries move up until one is larger than v, which takes its place
        const uint64_t rise = Lanes::vote(pn.count <= v.count) & act;
        const uint32_t is = (uint32_t)__builtin_popcountll(rise);
        const bool mv = ln < is;
        const HeapEntry moved{mv ? pn.count : v.count, mv ? pn.node : v.node};
        if (ln <= is) Lanes::entry(h, pk) = moved;
        // the new count one level down the path: what moved there, or what was there below v
        const uint32_t below = Lanes::next(moved.count, 0u);  // (paths are shorter than a row)
        const uint32_t now = mv ? below : pn.count;
        const uint32_t nb = (uint32_t)Lanes::vote((right ? sib : now) >= (right ? now : sib));
        top = changed(top, e1, nb);
        if (Deep) set_subtree(e1 - 64u, changed(sub, 64u | (E & 63u), nb >> 6));
        return HeapEntry{Lanes::read(moved.count, 0), Lanes::read(moved.node, 0)};
    }
    // the last of len entries takes the top's place; returns the new top
    CCA_HD HeapEntry pop(HeapEntry* h, int len) {
        const HeapEntry v = Lanes::entry(h, (uint32_t)len);
        if (len <= 1) return v;
        return len > 128 ? pop_path<true>(h, (uint32_t)len - 1u, v) : pop_path<false>(h, (uint32_t)len - 1u, v);
    }
    // v at the new 1-based position Q; lane d holds the ancestor at depth d.  Deep: Q >= 128.
    template <bool Deep>
    CCA_HD HeapEntry push_chain(HeapEntry* h, uint32_t Q, HeapEntry v, HeapEntry top_entry) {
        const uint32_t ln = (uint32_t)Lanes::lane(), T = 31u - (uint32_t)__builtin_clz(Q);
        const uint64_t act = (1ull << T) - 1ull;
        const uint32_t cq = Q >> ((T - ln - 1u) & 31u);  // the chain's node one level down
        const uint32_t c = cq > 2u ? cq : 2u;            // (any node in range for the lanes past the chain)
        const HeapEntry e = Lanes::entry(h, c >> 1);
        const uint32_t sib = Lanes::entry(h, c ^ 1u).count;
        const uint64_t sink = Lanes::vote(v.count < e.count) & act;  // the ancestors that move down
        const uint32_t at = (uint32_t)__builtin_ctzll(sink | (1ull << T));  // v's depth
        const bool mv = ln >= at;
        if (mv & (ln < T)) Lanes::entry(h, c) = e;
        Lanes::entry(h, Q >> (T - at)) = v;
        // the new count one level down the chain: an ancestor that moved, v, or what was there above v
        const uint32_t ec = ln < T ? e.count : 0xFFFFFFFFu;
        const uint32_t below = Lanes::next(ec, 0xFFFFFFFFu);
        const uint32_t now = mv ? ec : (v.count < below ? v.count : below);
        const bool odd = (c & 1u) != 0u;
        const uint32_t nb = (uint32_t)Lanes::vote((odd ? sib : now) >= (odd ? now : sib)), E = Q << (12 - T), e1 = E >> 6;
        // nodes below depth T - 1 on E's leftmost way down have no two children
        top = changed(top, e1, nb);
        if (Deep) set_subtree(e1 - 64u, changed(subtree(e1 - 64u), 64u | (E & 63u), nb >> 6));
        return at == 0 ? v : top_entry;
    }
    // v as entry number pos + 1; returns the new top
    CCA_HD HeapEntry push(HeapEntry* h, int pos, HeapEntry v, HeapEntry top_entry) {
        const uint32_t Q = (uint32_t)pos + 1u;
        return Q >= 128u ? push_chain<true>(h, Q, v, top_entry) : push_chain<false>(h, Q, v, top_entry);
    }
};

}  // namespace design
}  // namespace cca
