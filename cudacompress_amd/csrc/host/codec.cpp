// Host orchestration of the entropy coder: the equivalent of src/cudaCompress/Encode.cpp:208-917, for
// bitstreams in host memory.  The streaming passes are the device coder's (hip/coder.hip,
// hip/decoder.hip); the tables are designed here, where a merge takes 0.14 us (65,441 symbols, 8.9 ms)
// instead of the 0.9 us of a wave's serial chain, so a call of a few tables ends sooner.
//
// Encode, for all streams of a volume at once:
//   1. upload of the stream list; the stats pass (zero-run pairs, histograms)     -> sync #1: histograms
//   2. table design on the host (libstdc++ heap/sort, as the reference), exact bit counts from
//      histogram x length, the layout of every section (Encode.cpp:402-463 rl, :751-782 huff)
//   3. one upload (sequence records, symbols in codeword order and, for small alphabets, the code tables,
//      which the device makes of the symbols otherwise); the pack writes the sections in place -> sync #2:
//      words
// The reference does >= streams + 6 host synchronisations per encodeRLHuff, per level of a volume.
//
// Decode walks the sections' heads on the host (counts, sizes, as Encode.cpp:522-621; the symbol
// lists, unless they are few and short, and the codewords are left to the device), stages the sequence
// records and the bitstream in one pinned buffer, uploads it with a single copy and enqueues the table build,
// the block decode and the zero-run expansion.
#include "codec.hpp"

#include <algorithm>
#include <cstring>

#include "../hip/huff_design.hpp"
#include "batch.hpp"
#include "bitio.hpp"
#include "huffman_table.hpp"
#include "parallel.hpp"

namespace cca {
namespace {

// Bump allocator over a pinned host buffer mirrored by a device buffer.
struct Staging {
    size_t off = 0;
    template <class T>
    size_t push(size_t count) {
        off = align_up(off, 256);
        const size_t o = off;
        off += count * sizeof(T);
        return o;
    }
};

// Most arena words (64 MB) that are taken on the chance that every stream uses its whole alphabet, and the
// guess up to which none are: below a megabyte an allocation costs next to nothing and above 0.35 ms, more
// than to run the statistics again (first call of an instance on 32^3 floats 355 us with 0.7 MB and 1063 with
// 1.2; on a 64^3 lossless field, which needs 5.8 MB, the second run is 70 us) unless the call has many symbols
// (4096^2 of terrain: 1.1 ms).
constexpr uint64_t kArenaGuess = 1u << 24, kArenaSmall = 200000, kArenaSymbols = 1u << 23;
// Words that come down with the records at most, and that are pinned for it from the start (a megabyte; an
// allocation of pinned memory takes 0.02 or 0.35 ms, whatever its size, and each megabyte 0.4 ms to touch).
constexpr uint64_t kDownMost = 1u << 18;
// Bins of a call's alphabets up to which the code tables go up whole: 128 KB take about as long as the launch
// that makes them of the symbols (32^3 floats: 325 us with the tables, 335 with the launch; a 4096^2 terrain's
// alphabets are 4 MB).
constexpr uint64_t kDenseBins = 16384;

// A decode of at most so many sequences, symbols and blocks in all has its tables made here: the launch that
// makes them takes 7 us of the 45 to 70 that such a call has, two sequences 1 to 2 us (one stream of 1000
// symbols, zero runs: 71 us with the launch, 63 without).
constexpr uint32_t kHostTables = 4, kHostSymbols = 1024, kHostBlocks = 1024;

// Code table, lookup table, symbols and block offsets of a sequence, as k_dec_tables makes them.
void host_tables(const HeaderFormat& fmt, const uint32_t* words, uint64_t nbits, uint32_t nblk, DecSeq& s,
                 uint32_t* arena) {
    uint32_t cpl[32] = {0}, fc[32], fi[32];
    BitReader counts(words, nbits, s.hdr_bit + 5), symbols(words, nbits, s.sym_bit);
    for (uint32_t l = 0; l < s.nlen; l++) cpl[l] = counts.bits(fmt.count_bits);
    design::first_codes(cpl, (int)s.nlen, fc, fi);
    for (uint32_t l = 0; l < 32; l++) {
        const bool used = l < s.nlen && cpl[l] > 0;
        s.tab[l] = used ? (int32_t)fi[l] : -1;
        s.tab[32 + l] = used ? (int32_t)fc[l] : -1;
        s.tab[64 + l] = used ? (int32_t)(fc[l] + cpl[l] - 1) : -1;
    }
    uint32_t* lut = arena + s.lut_off;
    uint32_t* syms = lut + (1u << kDecLutBits);
    for (uint32_t k = 0; k < s.nsym; k++) syms[k] = symbols.bits(s.sb);
    // (length << 24) | symbol by the next lb bits; of the codes of a broken table the shorter one counts
    const uint32_t lb = std::min(s.nlen, kDecLutBits);
    std::fill(lut, lut + (1u << lb), 0u);
    for (uint32_t l = lb; l-- > 0;)
        for (uint64_t c = 0; c < cpl[l]; c++) {
            const uint64_t first = ((uint64_t)fc[l] + c) << (lb - l - 1), last = first + (1ull << (lb - l - 1));
            if (last > (1ull << lb)) break;
            const uint32_t sym = fi[l] + c < s.nsym ? syms[fi[l] + c] & 0xFFFFFFu : 0u;
            std::fill(lut + first, lut + last, (l + 1) << 24 | sym);
        }
    const uint16_t* incs = (const uint16_t*)(words + s.incs_off);
    for (uint32_t b = 0, at = 0; b < nblk; b++) arena[s.boff_off + b] = at += incs[b];
}

}  // namespace

void encode_items(cc_instance* I, int symSize, const std::vector<EncodeStream>& streams, uint32_t ncalls,
                  bool last_call_first) {
    DeviceGuard guard(I->device);
    hipStream_t st = I->stream;
    check_symbols(I, symSize);
    const uint32_t ns = (uint32_t)streams.size();
    std::vector<ItemSpec> items(ns);
    for (uint32_t i = 0; i < ns; i++) {
        const EncodeStream& s = streams[i];
        CCA_REQUIRE(s.in != nullptr || s.n == 0, CC_ERR_INVALID_ARG, "null stream");
        CCA_REQUIRE(s.start_bit < 32, CC_ERR_INVALID_ARG, "start bit offset >= 32");
        items[i] = ItemSpec{const_cast<void*>(s.in), s.n, s.rl, s.call};
    }
    const uint32_t cbs = I->cbs;
    const HeaderFormat fmt = header_format(I->dialect, I->log2);
    I->out_words = nullptr;
    I->out_count = 0;
    I->seg_begin.assign(ns, 0);
    I->seg_bits.assign(ns, 0);
    if (ns == 0) return;
    SectionTimer stage(I, 2);

    // ---- 1. pairs and histograms --------------------------------------------------------------
    stage("Encode: Histograms");
    DeviceCoder& D = I->coder;
    EncodeJob job;
    encode_upload(I, D, items, ncalls, symSize, job, st);
    const uint32_t nseq = job.nseq;
    // one device buffer: the coder's state, the sequence records, the arena
    const size_t o_seq = align_up(sizeof(CoderState), 64), o_arena = align_up(o_seq + sizeof(SeqInfo) * nseq, 256);
    // a guess, with a second run of the statistics where it was too small
    const uint64_t alphabet = I->dialect == CC_DIALECT_CPU ? 65536u : std::min<uint64_t>(1ull << I->log2, 65536u);
    uint64_t cap = 1024 + (uint64_t)nseq * (kStatBins + 2 * design_leaf_words());
    if (cap > kArenaSmall || job.total_syms >= kArenaSymbols)
        cap = std::max(cap, std::min(cap + ns * alphabet, kArenaGuess));
    cap = std::max(cap, I->enc_arena);
    unsigned char *d, *h;
    for (int attempt = 0;; attempt++) {
        d = (unsigned char*)I->d_enc.get(o_arena + 4 * cap);
        encode_stats(D, job, (SeqInfo*)(d + o_seq), (uint32_t*)(d + o_arena), cap, (CoderState*)d, st);
        // the state, the records and as much of the arena as the last call used come down together
        const uint64_t first = std::min(cap, std::max<uint64_t>(I->enc_down, 4096));
        h = (unsigned char*)I->h_down.get(o_arena + 4 * std::min<uint64_t>(cap, kDownMost));
        CCA_HIP(hipMemcpyAsync(h, d, o_arena + 4 * first, hipMemcpyDeviceToHost, st));
        CCA_HIP(hipStreamSynchronize(st));
        const CoderState s = *(const CoderState*)h;
        if (s.err == kErrScratch && attempt < 4) {
            cap = std::max<uint64_t>(2 * cap, s.scratch_used + s.scratch_used / 4);
            continue;
        }
        CCA_REQUIRE(s.err == kErrNone, CC_ERR_OUT_OF_MEMORY, "coder arena exhausted");
        const uint64_t used = std::min<uint64_t>(s.scratch_used, cap);
        if (used > first) {
            // (past kDownMost pinned for what comes down, not for the arena)
            const uint64_t have = I->h_down.cap < o_arena + 4 * used ? 0 : o_arena + 4 * first;
            h = (unsigned char*)I->h_down.get(o_arena + 4 * used);
            CCA_HIP(hipMemcpyAsync(h + have, d + have, o_arena + 4 * used - have, hipMemcpyDeviceToHost, st));
            CCA_HIP(hipStreamSynchronize(st));
        }
        I->enc_arena = cap;
        I->enc_down = std::min<uint64_t>(align_up(used, 4096), kDownMost);
        break;
    }
    std::vector<SeqInfo> seqs((const SeqInfo*)(h + o_seq), (const SeqInfo*)(h + o_seq) + nseq);
    const uint32_t* arena = (const uint32_t*)(h + o_arena);

    // ---- 2. table design and layout -------------------------------------------------------------
    stage("Encode: Design Huffman Tables");
    std::vector<EncTable> tables(nseq);
    std::vector<cc_status> rcs(nseq, CC_OK);
    std::vector<uint64_t> bits(nseq, 0);
    double work_us = 0;
    for (const SeqInfo& s : seqs) work_us += s.err ? 0.0 : 0.08 * s.nsym + 0.002 * s.smax;
    parallel_for(nseq, work_us, [&](size_t j) {
        const SeqInfo& s = seqs[j];
        if (s.err) return;
        const uint32_t* hist = arena + s.hist_off;
        rcs[j] = design_table(fmt.dialect, hist, s.smax, tables[j]);
        if (rcs[j] != CC_OK) return;
        uint64_t b = 0;
        const EncTable& t = tables[j];
        for (size_t l = 0, k = 0; l < t.count_per_length.size(); l++)
            for (uint32_t c = t.count_per_length[l]; c > 0; c--, k++) {
                const uint32_t sym = t.symbols[k];
                b += (uint64_t)(hist[sym] - (s.quirk && sym == 65535u ? 1u : 0u)) * (l + 1);  // the counted pad is not encoded
            }
        bits[j] = b;
    });
    // first sequence of every stream, and of every call (streams come grouped by call)
    std::vector<uint32_t> first_seq(ns), call_first(ncalls + 1, nseq);
    for (uint32_t i = 0, k = 0; i < ns; i++) {
        first_seq[i] = k;
        k += streams[i].rl ? 2 : 1;
    }
    for (uint32_t i = ns, c = ncalls; c-- > 0;) {
        call_first[c] = call_first[c + 1];
        while (i > 0 && streams[i - 1].call == c) call_first[c] = first_seq[--i];
    }
    for (uint32_t q = 0; q < ncalls; q++) {
        const uint32_t c = last_call_first ? ncalls - 1 - q : q;
        const uint32_t j0 = call_first[c], j1 = call_first[c + 1];
        // HuffmanTable.cu:409-419 (checked per design call)
        for (uint32_t j = j0; j < j1; j++)
            CCA_REQUIRE(seqs[j].err != kErrOverflow, CC_ERR_SYMBOL_OVERFLOW,
                        "symbol exceeds 2^log2HuffmanDistinctSymbolCountMax");
        for (uint32_t j = j0; j < j1; j++) {
            CCA_REQUIRE(rcs[j] == CC_OK, rcs[j], "Huffman codeword longer than 31 bits");
            if (fmt.dialect == CC_DIALECT_CPU)
                CCA_REQUIRE(tables[j].symbols.size() < (1u << 14), CC_ERR_SYMBOL_OVERFLOW,
                            "more than 16383 distinct symbols cannot be described in the CPU dialect header");
            CCA_REQUIRE(bits[j] < (1ull << 32), CC_ERR_INVALID_ARG, "coded stream exceeds 2^32 bits");
        }
    }
    // sections in stream order; the arena: every table's symbols in codeword order, then its codes and lengths
    // by symbol, which go up too or which the device makes, and the coding-block offsets, which the pack fills
    uint64_t pos = 0, up = 0, bins = 0;
    uint32_t most_syms = 0;
    for (uint32_t i = 0; i < ns; i++) {
        const EncodeStream& s = streams[i];
        I->seg_begin[i] = pos;
        if (s.rl) pos += 1 + (s.start_bit ? 1 : 0);  // the pair count, from a word boundary on
        for (uint32_t q = 0; q < (s.rl ? 2u : 1u); q++) {
            const uint32_t j = first_seq[i] + q;
            SeqInfo& r = seqs[j];
            const EncTable& t = tables[j];
            const uint64_t tb = table_bits(fmt, t), tw = (tb + 31) / 32;
            const uint64_t nblk = div_up(r.count, cbs);
            // a header that starts inside a word may reach one word further
            if (!s.rl) pos += (tb + s.start_bit + 31) / 32 - tw;
            r.out_off = pos;
            pos += tw + 1 + (bits[j] + 31) / 32 + (nblk + 1) / 2;
            r.nlen = (uint32_t)t.count_per_length.size();
            r.nsym = (uint32_t)t.symbols.size();
            r.bits = bits[j];
            for (uint32_t l = 0; l < 32; l++) r.cpl[l] = l < r.nlen ? t.count_per_length[l] : 0u;
            r.syms_off = up;
            up = align_up(up + std::max<uint32_t>(r.nsym, 1), 16);
            most_syms = std::max(most_syms, r.nsym);
            bins += r.smax + 1;
        }
        I->seg_bits[i] = (pos - I->seg_begin[i]) * 32;
    }
    const uint64_t total = pos;
    uint64_t arena_words = up;
    for (SeqInfo& r : seqs) {
        r.code_off = arena_words;
        arena_words = align_up(arena_words + 2ull * (r.smax + 1), 16);
    }
    const bool dense = bins <= kDenseBins;
    if (dense) up = arena_words;
    for (SeqInfo& r : seqs) {
        r.boff_off = arena_words;
        arena_words += align_up(std::max<uint32_t>(div_up(r.count, cbs), 1), 16);
    }

    // ---- 3. codewords ----------------------------------------------------------------------------
    stage("Encode: Huffman Encode");
    d = (unsigned char*)I->d_enc.get(o_arena + 4 * std::max(arena_words, cap));  // (what is there is not needed any more)
    unsigned char* u = (unsigned char*)I->h_up.get(o_arena + 4 * up);
    *(CoderState*)u = CoderState{0, total, 0, 0, 0};
    memcpy(u + o_seq, seqs.data(), sizeof(SeqInfo) * nseq);
    uint32_t* ua = (uint32_t*)(u + o_arena);
    for (uint32_t j = 0; j < nseq; j++) {
        const SeqInfo& r = seqs[j];
        const std::vector<uint32_t>& syms = tables[j].symbols;
        memcpy(ua + r.syms_off, syms.data(), 4ull * syms.size());
        if (!dense) continue;
        uint32_t fc[32], fi[32], *code = ua + r.code_off, *len = code + r.smax + 1;
        design::first_codes(r.cpl, (int)r.nlen, fc, fi);
        for (uint32_t l = 0; l < r.nlen; l++)
            for (uint32_t c = 0; c < r.cpl[l]; c++) {
                code[syms[fi[l] + c]] = fc[l] + c;
                len[syms[fi[l] + c]] = l + 1;
            }
    }
    CCA_HIP(hipMemcpyAsync(d, u, o_arena + 4 * up, hipMemcpyHostToDevice, st));
    if (!dense) coder_code_tables((const SeqInfo*)(d + o_seq), nseq, most_syms, (uint32_t*)(d + o_arena), st);
    uint32_t* dw = I->d_words.as<uint32_t>(std::max<uint64_t>(total, 1));
    encode_pack(D, job, (SeqInfo*)(d + o_seq), (uint32_t*)(d + o_arena), (CoderState*)d, dw, total, st);
    uint32_t* hw = I->h_words.as<uint32_t>(std::max<uint64_t>(total, 1));
    CCA_HIP(hipMemcpyAsync(hw, dw, 4 * total, hipMemcpyDeviceToHost, st));
    CCA_HIP(hipStreamSynchronize(st));

    // segments that start inside a word: zero bits where the caller's are, the header behind them
    stage("Encode: Bitstream Layout");
    for (uint32_t i = 0; i < ns; i++) {
        const EncodeStream& s = streams[i];
        if (!s.start_bit) continue;
        if (s.rl) {
            hw[I->seg_begin[i]] = 0;
            continue;
        }
        std::vector<uint32_t> head;
        BitWriter w(head);
        w.set_pos(s.start_bit);
        write_table(fmt, tables[first_seq[i]], w);
        memcpy(hw + I->seg_begin[i], head.data(), 4 * head.size());
    }
    I->out_words = hw;
    I->out_count = total;
}

void encode_streams(cc_instance* I, bool rl, int symSize, const void* const* streams, uint32_t ns, uint32_t n,
                    const uint32_t* startBits) {
    check_symbols(I, symSize);
    CCA_REQUIRE(ns == 0 || streams != nullptr, CC_ERR_INVALID_ARG, "null stream array");
    std::vector<EncodeStream> s(ns);
    for (uint32_t i = 0; i < ns; i++) s[i] = EncodeStream{streams[i], n, rl, 0, startBits ? startBits[i] : 0u};
    SectionTimer call(I, 1);
    if (ns) call(rl ? "Encode RLHuff" : "Encode Huff");
    encode_items(I, symSize, s, 1);
}

void decode_items(cc_instance* I, int symSize, const uint32_t* const* bsWords, const uint64_t* bsBits,
                  uint64_t* bsPos, uint32_t nbs, const std::vector<DecodeStream>& streams) {
    DeviceGuard guard(I->device);
    hipStream_t st = I->stream;
    check_symbols(I, symSize);
    CCA_REQUIRE(nbs >= 1 && bsWords && bsBits && bsPos, CC_ERR_INVALID_ARG, "no bitstream");
    const uint32_t ns = (uint32_t)streams.size();
    if (ns == 0) return;
    const uint32_t cbs = I->cbs;
    const HeaderFormat fmt = header_format(I->dialect, I->log2);
    SectionTimer stage(I, 2);
    stage("Decode: Read Tables + Upload");

    // ---- the sections' heads ------------------------------------------------------------------
    // Bit and word positions are kept from the first word of each bitstream that is read.
    std::vector<uint64_t> w0(nbs, ~0ull), w1(nbs, 0);
    std::vector<DecSeq> seqs;
    std::vector<DecItem> items(ns);
    std::vector<uint32_t> seq_bs;
    std::vector<DecPart> parts;
    auto read_coded = [&](BitReader& r, uint32_t bs, uint32_t item, uint32_t count) {
        DecSeq s{};
        s.hdr_bit = r.pos();
        s.nlen = r.bits(5);
        uint64_t codes = 0;
        for (uint32_t l = 0; l < s.nlen; l++) codes += r.bits(fmt.count_bits);
        s.nsym = r.bits(fmt.count_bits);
        s.sb = r.bits(fmt.symbits_bits);
        // HuffmanTable.cu:138-139: a stored 0 with more than one symbol means 16 (Symbol16 only)
        if (fmt.dialect == CC_DIALECT_GPU && fmt.symbits_bits == 4 && s.sb == 0 && s.nsym > 1) s.sb = 16;
        // lengths without a symbol code nothing: an empty table (the device refuses lengths and symbols that
        // do not fit, and would leave the output of a stream without a pair as it is)
        if (s.nsym == 0) s.nlen = 0;
        CCA_REQUIRE(s.sb <= 32 && r.ok(), CC_ERR_CORRUPT_STREAM, "malformed Huffman table header");
        s.sym_bit = r.pos();
        r.skip_bits((uint64_t)s.sb * s.nsym);
        CCA_REQUIRE(r.ok() && (s.nsym == 0 || s.nlen == 0 || codes == s.nsym), CC_ERR_CORRUPT_STREAM,
                    "malformed Huffman table header");
        const uint32_t nbits = r.aligned_u32();
        s.words_off = r.pos() >> 5;
        s.nwords_cw = (uint32_t)(((uint64_t)nbits + 31) / 32);
        r.skip_bits(32ull * s.nwords_cw);
        r.align32();
        s.incs_off = r.pos() >> 5;
        const uint16_t* incs = (const uint16_t*)r.word_ptr();
        const uint32_t noff = div_up(count, cbs);
        r.skip_aligned(noff, 2);
        CCA_REQUIRE(r.ok(), CC_ERR_CORRUPT_STREAM, "bitstream ends inside a coded stream");
        CCA_REQUIRE(count == 0 || s.nsym != 0, CC_ERR_CORRUPT_STREAM, "empty table for a non-empty stream");
        // the block offsets are running sums (unpackInc16CPU, PackInc.cu:222-229): the last is the largest
        const uint32_t tail = s.nsym > (1u << kDecLutBits) ? s.nsym - (1u << kDecLutBits) : 0u;
        const uint32_t np = std::max({1u, div_up(noff, kPartBlocks), div_up(tail, kPartSymbols)});
        uint64_t sum = 0;
        for (uint32_t k = 0; k < np; k++) {
            parts.push_back(DecPart{(uint32_t)seqs.size(), k, (uint32_t)sum, 0});
            const uint64_t end = std::min<uint64_t>(noff, (uint64_t)(k + 1) * kPartBlocks);
            for (uint64_t b = (uint64_t)k * kPartBlocks; b < end; b++) sum += incs[b];
        }
        CCA_REQUIRE(sum <= 32ull * s.nwords_cw, CC_ERR_CORRUPT_STREAM, "coding block offset beyond the codewords");
        s.count = count;
        s.item = item;
        seqs.push_back(s);
        seq_bs.push_back(bs);
    };
    uint64_t rl_elems = 0;
    std::vector<uint64_t> rl_off(ns, 0);
    for (uint32_t i = 0; i < ns; i++) {
        const DecodeStream& s = streams[i];
        const uint32_t b = s.bs;
        CCA_REQUIRE(b < nbs && bsWords[b], CC_ERR_INVALID_ARG, "bad bitstream index");
        BitReader r(bsWords[b], bsBits[b], bsPos[b]);
        w0[b] = std::min(w0[b], bsPos[b] >> 5);
        items[i] = DecItem{s.out, s.n, s.rl ? 1u : 0u, (uint32_t)seqs.size(), 0};
        uint32_t count = s.n;
        if (s.rl) {
            count = r.aligned_u32();
            CCA_REQUIRE(r.ok() && count <= s.n, CC_ERR_CORRUPT_STREAM, "run-length pair count exceeds the stream length");
            read_coded(r, b, i, count);
            rl_off[i] = rl_elems;
            rl_elems += align_up(std::max<uint32_t>(count, 1), 64);
        }
        read_coded(r, b, i, count);
        bsPos[b] = r.pos();
        w1[b] = std::max(w1[b], (r.pos() + 31) >> 5);
        CCA_REQUIRE(s.out != nullptr || s.n == 0, CC_ERR_INVALID_ARG, "null output stream");
    }
    const uint32_t nseq = (uint32_t)seqs.size();

    // ---- the upload and the arena ----------------------------------------------------------------
    uint32_t nlong = 0, nshort = 0, nchunks = 0;
    uint64_t total_syms = 0, arena = 0, total_nsym = 0, total_blk = 0;
    for (DecSeq& s : seqs) {
        const uint32_t nblk = div_up(s.count, cbs);
        total_nsym += s.nsym;
        total_blk += nblk;
        (dec_long(nblk) ? nlong : nshort) += dec_entries(nblk);
        s.boff_off = arena;
        s.lut_off = arena + align_up(std::max<uint32_t>(nblk, 1), 16);
        arena = s.lut_off + align_up((1u << kDecLutBits) + (uint64_t)s.nsym + 1, 16);
    }
    for (uint32_t i = 0; i < ns; i++) total_syms += items[i].n;
    for (uint32_t i = 0; i < ns; i++)  // an RLE stream without a pair still has its output cleared
        if (items[i].rl && items[i].n) nchunks += std::max(1u, rle_chunks(seqs[items[i].seq].count, true));
    const bool made_here = nseq <= kHostTables && total_nsym <= kHostSymbols && total_blk <= kHostBlocks;
    if (made_here) parts.clear();
    Staging s;
    const size_t o_state = s.push<CoderState>(1), o_seq = s.push<DecSeq>(nseq), o_item = s.push<DecItem>(ns);
    const size_t o_wseq = s.push<uint32_t>(nlong + nshort), o_wfirst = s.push<uint32_t>(nlong + nshort);
    const size_t o_ifirst = s.push<uint32_t>(ns + 1), o_part = s.push<DecPart>(parts.size());
    const size_t o_arena = s.push<uint32_t>(made_here ? arena + nchunks : 0);
    std::vector<size_t> o_words(nbs, 0);
    for (uint32_t b = 0; b < nbs; b++)
        if (w1[b] > w0[b]) o_words[b] = s.push<uint32_t>(w1[b] - w0[b]);
    const size_t total = s.off;
    // the first staging slot whose upload is done, or the next one in turn after a wait: a caller that waits
    // for its decodes uses one (a volume is one decode, and four slots of its size are four times its words
    // pinned, each megabyte 0.4 ms to touch for the first time)
    int slot = 0;
    while (slot < kDecodeRing && hipEventQuery(I->dec_event[slot]) != hipSuccess) slot++;
    if (slot > 0) (void)hipGetLastError();  // "not ready" is no error of this call
    if (slot == kDecodeRing) {
        slot = I->dec_slot;
        CCA_HIP(hipEventSynchronize(I->dec_event[slot]));
    }
    I->dec_slot = (slot + 1) % kDecodeRing;
    unsigned char* h = (unsigned char*)I->h_dec_stage[slot].get(total);
    unsigned char* d = (unsigned char*)I->d_dec_stage.get(total);
    unsigned char* dsym = (unsigned char*)I->d_dec_sym.get(std::max<uint64_t>(rl_elems, 1) * symSize);
    unsigned char* dzc = (unsigned char*)I->d_dec_zc.get(std::max<uint64_t>(rl_elems, 1) * symSize);

    *(CoderState*)(h + o_state) = CoderState{};
    uint32_t* hws = (uint32_t*)(h + o_wseq);
    uint32_t* hwf = (uint32_t*)(h + o_wfirst);
    uint32_t* hif = (uint32_t*)(h + o_ifirst);
    uint32_t wl = 0, ws = nlong;
    for (uint32_t j = 0; j < nseq; j++) {
        DecSeq& q = seqs[j];
        const uint32_t b = seq_bs[j], i = q.item;
        if (made_here) host_tables(fmt, bsWords[b], bsBits[b], div_up(q.count, cbs), q, (uint32_t*)(h + o_arena));
        q.base = (const uint32_t*)(d + o_words[b]);
        q.nwords = w1[b] - w0[b];
        q.hdr_bit -= 32 * w0[b];
        q.sym_bit -= 32 * w0[b];
        q.words_off -= w0[b];
        q.incs_off -= w0[b];
        q.out = !items[i].rl ? items[i].out : (j == items[i].seq ? dsym : dzc) + rl_off[i] * symSize;
        add_block_entries(j, div_up(q.count, cbs), hws, hwf, wl, ws);
    }
    hif[0] = 0;
    for (uint32_t i = 0; i < ns; i++)
        hif[i + 1] = hif[i] + (items[i].rl && items[i].n ? std::max(1u, rle_chunks(seqs[items[i].seq].count, true)) : 0u);
    memcpy(h + o_seq, seqs.data(), sizeof(DecSeq) * nseq);
    memcpy(h + o_item, items.data(), sizeof(DecItem) * ns);
    memcpy(h + o_part, parts.data(), sizeof(DecPart) * parts.size());
    for (uint32_t b = 0; b < nbs; b++)
        if (w1[b] > w0[b]) memcpy(h + o_words[b], bsWords[b] + w0[b], 4 * (w1[b] - w0[b]));
    uint32_t* scratch =
        made_here ? (uint32_t*)(d + o_arena) : I->d_dec_arena.as<uint32_t>(arena + std::max<uint32_t>(nchunks, 1));
    CCA_HIP(hipMemcpyAsync(d, h, total, hipMemcpyHostToDevice, st));
    CCA_HIP(hipEventRecord(I->dec_event[slot], st));

    stage("Decode: Huffman Decode");
    const RleChunks rc{(const uint32_t*)(d + o_ifirst), nchunks, scratch + arena};
    const CoderParams p = params_of(I);
    coder_decode_parsed((DecSeq*)(d + o_seq), nseq, p, symSize, scratch, (CoderState*)(d + o_state),
                        (const DecItem*)(d + o_item), (const uint32_t*)(d + o_wseq), (const uint32_t*)(d + o_wfirst),
                        nlong + nshort, nlong, (const DecPart*)(d + o_part), (uint32_t)parts.size(), total_syms, rc, st);
    if (nchunks) {
        stage("Decode: Run Length Decode");
        coder_decode_expand((const DecItem*)(d + o_item), ns, (DecSeq*)(d + o_seq), symSize, rc,
                            (CoderState*)(d + o_state), total_syms, st);
    }
}

void decode_streams(cc_instance* I, bool rl, int symSize, const uint32_t* const* bsWords, const uint64_t* bsBits,
                    uint64_t* bsPos, uint32_t nbs, const uint32_t* s2b, void* const* outs, uint32_t ns, uint32_t n) {
    check_symbols(I, symSize);
    CCA_REQUIRE(ns == 0 || outs != nullptr, CC_ERR_INVALID_ARG, "null output array");
    std::vector<DecodeStream> s(ns);
    for (uint32_t i = 0; i < ns; i++) s[i] = DecodeStream{outs[i], n, rl, s2b ? s2b[i] : 0u};
    SectionTimer call(I, 1);
    if (ns) call(rl ? "Decode RLHuff" : "Decode Huff");
    decode_items(I, symSize, bsWords, bsBits, bsPos, nbs, s);
}

}  // namespace cca
