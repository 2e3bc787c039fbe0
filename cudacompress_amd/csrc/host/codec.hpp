// Entropy-coder orchestration (host side of encodeRLHuff/encodeHuff/decodeRLHuff/decodeHuff).
#pragma once

#include <vector>

#include "instance.hpp"

namespace cca {

// One symbol stream of an encode: the streams of one `call` fail together, in call order.
struct EncodeStream {
    const void* in;
    uint32_t n;
    bool rl;
    uint32_t call;
    uint32_t start_bit;  // bits of the segment's first word that belong to the caller (0..31)
};
// Encodes every stream into one word array, segment after segment, left in inst->out_words /
// seg_begin / seg_bits.  last_call_first: the order in which failing calls are reported.  Throws cca::Error.
void encode_items(cc_instance* inst, int symSize, const std::vector<EncodeStream>& streams, uint32_t ncalls,
                  bool last_call_first = false);

// One stream of a decode: the next of its kind in bitstream `bs`.
struct DecodeStream {
    void* out;
    uint32_t n;
    bool rl;
    uint32_t bs;
};
// Decodes the streams in order; positions advanced.  Work is left enqueued on inst->stream.
void decode_items(cc_instance* inst, int symSize, const uint32_t* const* bsWords, const uint64_t* bsBits,
                  uint64_t* bsPos, uint32_t nbs, const std::vector<DecodeStream>& streams);

// One encodeRLHuff / encodeHuff (decodeRLHuff / decodeHuff) call.
void encode_streams(cc_instance* inst, bool rl, int symSize, const void* const* streams, uint32_t ns, uint32_t n,
                    const uint32_t* startBits);
void decode_streams(cc_instance* inst, bool rl, int symSize, const uint32_t* const* bsWords, const uint64_t* bsBits,
                    uint64_t* bsPos, uint32_t nbs, const uint32_t* s2b, void* const* outs, uint32_t ns, uint32_t n);

}  // namespace cca
