// Volume codecs built on the library API, restating the caller layouts of
// src/examples/CompressVolume.cpp (compressVolumeFloat :313-409, decompressVolumeFloat :412-516,
// compressVolumeLossless :234-277, decompressVolumeLossless :279-309,
// compressVolumeFloatQuantFirst :651-757, decompressVolumeFloatQuantFirst :759-856, the
// multi-channel decoders decompressVolumeFloatMultiChannel :518-648 and
// decompressVolumeFloatQuantFirstMultiChannel :863-985) and, for 2D lossless input, the three-band
// layout of src/examples/CompressHeightfield.cpp:116-126.
//
// Differences from the reference callers, none of which changes the bitstream:
//  * the transforms come first and every level's streams are coded in one go (the reference codes
//    level by level, each with its synchronisations); a 9/7 volume is transformed as a brick of one;
//  * every kernel runs on the instance stream (the reference quantizes on the default stream);
//  * decode outputs are not cleared first (decodeRLHuff here writes every element);
//  * 2D lossless input (sizeZ == 1) uses 3 highpass bands per level -- compressVolumeLossless
//    itself only handles 3D (it would compute a zero blockSizeZ);
//  * decompressVolumeFloatQuantFirst starts its inverse transforms from the buffer holding the
//    coarsest level's coefficients; the reference starts from buffer numLevels % 2, the same
//    buffer for an even level count (an odd count reads a buffer its decode did not fill); its
//    multi-channel form also carries that index from one channel to the next;
//  * the multi-channel decoders give each channel exactly its single-channel decode.
#include "volume.hpp"

#include <algorithm>
#include <cstring>

#include "../kernels.hpp"
#include "bricks.hpp"
#include "codec.hpp"

namespace cca {
namespace {

struct Band {
    uint32_t x, y, z;
};
Band band_of(uint32_t block, bool is3d) {  // CompressVolume.cpp:375-379, CompressHeightfield.cpp:119-121
    if (is3d) return Band{block % 2, block / 2 % 2, block / 4};
    return Band{block % 2, block / 2, 0};
}

// Symbol streams of a 3D volume in bitstream order: the lowpass band, then 7 bands a level from the
// coarsest, stream k from element at[k] of the symbol buffer on.
struct VolumeStreams {
    std::vector<uint64_t> at;
    std::vector<uint32_t> n, call;
    std::vector<bool> rl;
    uint64_t elems = 0;
    VolumeStreams(uint64_t volume, uint32_t levels, bool rle_only_lvl0) {
        auto add = [&](uint64_t count, bool zero_runs, uint32_t c) {
            at.push_back(elems);
            n.push_back((uint32_t)count);
            rl.push_back(zero_runs);
            call.push_back(c);
            elems += align_up(count, 64);
        };
        add(volume >> (3 * levels), false, 0);
        for (uint32_t level = levels; level-- > 0;)
            for (uint32_t b = 1; b <= 7; b++) add(volume >> (3 * (level + 1)), !(level > 0 && rle_only_lvl0), levels - level);
    }
    // stream of band b (1..7) of `level`, and the lowpass one
    uint32_t band(uint32_t levels, uint32_t level, uint32_t b) const { return 1 + 7 * (levels - 1 - level) + b - 1; }
};

void check_volume(uint32_t sx, uint32_t sy, uint32_t sz, uint32_t levels) {
    CCA_REQUIRE(levels >= 1 && levels < 32, CC_ERR_INVALID_ARG, "numLevels must be >= 1");
    CCA_REQUIRE(sz > 1, CC_ERR_INVALID_ARG, "the volume codecs for floats are 3D");
    const uint32_t f_all = 1u << levels;
    CCA_REQUIRE(sx % f_all == 0 && sy % f_all == 0 && sz % f_all == 0, CC_ERR_INVALID_ARG,
                "sizes must be divisible by 2^numLevels");
}

// Volumes as bricks: their levels' transforms with the quantizer fused, the streams in bitstream order.
std::vector<ItemSpec> volume_bricks(cc_instance* I, BrickJob& job, uint32_t levels, int symSize, bool rle_only_lvl0) {
    job.L = levels;
    job.symSize = symSize;
    std::vector<ItemSpec> items = bricks_transforms_layout(I->batch, job);
    for (size_t k = 0; k < items.size(); k++)  // streams 1 .. 7 (levels - 1) of a brick: levels above 0
        if (rle_only_lvl0 && k % (1 + 7 * levels) <= 7 * (levels - 1)) items[k].rl = false;
    return items;
}

// Volumes too large for 32-bit element offsets: pitched levels in two buffers.
void compress_volume_float_large(cc_instance* I, const float* image, uint32_t sx, uint32_t sy, uint32_t sz,
                                 uint32_t levels, float q0, const VolumeStreams& vs, int symSize) {
    hipStream_t st = I->stream;
    const uint64_t elems = (uint64_t)sx * sy * sz;
    float* dwt[2] = {I->d_vol[0].as<float>(elems), I->d_vol[1].as<float>(elems)};
    unsigned char* sym = (unsigned char*)I->d_vol[2].get(vs.elems * symSize);
    int d = 0;
    dwt97_forward(dwt[d], dwt[1 - d], dwt[d], image, (int)sx, (int)sy, (int)sz, 1, 0, 0, 0, 0, st);
    uint32_t f = 2;
    for (uint32_t level = 1; level < levels; level++) {
        dwt97_forward(dwt[1 - d], dwt[d], dwt[1 - d], dwt[d], (int)(sx / f), (int)(sy / f), (int)(sz / f), 1, (int)sx,
                      (int)(sx * sy), (int)sx, (int)(sx * sy), st);
        d = 1 - d;
        f *= 2;
    }
    // lowpass band (CompressVolume.cpp:353-362), highpass bands, coarsest level first (:365-402)
    quantize_to_symbols(sym, symSize, dwt[d], false, sx / f, sy / f, sz / f, q0 / float(f / 2), sx, sx * sy, 0, st);
    for (uint32_t level = levels; level-- > 0; f /= 2, d = 1 - d) {
        const uint32_t bx = sx / f, by = sy / f, bz = sz / f;
        for (uint32_t b = 1; b <= 7; b++) {
            const Band bd = band_of(b, true);
            const uint64_t off = bd.x * bx + (uint64_t)bd.y * by * sx + (uint64_t)bd.z * bz * sx * sy;
            quantize_to_symbols(sym + vs.at[vs.band(levels, level, b)] * symSize, symSize, dwt[d] + off, false, bx, by,
                                bz, q0 / float(f / 2), sx, sx * sy, 0, st);
        }
    }
    std::vector<EncodeStream> streams;
    for (size_t k = 0; k < vs.n.size(); k++)
        streams.push_back(EncodeStream{sym + vs.at[k] * symSize, vs.n[k], vs.rl[k], vs.call[k], 0});
    encode_items(I, symSize, streams, levels + 1);
}

void decompress_volume_float_large(cc_instance* I, float* image, const void* sym, const VolumeStreams& vs, uint32_t sx,
                                   uint32_t sy, uint32_t sz, uint32_t levels, float q0, int symSize) {
    hipStream_t st = I->stream;
    const uint64_t elems = (uint64_t)sx * sy * sz;
    float* dwt[2] = {I->d_vol[0].as<float>(elems), I->d_vol[1].as<float>(elems)};
    // device table of every level's 7 band pointers for the fused dequantize + IDWT
    const void** hptr = I->h_vol_ptrs.as<const void*>(7 * levels);
    for (uint32_t k = 0; k < 7 * levels; k++) hptr[k] = (const unsigned char*)sym + vs.at[1 + k] * symSize;
    const void** dptr = I->d_vol_ptrs.as<const void*>(7 * levels);
    CCA_HIP(hipMemcpyAsync(dptr, hptr, sizeof(void*) * 7 * levels, hipMemcpyHostToDevice, st));
    uint32_t f = 1u << levels;
    unquantize_from_symbols(image, sym, symSize, sx / f, sy / f, sz / f, q0 / float(f / 2), sx, sx * sy, 0, st);
    for (uint32_t level = levels; level-- > 0;) {
        f /= 2;
        dwt97_inverse_from_symbols(image, dwt[1], dwt[0], image, dptr + 7 * (levels - 1 - level), symSize, q0 / float(f),
                                   (int)(sx / f), (int)(sy / f), (int)(sz / f), 1, (int)sx, (int)(sx * sy), (int)sx,
                                   (int)(sx * sy), st);
    }
    // the pointer table upload must finish before the pinned copy is rewritten
    CCA_HIP(hipStreamSynchronize(st));
}

}  // namespace

void compress_volume_float(cc_instance* I, const float* image, uint32_t sx, uint32_t sy, uint32_t sz,
                           uint32_t levels, float q0, bool rle_only_lvl0, int symSize) {
    DeviceGuard guard(I->device);
    check_volume(sx, sy, sz, levels);
    CCA_REQUIRE(image, CC_ERR_INVALID_ARG, "null volume");
    check_symbols(I, symSize);
    const uint64_t elems = (uint64_t)sx * sy * sz;
    SectionTimer call(I, 1);
    if (!bricks_serve(I, elems, levels)) {
        call("Encode RLHuff");
        compress_volume_float_large(I, image, sx, sy, sz, levels, q0, VolumeStreams(elems, levels, rle_only_lvl0), symSize);
        return;
    }
    BrickJob job;
    job.bricks = {cc_brick{image, nullptr, sx, sy, sz, q0}};
    const std::vector<ItemSpec> items = volume_bricks(I, job, levels, symSize, rle_only_lvl0);
    bricks_transforms_upload(I, I->batch, job, I->stream);
    bricks_forward_launch(job, I->stream);
    call("Encode RLHuff");
    std::vector<EncodeStream> streams;
    for (size_t k = 0; k < items.size(); k++)  // (the lowpass call, then one a level)
        streams.push_back(EncodeStream{items[k].ptr, items[k].n, items[k].rl, k ? 1 + ((uint32_t)k - 1) / 7 : 0u, 0});
    encode_items(I, symSize, streams, levels + 1);
}

void decompress_volume_float(cc_instance* I, float* image, uint32_t sx, uint32_t sy, uint32_t sz, uint32_t levels,
                             const uint32_t* words, uint64_t nbits, float q0, bool rle_only_lvl0, int symSize) {
    const VolumeChannelIn ch{image, words, nbits, q0};
    decompress_volume_float_multichannel(I, &ch, 1, sx, sy, sz, levels, rle_only_lvl0, symSize);
}

namespace {
// Streams of a lossless field: the lowpass band, then 3 (2D) or 7 (3D) bands a level from the coarsest;
// a level's bands lie one after the other, from element at[level] of the symbol buffer on.
struct LosslessLayout {
    uint32_t nb, levels;
    std::vector<uint64_t> at, per_band, low;  // per level: first band, elements of a band, its lowpass in the low buffer
    uint64_t sym_elems = 0, low_elems = 0;
    LosslessLayout(uint32_t sx, uint32_t sy, uint32_t sz, uint32_t levels_) : nb(sz > 1 ? 7 : 3), levels(levels_) {
        at.resize(levels);
        per_band.resize(levels);
        low.resize(levels);
        for (uint32_t l = 0; l < levels; l++) {
            const uint32_t f = 2u << l;
            per_band[l] = (uint64_t)(sx / f) * (sy / f) * (sz > 1 ? sz / f : 1);
            low[l] = low_elems;
            low_elems += align_up(per_band[l], 64);
        }
        sym_elems = align_up(per_band[levels - 1], 64);
        for (uint32_t l = levels; l-- > 0;) {
            at[l] = sym_elems;
            sym_elems += nb * align_up(per_band[l], 64);
        }
    }
    uint64_t stride(uint32_t level) const { return align_up(per_band[level], 64); }
    // f(symbol offset, count, zero runs, call) for every stream in bitstream order
    template <class F>
    void streams(F f) const {
        f(0, (uint32_t)per_band[levels - 1], false, 0u);
        for (uint32_t l = levels; l-- > 0;)
            for (uint32_t b = 0; b < nb; b++) f(at[l] + b * stride(l), (uint32_t)per_band[l], true, levels - l);
    }
};
void check_lossless(cc_instance* I, uint32_t sx, uint32_t sy, uint32_t sz, uint32_t levels) {
    CCA_REQUIRE(I->log2 <= 16, CC_ERR_INVALID_ARG, "lossless volumes use Symbol16 (log2 <= 16)");
    CCA_REQUIRE(levels >= 1 && levels < 32, CC_ERR_INVALID_ARG, "numLevels must be >= 1");
    const uint32_t f_all = 1u << levels;
    CCA_REQUIRE(sx % f_all == 0 && sy % f_all == 0 && (sz <= 1 || sz % f_all == 0), CC_ERR_INVALID_ARG,
                "sizes must be divisible by 2^numLevels");
}
}  // namespace

// compressVolumeLosslessOneLevel per level, CompressVolume.cpp:84-150 (3D) / compressHeightfieldOneLevel's
// band layout (2D)
void compress_volume_lossless(cc_instance* I, const int16_t* image, uint32_t sx, uint32_t sy, uint32_t sz,
                              uint32_t levels) {
    DeviceGuard guard(I->device);
    hipStream_t st = I->stream;
    check_lossless(I, sx, sy, sz, levels);
    const bool is3d = sz > 1;
    const uint64_t elems = (uint64_t)sx * sy * sz;
    const LosslessLayout lay(sx, sy, sz, levels);
    int16_t* dwt0 = I->d_vol[0].as<int16_t>(elems);
    int16_t* dwt1 = I->d_vol[1].as<int16_t>(elems);
    uint16_t* sym = I->d_vol[2].as<uint16_t>(lay.sym_elems);
    int16_t* low = I->d_vol[3].as<int16_t>(lay.low_elems);
    for (uint32_t level = 0; level < levels; level++) {
        const uint32_t cx = sx >> level, cy = sy >> level, cz = is3d ? sz >> level : 1;
        dwt53_forward(dwt1, dwt0, level == 0 ? image : low + lay.low[level - 1], (int)cx, (int)cy, (int)cz, 0, 0, 0, 0, st);
        const bool last = level + 1 == levels;
        symbolize_level(sym + lay.at[level], lay.stride(level), last ? sym : nullptr, last ? nullptr : low + lay.low[level],
                        dwt1, cx, cy, cz, cx, (uint64_t)cx * cy, st);
    }
    std::vector<EncodeStream> streams;
    lay.streams([&](uint64_t off, uint32_t n, bool rl, uint32_t call) {
        streams.push_back(EncodeStream{sym + off, n, rl, call, 0});
    });
    SectionTimer call(I, 1);
    call("Encode RLHuff");
    encode_items(I, 2, streams, levels + 1, true);
}

// decompressVolumeLosslessOneLevel per level, CompressVolume.cpp:152-226
void decompress_volume_lossless(cc_instance* I, int16_t* image, uint32_t sx, uint32_t sy, uint32_t sz,
                                uint32_t levels, const uint32_t* words, uint64_t nbits) {
    DeviceGuard guard(I->device);
    hipStream_t st = I->stream;
    check_lossless(I, sx, sy, sz, levels);
    const bool is3d = sz > 1;
    const uint64_t elems = (uint64_t)sx * sy * sz;
    const LosslessLayout lay(sx, sy, sz, levels);
    int16_t* dwt0 = I->d_vol[0].as<int16_t>(elems);
    int16_t* dwt1 = I->d_vol[1].as<int16_t>(elems);
    uint16_t* sym = I->d_vol[2].as<uint16_t>(lay.sym_elems);
    int16_t* low = I->d_vol[3].as<int16_t>(lay.low_elems);
    std::vector<DecodeStream> streams;
    lay.streams([&](uint64_t off, uint32_t n, bool rl, uint32_t) { streams.push_back(DecodeStream{sym + off, n, rl, 0}); });
    uint64_t pos = 0;
    {
        SectionTimer call(I, 1);
        call("Decode RLHuff");
        decode_items(I, 2, &words, &nbits, &pos, 1, streams);
    }
    for (uint32_t level = levels; level-- > 0;) {
        const uint32_t cx = sx >> level, cy = sy >> level, cz = is3d ? sz >> level : 1;
        const bool last = level + 1 == levels;
        unsymbolize_level(dwt1, sym + lay.at[level], lay.stride(level), last ? sym : nullptr,
                          last ? nullptr : low + lay.low[level], cx, cy, cz, cx, (uint64_t)cx * cy, st);
        dwt53_inverse(level == 0 ? image : low + lay.low[level - 1], dwt0, dwt1, (int)cx, (int)cy, (int)cz, 0, 0, 0, 0, st);
    }
}

void compress_volume_float_quant_first(cc_instance* I, const float* image, uint32_t sx, uint32_t sy, uint32_t sz,
                                       uint32_t levels, float step, bool rle_only_lvl0) {
    DeviceGuard guard(I->device);
    hipStream_t st = I->stream;
    CCA_REQUIRE(I->log2 <= 16, CC_ERR_INVALID_ARG, "QuantFirst volumes use Symbol16 (log2 <= 16)");
    CCA_REQUIRE(levels >= 1 && sz > 1, CC_ERR_INVALID_ARG, "QuantFirst volumes are 3D with numLevels >= 1");
    const uint32_t f_all = 1u << levels;
    CCA_REQUIRE(sx % f_all == 0 && sy % f_all == 0 && sz % f_all == 0, CC_ERR_INVALID_ARG,
                "sizes must be divisible by 2^numLevels");
    const uint64_t elems = (uint64_t)sx * sy * sz;
    const VolumeStreams vs(elems, levels, rle_only_lvl0);
    int16_t* dwt[2] = {I->d_vol[0].as<int16_t>(elems), I->d_vol[1].as<int16_t>(elems)};
    uint16_t* sym = I->d_vol[2].as<uint16_t>(vs.elems);
    // uniform quantization of the whole volume (CompressVolume.cpp:685-687)
    quantize_to_short(dwt[0], image, sx, sy, sz, step, sx, sx * sy, 1, st);
    // level l's coefficients are in dwt[1 - l % 2]; its bands become symbols before the next level but one
    // reuses it
    int16_t* buf = I->d_vol[3].as<int16_t>(elems);
    for (uint32_t level = 0; level < levels; level++) {
        const uint32_t f = 1u << level;
        const int d = (int)(level & 1);
        dwt53_forward(dwt[1 - d], buf, dwt[d], (int)(sx / f), (int)(sy / f), (int)(sz / f), (int)sx, (int)(sx * sy),
                      (int)sx, (int)(sx * sy), st);
        symbolize_level(sym + vs.at[vs.band(levels, level, 1)], align_up(vs.n[vs.band(levels, level, 1)], 64),
                        level + 1 == levels ? sym : nullptr, nullptr, dwt[1 - d], sx / f, sy / f, sz / f, sx,
                        (uint64_t)sx * sy, st);
    }
    std::vector<EncodeStream> streams;
    for (size_t k = 0; k < vs.n.size(); k++)
        streams.push_back(EncodeStream{sym + vs.at[k], vs.n[k], vs.rl[k], vs.call[k], 0});
    SectionTimer call(I, 1);
    call("Encode RLHuff");
    encode_items(I, 2, streams, levels + 1);
}

void decompress_volume_float_quant_first(cc_instance* I, float* image, uint32_t sx, uint32_t sy, uint32_t sz,
                                         uint32_t levels, const uint32_t* words, uint64_t nbits, float step,
                                         bool rle_only_lvl0) {
    const VolumeChannelIn ch{image, words, nbits, step};
    decompress_volume_float_quant_first_multichannel(I, &ch, 1, sx, sy, sz, levels, rle_only_lvl0);
}

namespace {

void check_channels(cc_instance* I, const VolumeChannelIn* ch, uint32_t nch, uint32_t sx, uint32_t sy, uint32_t sz,
                    uint32_t levels) {
    CCA_REQUIRE(nch >= 1 && ch, CC_ERR_INVALID_ARG, "no channels");
    check_volume(sx, sy, sz, levels);
    for (uint32_t c = 0; c < nch; c++)
        CCA_REQUIRE(ch[c].image && ch[c].words, CC_ERR_INVALID_ARG, "null channel buffer");
}

// Bitstream cursors of the channels.
struct ChannelStreams {
    std::vector<const uint32_t*> words;
    std::vector<uint64_t> nbits, pos;
    ChannelStreams(const VolumeChannelIn* ch, uint32_t nch) : nbits(nch), pos(nch, 0) {
        for (uint32_t c = 0; c < nch; c++) {
            words.push_back(ch[c].words);
            nbits[c] = ch[c].nbits;
        }
    }
    void decode(cc_instance* I, int symSize, const std::vector<DecodeStream>& streams) {
        decode_items(I, symSize, words.data(), nbits.data(), pos.data(), (uint32_t)words.size(), streams);
    }
};

// Most work buffers (bytes) that the channels of a float decode have between them, one channel's at least:
// 8.6 bytes a voxel for each that is transformed at a time.  A channel that needs a good part of this keeps
// the chip busy by itself, and three of 512^3 would hold 3.4 GB.
constexpr uint64_t kChannelWork = 1u << 27;

}  // namespace

void decompress_volume_float_multichannel(cc_instance* I, const VolumeChannelIn* ch, uint32_t nch, uint32_t sx,
                                          uint32_t sy, uint32_t sz, uint32_t levels, bool rle_only_lvl0,
                                          int symSize) {
    DeviceGuard guard(I->device);
    hipStream_t st = I->stream;
    check_channels(I, ch, nch, sx, sy, sz, levels);
    check_symbols(I, symSize);
    const uint64_t elems = (uint64_t)sx * sy * sz;
    SectionTimer call(I, 1);
    call("Decode RLHuff");
    ChannelStreams cs(ch, nch);
    std::vector<DecodeStream> streams;
    if (!bricks_serve(I, elems * nch, levels)) {
        const VolumeStreams vs(elems, levels, rle_only_lvl0);
        unsigned char* sym = (unsigned char*)I->d_vol[2].get(nch * vs.elems * symSize);
        for (uint32_t c = 0; c < nch; c++)
            for (size_t k = 0; k < vs.n.size(); k++)
                streams.push_back(DecodeStream{sym + (c * vs.elems + vs.at[k]) * symSize, vs.n[k], vs.rl[k], c});
        cs.decode(I, symSize, streams);
        for (uint32_t c = 0; c < nch; c++)
            decompress_volume_float_large(I, ch[c].image, sym + c * vs.elems * symSize, vs, sx, sy, sz, levels, ch[c].step,
                                          symSize);
        return;
    }
    // the channels are bricks of one batch, or of several that take turns with the work buffers
    const uint32_t at_once = (uint32_t)std::max<uint64_t>(1, kChannelWork / brick_work_bytes(elems, levels));
    std::vector<BrickJob> jobs;
    I->batch.d_bsym.get(nch * align_up(elems, 64) * symSize);
    for (uint32_t c = 0; c < nch; c += at_once) {
        BrickJob job;
        job.sym_base = c * align_up(elems, 64);
        for (uint32_t k = c; k < std::min(nch, c + at_once); k++)
            job.bricks.push_back(cc_brick{nullptr, ch[k].image, sx, sy, sz, ch[k].step});
        for (const ItemSpec& it : volume_bricks(I, job, levels, symSize, rle_only_lvl0))
            streams.push_back(DecodeStream{it.ptr, it.n, it.rl, c + it.call});
        jobs.push_back(std::move(job));
    }
    bricks_transforms_upload(I, I->batch, jobs[0], st);
    // the level tables' upload must finish before the pinned copy is rewritten
    try {
        cs.decode(I, symSize, streams);
    } catch (...) {
        (void)hipStreamSynchronize(st);
        throw;
    }
    for (size_t j = 0; j < jobs.size(); j++) {
        if (j) bricks_transforms_upload(I, I->batch, jobs[j], st);
        bricks_inverse_launch(jobs[j], st);
        CCA_HIP(hipStreamSynchronize(st));
    }
}

void decompress_volume_float_quant_first_multichannel(cc_instance* I, const VolumeChannelIn* ch, uint32_t nch,
                                                      uint32_t sx, uint32_t sy, uint32_t sz, uint32_t levels,
                                                      bool rle_only_lvl0) {
    DeviceGuard guard(I->device);
    hipStream_t st = I->stream;
    CCA_REQUIRE(I->log2 <= 16, CC_ERR_INVALID_ARG, "QuantFirst volumes use Symbol16 (log2 <= 16)");
    check_channels(I, ch, nch, sx, sy, sz, levels);
    const uint64_t elems = (uint64_t)sx * sy * sz;
    const VolumeStreams vs(elems, levels, rle_only_lvl0);
    int16_t* dwt[2] = {I->d_vol[0].as<int16_t>(elems), I->d_vol[1].as<int16_t>(elems)};
    uint16_t* sym = I->d_vol[2].as<uint16_t>(nch * vs.elems);
    int16_t* buf = I->d_vol[3].as<int16_t>(elems);
    SectionTimer call(I, 1);
    call("Decode RLHuff");
    ChannelStreams cs(ch, nch);
    std::vector<DecodeStream> streams;
    for (uint32_t c = 0; c < nch; c++)
        for (size_t k = 0; k < vs.n.size(); k++)
            streams.push_back(DecodeStream{sym + c * vs.elems + vs.at[k], vs.n[k], vs.rl[k], c});
    cs.decode(I, 2, streams);
    // a channel at a time: each level's coefficients from its symbols around the level above's output,
    // alternating buffers from dwt[0] (CompressVolume.cpp:794-838)
    for (uint32_t c = 0; c < nch; c++) {
        const uint16_t* s = sym + c * vs.elems;
        int d = 0;
        for (uint32_t level = levels; level-- > 0; d = 1 - d) {
            const uint32_t f = 1u << level;
            unsymbolize_level(dwt[d], s + vs.at[vs.band(levels, level, 1)], align_up(vs.n[vs.band(levels, level, 1)], 64),
                              level + 1 == levels ? s : nullptr, nullptr, sx / f, sy / f, sz / f, sx, (uint64_t)sx * sy, st);
            dwt53_inverse(dwt[1 - d], buf, dwt[d], (int)(sx / f), (int)(sy / f), (int)(sz / f), (int)sx,
                          (int)(sx * sy), (int)sx, (int)(sx * sy), st);
        }
        unquantize_from_short(ch[c].image, dwt[d], sx, sy, sz, ch[c].step, sx, sx * sy, 1, st);
    }
}

}  // namespace cca
