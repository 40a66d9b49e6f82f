// Host-side entry points of the HIP kernels, and the device workspace they draw from.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cstdlib>
#include <stdexcept>
#include <string>
#include <vector>

#include "fz_common.h"

namespace fz {

// Bump allocator over device blocks; reset at the start of each call. reserve() sizes the arena
// for a call (one block when it grows while empty); take() adds a block when the current ones are
// full, so an estimate below the true need costs an allocation but never a failure, and a grown
// arena is not freed (hipFree synchronizes the whole device). Positions (used(), rewind(), peak())
// count through the blocks in order.
//
// A bound arena (bind()) draws from one region of device memory the caller owns and never
// allocates: a take() beyond the region throws instead of adding a block.
//
// side() gives memory that a call can do without, to one user a call: the end of the last block where the
// call leaves it free, else a region beside the blocks.
class DevArena {
   public:
    ~DevArena() { release(); }
    void bind(void* p, size_t bytes) {
        release();
        blocks_.push_back(Block{p, bytes & ~size_t(255)});
        cap_ = bytes & ~size_t(255);
        bound_ = true;
    }
    void reserve(size_t bytes) {
        bytes = (bytes + 255) & ~size_t(255);
        if (bytes <= cap_ || bound_) return;  // a bound arena cannot grow: its takes throw instead
        if (used_ == 0 && !blocks_.empty() && blocks_[0].cap < bytes) drop_blocks();  // regrow as one block
        if (blocks_.empty()) add_block(bytes);
        else add_block(bytes - cap_);
    }
    void reset() {
        cur_ = 0;
        off_ = 0;
        used_ = side_used_ = tail_ = 0;
    }
    template <typename T>
    T* take(size_t count) {
        const size_t bytes = ((count * sizeof(T)) + 255) & ~size_t(255);
        while (cur_ < blocks_.size() && off_ + bytes > open(cur_)) {  // the rest of this block is skipped
            used_ += blocks_[cur_].cap - off_;
            cur_++;
            off_ = 0;
        }
        if (cur_ == blocks_.size()) add_block(std::max(bytes, std::max<size_t>(size_t(256) << 20, cap_ / 2)));
        T* p = reinterpret_cast<T*>(static_cast<char*>(blocks_[cur_].p) + off_);
        off_ += bytes;
        used_ += bytes;
        peak_ = std::max(peak_, used_ + side_used_);
        return p;
    }
    // The most that side() may give, when `after` bytes of takes are still to come.
    size_t side_room(size_t after) const {
        size_t most = side_most_;
        if (bound_) most = blocks_.empty() || cur_ > 0 || off_ + after > blocks_[0].cap ? 0 : blocks_[0].cap - off_ - after;
        // FALCONS_SIDE_BYTES: a test switch
        if (const char* e = getenv("FALCONS_SIDE_BYTES")) most = std::min<size_t>(most, std::strtoull(e, nullptr, 10));
        return most;
    }
    void set_side_most(size_t bytes) { side_most_ = bytes; }
    // Null where there is no room (side_room) or the device has no such memory. A region is kept for the
    // next call and regrown for a larger one: to twice the need, 256 MB at least, and `most` at most, as the
    // hipFree that goes with it waits for the whole device.
    void* side(size_t bytes, size_t after, size_t most) {
        bytes = (bytes + 255) & ~size_t(255);
        const size_t room = side_room(after);
        if (bytes > room) return nullptr;
        if (bound_) return take<uint8_t>(bytes);
        const size_t last = blocks_.size() - 1;
        if (!tail_ && cur_ < blocks_.size() &&
            bytes + (cur_ == last ? off_ + after : 0) <= blocks_[last].cap) {
            tail_ = bytes;
            tail_block_ = last;
            side_used_ = bytes;
            peak_ = std::max(peak_, used_ + side_used_);
            return static_cast<char*>(blocks_[last].p) + (blocks_[last].cap - bytes);
        }
        if (bytes > side_.cap) {
            drop_side();
            const size_t cap = std::max(bytes, std::min(std::min(room, most), std::max(2 * bytes, size_t(256) << 20)));
            void* p = nullptr;
            if (hipMalloc(&p, cap) != hipSuccess) {
                (void)hipGetLastError();  // it is the caller's to go another way
                return nullptr;
            }
            side_ = Block{p, cap};
        }
        side_used_ = bytes;
        peak_ = std::max(peak_, used_ + side_used_);
        return side_.p;
    }
    size_t used() const { return used_; }
    // most taken at once since the last clear_peak()
    size_t peak() const { return peak_; }
    void clear_peak() { peak_ = used_ + side_used_; }
    // Gives back everything taken after `mark` (a value of used()); the caller has finished with it
    // in stream order.
    void rewind(size_t mark) {
        if (mark > used_) return;
        size_t base = 0;
        for (size_t k = 0; k < blocks_.size(); k++) {
            if (mark <= base + blocks_[k].cap) {
                cur_ = k;
                off_ = mark - base;
                used_ = mark;
                return;
            }
            base += blocks_[k].cap;
        }
    }
    size_t capacity() const { return cap_ + side_.cap; }
    size_t side_capacity() const { return side_.cap; }
    void release() {
        drop_blocks();
        drop_side();
    }

   private:
    struct Block {
        void* p = nullptr;
        size_t cap = 0;
    };
    // What takes may use of block k.
    size_t open(size_t k) const { return blocks_[k].cap - (tail_ && k == tail_block_ ? tail_ : 0); }
    void drop_blocks() {
        if (!bound_)
            for (Block& b : blocks_) (void)hipFree(b.p);
        blocks_.clear();
        cap_ = used_ = off_ = tail_ = 0;
        cur_ = 0;
        bound_ = false;
    }
    void drop_side() {
        if (side_.p) (void)hipFree(side_.p);
        side_ = Block{};
        side_used_ = 0;
    }
    void add_block(size_t bytes) {
        bytes = (bytes + 255) & ~size_t(255);
        if (bound_)
            throw std::length_error("the call needs more device workspace than the bound region holds (" +
                                    std::to_string(cap_) + " bytes)");
        void* p = nullptr;
        FZ_HIP(hipMalloc(&p, bytes));
        blocks_.push_back(Block{p, bytes});
        cap_ += bytes;
    }
    std::vector<Block> blocks_;
    Block side_;
    size_t cap_ = 0, used_ = 0, off_ = 0, peak_ = 0, cur_ = 0, side_used_ = 0, tail_ = 0, tail_block_ = 0;
    size_t side_most_ = ~size_t(0) / 2;
    bool bound_ = false;
};

// interpolation kernels (fz_interp.hip)
void interp_pass(int dtype, bool decomp, const PassDesc& p, void* data, int16_t* codes, void* escval,
                 const LevelEb* lv, int avx2, const uint64_t* esc_idx, uint64_t nesc, const void* unpred,
                 hipStream_t st);
// One level of a 3D or 2D direction-0 field: the z pass, then the y and x passes in one launch (or
// as separate passes when a row is too wide for the tiles' LDS). In place, like interp_pass.
void interp_level(int dtype, bool decomp, const LevelDesc& level, void* data, int16_t* codes, void* escval,
                  const LevelEb* lv, int avx2, const uint64_t* esc_idx, uint64_t nesc, const void* unpred,
                  hipStream_t st);
void interp_first(int dtype, bool decomp, void* data, int16_t* codes, void* escval, const double* eb_dev,
                  const uint64_t* esc_idx, uint64_t nesc, const void* unpred, hipStream_t st);
void interp_anchors(int dtype, bool decomp, void* data, void* unpred, const uint64_t cnt[3], const uint64_t str[3],
                    hipStream_t st);
void level_constants(const double* eb_dev, const double* ratio_dev, int mode, int levels, LevelEb* out,
                     hipStream_t st);
size_t minmax_scratch_bytes();
void abs_error_bound(int dtype, const void* data, uint64_t n, int simd, int mode, double abs_in, double rel,
                     double psnr_factor, void* scratch, double* eb_dev, hipStream_t st);
size_t select_escapes_scratch(uint64_t n);
void select_escapes(const int16_t* codes, uint64_t n, uint64_t* out_idx, uint64_t* nsel_dev, void* scratch,
                    hipStream_t st);
void gather_escapes(int dtype, const uint64_t* idx, const uint64_t* nsel_dev, uint64_t max_n, const void* escval,
                    void* out, hipStream_t st);

// entropy coder (fz_entropy.hip)
struct EntropyStats {
    int method = 0, use_delta = 0;
};
// Capacity that always holds the encoder output for n codes: order-1 tANS spends at most 13 bits on
// a symbol and 2 side-stream bytes on an escaped code; RLE+FSE at most 3 bytes per code; plus the
// per-segment and per-block headers and tables.
inline size_t entropy_encode_bound(uint64_t n) { return (size_t)n * 4 + (1u << 20); }
// A second stream for work that can run beside the main one (null: run on the main stream), with the
// two events that fork it from and join it back to the main stream.
struct AuxStream {
    hipStream_t stream = nullptr;
    hipEvent_t fork = nullptr, join = nullptr;
};
// Encodes n codes (device) into out (device, capacity out_cap; std::length_error, before any write
// past it, when the output would not fit). Returns the byte count of
// [u8 method|delta<<7][u16 lo][u16 mode][payload] (RleFseEncoder::save + ::encode). With a second
// stream, the order-1 escape side streams are coded on it, beside the chains.
size_t entropy_encode(const int16_t* codes, uint64_t n, uint8_t* out, size_t out_cap, DevArena& ws, hipStream_t st,
                      EntropyStats* stats, const AuxStream& aux = AuxStream{});
// Host-side check of an entropy stream's headers and framing (throws std::invalid_argument).
void entropy_check(const uint8_t* host, size_t len, uint64_t n);
// Decodes the encoder bytes (host copy `host`, device copy `dev`, length len) into n codes (device).
void entropy_decode(const uint8_t* host, const uint8_t* dev, size_t len, uint64_t n, int16_t* codes, DevArena& ws,
                    hipStream_t st, const AuxStream& aux);

// The same in three parts, for the batched decompress, which decodes the FSE blocks and the
// order-1 decoder's sequential chains of many calls in shared launches: start parses the stream
// and decodes the FSE-coded class bytes, or hands their blocks to an FseBatch; middle decodes the
// rest, handing the sequential chains to a DenseBatch when given; end finishes the codes. The caller
// orders the streams: fse_batch_run and dense_batch_run run after every call's previous part, and
// the next part after them. Without batches, start and middle decode everything themselves.
struct FseBatch;
FseBatch* fse_batch_create();
void fse_batch_destroy(FseBatch* b);
void fse_batch_run(FseBatch* b, DevArena& ws, hipStream_t st);
void fse_batch_clear(FseBatch* b);  // after fse_batch_run's launches have finished
struct DenseBatch;
DenseBatch* dense_batch_create();
void dense_batch_destroy(DenseBatch* b);
size_t dense_batch_size(DenseBatch* b);
// Before the calls hand over chains: the device memory that is free, of which split chains get a part.
void dense_batch_limit(DenseBatch* b, size_t free_bytes);
// Throws, with nothing launched, where the memory for the chains cannot be had.
void dense_batch_run(DenseBatch* b, DevArena& ws, hipStream_t st, const AuxStream& aux);
void dense_batch_clear(DenseBatch* b);  // after dense_batch_run's launches have finished
struct EntropyCall;
EntropyCall* entropy_call_new();
void entropy_call_free(EntropyCall* e);
void entropy_decode_start(EntropyCall* e, const uint8_t* host, const uint8_t* dev, size_t len, uint64_t n,
                          int16_t* codes, DevArena& ws, hipStream_t st, FseBatch* defer);
void entropy_decode_middle(EntropyCall* e, DevArena& ws, hipStream_t st, const AuxStream& aux, DenseBatch* defer);
void entropy_decode_end(EntropyCall* e, DevArena& ws, hipStream_t st);

}  // namespace fz
