// host_rows.h -- a row of logits on its way to the caller: a launch stores it piece by piece into pinned memory, each piece with a word behind it, and the host copies a piece as soon as its word is
// there.  What it takes the place of: a wait for the whole stream (its signal and the wake-up are 4 us behind the last store) and then one copy of the row (32000 floats 3 us, 128256 12 us, 14 KB a
// microsecond), which now goes on under the launch's own stores.
#pragma once
#include <chrono>
#include <cstring>
#include <vector>
#include "../../../include/ntk.h"
#include "../../../include/ntk_layers.h"

namespace nt {

class HostRows {
public:
    HostRows() = default;
    HostRows(const HostRows&) = delete;
    HostRows& operator=(const HostRows&) = delete;
    ~HostRows() { clear(); }
    void alloc(size_t floats) {
        clear();
        row_ = static_cast<float*>(nt_hip_malloc_host(floats * sizeof(float)));
        there_ = static_cast<unsigned*>(nt_hip_malloc_host(ntk_copy_out_words(floats) * sizeof(unsigned)));
        if (!row_ || !there_) { clear(); return; }
        memset(there_, 0, ntk_copy_out_words(floats) * sizeof(unsigned));
        floats_ = floats;
    }
    void clear() {
        if (row_) nt_hip_free_host(row_);
        if (there_) nt_hip_free_host(there_);
        row_ = nullptr; there_ = nullptr; floats_ = 0;
    }
    explicit operator bool() const { return row_ != nullptr; }
    // dev[floats] behind everything queued on `stream` -> host; bump (optional): a device word that the same launch adds one to
    int fetch(float* host, const float* dev, int* bump, void* stream) {
        if (++turn_ == 0) ++turn_;
        const int st = ntk_copy_out_pieces(row_, dev, floats_, there_, turn_, bump, stream);
        if (st != NTK_OK) return st;
        const size_t pieces = ntk_copy_out_words(floats_), per = NTK_COPY_OUT_PIECE;
        bool waited = false;
        std::chrono::steady_clock::time_point t0{};
        for (size_t i = 0; i < pieces; ++i) {
            for (unsigned spins = 1; __atomic_load_n(there_ + i, __ATOMIC_ACQUIRE) != turn_; ++spins) {
                if (waited) return NTK_E_LAUNCH;           // the stream is idle and the word is not there
#if defined(__x86_64__) || defined(__i386__)
                __builtin_ia32_pause();
#endif
                if ((spins & 0xFFFFu) != 0) continue;
                const auto now = std::chrono::steady_clock::now();
                if (t0 == std::chrono::steady_clock::time_point{}) t0 = now;
                else if (now - t0 > std::chrono::seconds(2)) {      // a long pass, or one that failed: what the stream says
                    const int s = ntk_stream_synchronize(stream);
                    if (s != NTK_OK) return s;
                    waited = true;
                }
            }
            const size_t at = i * per;
            memcpy(host + at, row_ + at, (at + per < floats_ ? per : floats_ - at) * sizeof(float));
        }
        return NTK_OK;
    }

private:
    float* row_ = nullptr;
    unsigned* there_ = nullptr;
    size_t floats_ = 0;
    unsigned turn_ = 0;
};

}  // namespace nt
