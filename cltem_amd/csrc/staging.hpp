// Pinned staging memory for copies from and to pageable host memory.  Host code only, written over
// the runtime's calls (RT: HIP's in engine_internal.hpp), so that it also runs without a GPU.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstring>
#include <mutex>

namespace mse_rt {

constexpr int kStages = 4;
constexpr size_t kStageBytes = size_t(4) << 20, kStageChunk = size_t(1) << 20;
constexpr int kStageChunks = (int)(kStageBytes / kStageChunk);

// The stream whose copies are staged: an engine's.  Its events belong to its device, the buffers to
// none, so that every device's engines share them.
template <class RT>
struct StageLane {
    typename RT::Stream stream{};
    typename RT::Event done[kStageChunks] = {};  // the last transfer of each chunk of the buffer in hand
    StageLane() = default;
    StageLane(const StageLane&) = delete;
    StageLane& operator=(const StageLane&) = delete;
    ~StageLane() {
        for (auto ev : done)
            if (ev) RT::drop_event(ev);
    }
    // the events, made on first use (on the current device)
    bool ready() {
        for (auto& ev : done)
            if (!ev && !RT::make_event(&ev)) return false;
        return true;
    }
};

// At most kStages buffers of kStageBytes, made on first use, shared by all engines and threads of
// the process, whatever their devices, and given back when the last engine is destroyed.
template <class RT>
struct StagePool {
    struct Stage {
        unsigned char* p = nullptr;
        bool taken = false;
    };

    // a free buffer; NULL while there is none
    Stage* take() {
        std::lock_guard<std::mutex> lk(mu);
        Stage* empty = nullptr;
        for (Stage& s : stages) {
            if (s.taken) continue;
            if (s.p) {
                s.taken = true;
                return &s;
            }
            empty = &s;
        }
        if (!empty || !RT::pin(&empty->p, kStageBytes)) return nullptr;  // the copy goes without
        empty->taken = true;
        return empty;
    }
    void give_back(Stage* s) {
        std::lock_guard<std::mutex> lk(mu);
        s->taken = false;
    }
    void engine_made() {
        std::lock_guard<std::mutex> lk(mu);
        ++engines;
    }
    void engine_gone() {
        std::lock_guard<std::mutex> lk(mu);
        if (--engines == 0)
            for (Stage& s : stages)
                if (!s.taken) release(s);
    }

private:
    static void release(Stage& s) {
        if (s.p) RT::unpin(s.p);
        s = Stage();
    }
    std::mutex mu;
    Stage stages[kStages];
    int engines = 0;
};

// One copy's hold on a buffer (none while all are taken: more threads copying than buffers).  Its
// transfers go through to_device and to_host; on every way out, an exception's too, the buffer goes
// back to the pool only when they have finished.  One whose stream can no longer be waited for
// stays out of the pool.
template <class RT>
struct StageHold {
    StagePool<RT>& pool;
    StageLane<RT>& lane;
    typename StagePool<RT>::Stage* s;
    bool in_flight = false;  // a transfer may be using the buffer

    StageHold(StagePool<RT>& pool, StageLane<RT>& lane, bool wanted = true)
        : pool(pool), lane(lane), s(wanted && lane.ready() ? pool.take() : nullptr) {}
    ~StageHold() {
        if (s && (!in_flight || RT::try_sync(lane.stream))) pool.give_back(s);
    }
    StageHold(const StageHold&) = delete;
    StageHold& operator=(const StageHold&) = delete;

    void to_device(void* dst, size_t at, size_t bytes) {
        in_flight = true;
        RT::to_device(dst, s->p + at, bytes, lane.stream);
    }
    void to_host(size_t at, const void* src, size_t bytes) {
        in_flight = true;
        RT::to_host(s->p + at, src, bytes, lane.stream);
    }
    void record(int part) { RT::record(lane.done[part], lane.stream); }
    void wait(int part) { RT::wait(lane.done[part]); }
    void sync() {
        RT::sync(lane.stream);
        in_flight = false;
    }
};

// Copies by the lane's stream, complete on return.
template <class RT>
void staged_download(StagePool<RT>& pool, StageLane<RT>& lane, void* dst, const void* src, size_t bytes) {
    StageHold<RT> hold(pool, lane);
    if (!hold.s) {
        RT::to_host(dst, src, bytes, lane.stream);
        RT::sync(lane.stream);
        return;
    }
    if (bytes <= kStageChunk) {
        hold.to_host(0, src, bytes);
        hold.sync();
        std::memcpy(dst, hold.s->p, bytes);
        return;
    }
    // chunk i lands in part i % kStageChunks while the chunks before it are copied out
    const size_t n = (bytes + kStageChunk - 1) / kStageChunk;
    for (size_t i = 0; i < n + kStageChunks - 1; ++i) {
        if (i >= (size_t)kStageChunks - 1) {
            const size_t j = i - (kStageChunks - 1), at = j * kStageChunk;
            const int part = (int)(j % kStageChunks);
            hold.wait(part);
            if (j == n - 1) hold.in_flight = false;
            std::memcpy((unsigned char*)dst + at, hold.s->p + part * kStageChunk, std::min(kStageChunk, bytes - at));
        }
        if (i < n) {
            const size_t at = i * kStageChunk;
            const int part = (int)(i % kStageChunks);
            hold.to_host(part * kStageChunk, (const unsigned char*)src + at, std::min(kStageChunk, bytes - at));
            hold.record(part);
        }
    }
}

template <class RT>
void staged_upload(StagePool<RT>& pool, StageLane<RT>& lane, void* dst, const void* src, size_t bytes) {
    StageHold<RT> hold(pool, lane);
    if (!hold.s) {
        RT::to_device(dst, src, bytes, lane.stream);
        RT::sync(lane.stream);
        return;
    }
    for (size_t at = 0, i = 0; at < bytes; at += kStageChunk, ++i) {
        const int part = (int)(i % kStageChunks);
        const size_t len = std::min(kStageChunk, bytes - at);
        if (i >= (size_t)kStageChunks) hold.wait(part);
        std::memcpy(hold.s->p + part * kStageChunk, (const unsigned char*)src + at, len);
        hold.to_device((unsigned char*)dst + at, part * kStageChunk, len);
        hold.record(part);
    }
    hold.sync();
}

}  // namespace mse_rt
