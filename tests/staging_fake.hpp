// A stand-in for the runtime under cltem_amd/csrc/staging.hpp: streams are queues of copies that
// run only when somebody waits for them, so a buffer reused too early shows in the bytes.  Calls
// can be made to fail.
#pragma once
#include <cstdio>
#include <cstdlib>
#include <deque>
#include <functional>
#include <stdexcept>
#include <vector>

#include "staging.hpp"

struct FakeStream {
    int device = 0;
    std::deque<std::function<void()>> queue;
    size_t done = 0, issued = 0;
    void run_to(size_t n) {
        while (done < n) {
            queue.front()();
            queue.pop_front();
            ++done;
        }
    }
};
struct FakeEvent {
    int device = 0;
    FakeStream* stream = nullptr;
    size_t at = 0;
};

struct Fake {
    using Stream = FakeStream*;
    using Event = FakeEvent*;
    static inline int device = 0;          // the current device
    static inline int fail_record = -1;    // the record call that fails, counted down
    static inline bool fail_pin = false;
    static inline int pinned = 0, direct = 0, events = 0;
    static inline std::vector<std::pair<unsigned char*, size_t>> pins;
    static bool is_pinned(const void* p) {
        for (auto& r : pins)
            if ((unsigned char*)p >= r.first && (unsigned char*)p < r.first + r.second) return true;
        return false;
    }
    static bool pin(unsigned char** p, size_t n) {
        if (fail_pin) return false;
        *p = (unsigned char*)std::malloc(n);
        pins.push_back({*p, n});
        ++pinned;
        return true;
    }
    static void unpin(unsigned char* p) {
        for (size_t i = 0; i < pins.size(); ++i)
            if (pins[i].first == p) {
                pins.erase(pins.begin() + i);
                break;
            }
        std::free(p);
        --pinned;
    }
    static bool make_event(FakeEvent** ev) {
        *ev = new FakeEvent{device};
        ++events;
        return true;
    }
    static void drop_event(FakeEvent* ev) {
        delete ev;
        --events;
    }
    static void copy(void* dst, const void* src, size_t n, FakeStream* st) {
        st->queue.push_back([=] { std::memcpy(dst, src, n); });
        ++st->issued;
    }
    static void to_host(void* dst, const void* src, size_t n, FakeStream* st) {
        if (!is_pinned(dst)) ++direct;
        copy(dst, src, n, st);
    }
    static void to_device(void* dst, const void* src, size_t n, FakeStream* st) {
        if (!is_pinned(src)) ++direct;
        copy(dst, src, n, st);
    }
    static void record(FakeEvent* ev, FakeStream* st) {
        if (fail_record == 0) {
            fail_record = -1;
            throw std::runtime_error("record");
        }
        if (fail_record > 0) --fail_record;
        if (ev->device != st->device) throw std::runtime_error("event of another device");
        ev->stream = st;
        ev->at = st->issued;
    }
    static void wait(FakeEvent* ev) {
        if (ev->stream) ev->stream->run_to(ev->at);
    }
    static void sync(FakeStream* st) { st->run_to(st->issued); }
    static bool try_sync(FakeStream* st) {
        sync(st);
        return true;
    }
};

#define CHECK(c)                                                    \
    do {                                                            \
        if (!(c)) {                                                 \
            std::printf("line %d: %s\n", __LINE__, #c);             \
            std::exit(1);                                           \
        }                                                           \
    } while (0)
