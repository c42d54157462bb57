"""The staging memory of host copies (cltem_amd/csrc/staging.hpp) over a stand-in runtime whose
transfers run only when they are waited for: no GPU."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "cltem_amd", "csrc")

COMMON = r"""
#include "staging_fake.hpp"
using namespace mse_rt;
using Bytes = std::vector<unsigned char>;
Bytes pattern(size_t n, int seed) {
    Bytes b(n);
    for (size_t i = 0; i < n; ++i) b[i] = (unsigned char)((i * 2654435761u >> 7) + seed);
    return b;
}
"""

# copies of one byte, a chunk, a buffer and more, each way, equal byte for byte; the pool gives its
# memory back with the last engine
COPIES = r"""
int main() {
    StagePool<Fake> pool;
    FakeStream st;
    {
        StageLane<Fake> lane;
        lane.stream = &st;
        pool.engine_made();
        for (size_t n : {size_t(1), size_t(4099), kStageChunk - 1, kStageChunk, kStageChunk + 1, kStageBytes,
                         kStageBytes + 5, 3 * kStageBytes + 77}) {
            const Bytes a = pattern(n, 1);
            Bytes dev(n), back(n);
            staged_upload(pool, lane, dev.data(), a.data(), n);
            CHECK(dev == a);
            const Bytes b = pattern(n, 2);
            staged_download(pool, lane, back.data(), b.data(), n);
            CHECK(back == b);
        }
        CHECK(Fake::direct == 0 && Fake::pinned == 1);
        Fake::fail_pin = true;  // no pinned memory: the copy goes without
        StagePool<Fake> none;
        Bytes c = pattern(kStageBytes + 3, 3), d(c.size());
        staged_upload(none, lane, d.data(), c.data(), c.size());
        CHECK(d == c && Fake::direct == 1);
        Fake::fail_pin = false;
    }
    pool.engine_gone();
    CHECK(Fake::pinned == 0 && Fake::events == 0);
}
"""

# a copy that ends in an exception with a transfer still in flight: its buffer must not be in
# another copy's hands before that transfer has read (or written) it
IN_FLIGHT = r"""
enum { UPLOAD, DOWNLOAD, HELD_UP, HELD_DOWN };
int main() {
    for (int kind = 0; kind < 4; ++kind)
        for (int at = 0; at < 3; ++at) {
            StagePool<Fake> pool;
            FakeStream s1, s2;
            StageLane<Fake> l1, l2;
            l1.stream = &s1;
            l2.stream = &s2;
            const size_t n = 2 * kStageChunk + 9;
            const Bytes a = pattern(n, 1), b = pattern(n, 2);
            Bytes dev(n), dev2(n);
            bool threw = false;
            try {
                if (kind == UPLOAD || kind == DOWNLOAD) {
                    Fake::fail_record = at;
                    if (kind == UPLOAD)
                        staged_upload(pool, l1, dev.data(), a.data(), n);
                    else
                        staged_download(pool, l1, dev.data(), a.data(), n);
                } else {
                    StageHold<Fake> hold(pool, l1);
                    if (kind == HELD_UP) {
                        std::memcpy(hold.s->p, a.data(), n);
                        hold.to_device(dev.data(), 0, n);
                    } else {
                        hold.to_host(0, a.data(), n);
                    }
                    throw std::runtime_error("between the transfer and its wait");
                }
            } catch (const std::runtime_error&) {
                threw = true;
            }
            CHECK(threw);
            // another engine's copy through the same pool, then the first stream's transfers
            staged_upload(pool, l2, dev2.data(), b.data(), n);
            CHECK(dev2 == b);
            StageHold<Fake> other(pool, l2);
            const Bytes held(other.s->p, other.s->p + n);
            Fake::sync(&s1);
            CHECK(Bytes(other.s->p, other.s->p + n) == held);  // no late transfer into it
            const size_t moved = kind == HELD_UP ? n : kind == UPLOAD ? std::min(n, (at + 1) * kStageChunk) : 0;
            CHECK(Bytes(dev.begin(), dev.begin() + moved) == Bytes(a.begin(), a.begin() + moved));
        }
}
"""

# engines on more devices than the pool has buffers, in turn: every one's copies are staged, with
# events of its own device
DEVICES = r"""
int main() {
    StagePool<Fake> pool;
    constexpr int devices = 2 * kStages + 1;
    for (int round = 0; round < 3; ++round)
        for (int d = 0; d < devices; ++d) {
            Fake::device = d;
            static FakeStream st[devices];
            static StageLane<Fake> lane[devices];
            st[d].device = d;
            lane[d].stream = &st[d];
            const Bytes a = pattern(2 * kStageChunk + 3, d + round);
            Bytes dev(a.size()), back(a.size());
            staged_upload(pool, lane[d], dev.data(), a.data(), a.size());
            staged_download(pool, lane[d], back.data(), dev.data(), a.size());
            CHECK(back == a);
            CHECK(Fake::direct == 0);
        }
    CHECK(Fake::pinned <= kStages);
}
"""


def run(tmp_path, body):
    src = tmp_path / "t.cpp"
    src.write_text(COMMON + body)
    exe = str(tmp_path / "t")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-I" + HERE, "-I" + CSRC, "-o", exe, str(src), "-lpthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("body", [COPIES, IN_FLIGHT, DEVICES], ids=["copies", "in_flight", "devices"])
def test_staging(tmp_path, body):
    run(tmp_path, body)
