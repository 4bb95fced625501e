// The slots of a staged host transfer: one worker's chunks between pageable memory and the device. Free of HIP, so that the
// order of copies and waits, and what a failure leaves, can be checked without a GPU.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstring>

namespace lira {

// Moves the chunks first, first + step, ... (slot_bytes each, the last one shorter) of `bytes` bytes at host through the
// worker's SLOTS slots: it copies one slot while the link moves another. link.slot(j) is slot j's memory; link.copy(j,
// off, len) queues the slot's copy to or from the device at byte off, link.record(j) marks it, link.wait(j) waits for the
// mark and link.drain() for everything queued; they return Err, 0 for success. Every copy that was queued has completed on
// return, also after a failure.
template <int SLOTS, typename Err, typename Link>
Err stage_chunks(Link &link, char *host, size_t bytes, size_t slot_bytes, bool to_device, size_t first, size_t step) {
    const size_t chunks = (bytes + slot_bytes - 1) / slot_bytes;
    Err err = Err(0);
    size_t queued[SLOTS];  // the chunk in flight in each slot, or chunks
    for (size_t &q : queued) q = chunks;
    auto len = [&](size_t c) { return std::min(slot_bytes, bytes - c * slot_bytes); };
    auto finish = [&](int j) {  // wait for the slot's copy; on the way to the host its data moves on
        if (queued[j] == chunks) return;
        const Err e = link.wait(j);
        if (err == Err(0)) err = e;
        if (!to_device && err == Err(0)) std::memcpy(host + queued[j] * slot_bytes, link.slot(j), len(queued[j]));
        queued[j] = chunks;
    };
    int j = 0;
    for (size_t c = first; c < chunks && err == Err(0); c += step, j = (j + 1) % SLOTS) {
        finish(j);
        if (err != Err(0)) break;
        if (to_device) std::memcpy(link.slot(j), host + c * slot_bytes, len(c));
        err = link.copy(j, c * slot_bytes, len(c));
        if (err == Err(0)) err = link.record(j);
        if (err == Err(0)) queued[j] = c;
    }
    for (int k = 0; k < SLOTS; k++, j = (j + 1) % SLOTS) finish(j);
    // a copy that was queued but not marked, or whose wait failed, may still use its slot
    if (err != Err(0)) (void)link.drain();
    return err;
}

}  // namespace lira
