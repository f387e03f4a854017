// Pinned host memory: a context's block, and the box of each of its models.
#pragma once

#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <mutex>

#include "l2h_internal.h"

// Pinned host memory of a context for its models' boxes (HostBox), a few kilobytes each: made once, for pinning takes half a millisecond.  What does not
// fit is pinned by itself.
struct PinnedArena {
    static constexpr size_t UNIT = 4096, UNITS = 64;
    void *(*pin)(size_t) = nullptr;  // (nullptr: not to be had)
    void (*unpin)(void *) = nullptr;
    std::mutex lock;
    char *mem = nullptr;  // UNIT x UNITS, or none
    bool used[UNITS] = {};
    void open(void *(*pin_)(size_t), void (*unpin_)(void *)) {
        pin = pin_, unpin = unpin_;
        mem = (char *)pin(UNIT * UNITS);
    }
    void close() {
        if (mem) unpin(mem);
        mem = nullptr;
    }
    void *take(size_t bytes) {
        const size_t n = (bytes + UNIT - 1) / UNIT;
        std::lock_guard<std::mutex> hold(lock);
        for (size_t i = 0; mem && i + n <= UNITS; i++) {
            size_t k = 0;
            while (k < n && !used[i + k]) k++;
            if (k < n) continue;
            std::fill(used + i, used + i + n, true);
            return mem + i * UNIT;
        }
        return nullptr;
    }
    bool give(void *p, size_t bytes) {  // false: not from here
        std::lock_guard<std::mutex> hold(lock);
        const char *c = (const char *)p;
        if (!mem || c < mem || c >= mem + UNIT * UNITS) return false;
        const size_t i = (size_t)(c - mem) / UNIT, n = (bytes + UNIT - 1) / UNIT;
        std::fill(used + i, used + i + n, false);
        return true;
    }
};

// What a call hands to the device and gets back, in host memory that stays: pinned, so that kernels fetch and leave it themselves and the call waits once, at
// its end (from a call's own stack every copy was a wait).  One call of a model at a time uses it.
struct HostBox {
    DecodeCtl *ctl = nullptr;   // [2], and the prompt behind them, as on the device
    int32_t *prompt = nullptr;  // [n]
    int32_t *out = nullptr;     // [n] tokens
    int32_t *pick = nullptr;    // l2h_sample's
    unsigned *gave_up = nullptr;
    void *mem = nullptr;
    size_t bytes = 0;
    bool pinned = false;  // by itself (or from the context's arena, which knows)
    bool seen = false;    // kernels read and write it: it is pinned either way
    // for sequences of n tokens; a box that is there stays (a model is asked to finalize again after it failed).  false: no memory
    bool make(PinnedArena &arena, int64_t n) {
        if (mem) return true;
        static_assert(sizeof(DecodeCtl) % 16 == 0, "the prompt follows the control blocks");
        bytes = 2 * sizeof(DecodeCtl) + 2 * (size_t)n * 4 + 64;
        mem = arena.take(bytes);
        if (!mem) {
            mem = arena.pin(bytes);
            pinned = mem != nullptr;
        }
        seen = mem != nullptr;
        if (!mem) mem = malloc(bytes);  // (then copies wait, as they do from any memory of a program)
        if (!mem) return false;
        memset(mem, 0, bytes);
        ctl = (DecodeCtl *)mem;
        prompt = (int32_t *)(ctl + 2);
        out = prompt + n;
        pick = out + n;
        gave_up = (unsigned *)pick + 1;
        return true;
    }
    void release(PinnedArena &arena) {
        if (mem && !arena.give(mem, bytes)) {
            if (pinned)
                arena.unpin(mem);
            else
                free(mem);
        }
        *this = HostBox();
    }
};
