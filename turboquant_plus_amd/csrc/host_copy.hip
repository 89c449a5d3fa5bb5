// Large host arrays of the NumPy classes on their way between host memory and the device, by several threads of the caller's.
//
// A transfer is a job that lies in the caller's memory (tq_host_job).  Its array is cut into pieces, which the threads in
// tq_host_serve take until none are left; the thread in tq_host_drive moves the pinned slots between the device and the pieces'
// workers, takes pieces itself while it has nothing to move, and returns when every piece is done.  So a job needs no other thread
// to end, and no thread belongs to this file.
//
// What bounds it: the host's pages.  An int64 or float64 result of 32 MiB is fresh memory, which one thread fills at 14 - 23 GB/s
// and six at 57 where the link gives 56; pieces are a few MiB of the host array, so that no two threads clear the same huge page.
#include <hip/hip_runtime.h>
#include <linux/futex.h>
#include <sched.h>
#include <string.h>
#include <sys/syscall.h>
#include <unistd.h>

#include "tq_internal.h"

namespace {

constexpr int SLOTS = TQ_HOST_SLOTS;

template <typename T> T load(const T *p) { return __atomic_load_n(p, __ATOMIC_ACQUIRE); }

__attribute__((target("avx2"))) void widen_avx2(int64_t *dst, const uint8_t *src, int64_t n) {
#pragma clang loop vectorize_width(16)
    for (int64_t i = 0; i < n; ++i) dst[i] = src[i];
}
void widen_any(int64_t *dst, const uint8_t *src, int64_t n) {
    for (int64_t i = 0; i < n; ++i) dst[i] = src[i];
}
__attribute__((target("avx2"))) int64_t narrow_avx2(uint8_t *dst, const int64_t *src, int64_t n) {
    int64_t seen = 0;
#pragma clang loop vectorize_width(16)
    for (int64_t i = 0; i < n; ++i) {
        seen |= src[i];
        dst[i] = (uint8_t)src[i];
    }
    return seen;
}
int64_t narrow_any(uint8_t *dst, const int64_t *src, int64_t n) {
    int64_t seen = 0;
    for (int64_t i = 0; i < n; ++i) {
        seen |= src[i];
        dst[i] = (uint8_t)src[i];
    }
    return seen;
}
bool has_avx2() {
    static const bool yes = __builtin_cpu_supports("avx2");
    return yes;
}

// bytes of an element on the host and on the device
int host_bytes(const tq_host_job *j) { return j->kind == TQ_HOST_WIDEN || j->kind == TQ_HOST_NARROW ? 8 : 1; }

void do_piece(tq_host_job *j, int64_t p) {
    const int64_t at = p * j->piece, n = j->n - at < j->piece ? j->n - at : j->piece;
    char *host = (char *)j->host + at * host_bytes(j);
    char *slot = (char *)j->slots + (p % SLOTS) * j->piece;
    if (j->kind == TQ_HOST_WIDEN) {
        if (has_avx2()) widen_avx2((int64_t *)host, (const uint8_t *)slot, n);
        else widen_any((int64_t *)host, (const uint8_t *)slot, n);
    } else if (j->kind == TQ_HOST_NARROW) {
        const int64_t seen = has_avx2() ? narrow_avx2((uint8_t *)slot, (const int64_t *)host, n) : narrow_any((uint8_t *)slot, (const int64_t *)host, n);
        __atomic_fetch_or(&j->seen, seen, __ATOMIC_RELAXED);
    } else if (j->kind == TQ_HOST_FETCH) {
        memcpy(host, slot, n);
    } else {
        memcpy(slot, host, n);
    }
    __atomic_store_n(&j->slot_done[p % SLOTS], 1, __ATOMIC_RELEASE);
    __atomic_fetch_add(&j->done, 1, __ATOMIC_RELEASE);
}

// one piece, if there is one that may be worked on now
bool take(tq_host_job *j) {
    int64_t p = load(&j->next);
    while (p < load(&j->ready)) {
        if (__atomic_compare_exchange_n(&j->next, &p, p + 1, false, __ATOMIC_ACQ_REL, __ATOMIC_ACQUIRE)) {
            do_piece(j, p);
            return true;
        }
    }
    return false;
}

void pause_for(int &idle) {
    if (++idle < 64) __builtin_ia32_pause();
    else sched_yield();
}

}  // namespace

namespace {

void work(tq_host_job *j) {
    int idle = 0;
    while (load(&j->next) < j->n_pieces) {   // the last piece taken: nothing is left for this thread
        if (take(j)) idle = 0;
        else pause_for(idle);
    }
}

void ring(tq_host_session *s) {
    __atomic_fetch_add(&s->bell, 1, __ATOMIC_RELEASE);
    syscall(SYS_futex, &s->bell, FUTEX_WAKE_PRIVATE, 0x7FFFFFFF, nullptr, nullptr, 0);
}

// the stream's part of a job, and pieces in between
hipError_t move(tq_host_job *j, char *device, hipStream_t s) {
    int idle = 0;
    const bool down = j->kind == TQ_HOST_WIDEN || j->kind == TQ_HOST_FETCH;
    hipEvent_t ev[SLOTS];
    hipError_t err = hipSuccess;
    int made = 0;
    while (made < SLOTS && made < j->n_pieces && (err = hipEventCreateWithFlags(&ev[made], hipEventDisableTiming)) == hipSuccess) ++made;
    // sent: pieces handed to the stream; landed: of those, the ones the stream is done with
    int64_t sent = 0, landed = 0;
    auto send = [&] {
        const int64_t at = sent * j->piece, bytes = j->n - at < j->piece ? j->n - at : j->piece;
        char *slot = (char *)j->slots + (sent % SLOTS) * j->piece;
        err = down ? hipMemcpyAsync(slot, device + at, bytes, hipMemcpyDeviceToHost, s) : hipMemcpyAsync(device + at, slot, bytes, hipMemcpyHostToDevice, s);
        if (err == hipSuccess) err = hipEventRecord(ev[sent % SLOTS], s);
        ++sent;
    };
    auto poll = [&] {   // one more piece landed?
        if (landed == sent) return false;
        const hipError_t q = hipEventQuery(ev[landed % SLOTS]);
        if (q == hipErrorNotReady) {
            (void)hipGetLastError();   // or the next launch's check would report it
            return false;
        }
        if (q != hipSuccess) err = q;
        ++landed;
        return true;
    };
    auto allow = [&](int64_t upto) { __atomic_store_n(&j->ready, upto < j->n_pieces ? upto : j->n_pieces, __ATOMIC_RELEASE); };
    if (!down) allow(SLOTS);   // every slot is free
    while (err == hipSuccess && (down ? load(&j->done) < j->n_pieces : landed < j->n_pieces)) {
        bool moved = false;
        // down: into a slot whose earlier piece is worked off; up: a slot that is filled, by the piece after the one that landed
        if (sent < j->n_pieces && sent - SLOTS < landed && ((down && sent < SLOTS) || load(&j->slot_done[sent % SLOTS]))) {
            if (down) __atomic_store_n(&j->slot_done[sent % SLOTS], 0, __ATOMIC_RELAXED);
            send();
            moved = true;
        }
        if (err == hipSuccess && poll()) {
            if (down) {
                allow(landed);
            } else {   // that piece's slot may be filled again
                __atomic_store_n(&j->slot_done[(landed - 1) % SLOTS], 0, __ATOMIC_RELAXED);
                allow(landed + SLOTS);
            }
            moved = true;
        }
        if (moved || take(j)) idle = 0;
        else pause_for(idle);
    }
    if (err != hipSuccess) {
        // nobody takes another piece; those being worked on end, and so does the stream's use of the slots
        const int64_t taken = __atomic_exchange_n(&j->next, j->n_pieces, __ATOMIC_ACQ_REL);
        while (load(&j->done) < taken) pause_for(idle);
        (void)hipStreamSynchronize(s);
    }
    for (int i = 0; i < made; ++i) (void)hipEventDestroy(ev[i]);
    return err;
}

}  // namespace

extern "C" void tq_host_serve(tq_host_session *s) {
    for (;;) {
        const int32_t heard = load(&s->bell);
        if (load(&s->closed)) return;
        __atomic_fetch_add(&s->users, 1, __ATOMIC_SEQ_CST);   // before the look: tq_host_drive waits for users after it has taken the job away
        if (tq_host_job *j = __atomic_load_n(&s->job, __ATOMIC_SEQ_CST)) work(j);
        __atomic_fetch_sub(&s->users, 1, __ATOMIC_SEQ_CST);
        syscall(SYS_futex, &s->bell, FUTEX_WAIT_PRIVATE, heard, nullptr, nullptr, 0);   // returns at once if it rang meanwhile
    }
}

extern "C" void tq_host_close(tq_host_session *s) {
    __atomic_store_n(&s->closed, 1, __ATOMIC_RELEASE);
    ring(s);
}

extern "C" int tq_host_drive(tq_host_session *s, tq_host_job *j, void *device, void *stream) {
    if (s) {
        __atomic_store_n(&s->job, j, __ATOMIC_SEQ_CST);
        ring(s);
    }
    const hipError_t err = move(j, (char *)device, (hipStream_t)stream);
    if (s) {
        __atomic_store_n(&s->job, (tq_host_job *)nullptr, __ATOMIC_SEQ_CST);
        int idle = 0;
        while (__atomic_load_n(&s->users, __ATOMIC_SEQ_CST) > 0) pause_for(idle);
    }
    if (err == hipSuccess) return TQ_OK;
    tq_set_error("host copy: %s", hipGetErrorString(err));
    return TQ_ERR_HIP;
}
