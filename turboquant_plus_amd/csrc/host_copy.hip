// Large host arrays of the NumPy classes on their way between host memory and the device, by several threads of the caller's.
//
// A transfer is a job that lies in the caller's memory (tq_host_job).  Its array is cut into pieces, which the threads in
// tq_host_serve take; the thread in tq_host_drive moves the pinned slots between the device and the pieces' workers, takes pieces
// itself while it has nothing to move, and returns when every piece is done.  So a job needs no other thread to end, and no thread
// belongs to this file.
//
// The threads serve a board, on which every caller's job has a desk from the time that the stream is at it to its last piece; they go
// round the desks a piece at a time.  A thread that finds nothing for a while (the time between two arrays of a call: it takes longer
// to wake than a small piece to land) sleeps until the bell rings, which it does when a job comes and for every piece that becomes
// ready while somebody sleeps.  The driver waits in the runtime until the stream is at its job: 0.43 s of other work in front of a
// 32 MiB result, for which nine threads span 3.85 CPU-seconds, now take 0.43.
//
// What bounds it: fresh host pages, then the way through the slots.  A result of 32 to 64 MiB is fresh memory, which one thread fills
// at 12 to 18 GB/s, six at 46 to 65 and eight at 77 to 86 (the link gives 56); with the transfer int64 results of 32 MiB come at 36 to
// 45 GB/s of host bytes, float64 ones at 22 to 29, inputs go up at 30 to 34.  Pieces are a few MiB of the host array, so that no two
// threads clear the same huge page.
#include <errno.h>
#include <hip/hip_runtime.h>
#include <linux/futex.h>
#include <sched.h>
#include <string.h>
#include <sys/syscall.h>
#include <time.h>
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

constexpr int SPINS = 64;                  // of the driver, before it sleeps until its next piece has landed; of a serving thread, at a job
constexpr int64_t SERVE_CYCLES = 500000;   // of a serving thread, before it sleeps: 0.15 to 0.25 ms

void pause_for(int &idle) {
    if (++idle < SPINS) __builtin_ia32_pause();
    else sched_yield();
}

// wakes at most n of the sleeping threads; they count themselves before they look at the bell for the last time
void ring(tq_host_board *b, int n) {
    __atomic_fetch_add(&b->bell, 1, __ATOMIC_SEQ_CST);
    if (__atomic_load_n(&b->sleepers, __ATOMIC_SEQ_CST) > 0) syscall(SYS_futex, &b->bell, FUTEX_WAKE_PRIVATE, n, nullptr, nullptr, 0);
}

// A job's place on the board while it lives.  Without a board, or where every desk is taken, the driver does the whole job.
struct Desk {
    tq_host_board *board;
    tq_host_job *job;
    tq_host_desk *at = nullptr;
    void post() {   // others may look at the job from now on
        for (int i = 0; board && !at && i < TQ_HOST_DESKS; ++i) {
            int64_t free = 0;
            if (!__atomic_compare_exchange_n(&board->desk[i].taken, &free, 1, false, __ATOMIC_ACQ_REL, __ATOMIC_RELAXED)) continue;
            at = &board->desk[i];
            __atomic_store_n(&at->job, job, __ATOMIC_SEQ_CST);
        }
        if (at) ring(board, 0x7FFFFFFF);
    }
    void allow(int64_t upto) {   // pieces below `upto` may be worked on
        const int64_t was = job->ready, now = upto < job->n_pieces ? upto : job->n_pieces;
        __atomic_store_n(&job->ready, now, __ATOMIC_RELEASE);
        if (at && now > was) ring(board, (int)(now - was));
    }
    ~Desk() {
        if (!at) return;
        __atomic_store_n(&at->job, (tq_host_job *)nullptr, __ATOMIC_SEQ_CST);
        int idle = 0;
        while (__atomic_load_n(&at->users, __ATOMIC_SEQ_CST) > 0) pause_for(idle);
        __atomic_store_n(&at->taken, 0, __ATOMIC_RELEASE);
    }
};

// the stream's part of a job, and pieces in between
hipError_t move(tq_host_board *board, tq_host_job *j, char *device, hipStream_t s) {
    Desk desk{board, j};
    int idle = 0;
    const bool down = j->kind == TQ_HOST_WIDEN || j->kind == TQ_HOST_FETCH;
    hipEvent_t ev[SLOTS + 1];   // of the slots' pieces, and with a board one more
    hipError_t err = hipSuccess;
    const int events = (j->n_pieces < SLOTS ? (int)j->n_pieces : SLOTS) + (board ? 1 : 0);
    int made = 0;
    while (made < events && (err = hipEventCreateWithFlags(&ev[made], hipEventDisableTiming)) == hipSuccess) ++made;
    // sent: pieces handed to the stream; landed: of those, the ones the stream is done with
    int64_t sent = 0, landed = 0;
    auto send = [&] {
        const int64_t at = sent * j->piece, bytes = j->n - at < j->piece ? j->n - at : j->piece;
        char *slot = (char *)j->slots + (sent % SLOTS) * j->piece;
        err = down ? hipMemcpyAsync(slot, device + at, bytes, hipMemcpyDeviceToHost, s) : hipMemcpyAsync(device + at, slot, bytes, hipMemcpyHostToDevice, s);
        if (err == hipSuccess) err = hipEventRecord(ev[sent % SLOTS], s);
        ++sent;
    };
    auto poll = [&](bool wait) {   // one more piece landed?
        if (landed == sent) return false;
        hipError_t q = hipEventQuery(ev[landed % SLOTS]);
        if (q == hipErrorNotReady) {
            (void)hipGetLastError();   // or the next launch's check would report it
            if (!wait) return false;
            q = hipEventSynchronize(ev[landed % SLOTS]);
        }
        if (q != hipSuccess) err = q;
        ++landed;
        return true;
    };
    if (down) {
        // the first pieces follow what the stream has before them; the threads wake up while they travel (called ahead of that they
        // were slower, 2 x 4 x 4096 x 128 both ways 7.7 ms against 7.2)
        if (err == hipSuccess && board) err = hipEventRecord(ev[made - 1], s);
        while (err == hipSuccess && sent < SLOTS && sent < j->n_pieces) send();
        if (err == hipSuccess && board) err = hipEventSynchronize(ev[made - 1]);
    } else {
        desk.allow(SLOTS);   // every slot is free
    }
    if (err == hipSuccess) desk.post();
    while (err == hipSuccess && (down ? load(&j->done) < j->n_pieces : landed < j->n_pieces)) {
        bool moved = false;
        // down: into a slot whose earlier piece is worked off; up: a slot that is filled, by the piece after the one that landed
        if (sent < j->n_pieces && sent - SLOTS < landed && load(&j->slot_done[sent % SLOTS])) {
            if (down) __atomic_store_n(&j->slot_done[sent % SLOTS], 0, __ATOMIC_RELAXED);
            send();
            moved = true;
        }
        // with nothing else to do it sleeps until the next piece has landed: the stream has work of others before it, or is slower
        // than the threads.  (With a slot to fill or empty there are pieces in work, whose workers do not wake it.)
        const bool wait = !moved && idle >= SPINS && (down ? load(&j->done) == landed : load(&j->done) == sent);
        if (err == hipSuccess && poll(wait)) {
            if (down) {
                desk.allow(landed);
            } else {   // that piece's slot may be filled again
                __atomic_store_n(&j->slot_done[(landed - 1) % SLOTS], 0, __ATOMIC_RELAXED);
                desk.allow(landed + SLOTS);
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

// the board's users and the threads that serve it (or were sent to), in one word: a thread leaves only while there is no user
int64_t users_of(int64_t state) { return state >> 32; }
int32_t serving(int64_t state) { return (int32_t)(uint32_t)state; }

}  // namespace

extern "C" void tq_host_serve(tq_host_board *b) {
    unsigned first = 0;
    int64_t idle_since = 0;
    for (;;) {
        const int32_t heard = load(&b->bell);
        bool did = false;
        for (int k = 0; k < TQ_HOST_DESKS; ++k) {
            tq_host_desk *d = &b->desk[(first + k) % TQ_HOST_DESKS];
            if (!load(&d->job)) continue;
            __atomic_fetch_add(&d->users, 1, __ATOMIC_SEQ_CST);   // before the look that counts: the driver takes the job away and then waits for users
            if (tq_host_job *j = __atomic_load_n(&d->job, __ATOMIC_SEQ_CST)) {
                // some microseconds at a job whose next piece is not there yet: the threads' coming and going writes to the desk (without
                // this 7.6 ms instead of 7.2)
                bool took = take(j);
                for (int spin = 0; !took && spin < SPINS && load(&j->next) < j->n_pieces; ++spin) {
                    __builtin_ia32_pause();
                    took = take(j);
                }
                did |= took;
            }
            __atomic_fetch_sub(&d->users, 1, __ATOMIC_SEQ_CST);
        }
        ++first;
        const int64_t now = (int64_t)__builtin_ia32_rdtsc();
        if (did || !idle_since) {
            idle_since = now;
        } else if (now - idle_since < SERVE_CYCLES && users_of(load(&b->state)) > 0) {
            __builtin_ia32_pause();
        } else {
            // a board without users is left after a while: the next call may come soon, and a thread that leaves wants the interpreter
            // (2 x 4 x 4096 x 128 both ways 7.8 -> 7.3 ms, 1 x 8 x 2000 x 128 5.3 -> 5.05, against going at once)
            int64_t state = load(&b->state);
            const bool alone = users_of(state) <= 0;
            const timespec linger{0, 5000000};
            __atomic_fetch_add(&b->sleepers, 1, __ATOMIC_SEQ_CST);
            const long rang = syscall(SYS_futex, &b->bell, FUTEX_WAIT_PRIVATE, heard, alone ? &linger : nullptr, nullptr, 0);   // returns at once if it rang meanwhile
            const bool timed_out = rang < 0 && errno == ETIMEDOUT;
            __atomic_fetch_sub(&b->sleepers, 1, __ATOMIC_SEQ_CST);
            if (timed_out)
                while (users_of(state) <= 0)
                    if (__atomic_compare_exchange_n(&b->state, &state, state - 1, false, __ATOMIC_SEQ_CST, __ATOMIC_SEQ_CST)) return;
            idle_since = 0;
        }
    }
}

extern "C" int tq_host_open(tq_host_board *b, int threads) {
    int64_t state = load(&b->state), missing;
    do {
        missing = threads > serving(state) ? threads - serving(state) : 0;
    } while (!__atomic_compare_exchange_n(&b->state, &state, state + (1ll << 32) + missing, false, __ATOMIC_SEQ_CST, __ATOMIC_SEQ_CST));
    ring(b, 0x7FFFFFFF);
    return (int)missing;
}

extern "C" void tq_host_close(tq_host_board *b, int not_sent) {
    __atomic_fetch_sub(&b->state, (1ll << 32) + not_sent, __ATOMIC_SEQ_CST);
    ring(b, 0x7FFFFFFF);
}

extern "C" int tq_host_drive(tq_host_board *b, tq_host_job *j, void *device, void *stream) {
    const hipError_t err = move(b, j, (char *)device, (hipStream_t)stream);
    if (err == hipSuccess) return TQ_OK;
    tq_set_error("host copy: %s", hipGetErrorString(err));
    return TQ_ERR_HIP;
}
