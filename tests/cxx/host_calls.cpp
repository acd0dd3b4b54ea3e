// The host side of signing calls without a GPU: this program defines the HIP
// runtime functions that the library calls (its own definitions take
// precedence over libamdhip64's), so that it sees every launch, event and
// allocation and can make any of them fail.  Device pointers are addresses
// that nothing reads.
//   host_calls join      errors while a signing call is being enqueued
//   host_calls slots     the attempt slots that a signing context allocates
//   host_calls timing    the two durations of a timed call
// Prints what is wrong and exits with 1, or exits with 0.
// Run by tests/test_host_sign_calls.py.
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "cudilithium_amd.h"

namespace {

typedef void *Handle;
constexpr int FAIL = 999;  // hipErrorUnknown

enum Kind { LAUNCH, RECORD, WAIT, SYNC };
struct Op {
    Kind kind;
    Handle stream, event;
    bool ok;
};
std::vector<Op> ops;
long fail_at = -1;  // index of the operation that fails
int last_error = 0;
Handle caller = nullptr;

std::vector<size_t> allocations;  // sizes asked for
size_t largest = SIZE_MAX;        // larger device allocations fail

uintptr_t next_handle = 0x1000, next_address = uintptr_t(1) << 40;
Handle make_handle() { return reinterpret_cast<Handle>(next_handle += 0x10); }

int op(Kind kind, Handle stream, Handle event) {
    const bool ok = (long)ops.size() != fail_at;
    ops.push_back({kind, stream, event, ok});
    if (!ok) last_error = FAIL;
    return ok ? 0 : FAIL;
}

struct Dim3 {
    uint32_t x, y, z;
};
struct Config {
    Dim3 grid, block;
    size_t shared;
    Handle stream;
} config;

int wrong(const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vprintf(fmt, ap);
    va_end(ap);
    printf("\n");
    return 1;
}

}  // namespace

extern "C" {

int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, Handle stream) {
    config = {grid, block, shared, stream};
    return 0;
}
int __hipPopCallConfiguration(Dim3 *grid, Dim3 *block, size_t *shared, Handle *stream) {
    *grid = config.grid;
    *block = config.block;
    *shared = config.shared;
    *stream = config.stream;
    return 0;
}
int hipLaunchKernel(const void *, Dim3, Dim3, void **, size_t, Handle stream) { return op(LAUNCH, stream, nullptr); }
int hipGetLastError() {
    const int e = last_error;
    last_error = 0;
    return e;
}
int hipEventRecord(Handle event, Handle stream) { return op(RECORD, stream, event); }
int hipStreamWaitEvent(Handle stream, Handle event, unsigned) { return op(WAIT, stream, event); }
int hipStreamSynchronize(Handle stream) { return op(SYNC, stream, nullptr); }

int hipMalloc(void **p, size_t bytes) {
    allocations.push_back(bytes);
    if (bytes > largest) return last_error = 2;  // hipErrorOutOfMemory
    *p = reinterpret_cast<void *>(next_address);
    next_address += (bytes + 4095) / 4096 * 4096;
    return 0;
}
int hipFree(void *) { return 0; }
int hipHostMalloc(void **p, size_t bytes, unsigned) {
    *p = malloc(bytes);
    return *p ? 0 : 2;
}
int hipHostFree(void *p) {
    free(p);
    return 0;
}
int hipGetDevice(int *dev) {
    *dev = 0;
    return 0;
}
int hipDeviceGetAttribute(int *v, int, int) {
    *v = 256;
    return 0;
}
int hipStreamCreateWithFlags(Handle *s, unsigned) {
    *s = make_handle();
    return 0;
}
int hipEventCreateWithFlags(Handle *e, unsigned) {
    *e = make_handle();
    return 0;
}
int hipEventCreate(Handle *e) {
    *e = make_handle();
    return 0;
}
int hipEventDestroy(Handle) { return 0; }
int hipEventSynchronize(Handle) { return 0; }
// An event's time is the number of launches before it on its stream, a launch
// of the caller's stream taking 1 ms and one of any other 100 ms.
int hipEventElapsedTime(float *ms, Handle from, Handle to) {
    auto time = [](Handle event) {
        for (size_t i = ops.size(); i-- > 0;)
            if (ops[i].kind == RECORD && ops[i].event == event) {
                long n = 0;
                for (size_t j = 0; j < i; ++j) n += ops[j].kind == LAUNCH && ops[j].stream == ops[i].stream;
                return n * (ops[i].stream == caller ? 1L : 100L);
            }
        return -100000L;
    };
    *ms = (float)(time(to) - time(from));
    return 0;
}

}  // extern "C"

namespace {

uint8_t *device(size_t bytes) {
    void *p = nullptr;
    (void)hipMalloc(&p, bytes);
    return static_cast<uint8_t *>(p);
}

// one signing call of n items on `st`
int sign(dil_sign_ctx *ctx, int mode, size_t n, Handle st) {
    static uint8_t *buf = device(size_t(1) << 32);
    return dil_sign_device(ctx, buf, dil_signature_bytes(mode), buf, dil_secret_key_bytes(mode), buf,
                           reinterpret_cast<uint64_t *>(buf), reinterpret_cast<uint32_t *>(buf), n,
                           DIL_ENGINE_PERSISTENT, st);
}

// A call of two chains whose k-th operation fails returns an error, and the
// caller's stream still waits for whatever the second stream was given: the
// caller may free the buffers once its own stream has drained.
int join_after_errors() {
    int bad = 0;
    for (const int mode : {2, 3, 5}) {
        const size_t n = 16384;
        dil_sign_ctx *ctx = nullptr;
        if (dil_sign_ctx_create(&ctx, mode, n, n)) return wrong("context");
        const Handle st = make_handle();
        ops.clear();
        fail_at = -1;
        last_error = 0;
        if (sign(ctx, mode, n, st)) return wrong("mode %d: the call without a failure", mode);
        const size_t total = ops.size();
        size_t forked = 0;
        for (const Op &o : ops) forked += o.kind == LAUNCH && o.stream != st;
        if (!forked) return wrong("mode %d: nothing runs on a second stream", mode);
        for (size_t k = 0; k < total; ++k) {
            ops.clear();
            fail_at = (long)k;
            last_error = 0;
            if (!sign(ctx, mode, n, st)) bad |= wrong("mode %d: operation %zu of %zu failed unnoticed", mode, k, total);
            // last launch on another stream, and what was waited for after it
            long last = -1;
            for (size_t i = 0; i < ops.size(); ++i)
                if (ops[i].kind == LAUNCH && ops[i].stream != st && ops[i].ok) last = (long)i;
            if (last < 0) continue;
            bool joined = false;
            for (size_t i = (size_t)last + 1; i < ops.size(); ++i) {
                if (ops[i].ok && ops[i].kind == SYNC && ops[i].stream == ops[last].stream) joined = true;
                if (!ops[i].ok || ops[i].kind != RECORD || ops[i].stream != ops[last].stream) continue;
                for (size_t j = i + 1; j < ops.size(); ++j)
                    joined |= ops[j].ok && ops[j].kind == WAIT && ops[j].stream == st && ops[j].event == ops[i].event;
            }
            if (!joined)
                bad |= wrong("mode %d: operation %zu of %zu failed and the second stream was not joined", mode, k, total);
        }
        fail_at = -1;
        dil_sign_ctx_destroy(ctx);
    }
    return bad;
}

// A context allocates the slots that it was asked for; where the count is left
// to the library, no more than it documents, and no error if that much is not
// free.
int slots_allocated() {
    int bad = 0;
    struct Case {
        size_t max_batch, nslots, automatic;
    };
    const Case cases[] = {{1, 1, 32},          {17, 17, 544},         {333, 7, 8192},
                          {1000, 1000, 8192},  {4096, 8192, 8192},    {5000, 2500, 10000},
                          {16384, 16384, 32768}, {16384, 40000, 40000}, {40000, 40000, 65536}, {65536, 8192, 65536},
                          {262144, 65536, 65536}};
    for (const int mode : {2, 3, 5})
        for (const Case &c : cases)
            for (int form = 0; form < 5; ++form) {
                // exact, exact resident, automatic, automatic resident, automatic without memory for more
                const size_t slot = (dil_sign_temp_row_bytes(mode) + 255) / 256 * 256;
                const size_t want = form == 2 || form == 3 ? c.automatic : c.nslots;
                largest = SIZE_MAX;
                if (form == 4) {
                    if (c.automatic == c.nslots) continue;
                    largest = slot * c.automatic - 1;
                }
                allocations.clear();
                dil_sign_ctx *ctx = nullptr;
                const int e = form == 0   ? dil_sign_ctx_create(&ctx, mode, c.max_batch, c.nslots)
                              : form == 1 ? dil_sign_ctx_create_resident(&ctx, mode, c.max_batch, c.nslots)
                                          : dil_sign_ctx_create_auto(&ctx, mode, c.max_batch, c.nslots, form != 2);
                const size_t rows = allocations.empty() ? 0 : allocations[0];
                const size_t lists = (c.max_batch + 511) / 512 * 8192 + 8192;
                if (form == 4 && rows > largest) continue;  // the rows themselves do not fit
                long found = 0, more = 0;
                for (size_t i = 1; i < allocations.size(); ++i) {
                    found += allocations[i] == slot * want;
                    more += allocations[i] > slot * want && allocations[i] <= largest && allocations[i] != lists;
                }
                if (e || found != 1 || more)
                    bad |= wrong("mode %d, %zu items, %zu slots, form %d: status %d, %ld allocations of %zu slots, %ld larger",
                                 mode, c.max_batch, c.nslots, form, e, found, want, more);
                if (!e && dil_sign_ctx_slots(ctx) != want) bad |= wrong("the context reports other slots");
                if (form == 4 && hipGetLastError()) bad |= wrong("an error is left behind");
                if (!e) dil_sign_ctx_destroy(ctx);
            }
    largest = SIZE_MAX;
    return bad;
}

// The fixed stage of a call ends when it has ended on both streams.
int timed_calls() {
    int bad = 0;
    for (const size_t n : {1000, 16384}) {
        dil_sign_ctx *ctx = nullptr;
        if (dil_sign_ctx_create(&ctx, 3, n, n) || dil_sign_ctx_enable_timing(ctx, 1)) return wrong("context");
        caller = make_handle();
        ops.clear();
        if (sign(ctx, 3, n, caller)) return wrong("call");
        long all = 0, second = 0;
        for (const Op &o : ops) (o.stream == caller ? all : second) += o.kind == LAUNCH;
        float fixed = 0, loop = 0;
        const int e = dil_sign_ctx_timing(ctx, 0, &fixed, &loop);
        // two launches of the caller's stream (clearing the control words and
        // the stage), or one of the second stream
        const float want = second ? 100.f : 2.f;
        if (e || fixed != want || loop != (float)all - want)
            bad |= wrong("%zu items: status %d, fixed %g ms, loop %g ms of %ld launches", n, e, fixed, loop, all);
        if ((n >= 12288) != (second > 0)) bad |= wrong("%zu items: %ld launches on a second stream", n, second);
        dil_sign_ctx_destroy(ctx);
    }
    return bad;
}

}  // namespace

int main(int argc, char **argv) {
    const char *what = argc > 1 ? argv[1] : "";
    if (!strcmp(what, "join")) return join_after_errors();
    if (!strcmp(what, "slots")) return slots_allocated();
    if (!strcmp(what, "timing")) return timed_calls();
    return 2;
}
