// pool_test.cpp - the pool of tensors' memory (cyb_amd/csrc/pool.hip) against a HIP that only counts: when it waits for the
// device, what it keeps and gives back, and that no exception leaves it.  Runs without a GPU.
#include <cstdio>
#include <cstdlib>
#include <new>

#include "../../cyb_amd/csrc/pool.hip"

namespace {
int syncs = 0, mallocs = 0, event_waits = 0, failed = 0;
size_t device_limit = (size_t)1 << 40, in_use = 0;
bool no_memory = false;
}  // namespace

void* operator new(size_t n)
{
    if (no_memory) throw std::bad_alloc();
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

// device memory: a malloc'ed word that holds the size
extern "C" {
hipError_t hipMalloc(void** p, size_t n)
{
    mallocs++;
    if (in_use + n > device_limit) return hipErrorOutOfMemory;
    *p = std::malloc(sizeof(size_t));
    *static_cast<size_t*>(*p) = n;
    in_use += n;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    in_use -= *static_cast<size_t*>(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipDeviceSynchronize(void) { return syncs++, hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return *p = std::malloc(n), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = reinterpret_cast<hipEvent_t>(std::malloc(1)), hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return event_waits++, hipSuccess; }
}

#define CHECK(what)                                                              \
    do {                                                                         \
        if (!(what)) std::printf("line %d: %s\n", __LINE__, #what), failed++;    \
    } while (0)

using namespace cybq;

int main()
{
    constexpr size_t MB = (size_t)1 << 20;
    void *a = nullptr, *b = nullptr;
    size_t na = 0, nb = 0;
    CHECK(pool_retain(0) == hipSuccess);

    // where a block was used before against where it is written next: only default stream after default stream, and a block
    // that nothing used, go without a wait
    for (int used = kUnused; used <= kElsewhere; used++)
        for (int next = kDefaultStream; next <= kElsewhere; next++) {
            CHECK(pool_alloc(0, 4 * MB, kDefaultStream, &a, &na) == hipSuccess);
            pool_free(0, a, na, static_cast<UsedOn>(used));
            const int s0 = syncs, m0 = mallocs;
            CHECK(pool_alloc(0, 4 * MB, static_cast<UsedOn>(next), &b, &nb) == hipSuccess);
            CHECK(b == a && mallocs == m0);
            CHECK(syncs - s0 == (used == kElsewhere || (used == kDefaultStream && next == kElsewhere) ? 1 : 0));
            pool_free(0, b, nb, kUnused);
        }
    // one wait covers every block that was there
    CHECK(pool_alloc(0, 4 * MB, kDefaultStream, &a, &na) == hipSuccess && pool_alloc(0, 4 * MB, kDefaultStream, &b, &nb) == hipSuccess);
    pool_free(0, a, na, kElsewhere);
    pool_free(0, b, nb, kElsewhere);
    const int s0 = syncs;
    CHECK(pool_alloc(0, 4 * MB, kElsewhere, &a, &na) == hipSuccess && pool_alloc(0, 4 * MB, kElsewhere, &b, &nb) == hipSuccess && syncs == s0 + 1);
    pool_free(0, a, na, kUnused);
    pool_free(0, b, nb, kUnused);

    // sizes: at most a quarter larger than asked for, the smallest of those
    CHECK(pool_alloc(0, 100 * MB, kDefaultStream, &a, &na) == hipSuccess && pool_alloc(0, 90 * MB, kDefaultStream, &b, &nb) == hipSuccess);
    void *pa = a, *pb = b;
    pool_free(0, a, na, kUnused);
    pool_free(0, b, nb, kUnused);
    CHECK(pool_alloc(0, 81 * MB, kDefaultStream, &a, &na) == hipSuccess && a == pb && na == 90 * MB);
    CHECK(pool_alloc(0, 79 * MB, kDefaultStream, &b, &nb) == hipSuccess && b != pa && nb == 79 * MB);
    pool_free(0, a, na, kUnused);
    pool_free(0, b, nb, kUnused);

    // the bound: what is kept never passes it, and a block larger than it is not kept
    void* many[12];
    size_t size[12];
    for (int i = 0; i < 12; i++) CHECK(pool_alloc(0, (64 + i) * MB, kDefaultStream, &many[i], &size[i]) == hipSuccess);
    for (int i = 0; i < 12; i++) pool_free(0, many[i], size[i], kUnused);
    CHECK(in_use <= kPoolBytes);
    CHECK(pool_alloc(0, kPoolBytes + MB, kDefaultStream, &a, &na) == hipSuccess);
    pool_free(0, a, na, kUnused);
    CHECK(in_use <= kPoolBytes);
    // the device runs out: the kept blocks are given up for the call
    device_limit = 600 * MB;
    CHECK(in_use > 100 * MB && pool_alloc(0, 590 * MB, kDefaultStream, &a, &na) == hipSuccess && in_use == 590 * MB);
    pool_free(0, a, na, kUnused);
    device_limit = (size_t)1 << 40;

    // scan slots: distinct, the longest free one next, waited for before it is used again
    ScanSlot s[3];
    for (ScanSlot& t : s) CHECK(scan_acquire(0, &t) == hipSuccess && t.word && t.done);
    CHECK(s[0].word != s[1].word && s[1].word != s[2].word && s[0].done != s[1].done);
    scan_release(0, s[0]);
    for (int i = 0; i < 1021; i++) CHECK(scan_acquire(0, &s[1]) == hipSuccess && event_waits == 0);
    CHECK(scan_acquire(0, &s[1]) == hipSuccess && s[1].word == s[0].word && event_waits == 1);

    // no host memory: errors and blocks that are not kept, no exceptions
    CHECK(pool_alloc(0, 4 * MB, kDefaultStream, &a, &na) == hipSuccess);
    const size_t before = in_use;
    no_memory = true;
    CHECK(pool_retain(1) == hipErrorOutOfMemory);
    CHECK(scan_acquire(0, &s[2]) == hipErrorOutOfMemory);          // (none free: it wants another slab)
    pool_free(0, a, na, kUnused);
    for (int i = 0; i < 600; i++) scan_release(0, s[0]);           // (past what the queue has room for)
    no_memory = false;
    CHECK(in_use == before - na);
    CHECK(scan_acquire(0, &s[2]) == hipSuccess);

    // everything kept goes back when asked
    CHECK(pool_alloc(0, 4 * MB, kDefaultStream, &a, &na) == hipSuccess && pool_alloc(0, 5 * MB, kDefaultStream, &b, &nb) == hipSuccess);
    pool_free(0, a, na, kElsewhere);
    CHECK(pool_trim(0) == hipSuccess && in_use == nb);
    pool_free(0, b, nb, kUnused);
    CHECK(pool_trim(0) == hipSuccess && pool_trim(0) == hipSuccess && in_use == 0);

    // the last context takes everything with it; what is freed later goes back at once
    CHECK(pool_alloc(0, 4 * MB, kDefaultStream, &a, &na) == hipSuccess && pool_alloc(0, 4 * MB, kDefaultStream, &b, &nb) == hipSuccess);
    pool_free(0, a, na, kElsewhere);
    pool_release(0);
    CHECK(in_use == nb);
    pool_free(0, b, nb, kDefaultStream);
    CHECK(in_use == 0);
    std::printf(failed ? "FAILED\n" : "OK\n");
    return failed != 0;
}
