// Host check of the kept buffers against a model of the device's pool: the pool may hand a
// buffer back to the stream that allocated it at once, so a buffer that another stream's
// queued work uses must neither be freed nor be kept for others before that stream was
// waited for.  The HIP calls of the buffers are the model's own.
#include <cstdio>
#include <cstdlib>
#include <map>
#include <set>
#include <utility>

#include "hmg_internal.h"

namespace {
std::map<void*, hipStream_t> owner;  // allocating stream of every live buffer
std::map<void*, hipStream_t> user;   // stream whose queued work uses it
int unsafe = 0, freed = 0;
}  // namespace

extern "C" {
hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t* d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipMallocAsync(void** p, size_t, hipStream_t s)
{
    *p = std::malloc(64);
    owner[*p] = s;
    return hipSuccess;
}
hipError_t hipFreeAsync(void* p, hipStream_t s)
{
    if (user.count(p) && !(owner[p] == s && user[p] == s)) unsafe++;
    freed++;
    owner.erase(p);
    user.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s)
{
    for (auto it = user.begin(); it != user.end();) it = it->second == s ? user.erase(it) : std::next(it);
    return hipSuccess;
}
}

#define CHECK(x)                                        \
    do {                                                \
        if (!(x)) {                                     \
            std::printf("line %d: %s\n", __LINE__, #x); \
            return 1;                                   \
        }                                               \
    } while (0)

int main()
{
    using namespace hmg;
    using Buf = DevBuf<unsigned char>;
    const hipStream_t A = (hipStream_t)16, B = (hipStream_t)32, C = (hipStream_t)48;
    const size_t n = (size_t)1 << 20;
    void* first;
    {
        // allocated on A, kept when A has been waited for
        AllocScope scope(A);
        Buf x;
        CHECK(x.alloc(n) == HMG_OK);
        first = x.p;
        user[x.p] = A;
        (void)hipStreamSynchronize(A);
        IdleScope idle(true);
        x.release();
    }
    CHECK(freed == 0);
    for (int round = 0; round < 3; round++) {
        // a temporary on B, released behind B's work: neither freed nor anybody else's yet
        AllocScope scope(B);
        Buf y, moved;
        CHECK(y.alloc(n) == HMG_OK && y.p == first);
        user[y.p] = B;
        moved = std::move(y);
        if (round == 1)
            CHECK(moved.alloc(4 * n) == HMG_OK);  // grown: the old one is released
        else
            moved.release();
        CHECK(unsafe == 0 && freed == 0 && user.count(first));
        {
            Buf z;
            hipStream_t prev = g_alloc_stream;
            g_alloc_stream = C;  // (no scope: its end would wait)
            CHECK(z.alloc(n) == HMG_OK && z.p != first);
            g_alloc_stream = prev;
            (void)hipStreamSynchronize(C);
            z.release();
            freed = 0;
        }
        if (round == 2) {
            (void)hipStreamSynchronize(B);
            idle_settle(B);
            Buf w;
            CHECK(w.alloc(n) == HMG_OK && w.p == first);
        }
        if (round == 1) {
            user[moved.p] = B;
            moved.release();  // its own stream's buffer: freed in stream order
            CHECK(freed == 1 && unsafe == 0);
            freed = 0;
        }
    }
    CHECK(!user.count(first));  // the scope waited for B
    {
        // without a scope the release waits itself
        Buf x;
        {
            AllocScope scope(C);
            CHECK(x.alloc(n) == HMG_OK && x.p == first);
        }
        user[x.p] = C;
        x.release();
        CHECK(!user.count(first) && unsafe == 0);
    }
    std::puts("ok");
    return 0;
}
