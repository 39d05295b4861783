// Host check of hmg_set_option on an engine that stands alone: the near field's LDS
// reservation can be set and given back to the kernel's own choice.
#include <cstdio>

#include "hmg_internal.h"

#define CHECK(x)                                    \
    do {                                            \
        if (!(x)) {                                 \
            std::printf("line %d: %s\n", __LINE__, #x); \
            return 1;                               \
        }                                           \
    } while (0)

int main()
{
    using namespace hmg;
    Engine e;
    h_matrix_data d{};
    d.engine = &e;
    const int own = e.near_lds_pad;
    CHECK(own == -1 && e.near_pad(12345) == 12345);
    for (const int v : {0, 4096, 128 * 1024}) {
        CHECK(hmg_set_option(&d, HMG_OPT_NEAR_LDS_BYTES, v) == HMG_OK);
        CHECK(e.near_pad(12345) == v);
    }
    CHECK(hmg_set_option(&d, HMG_OPT_NEAR_LDS_BYTES, 128 * 1024 + 1) == HMG_ERR_INVALID);
    CHECK(hmg_set_option(&d, HMG_OPT_NEAR_LDS_BYTES, -2) == HMG_ERR_INVALID);
    CHECK(e.near_pad(12345) == 128 * 1024);
    CHECK(hmg_set_option(&d, HMG_OPT_NEAR_LDS_BYTES, -1) == HMG_OK);
    CHECK(e.near_pad(12345) == 12345);
    std::puts("ok");
    return 0;
}
