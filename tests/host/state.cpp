// Host check of the state that a captured product is compared with: two H-matrices that
// stand in the same struct one after the other, with equal buffers, have different states.
#include <cstdio>
#include <new>

#include "hmg_internal.h"

int main()
{
    using namespace hmg;
    alignas(Engine) static unsigned char room[sizeof(Engine)];
    h_matrix_data d{};
    std::vector<std::vector<const void*>> seen;
    for (int life = 0; life < 3; life++) {
        Engine* e = new (room) Engine();
        d.engine = e;
        for (int change = 0; change < 3; change++) {
            seen.push_back(product_state(&d, *e));
            if (hmg_set_option(&d, HMG_OPT_SERIALIZE, 0) != HMG_OK) return 2;
        }
        e->~Engine();
    }
    for (size_t i = 0; i < seen.size(); i++)
        for (size_t j = i + 1; j < seen.size(); j++)
            if (seen[i] == seen[j]) {
                std::printf("states %zu and %zu are equal\n", i, j);
                return 1;
            }
    std::puts("ok");
    return 0;
}
