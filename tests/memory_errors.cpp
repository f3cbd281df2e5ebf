// Which errors of an optional structure's construction are done without (ifMemoryAllows): those of memory, on the host and on
// the device, and no others.
#include <cstdio>

#include "host_util.h"

using namespace spgvbd;

template <class E>
static bool passes(const E &e)
{
    try {
        ifMemoryAllows([&] { throw e; });
        return false;
    } catch (const E &) {
        return true;
    }
}

int main()
{
    int wrong = 0;
    wrong += !ifMemoryAllows([] {});
    wrong += ifMemoryAllows([] { throw std::bad_alloc(); });
    wrong += ifMemoryAllows([] { throw DeviceMemoryError(SPG_VBD_ERR_HIP, "hipMalloc: out of memory"); });
    wrong += !passes(VbdError(SPG_VBD_ERR_HIP, "tile records launch: invalid configuration"));
    wrong += !passes(std::runtime_error("another"));
    printf("%d wrong\n", wrong);
    return wrong;
}
