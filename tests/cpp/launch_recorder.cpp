// Preloaded into a process of the CPU tests: kernel launches are written down instead of being made, so that a test can
// see which kernel a call would launch, with which grid, workgroup and LDS size, without a GPU.
#include <stddef.h>
#include <stdint.h>
#include <string.h>

#include <map>
#include <string>
#include <vector>

struct Dim3 {
    uint32_t x, y, z;
};

namespace {
struct Launch {
    std::string name;
    uint32_t grid[3], block[3];
    size_t lds;
};
std::map<const void *, std::string> &names()
{
    static std::map<const void *, std::string> m;
    return m;
}
std::vector<Launch> &launches()
{
    static std::vector<Launch> v;
    return v;
}
} // namespace

extern "C" {

// (not handed on to the runtime: nothing of this process is ever launched)
void __hipRegisterFunction(void **, const void *host, char *, const char *device_name, unsigned, void *, void *, void *, void *, int *)
{
    names()[host] = device_name;
}

static Dim3 g_grid, g_block;
static size_t g_lds;

int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t lds, void *)
{
    g_grid = grid;
    g_block = block;
    g_lds = lds;
    return 0;
}

int __hipPopCallConfiguration(Dim3 *grid, Dim3 *block, size_t *lds, void **stream)
{
    *grid = g_grid;
    *block = g_block;
    *lds = g_lds;
    *stream = nullptr;
    return 0;
}

int hipLaunchKernel(const void *f, Dim3 grid, Dim3 block, void **, size_t lds, void *)
{
    launches().push_back(Launch{ names()[f], { grid.x, grid.y, grid.z }, { block.x, block.y, block.z }, lds });
    return 0;
}

int hipFuncSetAttribute(const void *, int, int) { return 0; }
int hipGetLastError() { return 0; }

int recorder_count() { return (int)launches().size(); }
const char *recorder_name(int i) { return launches()[i].name.c_str(); }
void recorder_sizes(int i, uint32_t *grid, uint32_t *block, uint64_t *lds)
{
    memcpy(grid, launches()[i].grid, 12);
    memcpy(block, launches()[i].block, 12);
    *lds = launches()[i].lds;
}
void recorder_clear() { launches().clear(); }
}
