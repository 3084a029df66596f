/* Stands in for the HIP runtime behind a library built by hipcc: nothing is launched, each launch is written down.  Loaded
 * (RTLD_GLOBAL) before the library, in a process that has no use for a GPU. */
#include <stddef.h>
#include <stdint.h>
#include <string.h>

typedef struct {
    uint32_t x, y, z;
} dim3;

typedef struct {
    const char* name;
    dim3 grid, block;
    size_t lds;
} launch;

enum { MOST = 4096 };
static const void* registered[MOST];
static const char* names[MOST];
int n_registered;
static dim3 config_grid, config_block;
static size_t config_lds;
static void* config_stream;

launch launches[MOST];
int n_launches;

void** __hipRegisterFatBinary(const void* data)
{
    static void* handle;
    (void)data;
    return &handle;
}
void __hipUnregisterFatBinary(void** modules) { (void)modules; }
void __hipRegisterVar(void** modules, void* var, char* host, char* device, int ext, size_t size, int constant, int global)
{
    (void)modules, (void)var, (void)host, (void)device, (void)ext, (void)size, (void)constant, (void)global;
}
void __hipRegisterFunction(void** modules, const void* host, char* device, const char* name, unsigned limit, void* tid, void* bid, void* bd, void* gd, int* ws)
{
    (void)modules, (void)device, (void)limit, (void)tid, (void)bid, (void)bd, (void)gd, (void)ws;
    if (n_registered < MOST) registered[n_registered] = host, names[n_registered++] = name;
}
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, void* stream)
{
    config_grid = grid, config_block = block, config_lds = lds, config_stream = stream;
    return 0;
}
int __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, void** stream)
{
    *grid = config_grid, *block = config_block, *lds = config_lds, *stream = config_stream;
    return 0;
}
int hipLaunchKernel(const void* host, dim3 grid, dim3 block, void** args, size_t lds, void* stream)
{
    (void)args, (void)stream;
    for (int i = 0; i < n_registered; ++i)
        if (registered[i] == host && n_launches < MOST) {
            launches[n_launches].name = names[i];
            launches[n_launches].grid = grid, launches[n_launches].block = block, launches[n_launches++].lds = lds;
        }
    return 0;
}
int hipGetLastError(void) { return 0; }
