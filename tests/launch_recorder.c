/* Stands in for the HIP runtime's launch entry points in a process without a GPU, so that a test can see what the library
 * would launch: kernel name, grid and block of every launch, and the split count that a combine launch is given.  Nothing
 * runs.  Loaded with RTLD_GLOBAL in front of the library (tests/launch_recorder.py). */
#include <hip/hip_runtime_api.h>
#include <string.h>

enum { kMaxKernels = 4096, kMaxLaunches = 16 };
static const void *handles[kMaxKernels];
static const char *names[kMaxKernels];
static int kernels;

struct launch {
    const char *name;
    unsigned long long groups, threads;
    int split_count; /* of a combine launch: its last argument; 0 otherwise */
};
static struct launch launches[kMaxLaunches];
static int launched;

void __hipRegisterFunction(void **modules, const void *handle, char *device_function, const char *name, unsigned limit, void *tid,
                           void *bid, void *block, void *grid, int *wsize)
{
    (void)modules, (void)device_function, (void)limit, (void)tid, (void)bid, (void)block, (void)grid, (void)wsize;
    if (kernels < kMaxKernels) handles[kernels] = handle, names[kernels++] = name;
}

hipError_t hipLaunchKernel(const void *handle, dim3 grid, dim3 block, void **args, size_t lds, hipStream_t stream)
{
    (void)lds, (void)stream;
    struct launch l = {"?", (unsigned long long)grid.x * grid.y * grid.z, (unsigned long long)block.x * block.y * block.z, 0};
    for (int i = 0; i < kernels; ++i)
        if (handles[i] == handle) l.name = names[i];
    if (strstr(l.name, "combine_kernel")) l.split_count = *(const int *)args[8];
    if (launched < kMaxLaunches) launches[launched++] = l;
    /* the runtime's own limits */
    return l.groups > 0x7fffffffull || l.groups * l.threads > 0xffffffffull ? hipErrorInvalidConfiguration : hipSuccess;
}

hipError_t hipGetDevice(int *device)
{
    *device = 0;
    return hipSuccess;
}

hipError_t hipGetDeviceProperties(hipDeviceProp_t *prop, int device)
{
    (void)device;
    memset(prop, 0, sizeof(*prop));
    strcpy(prop->gcnArchName, "gfx950");
    return hipSuccess;
}

hipError_t hipFuncSetAttribute(const void *handle, hipFuncAttribute attribute, int value)
{
    (void)handle, (void)attribute, (void)value;
    return hipSuccess;
}

void recorder_clear(void) { launched = 0; }
int recorder_count(void) { return launched; }
const char *recorder_name(int i) { return launches[i].name; }
unsigned long long recorder_groups(int i) { return launches[i].groups; }
unsigned long long recorder_threads(int i) { return launches[i].threads; }
int recorder_split_count(int i) { return launches[i].split_count; }
