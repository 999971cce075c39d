// runtime.cpp — HIP error mapping, device selection and buffers.
#include <atomic>
#include "runtime.hpp"

#include <cstring>
#include <string>

namespace nut {

namespace {

thread_local std::string g_last_error;
thread_local int g_device = 0;
thread_local bool g_device_ready = false;

} // namespace

void set_last_error(const char *message) { g_last_error = message; }
const char *last_error() { return g_last_error.c_str(); }

void fail_hip(hipError_t error, const char *what)
{
    fail(NUT_EDEVICE, std::string(what) + ": " + hipGetErrorString(error));
}

void check_launch(const char *what)
{
    const hipError_t error = hipGetLastError();
    if (error != hipSuccess)
        fail_hip(error, what);
}

int select_device(int device)
{
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess)
        count = 0;
    if (device < 0 || device >= count)
        fail(NUT_EDEVICE, "no such HIP device");
    hipDeviceProp_t props;
    hip_check(hipGetDeviceProperties(&props, device), "hipGetDeviceProperties");
    if (std::strncmp(props.gcnArchName, "gfx950", 6) != 0)
        fail(NUT_EDEVICE, std::string("device is ") + props.gcnArchName +
                              ", this library is built for gfx950");
    hip_check(hipSetDevice(device), "hipSetDevice");
    g_device = device;
    g_device_ready = true;
    return device;
}

void ensure_device()
{
    if (g_device_ready) {
        hip_check(hipSetDevice(g_device), "hipSetDevice");
        return;
    }
    select_device(g_device);
}

namespace {
std::atomic<unsigned long long> g_allocations{0};
}

unsigned long long device_allocations() { return g_allocations.load(); }

void count_device_allocation() { g_allocations.fetch_add(1); }

namespace {
thread_local unsigned g_skip_allocations = 0, g_fail_allocations = 0;

bool injected_failure()
{
    if (g_fail_allocations == 0)
        return false;
    if (g_skip_allocations > 0) {
        g_skip_allocations--;
        return false;
    }
    g_fail_allocations--;
    return true;
}
} // namespace

void fail_allocations(unsigned skip, unsigned count)
{
    g_skip_allocations = skip;
    g_fail_allocations = count;
}

hipError_t DeviceBuffer::replace(size_t bytes)
{
    release();
    if (bytes == 0)
        bytes = 1;
    void *p = nullptr;
    const hipError_t error = injected_failure() ? hipErrorOutOfMemory : hipMalloc(&p, bytes);
    if (error != hipSuccess) {
        (void)hipGetLastError(); // not the next launch's error
        return error;
    }
    count_device_allocation();
    ptr_ = p;
    bytes_ = bytes;
    return hipSuccess;
}

void DeviceBuffer::allocate(size_t bytes) { hip_check(replace(bytes), "hipMalloc"); }

bool DeviceBuffer::try_allocate(size_t bytes) { return replace(bytes) == hipSuccess; }

void DeviceBuffer::release()
{
    if (ptr_ != nullptr)
        (void)hipFree(ptr_);
    ptr_ = nullptr;
    bytes_ = 0;
}

void PinnedBuffer::allocate(size_t bytes)
{
    release();
    hip_check(hipHostMalloc(&ptr_, bytes, hipHostMallocMapped), "hipHostMalloc");
}

void PinnedBuffer::release()
{
    if (ptr_ != nullptr)
        (void)hipHostFree(ptr_);
    ptr_ = nullptr;
}

} // namespace nut
