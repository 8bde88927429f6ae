// The host side of a mesh's read-back (leven_amd/csrc/lvn_readback.cpp) on the CPU, with the
// HIP calls that it makes replaced by ones that know three kinds of memory: pinned, ordinary, and
// a buffer that begins in pinned memory and runs past its end.  A kernel or a runtime copy that
// would write a pinned buffer past its allocation is reported, and the meshes must arrive.
#include "../../leven_amd/csrc/lvn_runtime.h"

#include <cstdlib>
#include <cstring>

static char* g_pinned = nullptr;  // the one pinned allocation; ordinary memory follows it
static size_t g_pinned_bytes = 0;
static int g_launches = 0, g_copies = 0, g_bad = 0;

static bool in_pinned(const void* p) {
    return static_cast<const char*>(p) >= g_pinned && static_cast<const char*>(p) < g_pinned + g_pinned_bytes;
}
static void write_checked(void* dst, const void* src, size_t bytes) {
    if (bytes && in_pinned(dst) && !in_pinned(static_cast<char*>(dst) + bytes - 1)) {
        ++g_bad;
        return;
    }
    std::memcpy(dst, src, bytes);
}

extern "C" {
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    std::memset(a, 0, sizeof(*a));
    if (!in_pinned(p)) return hipErrorInvalidValue;
    a->type = hipMemoryTypeHost;
    a->devicePointer = const_cast<void*>(p);
    a->hostPointer = const_cast<void*>(p);
    return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t* base, size_t* size, hipDeviceptr_t p) {
    if (!in_pinned(p)) return hipErrorNotFound;
    *base = g_pinned;
    *size = g_pinned_bytes;
    return hipSuccess;
}
hipError_t hipMemcpy(void* dst, const void* src, size_t bytes, hipMemcpyKind) {
    ++g_copies;
    write_checked(dst, src, bytes);
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
}

namespace lvn {
void launch_copy_mesh(const MeshCopy& c, hipStream_t) {
    ++g_launches;
    for (int i = 0; i < 3; ++i) write_checked(c.dst[i], c.src[i], c.bytes[i]);
}
}  // namespace lvn

int main() {
    const size_t len[3] = {4800, 1200, 960}, pinned = 8192, total = 65536;
    char* mem = static_cast<char*>(std::aligned_alloc(4096, total));
    char src[3][4800];
    for (int k = 0; k < 3; ++k)
        for (size_t i = 0; i < len[k]; ++i) src[k][i] = (char)(17 * k + 3 * i + 1);
    g_pinned = mem;
    g_pinned_bytes = pinned;
    // where array k starts: within the pinned memory, over its end by `over` bytes, or behind it
    struct Case {
        const char* name;
        long at[3];
        int launches, copies;
    };
    const Case cases[] = {
        {"all pinned", {0, 4800, 6000}, 1, 0},
        {"one to the last byte", {(long)(pinned - 4800), 0, 1200}, 1, 0},
        {"vertices over the end", {(long)(pinned - 480), 0, 1200}, 0, 3},
        {"vertices one word over", {(long)(pinned - 4796), 0, 1200}, 0, 3},
        {"triangles over the end", {0, (long)(pinned - 4), 4800}, 0, 3},
        {"seam nodes over the end", {0, 4800, (long)(pinned - 956)}, 0, 3},
        {"ordinary", {20000, 30000, 40000}, 0, 3},
        {"odd address", {2, 4804, 6004}, 0, 3},
    };
    int failed = 0;
    for (const Case& c : cases) {
        std::memset(mem, 0x5A, total);
        g_launches = g_copies = g_bad = 0;
        char* out[3] = {mem + c.at[0], mem + c.at[1], mem + c.at[2]};
        const int r = lvn::read_mesh(src[0], len[0], src[1], len[1], src[2], len[2],
                                     reinterpret_cast<lvn_vertex*>(out[0]), reinterpret_cast<int32_t*>(out[1]),
                                     reinterpret_cast<lvn_seam_node*>(out[2]), nullptr);
        bool same = true;
        for (int k = 0; k < 3; ++k) same = same && !std::memcmp(out[k], src[k], len[k]);
        const bool ok = r == LVN_OK && same && !g_bad && g_launches == c.launches && g_copies == c.copies;
        printf("%s: %s (result %d, same %d, writes past the pinned end %d, launches %d, copies %d)\n", ok ? "ok" : "FAIL",
               c.name, r, (int)same, g_bad, g_launches, g_copies);
        failed += !ok;
    }
    std::free(mem);
    return failed != 0;
}
