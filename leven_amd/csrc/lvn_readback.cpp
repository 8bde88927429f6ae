// lvn_readback.cpp — finished meshes from device memory into a caller's host buffers (host code).

#include "lvn_runtime.h"

#include <cstring>
#include <new>
#include <vector>

namespace lvn {

// Where the device sees the pinned host memory that begins at p, and in *held how many bytes
// of it there are from there; null for any other memory.
static char* pinned_view(void* p, size_t* held) {
    *held = 0;
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();  // memory the runtime does not know
        return nullptr;
    }
    if (at.type != hipMemoryTypeHost || !at.devicePointer) return nullptr;
    char* const d = static_cast<char*>(at.devicePointer);
    hipDeviceptr_t base = nullptr;
    size_t size = 0;
    if (hipMemGetAddressRange(&base, &size, d) != hipSuccess) {
        (void)hipGetLastError();
        return d;
    }
    const char* const b = static_cast<const char*>(base);
    if (d >= b && d < b + size) *held = (size_t)(b + size - d);
    return d;
}

// A kernel writes only into pinned buffers that their allocation holds to the end: one that
// begins in pinned memory and runs past it (a caller may have registered a part of its memory)
// is copied through ordinary memory, since neither a kernel nor the runtime's copy may run on
// past the mapping.
int read_mesh(const char* verts, size_t bv, const char* tris, size_t bt, const char* seams, size_t bs, lvn_vertex* v,
              int32_t* tri, lvn_seam_node* sn, hipStream_t s) {
    MeshCopy c = {{verts, tris, seams}, {nullptr, nullptr, nullptr}, {v ? bv : 0, tri ? bt : 0, sn ? bs : 0}};
    void* out[3] = {v, tri, sn};
    size_t held[3] = {0, 0, 0};
    bool pinned = true;
    for (int i = 0; i < 3; ++i) {
        if (!c.bytes[i]) continue;
        c.dst[i] = pinned_view(out[i], &held[i]);
        pinned = pinned && c.dst[i] && ((uintptr_t)c.dst[i] & 3) == 0 && c.bytes[i] <= held[i];
    }
    if (c.bytes[0] + c.bytes[1] + c.bytes[2] == 0) return LVN_OK;
    if (pinned) {
        launch_copy_mesh(c, s);
        LVN_HIP(hipGetLastError());
        LVN_HIP(hipStreamSynchronize(s));
        return LVN_OK;
    }
    std::vector<char> part;
    for (int i = 0; i < 3; ++i) {
        if (!c.bytes[i]) continue;
        if (!c.dst[i] || c.bytes[i] <= held[i]) {
            LVN_HIP(hipMemcpy(out[i], c.src[i], c.bytes[i], hipMemcpyDeviceToHost));
            continue;
        }
        try {
            part.resize(c.bytes[i]);
        } catch (const std::bad_alloc&) {
            return LVN_ERR_NOMEM;
        }
        LVN_HIP(hipMemcpy(part.data(), c.src[i], c.bytes[i], hipMemcpyDeviceToHost));
        std::memcpy(out[i], part.data(), c.bytes[i]);
    }
    return LVN_OK;
}

}  // namespace lvn
