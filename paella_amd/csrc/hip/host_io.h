#pragma once
// Device memory that the host reads and writes itself, through the PCIe aperture.
//
// Copies between a request's buffers and pageable host memory: the runtime's take two copies and a wait, these one.  Input, streaming
// stores: 4 KB 0.3 us against 13, 602 KB 13.5 against 30, 1.07 MB 25 against 60.  Output, streaming loads (ordinary ones fetch 4 or 8
// bytes a trip): 4 KB 2.3 us against 13; from about 32 KB on the runtime's copy is as fast.

#include <cstddef>

namespace paella {

// Lets the host address `p`, the start of an allocation of device memory; false where the platform does not.
bool host_map_device(void* p);
// Host to mapped device memory (dst 64-byte aligned); a kernel whose doorbell is rung afterwards, by whatever thread the request is handed
// to, reads the data.
void host_store(void* dst, const void* src, size_t bytes);
// The same by the library's copy thread, as paella_host_copy_submit.
int host_store_submit(void* dst, const void* src, size_t bytes, void (*done)(void*), void* arg);
// Mapped device memory to the host, once the kernels that wrote it (through to memory) have finished.  src 64-byte aligned.
void host_load(void* dst, const void* src, size_t bytes);

}  // namespace paella
