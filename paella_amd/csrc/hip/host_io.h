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
// Host to mapped device memory (dst 64-byte aligned).  A kernel that this thread launches afterwards reads the data: stores through the
// aperture are posted, that is, the core is done with them before they are in memory, but the fence behind them keeps them ahead of
// whatever the core stores to the device later, and posted writes keep their order on the link.  So they arrive ahead of the doorbell, and
// ahead of a direct-dispatch kernel's arguments, which take the same way.  The packet that the doorbell announces lies in host memory,
// and the answer to its fetch comes down the same link, on which completions do not overtake posted writes: the packet processor cannot
// have a kernel's packet before the device has its input.
void host_store(void* dst, const void* src, size_t bytes);
// Waits until what host_store wrote is in memory: a read does not overtake the stores on its way to the device.  For a thread whose
// stores another core may follow with a doorbell within a microsecond, so that nothing rests on the order between two cores' stores.
// 1.2 to 2 us on the copy thread: a lone served request of ResNet-18 163 -> 164.5 us, nothing under load (4096 of them 216.1 -> 216.0 ms).  The
// calling thread's own launches do without (a small CNN's request 27.6 -> 29.3 us with it, ResNet-18's 166.5 -> 168, Inception-v3's 403 -> 405).
void host_settle(const void* dst, size_t bytes);
// The same by the library's copy thread, as paella_host_copy_submit.
int host_store_submit(void* dst, const void* src, size_t bytes, void (*done)(void*), void* arg);
// Mapped device memory to the host, once the kernels that wrote it (through to memory) have finished.  src 64-byte aligned.
void host_load(void* dst, const void* src, size_t bytes);

}  // namespace paella
