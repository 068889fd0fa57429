// pbf_transfer.hip -- copies between a caller's ordinary memory and the device.
//
// They go through a small block of pinned memory of the object: the host
// copies a chunk while the device moves the others.  Copies straight from and
// to pageable memory cost more, most of all where the runtime takes 100 to 200
// us for 64 to 400 KB, as it does in some processes.  Measured, us for a call
// that sets / reads an array, its reordering kernel and the wait included (in
// brackets with the runtime's copies):
//      12 KB     14 /   14   (21 /   28)
//     393 KB     31 /   38   (33 to 175 / 40 to 195)
//     1.6 MB     70 /   90   (77 /  110)
//     3.1 MB    125 /  170  (121 /  197)
//    12.6 MB    337 /  495  (375 /  735)
//      34 MB    900 /  960 (1000 / 1930)
//     101 MB   2580 / 2550 (3480 / 5800, into fresh pages 9800)
// (For some tens of milliseconds after much device memory was given back, the
// copy engines clear it: copies of either kind then take up to four times as
// long.)
// Bound: PCIe (12.6 MB alone take 228 us from pinned memory), the host's copy
// next to it, and some 15 us a queued copy, which is why chunks are large.  (A
// kernel that copies instead of the copy engine: 385 us up and 480 down at 12.6 MB.)
//
// Memory that the caller has pinned takes no part in this: the copy engine
// reads and writes it as it is, 257 / 266 us for 12.6 MB against 346 / 515
// through the staging memory.
#include <algorithm>
#include <cstring>
#include <thread>

#include "pbf_internal.h"

namespace pbf {

Memory memory_of(const void* p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return Memory::kPageable;
  }
  switch (a.type) {
    case hipMemoryTypeUnregistered: return Memory::kPageable;
    case hipMemoryTypeHost: return Memory::kPinned;
    default: return Memory::kDevice;
  }
}

int HostStage::create(uint64_t most, uint64_t slot) {
  // (two slots from 1 MB on, so that the host's copy of one chunk goes next to
  // the device's of the other: 1.6 MB up take 84 us in one piece)
  const bool halves = most > kSlot / 2 && most <= slot;
  slot_bytes = std::min<uint64_t>(slot, ((halves ? (most + 1) / 2 : most) + 255) / 256 * 256);
  const uint64_t slots = std::min<uint64_t>(kSlots, (most + slot_bytes - 1) / slot_bytes);
  int rc = check_hip(hipGetDevice(&device), "hipGetDevice");
  if (!rc) rc = check_hip(hipHostMalloc((void**)&pin, slots * slot_bytes), "hipHostMalloc");
  for (uint64_t i = 0; !rc && i < slots; ++i)
    rc = check_hip(hipEventCreateWithFlags(&done[i], hipEventDisableTiming), "hipEventCreate");
  if (!rc) nslots = (uint32_t)slots;
  return rc;
}

void HostStage::destroy() {
  for (hipEvent_t& e : done) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  if (pin) (void)hipHostFree(pin);
  pin = nullptr;
  nslots = 0;
}

// A part of a transfer, through slots [first, first + count): chunk by chunk,
// the host's copy of one next to the device's copy of the others.
hipError_t HostStage::upload_part(unsigned char* dev, const unsigned char* host, uint64_t bytes, uint64_t chunk,
                                  uint32_t first, uint32_t count, hipStream_t s) {
  uint32_t k = 0;
  for (uint64_t at = 0; at < bytes; at += chunk, ++k) {
    const uint64_t len = std::min(chunk, bytes - at);
    const uint32_t i = first + k % count;
    hipError_t e;
    if (k >= count && (e = hipEventSynchronize(done[i])) != hipSuccess) return e;
    std::memcpy(pin + i * slot_bytes, host + at, len);
    if ((e = hipMemcpyAsync(dev + at, pin + i * slot_bytes, len, hipMemcpyHostToDevice, s)) != hipSuccess) return e;
    if (at + chunk * count < bytes && (e = hipEventRecord(done[i], s)) != hipSuccess) return e;  // (a later chunk waits)
  }
  return hipSuccess;
}

hipError_t HostStage::download_part(unsigned char* host, const unsigned char* dev, uint64_t bytes, uint64_t chunk,
                                    uint32_t first, uint32_t count, hipStream_t s) {
  const uint32_t chunks = (uint32_t)((bytes + chunk - 1) / chunk);
  auto length = [&](uint32_t k) { return std::min(chunk, bytes - (uint64_t)k * chunk); };
  auto queue = [&](uint32_t k) {
    const uint32_t i = first + k % count;
    const hipError_t e = hipMemcpyAsync(pin + i * slot_bytes, dev + (uint64_t)k * chunk, length(k),
                                        hipMemcpyDeviceToHost, s);
    return e != hipSuccess ? e : hipEventRecord(done[i], s);
  };
  hipError_t e;
  if (chunks == 1) {
    if ((e = hipMemcpyAsync(pin + first * slot_bytes, dev, bytes, hipMemcpyDeviceToHost, s)) != hipSuccess) return e;
    if ((e = hipStreamSynchronize(s)) != hipSuccess) return e;
    std::memcpy(host, pin + first * slot_bytes, bytes);
    return hipSuccess;
  }
  for (uint32_t k = 0; k < std::min(chunks, count); ++k)
    if ((e = queue(k)) != hipSuccess) return e;
  for (uint32_t k = 0; k < chunks; ++k) {
    const uint32_t i = first + k % count;
    if ((e = hipEventSynchronize(done[i])) != hipSuccess) return e;
    std::memcpy(host + (uint64_t)k * chunk, pin + i * slot_bytes, length(k));
    if (k + count < chunks && (e = queue(k + count)) != hipSuccess) return e;
  }
  return hipSuccess;
}

// Long transfers in `parts` parts, all but the first by threads of this call
// (one thread copies 12.6 MB in 220 us into pinned memory and in 420 us out of
// it, about as long as the device takes), through their own slots.
template <class Part>
hipError_t HostStage::in_parts(uint64_t bytes, Part part) {
  const uint32_t parts = !threaded(bytes) ? 1u : (bytes < kFour ? 2u : 4u);
  const uint64_t share = (bytes / parts + 255) / 256 * 256;
  const uint32_t count = nslots / parts;
  const uint64_t chunk = slot_bytes;
  std::thread threads[3];
  hipError_t e[4] = {hipSuccess, hipSuccess, hipSuccess, hipSuccess};
  auto run = [&](uint32_t t) {
    const uint64_t at = t * share, len = t + 1 == parts ? bytes - at : share;
    e[t] = part(at, len, chunk, t * count, count);
  };
  for (uint32_t t = 1; t < parts; ++t) {
    try {
      threads[t - 1] = std::thread([&, t] {
        if ((e[t] = hipSetDevice(device)) == hipSuccess) run(t);
      });
    } catch (...) {  // no thread to be had
      run(t);
    }
  }
  run(0);
  for (std::thread& t : threads)
    if (t.joinable()) t.join();
  for (hipError_t x : e)
    if (x != hipSuccess) return x;
  return hipSuccess;
}

// What a small object's few slots do not hold (many samples of a warm-start
// model) would go through them chunk by chunk with a wait for each: 4 MB of
// samples took 360 us through one slot of 1 MB, 160 by the runtime.  (A second
// round of two slots is about as fast as the runtime's copies of 1 to 2 MB,
// which take 400 us where the caller makes and gives back an array a call.)
int HostStage::upload(void* dev, const void* host, uint64_t bytes, hipStream_t s, uint32_t slot) {
  if (slot)
    return check_hip(upload_part((unsigned char*)dev, (const unsigned char*)host, bytes, slot_bytes, slot, nslots - slot, s),
                     "upload");
  if (!fits(bytes)) return check_hip(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s), "upload");
  return check_hip(in_parts(bytes, [&](uint64_t at, uint64_t len, uint64_t chunk, uint32_t first, uint32_t count) {
                     return upload_part((unsigned char*)dev + at, (const unsigned char*)host + at, len, chunk, first,
                                        count, s);
                   }), "upload");
}

int HostStage::download(void* host, const void* dev, uint64_t bytes, hipStream_t s) {
  if (!fits(bytes)) {
    const int rc = check_hip(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s), "download");
    return rc ? rc : check_hip(hipStreamSynchronize(s), "download");
  }
  return check_hip(in_parts(bytes, [&](uint64_t at, uint64_t len, uint64_t chunk, uint32_t first, uint32_t count) {
                     return download_part((unsigned char*)host + at, (const unsigned char*)dev + at, len, chunk, first,
                                          count, s);
                   }), "download");
}

}  // namespace pbf
