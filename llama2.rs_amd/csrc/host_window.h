// Device memory that the host writes over the bus: when its writes are there.
#pragma once
#include <emmintrin.h>
#include <stdint.h>

// What the calling thread has written through a mapping of device memory is in that memory when this returns, so that a kernel launched behind it
// reads it.  `flush` is the register that flushes the device's host data path (hipDeviceAttributeHdpMemFlushCntl).  The fence alone empties
// the processor's write-combining buffers into writes posted on the bus, and the launch says nothing of those: its packet is in host memory.
// The register is written behind them (posted writes to a device stay in order) and flushes what the data path still holds; it is read
// back, for a read passes no posted write and has its answer when all of them have arrived; mfence keeps the launch behind that answer.
// Takes 1.1 us (64 KB with the fence alone 1.6, with this 2.7; the last place written read back in the register's place 2.9), 1.4 of a call for one column of
// 4096x4096 (17.9 -> 19.3).
static inline void window_written(volatile uint32_t *flush) {
    _mm_sfence();
    *flush = 1;
    (void)*flush;
    _mm_mfence();
}
