// Internal to libusagi_bsa.so: the error state shared by its translation units.
#ifndef USAGI_BSA_INTERNAL_H
#define USAGI_BSA_INTERNAL_H

// Records a formatted message for usagi_bsa_last_error() on the calling thread; returns code.
__attribute__((visibility("hidden"), format(printf, 2, 3))) int usagi_bsa_fail(int code,
                                                                               const char* fmt,
                                                                               ...);

// Empties the calling thread's message (every entry point starts with it).
__attribute__((visibility("hidden"))) void usagi_bsa_clear_error(void);

// A kernel of bsa_ksplit.hip and its workgroup size.
struct SmallKernel {
  const void* fn;
  unsigned threads;
};

// The kernel for a dtype, a row source (kRows of bsa_device.h) and 32, 64 or 128 query rows per
// workgroup.
__attribute__((visibility("hidden"))) SmallKernel usagi_bsa_small_kernel(bool bf16, int rows,
                                                                         int query_rows);

#endif  // USAGI_BSA_INTERNAL_H
