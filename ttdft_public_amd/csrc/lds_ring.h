// Device helpers of kernels that keep a ring of LDS stages filled by
// global->LDS loads while earlier stages are multiplied.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ttdft {

typedef __attribute__((address_space(3))) void lds_void;

// s_waitcnt immediate: vmcnt in bits [3:0] and [15:14], expcnt [6:4], lgkmcnt [11:8].
// Waits until at most n vector-memory operations of this wave are outstanding
// and all LDS operations are done.
#define TT_WAIT_VM_LDS(n)                                                                   \
    do {                                                                                    \
        asm volatile("" ::: "memory");                                                      \
        __builtin_amdgcn_s_waitcnt(((n) & 15) | ((((n) >> 4) & 3) << 14) | (7 << 4) | (0 << 8)); \
    } while (0)
#define TT_WAIT_ALL() __builtin_amdgcn_s_waitcnt(0)

// Workgroup barrier without the memory fence of __syncthreads(): that fence
// would also wait for the loads still in flight into LDS.  The waits the
// barrier needs are issued explicitly before it; the empty asm keeps the
// compiler from moving memory operations across.
__device__ __forceinline__ void line_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// One 16-byte load per lane from p straight into LDS at dst + 16 lane.
__device__ __forceinline__ void load_lds_16(const void *p, void *dst) {
#if defined(__HIP_DEVICE_COMPILE__)
    // (the host pass of a .hip file rejects the 16-byte form of this builtin)
    __builtin_amdgcn_global_load_lds(p, (lds_void *)dst, 16, 0, 0);
#else
    (void)p;
    (void)dst;
#endif
}

// LDS byte address of a shared-memory pointer
__device__ __forceinline__ unsigned lds_addr(const void *p) { return (unsigned)(uintptr_t)p; }

// Two, three or four 16-byte LDS loads from the given addresses (plus
// offsets), completed inside the asm block; every output is used by the
// caller.  Outputs are early-clobber: a load may return while a later load
// still reads an address register.  Written as asm because the compiler
// cannot tell these reads apart from the global->LDS loads into the other
// stages and would otherwise wait for all of those first.
typedef float v4f_t __attribute__((ext_vector_type(4)));

template <int O1, int O2>
__device__ __forceinline__ void lds_read3(unsigned a, v4f_t &x, v4f_t &y, v4f_t &z) {
    asm volatile("ds_read_b128 %0, %3\n\tds_read_b128 %1, %3 offset:%4\n\t"
                 "ds_read_b128 %2, %3 offset:%5\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(x), "=&v"(y), "=&v"(z)
                 : "v"(a), "i"(O1), "i"(O2));
}
__device__ __forceinline__ void lds_read4(unsigned a, unsigned b, unsigned c, unsigned d, v4f_t &x,
                                          v4f_t &y, v4f_t &z, v4f_t &w) {
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %6\n\t"
                 "ds_read_b128 %3, %7\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(x), "=&v"(y), "=&v"(z), "=&v"(w)
                 : "v"(a), "v"(b), "v"(c), "v"(d));
}

}  // namespace ttdft
