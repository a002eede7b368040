// Loads that go from global memory to LDS without passing through registers, and LDS reads that
// transpose on the way out (gfx950).
//
// The DMA is issued from an asm statement and waited for by one: the compiler's own counting knows
// nothing of it, which is what a pipeline of several stages needs (it would put a wait for
// everything in flight in front of every LDS read that may alias a stage).  No register receives
// anything, so there is nothing for the compiler to reuse too early; the address is read at issue.
// (Other passes than the device's: the same effect by copies.)
#ifndef K_LDS_DMA_H
#define K_LDS_DMA_H

#if defined(__HIP_DEVICE_COMPILE__)
#define NCHIP_LDS __attribute__((address_space(3)))
#else
#define NCHIP_LDS
#endif

typedef short lds_short4 __attribute__((ext_vector_type(4)));

// 16 bytes per lane: lane l's from base + off go to lds + 16 l bytes.  lds and base are the same in
// all lanes of the wavefront; every lane takes part.
__device__ __forceinline__ void lds_dma16(uint16_t NCHIP_LDS *lds, const void *base, uint32_t off)
{
#if defined(__HIP_DEVICE_COMPILE__)
    const uint32_t at = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)lds);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)base);
    const uint32_t up = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uintptr_t)base >> 32));
    uint64_t from;
    uint32_t m0; // (an output, for the compiler to know: it warns of a clobber, the register being reserved)
    // (the base is copied by the scalar unit: a vector instruction's scalar result may not be read by
    // a memory instruction right behind it; the copy is also the slot that the load needs after m0)
    asm volatile("s_mov_b32 m0, %2\n\ts_mov_b64 %0, %3\n\tglobal_load_lds_dwordx4 %4, %0"
                 : "=&s"(from), "={m0}"(m0) : "s"(at), "s"((uint64_t)lo | (uint64_t)up << 32), "v"(off) : "memory");
#else
    memcpy(lds + 8 * (threadIdx.x & 63), (const char *)base + off, 16);
#endif
}

// The same from 64-bit offsets, for rows more than 4 GiB apart.
__device__ __forceinline__ void lds_dma16(uint16_t NCHIP_LDS *lds, const void *base, uint64_t off)
{
#if defined(__HIP_DEVICE_COMPILE__)
    const uint32_t at = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)lds);
    uint32_t m0;
    // (the wait is the slot that the load needs after m0)
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off"
                 : "={m0}"(m0) : "s"(at), "v"((uint64_t)(uintptr_t)base + off) : "memory");
#else
    memcpy(lds + 8 * (threadIdx.x & 63), (const char *)base + off, 16);
#endif
}

// Waits until at most LEFT of this wavefront's vector-memory instructions are in flight (they
// complete in order) and its LDS reads are done, then for the other wavefronts of the workgroup.
template <int LEFT>
__device__ __forceinline__ void lds_dma_barrier()
{
    static_assert(LEFT >= 0 && LEFT <= 63, "six bits");
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(LEFT) : "memory");
#else
    __syncthreads();
#endif
}

// Four 16-bit values of one column: the 16 lanes of a row of lanes address 4 rows of 16 values, lane
// 4 r + c the values 4 c .. 4 c + 3 of row r, and lane j receives value j of the four rows.
__device__ __forceinline__ uint2 lds_read_columns(const uint16_t NCHIP_LDS *p)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4 NCHIP_LDS *)p));
#else
    uint32_t w[2];
    memcpy(w, p, 8);
    uint16_t r[4];
    const int lane = threadIdx.x & 63;
    for (int row = 0; row < 4; row++) {
        const int from = (lane & 48) + 4 * row + ((lane & 15) >> 2);
        const uint32_t lo = __shfl(w[0], from, 64), hi = __shfl(w[1], from, 64);
        r[row] = (uint16_t)((lane & 2 ? hi : lo) >> (lane & 1) * 16);
    }
    return make_uint2(r[0] | (uint32_t)r[1] << 16, r[2] | (uint32_t)r[3] << 16);
#endif
}

#endif
