// launch.hpp — grid sizing and vector types shared by the ahead-of-time
// streaming kernels.
//
// Every streaming kernel here is written so that each store instruction of a
// wave writes one contiguous 1 KiB span (64 lanes x 16 bytes): on MI355X a
// wave that interleaves two 16-byte stores per lane (lane j writing bytes
// 32j..32j+15 and then 32j+16..32j+31) ran 15-20% slower on a 1:2
// read:write stream than the contiguous form.
#ifndef MFH_LAUNCH_HPP
#define MFH_LAUNCH_HPP

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "common.hpp"
#include "codec.hpp"

namespace mfh {

typedef mfh_u32 u32x4 __attribute__((ext_vector_type(4)));
typedef mfh_u32 u32x2 __attribute__((ext_vector_type(2)));

// The same values in memory at any byte address.  Global loads and stores of
// 2 to 16 bytes work at any alignment on gfx950 (one instruction, as for an
// aligned address), so row slices, odd widths and tensors inside a file image
// take the kernels' whole-item paths like any other buffer.
typedef mfh_u32 u32x4_any __attribute__((ext_vector_type(4), aligned(1)));
typedef mfh_u32 u32x2_any __attribute__((ext_vector_type(2), aligned(1)));
typedef mfh_u32 u32_any __attribute__((aligned(1)));
typedef mfh_u16 u16_any __attribute__((aligned(1)));

constexpr int kBlock = 256;  // 4 wave64 per workgroup: families without a size setting

// Grid for `items` work items of `per_thread` items each in workgroups of
// `block` threads, capped at compute_units * blocks_per_cu(k); threads loop
// over the rest.  A dispatch counts its work-items in 32 bits, so grids stay
// below 2^32 / block.
inline unsigned grid_for(int64_t items, const Device* dev, Kern k, int per_thread = 1, int block = kBlock)
{
    int64_t threads = (items + per_thread - 1) / per_thread;
    int64_t need = (threads + block - 1) / block;
    int64_t cap = std::min<int64_t>((int64_t)dev->compute_units * blocks_per_cu(k), (int64_t(1) << 32) / block - 1);
    return (unsigned)std::max<int64_t>(1, std::min(need, cap));
}

// Runs f(std::integral_constant<int, BS>{}) with BS the workgroup size
// `threads` (64, 128 or 256; anything else runs 256), so that a launcher
// picks the kernel instantiation and its grid from one reading of the
// family's setting.
template <typename F>
int with_block(int threads, F&& f)
{
    switch (threads) {
    case 64: return f(std::integral_constant<int, 64>{});
    case 128: return f(std::integral_constant<int, 128>{});
    default: return f(std::integral_constant<int, 256>{});
    }
}

// with_block, plus 512-thread workgroups for the one family that runs them
// (the Int4 dequant).
template <typename F>
int with_block_to_512(int threads, F&& f)
{
    if (threads == 512) return f(std::integral_constant<int, 512>{});
    return with_block(threads, std::forward<F>(f));
}

int launch_status(const char* what);

// Loads of 16, 8, 4 and 2 bytes, non-temporal (global_load ... nt) where NT.
// Non-temporal loads pay where a kernel reads at least as many bytes as it
// writes (+4% on a 1:1 stream and +8% on 2:1), and for the FP8 dequant (+0.6%
// with its codes coming from HBM); the Int4 dequant (-0.8%) and the widening
// casts keep plain loads.
template <bool NT>
__device__ inline u32x4 load16(const void* p)
{
    const u32x4_any* q = static_cast<const u32x4_any*>(p);
    if constexpr (NT) return __builtin_nontemporal_load(q);
    else return *q;
}

template <bool NT>
__device__ inline u32x2 load8(const void* p)
{
    const u32x2_any* q = static_cast<const u32x2_any*>(p);
    if constexpr (NT) return __builtin_nontemporal_load(q);
    else return *q;
}

__device__ inline mfh_u32 load4(const void* p) { return *static_cast<const u32_any*>(p); }
__device__ inline mfh_u32 load2(const void* p) { return *static_cast<const u16_any*>(p); }

// Streaming stores (global_store ... nt).
__device__ inline void store16(void* p, u32x4 v) { __builtin_nontemporal_store(v, static_cast<u32x4_any*>(p)); }
__device__ inline void store8(void* p, u32x2 v) { __builtin_nontemporal_store(v, static_cast<u32x2_any*>(p)); }
__device__ inline void store4(void* p, mfh_u32 v) { __builtin_nontemporal_store(v, static_cast<u32_any*>(p)); }
__device__ inline void store2(void* p, mfh_u32 v) { __builtin_nontemporal_store((mfh_u16)v, static_cast<u16_any*>(p)); }

// Streaming 16-byte stores of a chunk: buffer stores with the non-temporal
// (nt) and sc1 cache-policy bits, addressed from the chunk's first item (the
// base is uniform across the block, so the descriptor lives in SGPRs).  On
// MI355X, with the inputs coming from HBM, nt|sc1 stores run the FP8 dequant
// (1:2 read:write) at 6.1-6.2 TB/s and the Int4 dequant (1:4) at 6.0-6.1,
// against 5.8 and 5.5 with plain stores; nt alone is 1-2% slower, sc1 alone
// 4-6%.  The descriptor's record count is the chunk's remaining bytes, so the
// hardware drops anything past the end of the output.  A base that is not
// dword-aligned (DWORDS = false) takes global stores (nt), which any address
// allows.  The kernel is compiled for one of the two: choosing per store put
// branches and both stores' code into every item, 0.1-0.2 us of each call whose
// few workgroups wait for instruction fetches (Int4, groups of 128 -> bf16 on
// MI355X: 2^16 elements 2.26 us, 2.46 so; 2^22 elements 3.09, 3.29 so).
template <bool DWORDS>
struct StreamOut {
    char* at;
    int64_t left;
    __amdgpu_buffer_rsrc_t rsrc;
    __device__ StreamOut(char* base, int64_t items_left)
        : at(base), left(items_left),
          rsrc(__builtin_amdgcn_make_buffer_rsrc(
              base, 0, (int)std::min<int64_t>(items_left * 16, 0x7fffffff), kBufferConfig))
    {
    }
    __device__ void store(int item, u32x4 v) const
    {
        if constexpr (DWORDS) __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, item * 16, 0, kCachePolicy);
        else if (item < left) store16(at + (int64_t)item * 16, v);
    }
    // Word 3 of a raw (untyped) gfx9 buffer descriptor.
    static constexpr int kBufferConfig = 0x00020000;
    // gfx950 buffer cache policy: bit 1 nt, bit 4 sc1.
    static constexpr int kCachePolicy = 2 | 16;
};

}  // namespace mfh

#endif  // MFH_LAUNCH_HPP
