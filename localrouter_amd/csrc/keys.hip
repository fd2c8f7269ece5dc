// Key compaction for attention under a key-padding mask (Kandinsky-6's attention.Call with mask = .keys,
// src/engines/kandinsky6/dit/attention.zig:21-27: a u8 per key, nonzero = keep; SDPA's additive 0 / -inf mask). The
// kept keys and their value rows are gathered, in order, into a workspace, and the attention runs over them:
// softmax over the kept keys equals softmax over all keys with the others at -inf.
//
// One launch: a block owns a range of source keys and a 1 KB slab of their rows' columns. It counts the kept keys before
// its range (the mask is a few KB, read from L2), which gives its first output slot, then copies its kept rows, 16 bytes a
// thread, all of a thread's loads in flight together. Bound by HBM on the rows (700 of 1,024 keys x 32 heads: 23 MB) and,
// at that size, by the launch; a scan launch in front of the gather (one workgroup) cost 3.2 us and the gap between.
#include "lr_common.h"
#include "lr_kernels.h"

namespace lr {
namespace {

constexpr int GT = 256;           // threads
constexpr int KEYS = 16;          // source keys per pass of a block
constexpr int SLAB = 64;          // 16-byte chunks of a row per block: one wave a row, four rows at a time
constexpr int KEYS_PER_THREAD = KEYS / (GT / SLAB);

// nonzero bytes of a word, a bit each at bits 7, 15, 23, 31
__device__ __forceinline__ uint32_t nonzero_bytes(uint32_t w) {
    return (((w & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w) & 0x80808080u;
}

// Kept keys of kmask[0 .. n), by the whole block (every thread gets the sum).
__device__ __forceinline__ int count_kept(const uint8_t* kmask, int n, int* red) {
    const int t = threadIdx.x;
    int cnt = 0, i0 = 0;
    if ((reinterpret_cast<uintptr_t>(kmask) & 15) == 0) {   // 16 bytes a thread at a time
        i0 = n & ~15;
        for (int i = 16 * t; i < i0; i += 16 * GT) {
            const u32x4 w = *reinterpret_cast<const u32x4*>(kmask + i);
#pragma unroll
            for (int j = 0; j < 4; ++j) cnt += __popc(nonzero_bytes(w[j]));
        }
    }
    for (int i = i0 + t; i < n; i += GT) cnt += kmask[i] != 0;
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) cnt += __shfl_xor(cnt, m, 64);
    if ((t & 63) == 0) red[t >> 6] = cnt;
    __syncthreads();
    return red[0] + red[1] + red[2] + red[3];
}

// Block (x, y): source keys [x * per, (x + 1) * per), column chunks [y * SLAB, (y + 1) * SLAB). Slots past the last kept
// key (the mask holds fewer than n_valid: a caller error) get zero rows, from the last range's blocks; kept keys past
// n_valid are left out.
__global__ __launch_bounds__(GT) void gather_kept_kernel(const uint16_t* k, const uint16_t* v, int64_t kv_rs,
                                                         const uint8_t* kmask, int nkeys, int n_valid, int per,
                                                         int row_chunks, uint16_t* kc, uint16_t* vc) {
    __shared__ int red[GT / 64];
    const int t = threadIdx.x, r = t / SLAB, c = blockIdx.y * SLAB + t % SLAB;
    const bool live = c < row_chunks;
    const int b = blockIdx.x * per, e = min(nkeys, b + per);
    const int lane = t & 63;
    int slot0 = 0;
    for (int k0 = b; k0 < e; k0 += KEYS) {
        // the pass's mask: bit i = key k0 + i is kept (lanes 0 .. KEYS - 1 of every wave)
        const int km = lane < KEYS && k0 + lane < e ? kmask[k0 + lane] : 0;
        const uint32_t keep = (uint32_t)__builtin_amdgcn_ballot_w64(km != 0);
        u32x4 kk[KEYS_PER_THREAD], vv[KEYS_PER_THREAD];
#pragma unroll
        for (int j = 0; j < KEYS_PER_THREAD; ++j) {
            const int i = r + (GT / SLAB) * j;
            if (((keep >> i) & 1) && live) {
                const int64_t src = (int64_t)(k0 + i) * kv_rs + 8 * c;
                kk[j] = *reinterpret_cast<const u32x4*>(k + src);
                vv[j] = *reinterpret_cast<const u32x4*>(v + src);
            }
        }
        if (k0 == b) slot0 = count_kept(kmask, b, red);   // beside the first rows' loads
#pragma unroll
        for (int j = 0; j < KEYS_PER_THREAD; ++j) {
            const int i = r + (GT / SLAB) * j, slot = slot0 + __popc(keep & ((1u << i) - 1));
            if (((keep >> i) & 1) && live && slot < n_valid) {
                const int64_t dst = ((int64_t)slot * row_chunks + c) * 8;
                *reinterpret_cast<u32x4*>(kc + dst) = kk[j];
                *reinterpret_cast<u32x4*>(vc + dst) = vv[j];
            }
        }
        slot0 += __popc(keep);
    }
    if (e == nkeys && live)
        for (int s = slot0 + r; s < n_valid; s += GT / SLAB) {
            const int64_t dst = ((int64_t)s * row_chunks + c) * 8;
            *reinterpret_cast<u32x4*>(kc + dst) = u32x4{0u, 0u, 0u, 0u};
            *reinterpret_cast<u32x4*>(vc + dst) = u32x4{0u, 0u, 0u, 0u};
        }
}

}  // namespace

hipError_t launch_compact_keys(const void* k, const void* v, int64_t kv_rs, const uint8_t* kmask, int nkeys,
                               int n_valid, int HK, void* kc, void* vc, hipStream_t stream) {
    const int row_chunks = HK * D / 8;
    // 16 keys a block up to 8,192 keys; beyond, more passes a block rather than more counts of the mask before it
    const int per = KEYS * ((nkeys + 8191) / 8192);
    const dim3 grid((unsigned)((nkeys + per - 1) / per), (unsigned)((row_chunks + SLAB - 1) / SLAB));
    hipLaunchKernelGGL(gather_kept_kernel, grid, dim3(GT), 0, stream, static_cast<const uint16_t*>(k),
                       static_cast<const uint16_t*>(v), kv_rs, kmask, nkeys, n_valid, per, row_chunks,
                       static_cast<uint16_t*>(kc), static_cast<uint16_t*>(vc));
    return hipGetLastError();
}

}  // namespace lr
