// Weights that later launches read, brought into the caches by compute units that a launch leaves idle.
#ifndef RMI_DEVICE_AHEAD_H
#define RMI_DEVICE_AHEAD_H

#include <hip/hip_runtime.h>
#include <stdint.h>

// A token's mixers are a few workgroups that wait for memory; meanwhile HBM and most of the compute units idle, and the product
// behind them is bound by HBM.  So such a launch gets a workgroup more for every compute unit that the mixers leave, which read
// what comes next and drop it.  28 layers of width 1024 in bf16, 12.6 MB of output weights and 25 MB of the next layer's input
// weights a layer, us a token behind 16 | 512 | 2048 | 4096 keys (where the mixers are 16 to 144 workgroups):
//   nothing fetched                        578 | 643 | 749 | 804
//   16 MB, 128 workgroups at any context   530 | 597 | 711 | 774
//   24 MB, 192 workgroups                  519 | 580 | 707 | 781
//   24 MB, a workgroup a unit left         522 | 583 | 693 | 761
//   32 MB, a workgroup a unit left         545 | 574 | 710 | 765     (all of the L2s: what the mixers read goes, too)
// In f32 and at widths of 2048 and 4096 the kept setting is within 3 % of the best of the five, and no token is slower for it.
// Qwen3's attention launch, with 64 workgroups that all read keys, lost by as much (11 -> 21 us) and fetches a few MB only.
// Workgroup b of the launch that reads a region reads its bytes [b chunk, (b + 1) chunk).  Workgroups go round the eight
// XCDs in turn, each with an L2 of its own: what workgroup b will read is read on the XCD b % 8.  Only a hint: if the
// workgroups go elsewhere, the bytes are still nearer than HBM.
constexpr uint32_t kAheadRegions = 2;
constexpr uint64_t kAheadBytes = 24u << 20;  // three quarters of all L2s
struct RmiAhead {
    struct Region {
        const void *p;
        uint32_t chunk, n;   // chunk: a multiple of 16 bytes
        uint32_t magic;      // 2^31 by a chunk's pieces of 16 bytes, rounded up
    } r[kAheadRegions];
    uint32_t n_regions;
    uint64_t bytes;
    // as many of n chunks as still fit
    void add(const void *p, size_t chunk, uint32_t n) {
        if (n_regions == kAheadRegions || chunk == 0 || chunk % 16 || chunk > kAheadBytes) return;
        const uint64_t fit = (kAheadBytes - bytes) / chunk;
        r[n_regions] = {p, uint32_t(chunk), fit < n ? uint32_t(fit) : n, uint32_t((uint64_t(1) << 31) / (chunk / 16) + 1)};
        bytes += chunk * uint64_t(r[n_regions].n);
        n_regions++;
    }
};
// workgroups for it beside `used` others: a multiple of the XCDs
inline uint32_t rmi_ahead_blocks(const RmiAhead &a, uint32_t used, uint32_t cus) { return a.bytes && used < cus ? (cus - used) / 8 * 8 : 0; }

// One of the launch's last workgroups, those from `first` on (all of them with THREADS threads).  An XCD's pieces of 16 bytes go
// round its workgroups a thread's piece each, so that all of them have the same to read and wait as rarely as it allows.  With a
// workgroup a chunk, whose last loads read nothing new and whose number is no multiple of the workgroups': 28 layers as above,
// us a token at 16 | 150 | 300 | 700 | 2048 positions 529 | 536 | 546 | 550 | 636, by pieces 516 | 532 | 542 | 552 | 606;
// sixteen loads instead of eight before a wait, or the regions side by side, take as long or up to 2 % longer.
template <uint32_t THREADS>
__device__ __forceinline__ void fetch_ahead(const RmiAhead &a, uint32_t first) {
    typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
    constexpr uint32_t kLoads = 8;
    const uint32_t xcd = blockIdx.x % 8, at0 = (blockIdx.x - first) / 8 * THREADS, step = (gridDim.x - first) / 8 * THREADS;
#pragma unroll
    for (uint32_t r = 0; r < kAheadRegions; r++) {
        const uint32_t c16 = a.r[r].chunk / 16, pieces = (a.r[r].n + 7 - xcd) / 8 * c16;  // of the chunks xcd, xcd + 8, ...
        for (uint32_t i0 = at0; i0 < pieces; i0 += kLoads * step) {
            u32x4_t x[kLoads];
#pragma unroll
            for (uint32_t k = 0; k < kLoads; k++) {
                const uint32_t i = i0 + threadIdx.x + k * step, at = i < pieces ? i : pieces - 1;
                uint32_t c = __umulhi(2 * at, a.r[r].magic), o = at - c * c16;
                if (int32_t(o) < 0) c--, o += c16;  // (the quotient is at most one too large: at < 2^31)
                x[k] = *reinterpret_cast<const u32x4_t *>(static_cast<const uint8_t *>(a.r[r].p) + (size_t(c * 8 + xcd) * c16 + o) * 16);
            }
#pragma unroll
            for (uint32_t k = 0; k < kLoads; k++) asm volatile("" ::"v"(x[k]));
        }
    }
}

#endif  // RMI_DEVICE_AHEAD_H
