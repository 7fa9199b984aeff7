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
// Qwen3's attention launch, with 64 workgroups that all read keys, lost by it (11 -> 21 us) and has none.
// Workgroup b of the launch that reads a region reads its bytes [b chunk, (b + 1) chunk).  Workgroups go round the eight
// XCDs in turn, each with an L2 of its own: what workgroup b will read is read on the XCD b % 8.  Only a hint: if the
// workgroups go elsewhere, the bytes are still nearer than HBM.
constexpr uint32_t kAheadRegions = 2;
constexpr uint64_t kAheadBytes = 24u << 20;  // three quarters of all L2s
struct RmiAhead {
    struct Region {
        const void *p;
        uint32_t chunk, n;  // chunk: a multiple of 16 bytes
    } r[kAheadRegions];
    uint32_t n_regions;
    uint64_t bytes;
    // as many of n chunks as still fit
    void add(const void *p, size_t chunk, uint32_t n) {
        if (n_regions == kAheadRegions || chunk == 0 || chunk % 16 || chunk > kAheadBytes) return;
        const uint64_t fit = (kAheadBytes - bytes) / chunk;
        r[n_regions] = {p, uint32_t(chunk), fit < n ? uint32_t(fit) : n};
        bytes += chunk * uint64_t(r[n_regions].n);
        n_regions++;
    }
};
// workgroups for it beside `used` others: a multiple of the XCDs
inline uint32_t rmi_ahead_blocks(const RmiAhead &a, uint32_t used, uint32_t cus) { return a.bytes && used < cus ? (cus - used) / 8 * 8 : 0; }

// One of the launch's last workgroups, those from `first` on (all of them with THREADS threads): a workgroup a chunk.
template <uint32_t THREADS>
__device__ __forceinline__ void fetch_ahead(const RmiAhead &a, uint32_t first) {
    typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
    constexpr uint32_t kLoads = 8;
    const uint32_t xcd = blockIdx.x % 8, unit = (blockIdx.x - first) / 8, units = (gridDim.x - first) / 8;
#pragma unroll
    for (uint32_t i = 0; i < kAheadRegions; i++) {
        const uint8_t *p = static_cast<const uint8_t *>(a.r[i].p);
        const uint32_t chunk = a.r[i].chunk, n = a.r[i].n;
        for (uint32_t b = unit * 8 + xcd; b < n; b += units * 8) {
            const uint8_t *c = p + size_t(b) * chunk;
            for (uint32_t o = threadIdx.x * 16; o < chunk; o += kLoads * THREADS * 16) {
                u32x4_t x[kLoads];
#pragma unroll
                for (uint32_t k = 0; k < kLoads; k++) {
                    const uint32_t at = o + k * THREADS * 16;
                    x[k] = *reinterpret_cast<const u32x4_t *>(c + (at < chunk ? at : o));
                }
#pragma unroll
                for (uint32_t k = 0; k < kLoads; k++) asm volatile("" ::"v"(x[k]));
            }
        }
    }
}

#endif  // RMI_DEVICE_AHEAD_H
