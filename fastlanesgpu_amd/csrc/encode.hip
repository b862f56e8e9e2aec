// GPU encoders: FastLanes bit-packing (plain or transposed), FastLanes delta
// and FastLanes RLE, each as plan -> scan -> pack over device buffers.
//
// Work-item t of a 256-work-item block serves lane t%32 of vector
// blockIdx.x*8 + t/32.  All of them read their vector in the coalesced layout
// of fls_rows.hpp (two whole lines per load instruction) and are bound by that
// read: the transposed bit-pack and the delta pack then move the values to
// their owning lanes through an LDS tile, the plans and the RLE pack need only
// neighbour-lane comparisons.
#include "fls/device/unpack.hpp"
#include "fls/device/wave.hpp"
#include "fls_encode.hpp"
#include "fls_pack.hpp"
#include "fls_rows.hpp"
#include "fls_runtime.hpp"
#include "fls_scan.hpp"

namespace fls {
namespace {

constexpr int kBlock = 256;
constexpr int kVecPerBlock = kBlock / 32;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------ bitpack
// Rows 32j + l of vector v minus base, rows past n zero (loaded as the last row
// and then cleared: a load under a condition is waited for before the next one,
// 32 round trips, and 100,003 values not read before took 14.0 us instead of 6.2).
// In normal order these are the lane's own rows; TRANSPOSED sends them through the LDS tile
// (the lane's row rsum_row(j) is element j of its chain).
template <int BW, bool TRANSPOSED>
__global__ __launch_bounds__(kBlock) void pack_kernel(const uint32_t* __restrict in, uint64_t n, uint32_t base,
                                                       uint32_t* __restrict out) {
    __shared__ uint32_t tile[TRANSPOSED ? kVecPerBlock : 1][TRANSPOSED ? kTile : 1];
    const uint64_t v = (uint64_t)blockIdx.x * kVecPerBlock + (threadIdx.x >> 5);
    const bool live = v * 1024u < n;
    const uint32_t l = dev::lane32();
    uint32_t x[32];
    if (live) {
        const uint64_t i0 = v * 1024u + l;
        if (v * 1024u + 1024u <= n) {
#pragma unroll
            for (int r = 0; r < 32; ++r) x[r] = __builtin_nontemporal_load(in + i0 + 32u * r) - base;
        } else {
#pragma unroll
            for (int r = 0; r < 32; ++r) x[r] = padded(in, n, i0 + 32u * r) - base;
#pragma unroll
            for (int r = 0; r < 32; ++r) x[r] = i0 + 32u * r < n ? x[r] : 0u;
        }
    }
    if constexpr (TRANSPOSED) {
        uint32_t* t = tile[threadIdx.x >> 5];
        if (live) rows_to_tile(x, t);
        wave_sync();
        const uint32_t c = chain_slot(l);
        if (live) {
#pragma unroll
            for (int j = 0; j < 32; ++j) x[dev::rsum_row(j)] = t[33 * c + j];
        }
    }
    if (live) pack_lane<BW>(x, out + v * (32u * BW));
}

// ------------------------------------------------------------------- delta
// Per vector: the width of its largest in-chain difference (chain start 0)
// and the 32 chain starts.  The starts sit in lane 0 and reach their lanes
// through 32 words of LDS.
__global__ __launch_bounds__(kBlock) void delta_plan_kernel(const uint32_t* __restrict in, uint64_t n,
                                                            uint64_t n_vec, uint32_t* __restrict bws,
                                                            uint32_t* __restrict words, uint32_t* __restrict bases,
                                                            ScanState state) {
    __shared__ __align__(16) uint32_t first[kVecPerBlock][32];
    scan_clear(state);
    const uint64_t v = (uint64_t)blockIdx.x * kVecPerBlock + (threadIdx.x >> 5);
    if (v >= n_vec) return;
    const uint32_t l = dev::lane32();
    uint32_t* f = first[threadIdx.x >> 5];
    uint32_t x[32], dor = 0;
    load_rows(in, n, v, x);
#pragma unroll
    for (int j = 0; j < 32; ++j) {
        const uint32_t up = dpp<kWaveShr1>(x[j]);  // element l-1 of chain j
        dor |= l ? x[j] - up : 0u;
    }
    if (l == 0) {
#pragma unroll
        for (int j = 0; j < 32; j += 4)
            *reinterpret_cast<u32x4*>(f + j) = u32x4{x[j], x[j + 1], x[j + 2], x[j + 3]};
    }
    const uint32_t bw = wid(h_or(dor));
    wave_sync();
    bases[v * 32u + l] = f[chain_slot(l)];
    if (l == 0) {
        bws[v] = bw;
        words[v] = 32u * bw;
    }
}

__global__ __launch_bounds__(kBlock) void delta_pack_kernel(const uint32_t* __restrict in, uint64_t n,
                                                            uint64_t n_vec, const fls_vmeta* __restrict vmeta,
                                                            uint32_t* __restrict out) {
    __shared__ uint32_t tile[kVecPerBlock][kTile];
    const uint64_t v = (uint64_t)blockIdx.x * kVecPerBlock + (threadIdx.x >> 5);
    const bool live = v < n_vec;
    uint32_t* t = tile[threadIdx.x >> 5];
    uint32_t x[32];
    fls_vmeta m = 0;
    if (live) {
        m = vmeta[v];
        load_rows(in, n, v, x);
        rows_to_tile(x, t);
    }
    wave_sync();
    if (!live) return;
    const uint32_t* chain = t + 33u * chain_slot(dev::lane32());
    uint32_t d[32];
    uint32_t prev = chain[0];
    d[0] = 0u;
#pragma unroll
    for (int j = 1; j < 32; ++j) {
        const uint32_t y = chain[j];
        d[dev::rsum_row(j)] = y - prev;
        prev = y;
    }
    pack_rows(d, out + FLS_VMETA_OFFSET(m), FLS_VMETA_BW(m));
}

// --------------------------------------------------------------------- RLE
// Run starts in original order, a ballot per chain: f(j, m, before) gets the
// chain's 32 start flags (bit e = element e starts a run), the same in every
// lane of the half-wave, and the number of runs started before the chain.
// Returns the vector's run count.
template <typename F>
__device__ __forceinline__ uint32_t rle_chains(const uint32_t (&x)[32], F&& f) {
    const uint32_t l = dev::lane32();
    const bool hi = (threadIdx.x & 32u) != 0;
    uint32_t before = 0, last = 0;
#pragma unroll
    for (int j = 0; j < 32; ++j) {
        const uint32_t up = dpp<kWaveShr1>(x[j]);  // element l-1 of chain j
        const bool st = l ? x[j] != up : (j == 0 || x[j] != last);
        const uint64_t b = __ballot(st);
        const uint32_t m = hi ? (uint32_t)(b >> 32) : (uint32_t)b;
        f(j, m, before);
        before += __builtin_popcount(m);
        const uint32_t e0 = (uint32_t)__builtin_amdgcn_readlane((int)x[j], 31);
        const uint32_t e1 = (uint32_t)__builtin_amdgcn_readlane((int)x[j], 63);
        last = hi ? e1 : e0;  // element 31 of chain j
    }
    return before;
}

__global__ __launch_bounds__(kBlock) void rle_plan_kernel(const uint32_t* __restrict in, uint64_t n, uint64_t n_vec,
                                                          uint32_t* __restrict words, fls_rle_meta* __restrict rmeta,
                                                          uint32_t* __restrict bases, uint32_t* __restrict ibws,
                                                          ScanState state) {
    __shared__ uint32_t first[kVecPerBlock][32];
    scan_clear(state);
    const uint64_t v = (uint64_t)blockIdx.x * kVecPerBlock + (threadIdx.x >> 5);
    if (v >= n_vec) return;
    const uint32_t l = dev::lane32();
    uint32_t* f = first[threadIdx.x >> 5];
    uint32_t x[32], vmin = 0xffffffffu, vmax = 0u, inner = 0u;
    load_rows(in, n, v, x);
#pragma unroll
    for (int j = 0; j < 32; ++j) {
        vmin = min(vmin, x[j]);
        vmax = max(vmax, x[j]);
    }
    const uint32_t n_runs = rle_chains(x, [&](int j, uint32_t m, uint32_t before) {
        if (l == 0) f[j] = before + (m & 1u) - 1u;  // run index of the chain's first row
        inner |= m & ~1u;
    });
    vmin = h_min(vmin);
    vmax = h_max(vmax);
    const uint32_t ibw = inner ? 1u : 0u;
    const uint32_t vbw = wid(vmax - vmin);
    wave_sync();
    bases[v * 32u + l] = f[chain_slot(l)];
    if (l == 0) {
        rmeta[v] = fls_rle_meta{vmin, (uint16_t)n_runs, (uint8_t)vbw, (uint8_t)ibw};
        words[v] = 32u * ibw + (n_runs * vbw + 31u) / 32u;
        ibws[v] = ibw;
    }
}

// Bit e of the low byte to bit 4e.
__device__ __forceinline__ uint32_t spread4(uint32_t b) {
    b = (b | (b << 12)) & 0x000f000fu;
    b = (b | (b << 6)) & 0x03030303u;
    return (b | (b << 3)) & 0x11111111u;
}

// A chain's start flags in element order to its index word: element e sits in
// row rsum_row(e) = 4 (e % 8) + {0, 2, 1, 3}[e / 8]; the chain's first element
// always has difference 0.
__device__ __forceinline__ uint32_t index_word(uint32_t m) {
    m &= ~1u;
    return spread4(m & 255u) | (spread4((m >> 8) & 255u) << 2) | (spread4((m >> 16) & 255u) << 1) |
           (spread4(m >> 24) << 3);
}

__global__ __launch_bounds__(kBlock) void rle_pack_kernel(const uint32_t* __restrict in, uint64_t n, uint64_t n_vec,
                                                          const fls_vmeta* __restrict vmeta,
                                                          const fls_rle_meta* __restrict rmeta,
                                                          uint32_t* __restrict out) {
    __shared__ uint32_t vals[kVecPerBlock][1024];  // run values by run index
    __shared__ uint32_t starts[kVecPerBlock][32];  // start flags by chain
    const uint64_t v = (uint64_t)blockIdx.x * kVecPerBlock + (threadIdx.x >> 5);
    if (v >= n_vec) return;  // every exchange below stays inside the half-wave
    const uint32_t l = dev::lane32();
    uint32_t* val = vals[threadIdx.x >> 5];
    uint32_t* msk = starts[threadIdx.x >> 5];
    uint32_t x[32];
    const fls_vmeta m = vmeta[v];
    const fls_rle_meta rm = rmeta[v];
    load_rows(in, n, v, x);
    const uint32_t upto = (2u << l) - 1u;  // elements 0..l
    rle_chains(x, [&](int j, uint32_t mj, uint32_t before) {
        if ((mj >> l) & 1u) val[before + __builtin_popcount(mj & upto) - 1u] = x[j];
        if (l == 0) msk[j] = mj;
    });
    wave_sync();
    uint32_t* vec_out = out + FLS_VMETA_OFFSET(m);
    const uint32_t ibw = FLS_VMETA_BW(m);
    if (ibw) vec_out[l] = index_word(msk[chain_slot(l)]);
    // linear LSB-first packing of (value - vbase) at vbw bits after the index
    // words; lane l builds words l, l+32, ...
    uint32_t* vals_out = vec_out + 32u * ibw;
    const uint32_t vbw = rm.vbw, nr = rm.n_runs;
    const uint32_t n_words = (nr * vbw + 31u) / 32u;
    for (uint32_t w = l; w < n_words; w += 32u) {
        uint32_t word = 0;
        const uint32_t bit0 = 32u * w;
        const uint32_t k0 = bit0 / vbw, k1 = min(nr - 1u, (bit0 + 31u) / vbw);
        for (uint32_t k = k0; k <= k1; ++k) {
            const uint32_t kb = k * vbw;  // first bit of value k
            const uint32_t y = val[k] - rm.vbase;
            if (kb >= bit0) {
                if (kb - bit0 < 32u) word |= y << (kb - bit0);
            } else {
                word |= y >> (bit0 - kb);
            }
        }
        vals_out[w] = word;
    }
}

// The planners' words and widths to offsets: see scan_vectors.
__global__ __launch_bounds__(kScanBlock) void scan_kernel(const uint32_t* __restrict words,
                                                          const uint32_t* __restrict bws, uint64_t n,
                                                          unsigned long long* __restrict state,
                                                          fls_vmeta* __restrict vmeta, uint64_t* __restrict total_out,
                                                          uint32_t* __restrict flagged) {
    scan_vectors([&](uint64_t i, uint32_t& w, uint32_t& bw) { w = words[i], bw = bws[i]; }, n, state, vmeta, total_out,
                 flagged);
}

template <bool TRANSPOSED>
struct PackTable {
    using Fn = void (*)(const uint32_t*, uint64_t, uint32_t, uint32_t*);
    template <int... B>
    static constexpr auto make(std::integer_sequence<int, B...>) {
        return std::array<Fn, sizeof...(B)>{&pack_kernel<B, TRANSPOSED>...};
    }
    static constexpr auto table = make(std::make_integer_sequence<int, 33>{});
};

}  // namespace

uint64_t scratch_words(uint64_t n_vec) {
    // bws[n_vec] + words[n_vec] (u32), then 8 bytes per 1,024 vectors, 256-byte
    // aligned: the scan's state (a sum per 1,024 vectors; its ticket is in the slack)
    const uint64_t nb = ceil_div(n_vec ? n_vec : 1, 1024);
    return ((2 * n_vec * 4 + 255) / 256 * 256 + nb * 8 + 255) / 4;
}

EncodeScratch encode_scratch(void* d_scratch, uint64_t n_vec) {
    EncodeScratch e;
    e.bws = static_cast<uint32_t*>(d_scratch);
    e.words = e.bws + n_vec;
    e.state.p = reinterpret_cast<unsigned long long*>(static_cast<char*>(d_scratch) + (2 * n_vec * 4 + 255) / 256 * 256);
    e.state.n = (uint32_t)(ceil_div(n_vec, kScanChunk) + 1);
    e.state.ticket = scan_ticket_word(n_vec);
    return e;
}

int scan_offsets(const EncodeScratch& e, uint64_t n_vec, fls_vmeta* vmeta, uint64_t* d_total, hipStream_t s,
                 uint32_t* d_flagged) {
    hipLaunchKernelGGL(scan_kernel, dim3(e.state.n - 1u), dim3(kScanBlock), 0, s, e.words, e.bws, n_vec, e.state.p,
                       vmeta, d_total, d_flagged);
    return check_launch();
}

}  // namespace fls

extern "C" {

uint64_t fls_encode_scratch_bytes(uint64_t n) { return 4u * fls::scratch_words(fls::ceil_div(n, 1024)); }

int fls_pack_column_device(const uint32_t* d_in, uint64_t n, uint32_t bw, uint32_t base, uint32_t flags,
                           uint32_t* d_out, void* stream) {
    using namespace fls;
    FLS_RETURN_IF(bw > 32, FLS_ERR_BW);
    if (n == 0 || bw == 0) return FLS_OK;
    FLS_RETURN_IF(!d_in || !d_out, FLS_ERR_NULL);
    const uint64_t blocks = ceil_div(ceil_div(n, 1024), kVecPerBlock);
    FLS_RETURN_IF(blocks > 0x7fffffffu, FLS_ERR_SIZE);
    auto fn = (flags & FLS_ENC_FLAG_TRANSPOSE) ? PackTable<true>::table[bw] : PackTable<false>::table[bw];
    hipLaunchKernelGGL(fn, dim3((uint32_t)blocks), dim3(kBlock), 0, as_stream(stream), d_in, n, base, d_out);
    return check_launch();
}

int fls_delta_plan_device(const uint32_t* d_in, uint64_t n, fls_vmeta* d_vmeta, uint32_t* d_bases,
                          uint64_t* d_total_words, void* d_scratch, void* stream) {
    using namespace fls;
    if (n == 0) return zero_u64(d_total_words, 1, as_stream(stream));
    FLS_RETURN_IF(!d_in || !d_vmeta || !d_bases || !d_total_words || !d_scratch, FLS_ERR_NULL);
    const uint64_t n_vec = ceil_div(n, 1024), blocks = ceil_div(n_vec, kVecPerBlock);
    FLS_RETURN_IF(blocks > 0x7fffffffu, FLS_ERR_SIZE);
    const EncodeScratch e = encode_scratch(d_scratch, n_vec);
    hipStream_t s = as_stream(stream);
    hipLaunchKernelGGL(delta_plan_kernel, dim3((uint32_t)blocks), dim3(kBlock), 0, s, d_in, n, n_vec, e.bws, e.words,
                       d_bases, e.state);
    if (const int rc = check_launch()) return rc;
    return scan_offsets(e, n_vec, d_vmeta, d_total_words, s);
}

int fls_delta_pack_device(const uint32_t* d_in, uint64_t n, const fls_vmeta* d_vmeta, uint32_t* d_out,
                          void* stream) {
    using namespace fls;
    if (n == 0) return FLS_OK;
    FLS_RETURN_IF(!d_in || !d_vmeta || !d_out, FLS_ERR_NULL);
    const uint64_t n_vec = ceil_div(n, 1024);
    hipLaunchKernelGGL(delta_pack_kernel, dim3((uint32_t)ceil_div(n_vec, kVecPerBlock)), dim3(kBlock), 0,
                       as_stream(stream), d_in, n, n_vec, d_vmeta, d_out);
    return check_launch();
}

int fls_rle_plan_device(const uint32_t* d_in, uint64_t n, fls_vmeta* d_vmeta, fls_rle_meta* d_rmeta,
                        uint32_t* d_bases, uint64_t* d_total_words, void* d_scratch, void* stream) {
    using namespace fls;
    if (n == 0) return zero_u64(d_total_words, 1, as_stream(stream));
    FLS_RETURN_IF(!d_in || !d_vmeta || !d_rmeta || !d_bases || !d_total_words || !d_scratch, FLS_ERR_NULL);
    const uint64_t n_vec = ceil_div(n, 1024), blocks = ceil_div(n_vec, kVecPerBlock);
    FLS_RETURN_IF(blocks > 0x7fffffffu, FLS_ERR_SIZE);
    const EncodeScratch e = encode_scratch(d_scratch, n_vec);
    hipStream_t s = as_stream(stream);
    hipLaunchKernelGGL(rle_plan_kernel, dim3((uint32_t)blocks), dim3(kBlock), 0, s, d_in, n, n_vec, e.words, d_rmeta,
                       d_bases, e.bws, e.state);
    if (const int rc = check_launch()) return rc;
    return scan_offsets(e, n_vec, d_vmeta, d_total_words, s);
}

int fls_rle_pack_device(const uint32_t* d_in, uint64_t n, const fls_vmeta* d_vmeta, const fls_rle_meta* d_rmeta,
                        uint32_t* d_out, void* stream) {
    using namespace fls;
    if (n == 0) return FLS_OK;
    FLS_RETURN_IF(!d_in || !d_vmeta || !d_rmeta || !d_out, FLS_ERR_NULL);
    const uint64_t n_vec = ceil_div(n, 1024);
    hipLaunchKernelGGL(rle_pack_kernel, dim3((uint32_t)ceil_div(n_vec, kVecPerBlock)), dim3(kBlock), 0,
                       as_stream(stream), d_in, n, n_vec, d_vmeta, d_rmeta, d_out);
    return check_launch();
}

}  // extern "C"
