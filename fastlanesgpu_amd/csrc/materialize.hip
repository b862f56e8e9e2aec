// Untranspose and decode-to-materialize on the GPU.
//
// transpose_i / transpose_o (fastlanes/src/transpose.cpp:4110-5135 and the
// inverse that transpose.cpp:5136-6161 is meant to be) over whole 1024-value
// vectors: each vector is staged in LDS with coalesced loads and written back
// through the permutation with coalesced stores.
//
// fls_decode_column_u32 turns a compressed column of any encoding into plain
// values for a downstream operator (the role of Crystal's BlockStore,
// crystal-opt/store.cuh:57-69, after a decode): in the order the column is
// stored, or in original row order, which untransposes DELTA / RLE / MIXED /
// transposed BITPACK columns on the fly so they line up with plain columns.
#include "fls/device/unpack.hpp"
#include "fls/device/wave.hpp"
#include "fls_columns.hpp"
#include "fls_materialize.hpp"
#include "fls_rle.hpp"
#include "fls_runtime.hpp"

namespace fls {
namespace {

constexpr int kTrBlock = 256;                 // 4 waves, one vector each
constexpr int kTrVecs = kTrBlock / 64;
constexpr uint32_t kTrPad = 1024u + 64u;      // words per staged vector

// LDS slot of index k: four padding words per 64 keep 16-byte groups aligned
// and the strided gathers of the permutation on distinct banks.
__device__ __forceinline__ uint32_t tr_slot(uint32_t k) { return k + 4u * (k >> 6); }

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// A wave per vector: four 16-byte loads per work-item (a work-item holds
// words 4t + 256j .. +3) into LDS in stored order, then four 16-byte stores
// of four consecutive output words, each gathered from LDS through the
// permutation.  (One word per load and per store, 16 each, took 205 us over
// 117,188 vectors.)
template <bool INVERSE>
__global__ __launch_bounds__(kTrBlock) void transpose_kernel(const uint32_t* __restrict in, uint64_t n_vec,
                                                             uint32_t* __restrict out) {
    __shared__ __align__(16) uint32_t stage[kTrVecs][kTrPad];
    const uint32_t w = threadIdx.x >> 6, t = threadIdx.x & 63u;
    uint32_t* st = stage[w];
    for (uint64_t g = blockIdx.x; g * kTrVecs < n_vec; g += gridDim.x) {
        const uint64_t v = g * kTrVecs + w;
        if (v < n_vec) {  // wave-uniform: one vector per wave
            const u32x4* src = reinterpret_cast<const u32x4*>(in + v * 1024u);
            u32x4 x[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) x[j] = __builtin_nontemporal_load(src + t + 64u * j);
#pragma unroll
            for (int j = 0; j < 4; ++j) *reinterpret_cast<u32x4*>(st + tr_slot(4u * t + 256u * j)) = x[j];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (v < n_vec) {
            u32x4* dst = reinterpret_cast<u32x4*>(out + v * 1024u);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                u32x4 y;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t p = 4u * t + 256u * j + i;
                    // transpose_i: position p holds original index untranspose_index(p);
                    // transpose_o: original index p sits at position transpose_index(p)
                    y[i] = st[tr_slot(INVERSE ? dev::transpose_index(p) : dev::untranspose_index(p))];
                }
                __builtin_nontemporal_store(y, dst + t + 64u * j);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// A grid of every vector group (over the resident set with a grid-stride loop
// the transpose measured 8-10 % slower; in materialize_kernel even a loop that
// runs once cost 127 VGPRs instead of 54, addresses hoisted out of it: 92.0 us
// against 88.1 for 120M delta rows).  Materialize's stores to aligned outputs are
// non-temporal (2-3 % faster there, 13 % slower in the transpose).  To other
// outputs they are not: every store instruction then ends in the middle of a
// line, which only the caches can put together again (120M delta rows 205 us
// non-temporal, 131 this way, stored order 187 and 101; 30M 45.5 and 22.1; 11
// bits transposed 192 and 117).
constexpr int kMatBlock = 256;          // 4 waves, two vectors per wave
constexpr int kMatVecs = kMatBlock / 32;
constexpr uint32_t kRowPad = 33u;       // words per 32 staged rows

// One vector per 32 lanes: decode (any encoding but RLE) into the lane's 32
// rows, then store.  ROWS with a transposed column: row r of lane l is original
// row untranspose_index(l + 32 r); the vector is staged in LDS by original row
// (33 words per 32 rows) and read back in row order, so the stores are
// coalesced.  ROWS writes rows < n_rows only; stored order writes whole
// vectors.  VEC (a 16-byte aligned output): the vector goes through the LDS
// stage in either order (stored order: word 32 r + l at its own index) and
// each work-item stores four consecutive words at a time.  Bound by the writes.
// The stage holds the whole vector, which leaves four blocks per CU: with half
// the stage and eight blocks the pure write streams were slower (120M delta
// rows 97 us against 88, stored order 48.2 against 45.1 for 60M), and so were
// three and two blocks (98.7 and 116 us).  MIXED: RLE vectors leave through
// rle_emit, whose latency wants the waves, so the rest go half the chains, or
// eight stored rows, at a time through a stage of that size (60M rows of mixed
// families: 64.4 us in row order and 63.1 stored, with the whole stage 71.0
// and 67.5; an all-bit-packed mixed column 71.6 against 70.2; with the packed
// words through the caches 50.7 and 49.1).  Half of every
// chain at a time (64-byte pieces) took 88 us: lines have to be filled by one
// instruction.
template <bool ROWS, bool VEC, bool MIXED, bool CACHED>
__global__ __launch_bounds__(kMatBlock) void materialize_kernel(const ColDev c, uint64_t n_rows, uint64_t n_vec,
                                                                uint32_t* __restrict out) {
    constexpr bool kStage = ROWS || VEC;
    // a mixed column's stage is the RLE stage, which holds 512 rows too
    constexpr uint32_t kRleWords = sizeof(RleLds) / 4u;
    constexpr uint32_t kStageWords = MIXED ? kRleWords : kStage ? 32u * kRowPad : 4u;
    static_assert(kRleWords >= 16u * kRowPad && kRleWords % 4u == 0, "512 rows fit, and the stage stays aligned");
    __shared__ __align__(16) uint32_t stage[kMatVecs][kStageWords];
    auto fence = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    const uint32_t l = dev::lane32();
    const uint32_t slot = threadIdx.x >> 5;
    const uint64_t v = (uint64_t)blockIdx.x * kMatVecs + slot;
    bool live = v < n_vec;
    uint32_t x[32];
    uint32_t* dst = out + v * 1024u;
    if (MIXED && live && ((uint32_t)c.vmeta[v] >> 6 & 3u) == FLS_MIX_RLE) {
        // an RLE vector of a mixed column goes straight to memory
        const fls_vmeta m = c.vmeta[v];
        const uint64_t ax = c.aux[v];
        const uint32_t* q = c.words + FLS_VMETA_OFFSET(m);
        const uint32_t ibw = (uint32_t)(ax >> 48) & 1u;
        const RleVector r{ibw, ldg(q + dev::lane32()), q + 32u, q + 32u + 32u * ibw, (uint32_t)(ax >> 32) & 0xffffu,
                          (uint32_t)m & 63u, (uint32_t)ax};
        rle_emit<ROWS, VEC>(r, *reinterpret_cast<RleLds*>(stage[slot]),
                            ROWS ? (uint32_t)min<uint64_t>(1024u, n_rows - v * 1024u) : 1024u, dst);
        live = false;  // done
    }
    if (live) decode_regs<false, CACHED>(c, v, x);
    auto put = [](uint32_t y, uint32_t* p) {  // one word: past the caches where whole lines are stored
        if constexpr (VEC) __builtin_nontemporal_store(y, p);
        else *p = y;
    };
    if constexpr (!kStage) {
        if (live) {
#pragma unroll
            for (int r = 0; r < 32; ++r) put(x[r], dst + 32u * r + l);
        }
    } else {
        const uint32_t rows = !live ? 0u : ROWS ? (uint32_t)min<uint64_t>(1024u, n_rows - v * 1024u) : 1024u;
        uint32_t* st = stage[slot];
        if (ROWS && !c.transposed) {
#pragma unroll
            for (int r = 0; r < 32; ++r)
                if (32u * r + l < rows) put(x[r], dst + 32u * r + l);
        } else if constexpr (!MIXED) {
            // the whole vector at once: by original row (ROWS) or by place
            if (live) {
#pragma unroll
                for (int r = 0; r < 32; ++r) {
                    const uint32_t i = ROWS ? dev::untranspose_index(l + 32u * r) : l + 32u * r;
                    st[i + (i >> 5)] = x[r];
                }
            }
            fence();
            if constexpr (VEC) {
                // rows 4l + 128j .. +3 per work-item: four LDS reads (on
                // distinct banks across the half-wave) and one 16-byte store
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const uint32_t r0 = 4u * l + 128u * (uint32_t)j;
                    const uint32_t* sp = st + r0 + (r0 >> 5);
                    if (r0 + 4u <= rows) {
                        __builtin_nontemporal_store(u32x4{sp[0], sp[1], sp[2], sp[3]},
                                                    reinterpret_cast<u32x4*>(dst + r0));
                    } else {
                        for (uint32_t i = 0; r0 + i < rows; ++i) dst[r0 + i] = sp[i];
                    }
                }
            } else {
#pragma unroll
                for (int r = 0; r < 32; ++r)
                    if (32u * r + l < rows) put(st[kRowPad * r + l], dst + 32u * r + l);
            }
        } else if constexpr (ROWS) {
            // the lane's chain is 32 consecutive rows: half of the chains (512
            // rows, 33 words of LDS per 32) at a time, so that every store
            // instruction fills whole lines
            const uint32_t ch = 2u * (l & 15u) + (l >> 4);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (live && (ch >> 4) == (uint32_t)h) {
#pragma unroll
                    for (int e = 0; e < 32; ++e) st[kRowPad * (ch & 15u) + e] = x[dev::rsum_row(e)];
                }
                fence();
                uint32_t* d = dst + 512u * h;
                const uint32_t here = rows > 512u * h ? rows - 512u * h : 0u;
                if constexpr (VEC) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const uint32_t r0 = 4u * l + 128u * (uint32_t)j;
                        const uint32_t* sp = st + r0 + (r0 >> 5);
                        if (r0 + 4u <= here) {
                            __builtin_nontemporal_store(u32x4{sp[0], sp[1], sp[2], sp[3]},
                                                        reinterpret_cast<u32x4*>(d + r0));
                        } else {
                            for (uint32_t i = 0; r0 + i < here; ++i) d[r0 + i] = sp[i];
                        }
                    }
                } else {
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if (32u * r + l < here) put(st[kRowPad * r + l], d + 32u * r + l);
                }
                fence();
            }
        } else {
            // eight rows at a time, 16-byte stores
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (live) {
#pragma unroll
                    for (int r = 0; r < 8; ++r) st[kRowPad * r + l] = x[8 * q + r];
                }
                fence();
                if (live) {
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const uint32_t p = 4u * l + 128u * (uint32_t)j;
                        const uint32_t* sp = st + p + (p >> 5);
                        __builtin_nontemporal_store(u32x4{sp[0], sp[1], sp[2], sp[3]},
                                                    reinterpret_cast<u32x4*>(dst + 256u * q + p));
                    }
                }
                fence();
            }
        }
    }
}

// An RLE column: see fls_rle.hpp.  Bound by two dependent round trips per
// vector, then the writes: seven to eight waves per SIMD (18.4 KB of LDS; 60M
// rows of mean run 8 55.8 us, and 63.8 with four waves).  67,109,641 such rows
// in row order: 97.7 us through the general kernel with a gather from memory
// per row, 61.3 here, and 48.3 with the index words through the caches, whose
// lines neighbouring vectors share (6.3 TB/s).  Stored order, 60M rows: 60.3
// with 1,024-run stages and one word per store, 55.2 here, 44.0 through the
// caches.
template <bool ROWS, bool VEC>
__global__ __launch_bounds__(kMatBlock) void rle_kernel(const ColDev c, uint64_t n_rows, uint64_t n_vec,
                                                        uint32_t* __restrict out) {
    __shared__ RleLds lds[kMatVecs];
    const uint64_t v = (uint64_t)blockIdx.x * kMatVecs + (threadIdx.x >> 5);
    if (v >= n_vec) return;
    const fls_vmeta m = ldg(c.vmeta + v);
    const fls_rle_meta rm = ldg(reinterpret_cast<const fls_rle_meta*>(c.aux) + v);
    const uint32_t* q = c.words + FLS_VMETA_OFFSET(m);
    const uint32_t ibw = FLS_VMETA_BW(m);
    const RleVector r{ibw, ldg(c.bases + v * 32u + dev::lane32()), q, q + 32u * ibw, rm.n_runs, rm.vbw, rm.vbase};
    rle_emit<ROWS, VEC>(r, lds[threadIdx.x >> 5], ROWS ? (uint32_t)min<uint64_t>(1024u, n_rows - v * 1024u) : 1024u,
                        out + v * 1024u);
}

template <bool ROWS, bool VEC, bool MIXED>
auto pick(const ColDev& c) {
    return c.cached ? materialize_kernel<ROWS, VEC, MIXED, true> : materialize_kernel<ROWS, VEC, MIXED, false>;
}

template <bool ROWS>
int launch_order(const ColDev& c, uint64_t n_rows, uint32_t* d_out, hipStream_t s) {
    const uint64_t n_vec = ceil_div(n_rows, 1024);
    const uint64_t work = ceil_div(n_vec, kMatVecs);  // a grid of every group
    FLS_RETURN_IF(work > 0x7fffffffu, FLS_ERR_SIZE);
    const bool vec = reinterpret_cast<uintptr_t>(d_out) % 16u == 0;  // 16-byte stores where the output allows them
    auto k = vec ? rle_kernel<ROWS, true> : rle_kernel<ROWS, false>;
    if (c.enc == FLS_ENC_MIXED)
        k = vec ? pick<ROWS, true, true>(c) : pick<ROWS, false, true>(c);
    else if (c.enc != FLS_ENC_RLE)
        k = vec ? pick<ROWS, true, false>(c) : pick<ROWS, false, false>(c);
    hipLaunchKernelGGL(k, dim3((uint32_t)work), dim3(kMatBlock), 0, s, c, n_rows, n_vec, d_out);
    return check_launch();
}

}  // namespace

int materialize(const ColDev& c, uint64_t n_rows, bool rows, uint32_t* d_out, hipStream_t s) {
    return rows ? launch_order<true>(c, n_rows, d_out, s) : launch_order<false>(c, n_rows, d_out, s);
}

}  // namespace fls

extern "C" {

int fls_transpose_u32(const uint32_t* d_in, uint64_t n_vec, uint32_t inverse, uint32_t* d_out, void* stream) {
    using namespace fls;
    if (n_vec == 0) return FLS_OK;
    FLS_RETURN_IF(!d_in || !d_out, FLS_ERR_NULL);
    FLS_RETURN_IF(d_in == d_out, FLS_ERR_ARG);
    FLS_RETURN_IF((reinterpret_cast<uintptr_t>(d_in) | reinterpret_cast<uintptr_t>(d_out)) % 16u, FLS_ERR_ARG);
    uint32_t grid = 0;
    const uint64_t work = ceil_div(n_vec, kTrVecs);  // a grid of every group
    FLS_RETURN_IF(work > 0x7fffffffu, FLS_ERR_SIZE);
    if (inverse) {
        grid = (uint32_t)work;
        hipLaunchKernelGGL(transpose_kernel<true>, dim3(grid), dim3(kTrBlock), 0, as_stream(stream), d_in, n_vec,
                           d_out);
    } else {
        grid = (uint32_t)work;
        hipLaunchKernelGGL(transpose_kernel<false>, dim3(grid), dim3(kTrBlock), 0, as_stream(stream), d_in, n_vec,
                           d_out);
    }
    return check_launch();
}

int fls_decode_column_u32(const fls_column* col, uint64_t n_rows, uint32_t order, uint32_t* d_out, void* stream) {
    using namespace fls;
    FLS_RETURN_IF(!col, FLS_ERR_NULL);
    FLS_RETURN_IF(order != FLS_ORDER_STORED && order != FLS_ORDER_ROWS, FLS_ERR_ARG);
    ColDev c{};
    if (const int st = to_dev_column(*col, n_rows, &c, true)) return st;
    if (n_rows == 0) return FLS_OK;
    FLS_RETURN_IF(!d_out, FLS_ERR_NULL);
    return materialize(c, n_rows, order == FLS_ORDER_ROWS, d_out, as_stream(stream));
}

}  // extern "C"
