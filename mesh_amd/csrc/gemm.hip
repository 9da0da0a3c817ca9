// Shard projection GEMMs on MFMA: C[M,N] = A[M,K] @ W[K,N].
//
// W (bf16 weights, reference [in, out] layout) is repacked once at upload into
// MFMA B-operand fragments of v_mfma_f32_32x32x16_bf16 (on gfx950 it issues
// at the rate of 16x16x32 with twice the work): fragment (nt, kt16) is 64
// lanes x 8 bf16, lane l holding W[16 kt16 + 8 (l / 32) + j][32 nt + l % 32],
// j < 8, stored contiguously; fragments of one 32-column tile are consecutive
// along K (kt16 < 2 ceil(K / 32), zero padded).  A wavefront streams its
// weights as perfectly coalesced 1 KiB loads.
// A (activations) arrives fragment-packed (a_pack_index: 1 KiB fragments of
// 32 rows x 16 columns) as bf16 -- or a hi + lo bf16 pair under
// ZR_FLAG_SPLIT_ACTIVATIONS -- written that way by the producing kernel.
// Matmul semantics: forward_pass.rs:1696-1714 (w_qkv / w_gate_up column
// concatenations), 2265 (O), 2290 (down), 2311 (LM head); f32 accumulation.
// The gate|up concatenation is interleaved per 32 columns so one 64-column
// pair holds matching gate and up values for the SwiGLU epilogue
// (silu(g) * u, forward_pass.rs:2286-2289).
#include "zr_internal.h"

#include <algorithm>
#include <cstdlib>

namespace zr {

size_t packed_weight_elems(int k, int n) {
    const size_t kt16 = 2 * (size_t)((k + 31) / 32), nt = (size_t)(n + 31) / 32;
    return kt16 * nt * 512;
}

// dst 32-column tile `nt_dst0 + i * tile_step` takes source columns
// [32 i, 32 i + 32) of src [K, n_src] (zero outside).
__global__ __launch_bounds__(256) void pack_weight_kernel(const uint16_t* __restrict__ src, int K, int n_src,
                                                          int KT16, int nt_dst0, int tile_step, int n_tiles,
                                                          uint16_t* __restrict__ dst) {
    const size_t gid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t total = (size_t)n_tiles * KT16 * 64;
    if (gid >= total) return;
    const int lane = (int)(gid % 64);
    const size_t frag = gid / 64;
    const int kt = (int)(frag % KT16);
    const int i = (int)(frag / KT16);
    const int nt = nt_dst0 + i * tile_step;
    const int n = i * 32 + (lane & 31);
    uint16_t* out = dst + (((size_t)nt * KT16 + kt) * 64 + lane) * 8;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int k = kt * 16 + (lane >> 5) * 8 + j;
        out[j] = (k < K && n < n_src) ? src[(size_t)k * n_src + n] : (uint16_t)0;
    }
}

static zr_status pack_into(zr_context* ctx, const uint16_t* src, int k, int n, int nt0, int step, uint16_t* dst) {
    const size_t bytes = (size_t)k * n * 2;
    const int KT16 = 2 * ((k + 31) / 32);
    uint16_t* tmp = nullptr;
    ZR_HIP(ctx, hipMalloc(&tmp, bytes));
    hipError_t e = hipMemcpyAsync(tmp, src, bytes, hipMemcpyDefault, ctx->stream);
    if (e == hipSuccess) {
        const int n_tiles = (n + 31) / 32;
        const size_t total = (size_t)n_tiles * KT16 * 64;
        hipLaunchKernelGGL(pack_weight_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, ctx->stream,
                           tmp, k, n, KT16, nt0, step, n_tiles, dst);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    (void)hipFree(tmp);
    if (e != hipSuccess) return set_err(ctx, ZR_E_HIP, "weight pack failed: %s", hipGetErrorString(e));
    return ZR_OK;
}

zr_status pack_weight(zr_context* ctx, const uint16_t* src, int k, int n, uint16_t** out) {
    const int* widths = &n;
    return pack_weight_concat(ctx, &src, widths, 1, k, out);
}

zr_status pack_weight_concat(zr_context* ctx, const uint16_t* const* srcs, const int* widths, int count,
                             int k, uint16_t** out) {
    int n_total = 0;
    for (int i = 0; i < count; ++i) {
        if (count > 1 && widths[i] % 32 != 0)
            return set_err(ctx, ZR_E_UNSUPPORTED, "concatenated projection width %d is not a multiple of 32",
                           widths[i]);
        n_total += widths[i];
    }
    uint16_t* dst = nullptr;
    ZR_HIP(ctx, hipMalloc(&dst, packed_weight_elems(k, n_total) * 2));
    int nt0 = 0;
    for (int i = 0; i < count; ++i) {
        zr_status rc = pack_into(ctx, srcs[i], k, widths[i], nt0, 1, dst);
        if (rc != ZR_OK) {
            (void)hipFree(dst);
            return rc;
        }
        nt0 += (widths[i] + 31) / 32;
    }
    *out = dst;
    return ZR_OK;
}

// Interleaved [gate | up]: tile 2b = gate columns [32b, 32b+32), tile 2b+1 = up.
zr_status pack_weight_gate_up(zr_context* ctx, const uint16_t* gate, const uint16_t* up, int k, int f,
                              uint16_t** out) {
    if (f % 32 != 0) return set_err(ctx, ZR_E_UNSUPPORTED, "ffn width %d is not a multiple of 32", f);
    uint16_t* dst = nullptr;
    ZR_HIP(ctx, hipMalloc(&dst, packed_weight_elems(k, 2 * f) * 2));
    zr_status rc = pack_into(ctx, gate, k, f, 0, 2, dst);
    if (rc == ZR_OK) rc = pack_into(ctx, up, k, f, 1, 2, dst);
    if (rc != ZR_OK) {
        (void)hipFree(dst);
        return rc;
    }
    *out = dst;
    return ZR_OK;
}

// silu(g) * u = g / (1 + e^-g) * u (runtime.rs:927-929, forward_pass.rs:2286-2289),
// one rounding per operation as written.
__device__ inline float swiglu(float g, float u) {
#pragma clang fp contract(off)
    return g / (1.0f + expf(-g)) * u;
}

// ------------------------------------------------------------------ GEMM
// v_mfma_f32_32x32x16_bf16: A fragment lane l holds A[row l % 32][k 8 (l / 32)
// + j]; the product lane l, element i is C[8 (i / 4) + 4 (l / 32) + i % 4][l % 32].
// Block tile BM x BN = (32 WAVES_M WM) x (32 WAVES_N WN); wave tile
// (32 WM) x (32 WN); a k-step covers 32 of K (two MFMA k-halves).
// Both operands go global -> LDS with `buffer_load_dwordx4 ... lds` (no
// registers): every 1 KiB MFMA fragment of a k-step -- A rows (hi, then lo)
// and weight tiles -- is one wave instruction, spread evenly over the
// block's waves.  STAGES-deep ring: halfway through step i a wave waits
// (vmcnt) for its own copies of stage i + 1, the block barrier publishes that
// stage to every wave and retires slot i (all of its reads have returned),
// and the copies of stage i + STAGES go into slot i.  The compiler does not
// order LDS reads after these copies, hence the explicit waits; on gfx950 a
// copy into LDS retires with vmcnt only (an lgkmcnt(0) wait does not cover
// it, measured), so the ring waits on vmcnt.  (Measured on
// the decode shapes: 4 or 5 stages instead of 3, streaming the weights into
// per-wave registers, staging both operands through registers + ds_write,
// or two k-steps per stage, are each no faster; the per-half register
// pipeline below is 3-8 % faster than reading each fragment just before
// its MFMAs.)
// Grid: 1-D, decoded so that the row blocks of one (column block, split)
// pair are dispatched 8 apart -- on the same XCD, one after the other -- and
// share that weight tile through its L2.  Pairs left over by 8 are spread
// tile by tile: as whole pairs they gave some XCDs up to a row of tiles more
// than the rest, often a pass over their 32 CUs  (170 tiles of
// 2560 columns, 2108 rows, K 2048: 90 us as two passes, 50 as one).
// SWIGLU = 1: single split; column tiles come in gate / up pairs (tile 2b is
// gate, 2b + 1 up, WN even) and silu(g) * u is written straight to H as the
// next GEMM's fragment-packed bf16 hi (+ lo when h_lo) operand [M, N / 2].
template <int WM, int WN, int WAVES_M, int WAVES_N, int HL, int STAGES, int SWIGLU>
__global__ __launch_bounds__(WAVES_M* WAVES_N * 64) void gemm_kernel(
    const uint16_t* __restrict__ A, int M, int K, const bf16x8* __restrict__ Wp, int KT, int NT,
    float* __restrict__ C, int N, int kt_per_split, int splits, int row_blocks, int col_blocks,
    size_t split_stride, uint16_t* __restrict__ H, int h_lo) {
    static_assert(!SWIGLU || WN % 2 == 0, "gate / up tile pairs");
    constexpr int NW = WAVES_M * WAVES_N;
    constexpr int BMT = WAVES_M * WM, BNT = WAVES_N * WN;
    constexpr int FA = HL * BMT * 2, FB = BNT * 2, FS = FA + FB;
    constexpr int PW = (FS + NW - 1) / NW;  // LDS copies per wave per stage
    constexpr int FSP = PW * NW;            // fragments per stage incl. padding
    constexpr int VM = PW;                  // vector-memory ops per wave per stage
    static_assert(STAGES >= 2 && STAGES <= 6, "stages");
    static_assert(VM * (STAGES - 2) < 64, "vmcnt range");
    typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
    __shared__ bf16x8 lds[STAGES][FSP][64];

    // (workgroups reach the 8 XCDs round-robin: XCD x runs the pairs x, x + 8,
    // ...; the tiles of the last, fewer than 8, go round all XCDs)
    // Branch-free and in one unsigned division: this stands before a block's
    // first copy.
    const unsigned x = blockIdx.x & 7, j = blockIdx.x >> 3;
    const unsigned groups = (unsigned)(col_blocks * splits), whole = (groups >> 3) * (unsigned)row_blocks;
    const bool left = j >= whole;
    const unsigned t = left ? (j - whole) * 8 + x : j, quot = t / (unsigned)row_blocks;
    const int rb = (int)(t - quot * (unsigned)row_blocks);
    const unsigned g = left ? (groups & ~7u) + quot : quot * 8 + x;
    if (g >= groups) return;  // padding block
    const int cb = (int)(g / (unsigned)splits), split = (int)g - cb * splits;

    // the wave index is uniform: readfirstlane keeps it (and every copy
    // offset derived from it) in scalar registers
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int wm_idx = wave / WAVES_N, wn_idx = wave - wm_idx * WAVES_N;
    const int m0 = rb * BMT * 32;
    const int nt_blk = cb * BNT;
    const int KT16 = 2 * KT;
    const int MT = (M + 31) / 32;  // row tiles of the packed A operand
    const int kt_begin = split * kt_per_split;
    const int nsteps = min(KT, kt_begin + kt_per_split) - kt_begin;

    // Copies are buffer loads into LDS: the lane's 16 B of a 1 KiB fragment
    // is a constant vector offset, the fragment's byte offset a scalar, so
    // the per-step address arithmetic stays in the scalar unit.  Offsets are
    // 32-bit: packed operands stay below 2 GiB (zr_context_create refuses
    // geometries past it; launch_gemm checks again).
    const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc((void*)Wp, 0, 0x7fffffff, 0x00020000);
    const int voff = lane * 16;
    auto issue = [&](int slot, int kt) {
#pragma unroll
        for (int i = 0; i < PW; ++i) {
            int f = i * NW + wave;
            const int fs = f < FS ? f : f - FS;  // padding rows repeat a real fragment
            if (fs < FA) {
                // fragment-packed A: row tile (clamped into the operand), k-slice 2 kt + kh
                const int kh = fs & 1, r = fs >> 1;
                const int hl = r / BMT, mt = min(m0 / 32 + (r - hl * BMT), MT - 1);
                const int off = (((hl * MT + mt) * KT16 + 2 * kt + kh) << 10);
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_void*)&lds[slot][f][0], 16, voff, off, 0, 0);
            } else {
                const int fb = fs - FA;
                const int nt = min(nt_blk + (fb >> 1), NT - 1);
                const int off = ((nt * KT16 + 2 * kt + (fb & 1)) << 10);
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_w, (lds_void*)&lds[slot][f][0], 16, voff, off, 0, 0);
            }
        }
    };

    f32x16 acc[WM][WN];
#pragma unroll
    for (int mt = 0; mt < WM; ++mt)
#pragma unroll
        for (int wn = 0; wn < WN; ++wn)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[mt][wn][i] = 0.0f;

    // fragments of one k-half (16 k) in registers: kh 0 / kh 1 alternate so
    // that one half's LDS reads are in flight while the other's MFMAs run
    auto load_frags = [&](int slot, int kh, bf16x8* fa, bf16x8* fb) {
#pragma unroll
        for (int wn = 0; wn < WN; ++wn) fb[wn] = lds[slot][FA + (wn_idx * WN + wn) * 2 + kh][lane];
#pragma unroll
        for (int mt = 0; mt < WM; ++mt)
#pragma unroll
            for (int hl = 0; hl < HL; ++hl)
                fa[mt * HL + hl] = lds[slot][((hl * BMT + wm_idx * WM + mt) << 1) + kh][lane];
    };
    constexpr int NM = WM * HL * WN;  // MFMAs per k-half
    auto mfmas = [&](const bf16x8* fa, const bf16x8* fb, int t0, int t1) {
#pragma unroll
        for (int t = 0; t < NM; ++t) {
            if (t < t0 || t >= t1) continue;
            const int mt = t / (HL * WN), hl = (t / WN) % HL, wn = t % WN;
            acc[mt][wn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[mt * HL + hl], fb[wn], acc[mt][wn], 0, 0, 0);
        }
    };
    bf16x8 fa0[WM * HL], fb0[WN], fa1[WM * HL], fb1[WN];

#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
        if (s < nsteps) issue(s, kt_begin + s);
    if (nsteps > 0) {
        ring_wait<VM, STAGES - 2>(min(STAGES - 2, nsteps - 1));
        if (STAGES - 1 < nsteps) issue(STAGES - 1, kt_begin + STAGES - 1);
        load_frags(0, 0, fa0, fb0);
    }
    // Step i: first MFMA of kh 0, the kh 1 reads, the other kh 0 MFMAs; the
    // ring barrier for step i + 1 (its copies landed, slot i free) and the
    // copy of stage i + STAGES into slot i; first MFMA of kh 1, the kh 0 reads
    // of step i + 1, the other kh 1 MFMAs.  The scheduling barriers keep the
    // reads where they are.  After the last step the barrier and the reads
    // are idle (the slot's data is not used).  Each accumulator still sums
    // (kh 0, hi), (kh 0, lo), (kh 1, hi), (kh 1, lo) per k-step, in k order.
    for (int i0 = 0; i0 < nsteps; i0 += STAGES) {
#pragma unroll
        for (int u = 0; u < STAGES; ++u) {
            const int i = i0 + u;
            if (i >= nsteps) break;
            mfmas(fa0, fb0, 0, 1);
            __builtin_amdgcn_sched_barrier(0);
            load_frags(u, 1, fa1, fb1);
            __builtin_amdgcn_sched_barrier(0);
            mfmas(fa0, fb0, 1, NM);
            ring_wait<VM, STAGES - 2>(max(0, min(STAGES - 2, nsteps - 2 - i)));
            if (i + STAGES < nsteps) issue(u, kt_begin + i + STAGES);
            mfmas(fa1, fb1, 0, 1);
            __builtin_amdgcn_sched_barrier(0);
            load_frags((u + 1) % STAGES, 0, fa0, fb0);
            __builtin_amdgcn_sched_barrier(0);
            mfmas(fa1, fb1, 1, NM);
        }
    }

    if constexpr (SWIGLU) {
        // Each 32 x 32 tile of H (silu(g) * u of a gate / up tile pair) goes
        // through a per-wave LDS tile (row pitch 33): written in the product's
        // layout (lane = column), read back as 8 consecutive columns of a row
        // per lane, which is one 16-byte run of the fragment-packed operand.
        // One store per plane and 8 values instead of 8 2-byte stores
        // (256-session decode step: the 2-byte stores cost 0.33 ms of GEMM).
        // F = N / 2 is a multiple of 32 (the planner's SwiGLU requires N % 64
        // == 0), so a run is either whole or past F.
        constexpr int TP = 32 * 33;
        static_assert((size_t)NW * TP * sizeof(float) <= sizeof(lds), "transpose tiles fit the ring");
        const int F = N / 2;
        const size_t plane = a_plane(M, F);
        float* tp = (float*)&lds[0][0][0] + wave * TP;
        __syncthreads();  // every wave is past its last ring read
#pragma unroll
        for (int mt = 0; mt < WM; ++mt)
#pragma unroll
            for (int p = 0; p < WN / 2; ++p) {
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    tp[(8 * (i >> 2) + 4 * (lane >> 5) + (i & 3)) * 33 + (lane & 31)] =
                        swiglu(acc[mt][2 * p][i], acc[mt][2 * p + 1][i]);
                __syncthreads();
                const int j0 = ((nt_blk + wn_idx * WN + 2 * p) >> 1) * 32;
                const int mb = m0 + (wm_idx * WM + mt) * 32;
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const int r = (lane + 64 * t) >> 2, grp = lane & 3;
                    const int m = mb + r, j = j0 + 8 * grp;
                    if (m < M && j < F) {
                        float x[8];
#pragma unroll
                        for (int e = 0; e < 8; ++e) x[e] = tp[r * 33 + 8 * grp + e];
                        const size_t o = a_pack_index(m, j, F);
                        *(bf16x8*)(H + o) = to_bf16x8(x, false);
                        if (h_lo) *(bf16x8*)(H + plane + o) = to_bf16x8(x, true);
                    }
                }
                __syncthreads();  // the tile is read before the next one is written
            }
    } else {
        float* out = C + (size_t)split * split_stride;
#pragma unroll
        for (int mt = 0; mt < WM; ++mt)
#pragma unroll
            for (int wn = 0; wn < WN; ++wn) {
                const int n = (nt_blk + wn_idx * WN + wn) * 32 + (lane & 31);
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int m = m0 + (wm_idx * WM + mt) * 32 + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
                    if (m < M && n < N) out[(size_t)m * N + n] = acc[mt][wn][i];
                }
            }
    }
}

// gate/up + SwiGLU for 9-32 rows (33-64: MT = 2) in one launch: K split over the 4
// waves of a workgroup instead of over workgroups (no slabs, no reduce
// kernel).  A workgroup owns one gate / up tile pair (64 columns of the
// interleaved product, 32 columns of H); wave w takes k-steps w, w + 4, ...
// through a ring of its own in LDS: it copies a step's 8 fragments (A hi / lo
// and both weight tiles, two k-halves each) with `buffer_load ... lds` and
// reads only what it copied, so its own vmcnt wait orders the ring and the
// waves never wait for one another until the end.  Each wave accumulates its
// steps in k order ((kh 0, hi), (kh 0, lo), (kh 1, hi), (kh 1, lo) per step);
// the four partial sums then meet in LDS and are added in wave order, and
// silu(g) * u goes to H as the next GEMM's fragment-packed bf16 hi (+ lo).
// Requires M <= 32 and KT % 4 == 0 (every wave the same number of steps).
// ring_wait without the block barrier: only this wave's copies order its ring
template <int N>
__device__ __forceinline__ void wave_copies_wait() {
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));  // vmcnt(N), expcnt(7), lgkmcnt(0)
    asm volatile("" ::: "memory");
}
template <int VM, int MAXA>
__device__ __forceinline__ void wave_ring_wait(int ahead) {
    if constexpr (MAXA > 0) {
        if (ahead >= MAXA) {
            wave_copies_wait<VM * MAXA>();
            return;
        }
        wave_ring_wait<VM, MAXA - 1>(ahead);
    } else {
        wave_copies_wait<0>();
    }
}

template <int STAGES, int HL, int MT>
__global__ __launch_bounds__(256) void gemm_swiglu_ksplit_kernel(const uint16_t* __restrict__ A, int M, int K,
                                                                const bf16x8* __restrict__ Wp, int KT, int N,
                                                                uint16_t* __restrict__ H, int h_lo) {
    constexpr int FW = 2 * HL * MT + 4;  // fragments per k-step: A (hl, row tile, kh), then weights (tile, kh)
    typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
    __shared__ bf16x8 lds[4][STAGES][FW][64];
    const int pair = blockIdx.x;  // weight tiles 2 pair (gate), 2 pair + 1 (up)
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int KT16 = 2 * KT;
    const int nsteps = KT / 4;
    const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc((void*)Wp, 0, 0x7fffffff, 0x00020000);
    const int voff = lane * 16;
    auto issue = [&](int slot, int step) {
        const int kt = step * 4 + wave;
#pragma unroll
        for (int hl = 0; hl < HL; ++hl)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int kh = 0; kh < 2; ++kh)  // row tile mt of the packed A operand (hi plane, then lo)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_void*)&lds[wave][slot][(hl * MT + mt) * 2 + kh][0],
                                                             16, voff, (((hl * MT + mt) * KT16 + 2 * kt + kh) << 10), 0,
                                                             0);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int kh = 0; kh < 2; ++kh)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_w,
                                                         (lds_void*)&lds[wave][slot][2 * HL * MT + t * 2 + kh][0], 16,
                                                         voff, (((2 * pair + t) * KT16 + 2 * kt + kh) << 10), 0, 0);
    };
    f32x16 acc[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[mt][t][i] = 0.0f;
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
        if (s < nsteps) issue(s, s);
    for (int i0 = 0; i0 < nsteps; i0 += STAGES) {
#pragma unroll
        for (int u = 0; u < STAGES; ++u) {
            const int i = i0 + u;
            if (i >= nsteps) break;
            // this wave's copies of step i have landed (later steps may still be in flight)
            wave_ring_wait<FW, STAGES - 2>(max(0, min(STAGES - 2, nsteps - 1 - i)));
            if (i + STAGES - 1 < nsteps) issue((u + STAGES - 1) % STAGES, i + STAGES - 1);
#pragma unroll
            for (int kh = 0; kh < 2; ++kh) {
                const bf16x8 bg = lds[wave][u][2 * HL * MT + kh][lane], bu = lds[wave][u][2 * HL * MT + 2 + kh][lane];
#pragma unroll
                for (int hl = 0; hl < HL; ++hl)
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) {
                        const bf16x8 a = lds[wave][u][(hl * MT + mt) * 2 + kh][lane];
                        acc[mt][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, bg, acc[mt][0], 0, 0, 0);
                        acc[mt][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, bu, acc[mt][1], 0, 0, 0);
                    }
            }
        }
    }
    // the four partial sums meet in LDS (the ring is free once every wave is past its last step)
    __syncthreads();
    float* red = (float*)&lds[0][0][0][0];  // [wave][row tile][tile][i][lane]
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) red[(((wave * MT + mt) * 2 + t) * 16 + i) * 64 + lane] = acc[mt][t][i];
    __syncthreads();
    // thread (i-group tid / 64, lane): elements i = 4 (tid / 64) .. + 3 of each row tile's accumulators
    const int F = N / 2;
    const size_t plane = a_plane(M, F);
    const int j = pair * 32 + (lane & 31);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int i = 4 * wave + q;
            const int m = 32 * mt + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
            float g = red[((mt * 2 + 0) * 16 + i) * 64 + lane], up = red[((mt * 2 + 1) * 16 + i) * 64 + lane];
#pragma unroll
            for (int w = 1; w < 4; ++w) {
                g += red[(((w * MT + mt) * 2 + 0) * 16 + i) * 64 + lane];
                up += red[(((w * MT + mt) * 2 + 1) * 16 + i) * 64 + lane];
            }
            if (m < M && j < F) {
                uint16_t hi, lo;
                split_bf16(swiglu(g, up), hi, lo);
                const size_t o = a_pack_index(m, j, F);
                H[o] = hi;
                if (h_lo) H[plane + o] = lo;
            }
        }
}

// At most kFewRows rows (one session's step, a few of them): the product is the
// stream of its weights, and the ring above copies a padded 32-row A tile, as
// many bytes as the weights themselves, beside them.  Here a workgroup of NW
// waves owns 16 columns (SWIGLU: 16 of H, a gate and an up tile), and the waves
// take consecutive runs of its k-steps.  Weights go straight to registers as
// v_mfma_f32_16x16x32_bf16 fragments: lane l = 16 q + i holds k 8 q + j of
// column i, one 16-byte run of the packed 32x32x16 fragment 2 kt + q / 2 (four
// 256-byte runs per wave load).  Of A only the MR rows (M rounded up to a power
// of two) are read, 16-byte runs packed 64 to a load, and pass through a
// per-wave LDS block to their fragments (as masked fragment loads, two per
// k-step beside one of weights, the address unit held the stream back).  The
// fragments' rows past MR repeat the others: their products are not stored.
// Rows past M and steps past the wave's run are loads past the buffer's end:
// zeros, and no memory traffic.  Two sets of U steps alternate, the next one in
// flight under the other's products; the waves' sums meet in LDS and are added
// in wave order.
// One session's TinyLlama step (517 tokens, us per launch, before / after):
// gate/up 14.1 / 11.9, LM head 27.3 / 23.6 (5.5 TB/s), QKV 5.2 / 5.0 and O, down
// 5.6 / 5.3, with 1-2 slabs instead of 11-16, which take the norms from 4.3 to
// 3.6; the step's kernels 1190 / 1080.  What is left is launch ramp: 8-46 MB at
// the rate of the LM head would take 1.5-8.4.
// Waves and steps per set (NW, U) tried: (4, 4), (8, 2), (8, 4), (4, 8); with
// 9-16 rows (and 16 in masked fragment loads) the tiles are faster (Llama-3, 16
// sessions 621 / 656 us per step of 4 layers).
constexpr int kFewRows = 8;
constexpr int kWeightCache = 2;  // nontemporal: read once per product
struct NormRows {
    const float *x, *res;
    int res_n;
    size_t res_stride;
    float* x_out;
    const float* gamma;
    float eps;
};
// block barrier for LDS data that leaves loads to registers in flight
__device__ __forceinline__ void lds_barrier() {
    wave_copies_wait<63>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
// NORM: A is rms_norm(x + residual) gamma (launch_norm_gemm): every workgroup
// reads the rows, their residual slabs and gamma (L2 hits, under its first
// weights' flight), normalises them as the norm kernel does and keeps them in
// LDS; workgroup 0 writes x + residual to x_out (another buffer: the rest still
// read x).  TinyLlama, one row: gate/up 11.9 us with or without, QKV 5.0 -> 5.8,
// and no norm launches of 3.6; the step 1.07 -> 0.95 ms.
template <int MR, int NW, int U, int HL, int SWIGLU, int NORM>
__global__ __launch_bounds__(NW * 64) void gemm_few_rows_kernel(const uint16_t* __restrict__ A, int M,
                                                                const uint16_t* __restrict__ Wp, int KT, int NT,
                                                                float* __restrict__ C, int N, int kt_per_split,
                                                                int splits, size_t split_stride,
                                                                uint16_t* __restrict__ H, NormRows nr) {
    constexpr int TW = SWIGLU ? 2 : 1;
    constexpr int NA = (U * HL * 4 * MR + 63) / 64;  // loads of A runs per set
    typedef __attribute__((__vector_size__(4 * sizeof(unsigned)))) unsigned u32x4;
    __shared__ f32x4 red[NW][TW][64];
    __shared__ u32x4 rows[NORM ? 1 : NW][NORM ? 1 : NA * 64];  // [step u][hi, lo][q][row]
    extern __shared__ bf16x8 normed[];                         // NORM: [k / 8][hi, lo][row]
    constexpr int KC = kNormCols / (8 * NW * 64);              // runs of 8 columns per thread
    f32x4 xv[MR][KC][2], gv[KC][2];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int col16 = blockIdx.x / splits, split = blockIdx.x - col16 * splits;
    const int q = lane >> 4, i16 = lane & 15;
    const unsigned plane_bytes = (unsigned)KT << 11;  // one 32-row or 32-column tile: 2 KT fragments of 1 KiB
    const __amdgpu_buffer_rsrc_t rsrc_a =
        __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, (int)(plane_bytes * HL), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_w =
        __builtin_amdgcn_make_buffer_rsrc((void*)Wp, 0, (int)(plane_bytes * (unsigned)NT), 0x00020000);
    constexpr unsigned kPast = 0x80000000u;  // beyond either buffer (both below 2 GiB)
    const unsigned tile0 = SWIGLU ? (unsigned)(col16 >> 1) * 2 : (unsigned)(col16 >> 1);
    const unsigned w0 = tile0 * plane_bytes + (unsigned)(q >> 1) * 1024 + (unsigned)(q & 1) * 512 +
                        (unsigned)(col16 & 1) * 256 + i16 * 16;
    // the lane's run of A load v: byte offset at step 0 and its step within the set (U: none)
    unsigned a0[NA];
    int au[NA];
#pragma unroll
    for (int v = 0; v < NA; ++v) {
        const int idx = v * 64 + lane, row = idx & (MR - 1), r = idx / MR, aq = r & 3, h = (r >> 2) % HL;
        au[v] = (r >> 2) / HL;
        a0[v] = (unsigned)h * plane_bytes + ((unsigned)au[v] << 11) + (unsigned)(aq >> 1) * 1024 +
                (unsigned)(aq & 1) * 512 + row * 16;
        if (row >= M || au[v] >= U) au[v] = 1 << 28;
    }
    // this wave's steps of the split's
    const int kb = split * kt_per_split, n = min(KT, kb + kt_per_split) - kb;
    const int s0 = kb + (int)((long)wave * n / NW), s1 = kb + (int)((long)(wave + 1) * n / NW);

    u32x4 wr[2][U][TW], ar[2][NA];
    auto load = [&](int set, int s) {
#pragma unroll
        for (int v = 0; v < (NORM ? 0 : NA); ++v)
            ar[set][v] = __builtin_amdgcn_raw_buffer_load_b128(
                rsrc_a, (int)(s + au[v] < s1 ? a0[v] + ((unsigned)s << 11) : kPast), 0, 0);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int t = 0; t < TW; ++t)
                wr[set][u][t] = __builtin_amdgcn_raw_buffer_load_b128(
                    rsrc_w, (int)(s + u < s1 ? w0 + t * plane_bytes + ((unsigned)(s + u) << 11) : kPast), 0,
                    kWeightCache);
    };
    f32x4 acc[TW];
#pragma unroll
    for (int t = 0; t < TW; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto products = [&](int set, int s) {
        if constexpr (!NORM) {
            // (one wave's LDS operations run in order; the fences keep the compiler's order the same)
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int v = 0; v < NA; ++v) rows[wave][v * 64 + lane] = ar[set][v];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int h = 0; h < HL; ++h) {
                bf16x8 fa;
                if constexpr (NORM)  // (a step past the wave's run repeats its last: its weights are zeros)
                    fa = normed[((min(s + u, s1 - 1) * 4 + q) * HL + h) * MR + (i16 & (MR - 1))];
                else
                    fa = __builtin_bit_cast(bf16x8, rows[wave][((u * HL + h) * 4 + q) * MR + (i16 & (MR - 1))]);
#pragma unroll
                for (int t = 0; t < TW; ++t)
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa, __builtin_bit_cast(bf16x8, wr[set][u][t]),
                                                                     acc[t], 0, 0, 0);
            }
    };
    const int chunks = KT * 4;  // runs of 8 columns
    f32x4 rv[MR][KC][2][2];
    if constexpr (NORM) {
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < KC; ++k) {
            const int ch = tid + k * NW * 64;
            const bool in = ch < chunks;
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                gv[k][p] = in ? *(const f32x4*)(nr.gamma + ch * 8 + 4 * p) : zero;
#pragma unroll
                for (int r = 0; r < MR; ++r) {
                    const size_t at = (size_t)r * KT * 32 + ch * 8 + 4 * p;
                    const bool ok = in && r < M;
                    xv[r][k][p] = ok ? *(const f32x4*)(nr.x + at) : zero;
#pragma unroll
                    for (int n2 = 0; n2 < 2; ++n2)
                        rv[r][k][p][n2] =
                            ok && n2 < nr.res_n ? *(const f32x4*)(nr.res + n2 * nr.res_stride + at) : zero;
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    load(0, s0);
    if constexpr (NORM) {
        __builtin_amdgcn_sched_barrier(0);
        __shared__ float ssum[MR][NW];
#pragma unroll
        for (int r = 0; r < MR; ++r) {
            float ss = 0.0f;
#pragma unroll
            for (int k = 0; k < KC; ++k) {
                const int ch = tid + k * NW * 64;
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    const size_t at = (size_t)r * KT * 32 + ch * 8 + 4 * p;
                    if (nr.res_n > 0) {
                        f32x4 sum = rv[r][k][p][0];
                        if (nr.res_n > 1) sum += rv[r][k][p][1];
                        for (int n2 = 2; n2 < nr.res_n; ++n2)
                            if (ch < chunks && r < M) sum += *(const f32x4*)(nr.res + n2 * nr.res_stride + at);
                        xv[r][k][p] += sum;
                        if (blockIdx.x == 0 && ch < chunks && r < M) *(f32x4*)(nr.x_out + at) = xv[r][k][p];
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) ss += xv[r][k][p][e] * xv[r][k][p][e];
                }
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
            if (lane == 0) ssum[r][wave] = ss;
        }
        lds_barrier();
#pragma unroll
        for (int r = 0; r < MR; ++r) {
            float total = 0.0f;
#pragma unroll
            for (int w = 0; w < NW; ++w) total += ssum[r][w];
            const float inv = 1.0f / sqrtf(total / (float)(KT * 32) + nr.eps);
#pragma unroll
            for (int k = 0; k < KC; ++k) {
                const int ch = tid + k * NW * 64;
                float y[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) y[e] = xv[r][k][e >> 2][e & 3] * inv * gv[k][e >> 2][e & 3];
                if (ch < chunks) {
                    normed[(ch * HL + 0) * MR + r] = to_bf16x8(y, false);
                    if (HL == 2) normed[(ch * HL + HL - 1) * MR + r] = to_bf16x8(y, true);
                }
            }
        }
        lds_barrier();
    }
    for (int s = s0; s < s1; s += 2 * U) {
        load(1, s + U);
        __builtin_amdgcn_sched_barrier(0);
        products(0, s);
        __builtin_amdgcn_sched_barrier(0);
        load(0, s + 2 * U);
        __builtin_amdgcn_sched_barrier(0);
        products(1, s + U);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int t = 0; t < TW; ++t) red[wave][t][lane] = acc[t];
    __syncthreads();
    // thread (m, column): element m % 4 of lane 16 (m / 4) + column
    const int m = tid >> 4, c = tid & 15;
    if (m >= M) return;  // (M <= 8 rows, at least 256 threads)
    float v[TW];
#pragma unroll
    for (int t = 0; t < TW; ++t) {
        v[t] = red[0][t][16 * (m >> 2) + c][m & 3];
#pragma unroll
        for (int w = 1; w < NW; ++w) v[t] += red[w][t][16 * (m >> 2) + c][m & 3];
    }
    const int j = col16 * 16 + c;
    if constexpr (SWIGLU) {
        const int F = N / 2;
        uint16_t hi, lo;
        split_bf16(swiglu(v[0], v[TW - 1]), hi, lo);
        const size_t o = a_pack_index(m, j, F);
        H[o] = hi;
        if (HL == 2) H[a_plane(M, F) + o] = lo;
    } else if (j < N) {
        C[(size_t)split * split_stride + (size_t)m * N + j] = v[0];
    }
}

// Sum of split-K slabs [S][M][N] with the epilogue.
// kEpiStore:  out_f32[m][n] = sum
// kEpiSwiGLU: N = 2F interleaved per 32 columns; h = silu(g) * u written as
//             bf16 hi (+ lo) [M, F] (the next GEMM's A operand) or f32.
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ ws, int S, int M, int N,
                                                            size_t split_stride, int epilogue,
                                                            float* __restrict__ out_f32,
                                                            uint16_t* __restrict__ out_bf16, int out_lo) {
#pragma clang fp contract(off)
    const int n_out = epilogue == kEpiSwiGLU ? N / 2 : N;
    const size_t total = (size_t)M * n_out;
    for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
         idx += (size_t)gridDim.x * blockDim.x) {
        const int m = (int)(idx / n_out), j = (int)(idx % n_out);
        float v;
        if (epilogue == kEpiSwiGLU) {
            const int gc = (j >> 5) * 64 + (j & 31);
            float g = 0.0f, u = 0.0f;
            for (int s = 0; s < S; ++s) {
                g += ws[s * split_stride + (size_t)m * N + gc];
                u += ws[s * split_stride + (size_t)m * N + gc + 32];
            }
            v = swiglu(g, u);
        } else {
            v = 0.0f;
            for (int s = 0; s < S; ++s) v += ws[s * split_stride + (size_t)m * N + j];
        }
        if (out_bf16) {  // fragment-packed A operand of the next GEMM
            uint16_t hi, lo;
            split_bf16(v, hi, lo);
            const size_t o = a_pack_index(m, j, n_out);
            out_bf16[o] = hi;
            if (out_lo) out_bf16[a_plane(M, n_out) + o] = lo;
        } else {
            out_f32[idx] = v;
        }
    }
}

// f32 [rows, K] -> fragment-packed bf16 hi (+ lo) (A operand of zr_gemm)
__global__ __launch_bounds__(256) void to_bf16_pair_kernel(const float* __restrict__ x, int rows, int K,
                                                           uint16_t* __restrict__ out, int with_lo) {
    const size_t n = (size_t)rows * K, plane = a_plane(rows, K);
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        uint16_t hi, lo;
        split_bf16(x[i], hi, lo);
        const size_t o = a_pack_index((int)(i / K), (int)(i % K), K);
        out[o] = hi;
        if (with_lo) out[plane + o] = lo;
    }
}

// fragment-packed bf16 hi (+ lo) [rows, K] -> f32 hi + lo (the value a GEMM
// operand stands for)
__global__ __launch_bounds__(256) void from_bf16_pair_kernel(const uint16_t* __restrict__ in, int rows, int K,
                                                             int with_lo, float* __restrict__ y) {
    const size_t n = (size_t)rows * K, plane = a_plane(rows, K);
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const size_t o = a_pack_index((int)(i / K), (int)(i % K), K);
        const float hi = __uint_as_float((uint32_t)in[o] << 16);
        y[i] = with_lo ? hi + __uint_as_float((uint32_t)in[plane + o] << 16) : hi;
    }
}

zr_status launch_from_bf16_pair(zr_context* ctx, const uint16_t* in, int rows, int K, int with_lo, float* y) {
    if (K % 32 != 0) return set_err(ctx, ZR_E_UNSUPPORTED, "GEMM operand width %d is not a multiple of 32", K);
    const size_t n = (size_t)rows * K;
    const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 16384);
    hipLaunchKernelGGL(from_bf16_pair_kernel, dim3(blocks), dim3(256), 0, ctx->stream, in, rows, K, with_lo, y);
    ZR_LAUNCH_CHECK(ctx);
    return ZR_OK;
}

zr_status launch_to_bf16_pair(zr_context* ctx, const float* x, int rows, int K, uint16_t* out, int with_lo) {
    if (K % 32 != 0) return set_err(ctx, ZR_E_UNSUPPORTED, "GEMM operand width %d is not a multiple of 32", K);
    const size_t n = (size_t)rows * K;
    const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 16384);
    hipLaunchKernelGGL(to_bf16_pair_kernel, dim3(blocks), dim3(256), 0, ctx->stream, x, rows, K, out, with_lo);
    ZR_LAUNCH_CHECK(ctx);
    return ZR_OK;
}

// Tile configurations: wave tile WM x WN 32x32 tiles, WAVES_M x WAVES_N waves.
struct GemmCfg {
    int wm, wn, waves_m, waves_n, stages;
    int bm() const { return waves_m * wm * 32; }
    int bn() const { return waves_n * wn * 32; }
};

static int device_cus() {
    static const int cus = [] {
        int v = 256, dev = 0;
        if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev);
        return v > 0 ? v : 256;
    }();
    return cus;
}

static bool swiglu_fused(int m, int epilogue) { return epilogue == kEpiSwiGLU && m > 64; }

// <= 64 rows of gate / up: SwiGLU in one launch with K split over the waves of
// a workgroup (gemm_swiglu_ksplit_kernel; two 32-row tiles above 32 rows)
static bool swiglu_ksplit(int m, int n, int k, int epilogue) {
    return epilogue == kEpiSwiGLU && m <= 64 && n % 64 == 0 && ((k + 31) / 32) % 4 == 0;
}

// At most kFewRows rows: gemm_few_rows_kernel, K split over workgroups as far
// as one pass over the CUs goes (single TinyLlama step: 128 workgroups for O
// and down 0.7 us more per product, two passes of splits 2 us more).
static bool few_rows(int m, int n, int epilogue) { return m <= kFewRows && (epilogue == kEpiStore || n % 64 == 0); }

struct GemmChoice {
    GemmCfg cfg;
    int splits;
};

// Split K as far as the grid fits one pass over the CUs, >= 4 k-steps per
// split, at most 16 splits.  More tiles than one pass: up to 4 splits when they
// fill the last pass better, in passes of unsplit blocks plus, per extra split,
// one more f32 slab written and read back (8 M N bytes at ~5 TB/s) against one
// pass of the hi + lo MFMA work (4 BM BN K per CU at ~1.2 PFLOP/s).
static GemmChoice one_pass(const GemmCfg& c, int m, int n, int k) {
    const int tiles = ((m + c.bm() - 1) / c.bm()) * ((n + c.bn() - 1) / c.bn());
    const int KT = (k + 31) / 32, cus = device_cus();
    if (tiles <= cus) return {c, std::max(1, std::min(std::min(16, cus / tiles), KT / 4))};
    const double slab = 480.0 * tiles / ((double)k * cus);
    GemmChoice best{c, 1};
    double least = 1e30;
    for (int s = 1; s <= 4 && s <= std::max(1, KT / 4); ++s) {
        const double cost = (double)(((size_t)tiles * s + cus - 1) / cus) / s + slab * (s - 1);
        if (cost < least - 1e-9) {
            least = cost;
            best.splits = s;
        }
    }
    return best;
}

// Tiles of products over many rows, priced two ways.
//
// By themselves: a block of a config takes `step` us per k-step of 32 (plus
// four of prologue and epilogue) in a full pass over its slots; a last pass
// over a share f of them takes alone + (1 - alone) f of that, less than a whole
// one because the chip clocks higher then (it runs these products at its power
// limit: full passes reach 1.34-1.44 PFLOP/s of MFMA work whatever the tile).
// Fitted to cold weights, hi + lo operands, 256-3000 rows, 2048-28672 columns,
// K 2048-14336; within 5 % of most of them.  With two blocks per CU, up to half
// of the slots run one to a CU.
//
// Beside other streams' kernels: those fill the CUs that a last pass leaves, so
// a product costs the CU time it takes, blocks x `busy` us per k-step (plus
// `fixed` steps) over the slots.  Three streams of one product each (the same
// sizes) are within 3 % of it.  Per element of the product 256 x 256 tiles take
// 0.91 and 64 x 256 ones 1.14 of the CU time of 128 x 256 tiles.
struct TileCost {
    GemmCfg cfg;
    int per_cu;
    float step, alone;
    struct { float busy, fixed; } store, fused;
};
static const TileCost kTileCosts[] = {
    {{2, 2, 2, 4, 3}, 1, 0.80f, 0.70f, {0.883f, 2.0f}, {0.863f, 5.6f}},  // 128 x 256
    {{2, 2, 3, 4, 3}, 1, 1.10f, 0.60f, {1.273f, 0.3f}, {1.232f, 6.7f}},  // 192 x 256, 12 waves
    {{2, 2, 4, 4, 3}, 1, 1.47f, 0.50f, {1.628f, 0.0f}, {1.564f, 7.1f}},  // 256 x 256, 16 waves
    {{2, 2, 1, 4, 3}, 2, 0.90f, 0.70f, {0.936f, 0.7f}, {0.986f, 0.0f}},  // 64 x 256, two blocks per CU
    {{2, 4, 2, 4, 3}, 1, 1.55f, 0.60f, {1.620f, 6.0f}, {1.620f, 6.0f}},  // 128 x 512
};

// us per float of a split-K slab past the first: written, then read by the
// product's consumer
constexpr float kSlabUs = 1.6e-6f;

// (both priced at whole 64-row units, so that a plan and its workspace change
// at their ends only)
static int tiles_of(const TileCost& t, int rows, int n) {
    return ((rows + t.cfg.bm() - 1) / t.cfg.bm()) * ((n + t.cfg.bn() - 1) / t.cfg.bn());
}

static float time_alone(const TileCost& t, int splits, int rows, int n, int k) {
    const int KT = (k + 31) / 32, slots = t.per_cu * device_cus();
    const int blocks = tiles_of(t, rows, n) * splits, full = blocks / slots;
    const float f = (float)(blocks - full * slots) / slots;
    float passes = (float)full;
    if (f > 0.0f) passes += t.per_cu == 2 && f <= 0.5f ? 0.45f + 0.15f * f : t.alone + (1.0f - t.alone) * f;
    return passes * t.step * ((KT + splits - 1) / splits + 4) + kSlabUs * rows * (float)n * (splits - 1);
}

static float cu_time(const TileCost& t, int splits, int rows, int n, int k, int epilogue) {
    const int KT = (k + 31) / 32;
    const auto& c = epilogue == kEpiStore ? t.store : t.fused;
    return (float)(tiles_of(t, rows, n) * splits) / (t.per_cu * device_cus()) * c.busy *
               ((KT + splits - 1) / splits + c.fixed) +
           kSlabUs * rows * (float)n * (splits - 1);
}

// The plan that is fastest by itself among those that take no more CU time
// than `most` does (the plan of one pass over the CUs).  Without that limit the
// tiles that fill a pass better are up to 6 % slower per microbatch where
// others run beside it (4 layers on three streams, us: Llama-3, 600 rows 2352
// against 2232 with it, 1400 rows 4722 / 4457; TinyLlama, 8 layers, 800 rows
// 1470 / 1428), and 0-5 % faster where none do.
// waits: no limit -- the caller waits for this microbatch, and nothing else of
// its context runs beside it (a 760-row Llama-3 prompt of 3 layers 2257 us with
// the limit, 2199 without).
static GemmChoice cheapest(int m, int n, int k, int epilogue, const GemmChoice& most, bool waits) {
    const int rows = (m + 63) / 64 * 64, KT = (k + 31) / 32, cus = device_cus();
    auto same = [](const GemmCfg& a, const GemmCfg& b) {
        return a.wm == b.wm && a.wn == b.wn && a.waves_m == b.waves_m && a.waves_n == b.waves_n;
    };
    float limit = 1e30f, least = 1e30f;
    for (const TileCost& t : kTileCosts)
        if (same(t.cfg, most.cfg)) {
            if (!waits) limit = cu_time(t, most.splits, rows, n, k, epilogue);
            least = time_alone(t, most.splits, rows, n, k);
        }
    GemmChoice best = most;
    for (const TileCost& t : kTileCosts) {
        const int tiles = tiles_of(t, rows, n);
        for (int s = 1; s <= (epilogue == kEpiStore ? 16 : 1); ++s) {
            if (s > 1 && KT / s < 4) break;
            if (s > 4 && tiles * s > 2 * cus) break;  // (bounds the workspace)
            const float us = time_alone(t, s, rows, n, k);
            if (us < least && cu_time(t, s, rows, n, k, epilogue) <= limit) {
                least = us;
                best = {t.cfg, s};
            }
        }
    }
    return best;
}

// The tile and K split of a product (measured with weights streamed from HBM
// and split activations; the decode steps are those of TinyLlama and Llama-3
// shapes).
static GemmChoice choose_tiles(int m, int n, int k, int epilogue, bool waits) {
    const bool store = epilogue == kEpiStore;
    // A vocabulary-wide head over 129-256 rows (the 256-session decode step):
    // 256 x 256 tiles in 16-wave blocks, four waves per SIMD (128256 columns:
    // 319 us against 339 us with 8-wave 256 x 256 blocks).
    if (m > 128 && m <= 256 && store && n >= 65536) return one_pass({2, 2, 4, 4, 3}, m, n, k);
    if (swiglu_fused(m, epilogue)) {
        // 65-128 rows: 64 x 256 tiles (two row blocks share each weight tile)
        // fill twice the CUs of one 128-row block (decode steps at 96 / 128
        // sessions -4.7 / -4.2 %)
        if (m <= 128) return {{2, 2, 1, 4, 3}, 1};
        // 129-256 rows: 128 x 256 tiles in 16-wave blocks (32 x 64 wave tiles,
        // four waves per SIMD to cover the copies' latency): GEMM class
        // 7.33-7.36 against 7.47-7.50 ms per 256-session step with 8 waves.
        // The store products measured slower in 16-wave blocks.  64 x 256 tiles
        // are faster by themselves where 128-row ones leave CUs idle (256 rows,
        // 11264 columns, K 2048: 35 / 45 us) and slower beside other streams
        // (steps of 208 sessions on three streams, 8 TinyLlama layers: 778 / 751
        // us; 4 layers of a Llama-3 shard: 1037 / 1011).
        if (m <= 256) {
            const GemmChoice w16 = {{1, 2, 4, 4, 3}, 1};
            if (!waits) return w16;
            const GemmChoice c = cheapest(m, n, k, epilogue, {{2, 2, 2, 4, 3}, 1}, true);
            return c.cfg.bm() == 128 && c.cfg.bn() == 256 ? w16 : c;
        }
        // 128 x 512 tiles once they alone fill two passes over the CUs
        const bool wide = ((m + 127) / 128) * ((n + 511) / 512) >= 2 * device_cus();
        return cheapest(m, n, k, epilogue, {wide ? GemmCfg{2, 4, 2, 4, 3} : GemmCfg{2, 2, 2, 4, 3}, 1}, waits);
    }
    // <= 32 rows: a 4-deep ring and one pass of splits over the CUs (TinyLlama
    // shapes at 32 rows, back to back with weights from HBM: QKV 4.84 us
    // against 5.27 with 3 stages and three blocks per CU, gate/up 15.6 against
    // 17.1 (2 slabs instead of 8 for the SwiGLU reduce), down 6.96 against
    // 7.48, LM head 26.8 unsplit against 28.2 + its reduce; O unchanged)
    if (m <= 32) return one_pass({1, 1, 1, 4, 4}, m, n, k);
    // 33-64 rows the same way on 64-row tiles (the tensor-parallel shard step
    // at 64 sessions: 12.6k -> 13.4k tokens/s against ~3 blocks per CU and 3
    // stages, whose 16 slabs each consumer read back)
    if (m <= 64) return one_pass({2, 1, 1, 4, 4}, m, n, k);
    // and the 65-128-row store products (QKV, O, down) on two or more 64-row
    // tiles: fewer split-K slabs for their consumers (decode steps at 96 / 128
    // sessions 10.5 -> 10.2 / 12.4 -> 11.3 ms; at 128 sessions the attention,
    // with RoPE inside, sums q from 2 QKV slabs instead of 10).  At 256 rows
    // the same plan costs the GEMMs what it saves their consumers.
    if (m <= 128 && store && n < 65536) return one_pass({2, 1, 1, 4, 4}, m, n, k);
    // vocabulary-wide heads: 256-row tiles read each weight tile once
    if (n >= 65536) return one_pass(m > 128 ? GemmCfg{2, 4, 4, 2, 3} : GemmCfg{2, 4, 2, 4, 3}, m, n, k);
    const GemmChoice plain = one_pass(n >= 16384 ? GemmCfg{2, 4, 2, 4, 3} : GemmCfg{2, 2, 2, 4, 3}, m, n, k);
    if (m <= 256) return plain;
    // More rows (us per product by itself / beside two more streams, one pass of
    // 128 x 256 tiles and up to 4 splits against this): Llama-3 at 2108 rows QKV
    // 202 / 186 against 187 / 179, O 150 / 129 against 137 / 115 and no slabs,
    // down 479 / 456 against 405 / 432, gate/up at 1000 408 / 394 against 380 /
    // 366; TinyLlama at 1000 gate/up 103 / 82 against 88 / 76, at 300 QKV 12.9 /
    // 11.5 against 12.4 / 8.6 with half the slabs.
    return cheapest(m, n, k, epilogue, plain, waits);
}

GemmPlan gemm_plan(int m, int n, int k, int epilogue, bool waits) {
    GemmPlan p;
    if (few_rows(m, n, epilogue)) {
        p.few_rows = true;
        p.KT = (k + 31) / 32;
        p.NT = (n + 31) / 32;
        p.row_blocks = 1;
        p.col_blocks = epilogue == kEpiSwiGLU ? n / 32 : (n + 15) / 16;
        const int splits = epilogue == kEpiSwiGLU ? 1 : std::max(1, std::min(device_cus() / p.col_blocks, p.KT / 32));
        p.kt_per_split = (p.KT + splits - 1) / splits;
        p.splits = (p.KT + p.kt_per_split - 1) / p.kt_per_split;
        p.direct = p.splits == 1;
        p.ws_floats = p.direct ? 0 : (size_t)p.splits * m * n;
        return p;
    }
    if (swiglu_ksplit(m, n, k, epilogue)) {
        p.KT = (k + 31) / 32;
        p.NT = (n + 31) / 32;
        p.row_blocks = 1;
        p.col_blocks = p.NT / 2;
        p.kt_per_split = p.KT;
        return p;  // one launch, no workspace
    }
    const GemmChoice ch = choose_tiles(m, n, k, epilogue, waits);
    const GemmCfg& c = ch.cfg;
    p.wm = c.wm;
    p.wn = c.wn;
    p.waves_m = c.waves_m;
    p.waves_n = c.waves_n;
    p.stages = c.stages;
    p.KT = (k + 31) / 32;
    p.NT = (n + 31) / 32;
    p.row_blocks = (m + c.bm() - 1) / c.bm();
    p.col_blocks = (p.NT + c.bn() / 32 - 1) / (c.bn() / 32);
    p.kt_per_split = (p.KT + ch.splits - 1) / ch.splits;
    p.splits = (p.KT + p.kt_per_split - 1) / p.kt_per_split;
    p.direct = p.splits == 1 && (epilogue == kEpiStore || swiglu_fused(m, epilogue));
    p.ws_floats = p.direct ? 0 : (size_t)p.splits * m * n;
    return p;
}

template <int WM, int WN, int WAVES_M, int WAVES_N, int STAGES, int HL, int SWIGLU = 0>
static void gemm_launch(const GemmPlan& p, hipStream_t stream, const uint16_t* a, int m, int k, const uint16_t* w,
                        float* c, int n, size_t split_stride, uint16_t* h = nullptr, int h_lo = 0) {
    const unsigned blocks = ((unsigned)p.row_blocks * (unsigned)p.col_blocks * (unsigned)p.splits + 7u) / 8u * 8u;
    hipLaunchKernelGGL((gemm_kernel<WM, WN, WAVES_M, WAVES_N, HL, STAGES, SWIGLU>), dim3(blocks),
                       dim3(WAVES_M * WAVES_N * 64), 0, stream, a, m, k, (const bf16x8*)w, p.KT, p.NT, c, n,
                       p.kt_per_split, p.splits, p.row_blocks, p.col_blocks, split_stride, h, h_lo);
}

template <int NW, int U, int HL, int SWIGLU>
static void few_rows_launch(const GemmPlan& p, hipStream_t stream, const uint16_t* a, int m, const uint16_t* w,
                            float* c, int n, size_t split_stride, uint16_t* h, const NormRows* nr = nullptr) {
    auto go = [&](auto kernel, size_t lds) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)(p.col_blocks * p.splits)), dim3(NW * 64), lds, stream, a, m, w,
                           p.KT, p.NT, c, n, p.kt_per_split, p.splits, split_stride, h, nr ? *nr : NormRows{});
    };
    static_assert(kFewRows == 8 && kNormRows == 2, "row counts below");
    if (nr) {
        if (m == 1) go(gemm_few_rows_kernel<1, NW, U, HL, SWIGLU, 1>, (size_t)p.KT * 64 * HL);
        else go(gemm_few_rows_kernel<2, NW, U, HL, SWIGLU, 1>, (size_t)p.KT * 128 * HL);
        return;
    }
    if (m == 1) go(gemm_few_rows_kernel<1, NW, U, HL, SWIGLU, 0>, 0);
    else if (m == 2) go(gemm_few_rows_kernel<2, NW, U, HL, SWIGLU, 0>, 0);
    else if (m <= 4) go(gemm_few_rows_kernel<4, NW, U, HL, SWIGLU, 0>, 0);
    else go(gemm_few_rows_kernel<8, NW, U, HL, SWIGLU, 0>, 0);
}

// Every workgroup normalises the rows for itself, from L2 and under the flight
// of its first weights: one or two rows cost a product 0-0.8 us where the norm
// launch took 3.6.  Llama-3 steps of 4 layers, us per step replayed on three
// streams / by itself: one row (gate/up 1792 workgroups of 16 KB per row and
// buffer) 470 / 597 inside, 485 / 628 with norm launches.  Past 2048 rows x
// workgroups the rows read again weigh beside the weights and nothing more is
// gained: two rows with gate/up's norms inside 494 / 614, outside 497 / 615.
bool norm_in_gemm(int m, int n, int k, int epilogue) {
    if (m < 1 || m > kNormRows || k > kNormCols || k % 32 != 0 || !few_rows(m, n, epilogue) ||
        2 * packed_weight_elems(k, n) > 0x7fffffffull)
        return false;
    const GemmPlan p = gemm_plan(m, n, k, epilogue);
    return p.direct && m * p.col_blocks <= 2048;
}

zr_status launch_norm_gemm(zr_context* ctx, const float* x, const Slabs& residual, float* x_out, const float* gamma,
                           const uint16_t* w_packed, float* c_f32, uint16_t* c_bf16, int m, int n, int k,
                           int epilogue) {
    if (!norm_in_gemm(m, n, k, epilogue) || x_out == x || (epilogue == kEpiSwiGLU ? !c_bf16 : !c_f32))
        return set_err(ctx, ZR_E_INVARIANT, "no normalising product for %d x %d x %d", m, n, k);
    const GemmPlan p = gemm_plan(m, n, k, epilogue);
    const bool split_act = (ctx->desc.flags & ZR_FLAG_SPLIT_ACTIVATIONS) != 0;
    const NormRows nr = {x, residual.ptr, residual.ptr ? residual.n : 0, residual.stride, x_out, gamma,
                         ctx->desc.rms_norm_eps};
    hipEvent_t ev;
    timing_mark_begin(ctx, kClassGemm, &ev);
    if (epilogue == kEpiSwiGLU) {
        if (split_act)
            few_rows_launch<4, 2, 2, 1>(p, ctx->stream, nullptr, m, w_packed, nullptr, n, 0, c_bf16, &nr);
        else
            few_rows_launch<4, 2, 1, 1>(p, ctx->stream, nullptr, m, w_packed, nullptr, n, 0, c_bf16, &nr);
    } else {
        if (split_act)
            few_rows_launch<4, 4, 2, 0>(p, ctx->stream, nullptr, m, w_packed, c_f32, n, 0, nullptr, &nr);
        else
            few_rows_launch<4, 4, 1, 0>(p, ctx->stream, nullptr, m, w_packed, c_f32, n, 0, nullptr, &nr);
    }
    ZR_LAUNCH_CHECK(ctx);
    timing_mark_end(ctx, kClassGemm, ev);
    return ZR_OK;
}

zr_status launch_gemm(zr_context* ctx, const uint16_t* a, const uint16_t* w_packed, float* c_f32,
                      uint16_t* c_bf16, int m, int n, int k, int epilogue, Slabs* deferred, bool waits) {
    if (deferred && (epilogue != kEpiStore || !c_f32 || c_bf16))
        return set_err(ctx, ZR_E_INVARIANT, "deferred split-K needs an f32 store epilogue");
    if (m <= 0) return ZR_OK;
    if (k % 32 != 0) return set_err(ctx, ZR_E_UNSUPPORTED, "GEMM K=%d must be a multiple of 32", k);
    // the kernel addresses its operands with 32-bit buffer offsets
    const size_t a_bytes = 2 * 2 * a_plane(m, k), w_bytes = 2 * packed_weight_elems(k, n);
    if (a_bytes > 0x7fffffffull || w_bytes > 0x7fffffffull)
        return set_err(ctx, ZR_E_UNSUPPORTED, "GEMM operands of %zu / %zu bytes exceed 2 GiB", a_bytes, w_bytes);
    const bool split_act = (ctx->desc.flags & ZR_FLAG_SPLIT_ACTIVATIONS) != 0;
    const GemmPlan p = gemm_plan(m, n, k, epilogue, waits);
    const bool in_launch = p.few_rows ? epilogue == kEpiSwiGLU : swiglu_ksplit(m, n, k, epilogue);
    if (in_launch && (!c_bf16 || c_f32 || deferred))
        return set_err(ctx, ZR_E_INVARIANT, "K-split SwiGLU (M=%d) writes the bf16 operand only", m);
    hipEvent_t ev;
    if (in_launch && p.few_rows) {
        timing_mark_begin(ctx, kClassGemm, &ev);
        if (split_act)
            few_rows_launch<4, 2, 2, 1>(p, ctx->stream, a, m, w_packed, nullptr, n, 0, c_bf16);
        else
            few_rows_launch<4, 2, 1, 1>(p, ctx->stream, a, m, w_packed, nullptr, n, 0, c_bf16);
        ZR_LAUNCH_CHECK(ctx);
        timing_mark_end(ctx, kClassGemm, ev);
        return ZR_OK;
    }
    if (in_launch) {
        timing_mark_begin(ctx, kClassGemm, &ev);
#define ZR_KSPLIT(HLV, MTV)                                                                                     \
    hipLaunchKernelGGL((gemm_swiglu_ksplit_kernel<3, HLV, MTV>), dim3(p.col_blocks), dim3(256), 0, ctx->stream, a, \
                       m, k, (const bf16x8*)w_packed, p.KT, n, c_bf16, HLV - 1)
        if (split_act) {
            if (m > 32)
                ZR_KSPLIT(2, 2);
            else
                ZR_KSPLIT(2, 1);
        } else {
            if (m > 32)
                ZR_KSPLIT(1, 2);
            else
                ZR_KSPLIT(1, 1);
        }
#undef ZR_KSPLIT
        ZR_LAUNCH_CHECK(ctx);
        timing_mark_end(ctx, kClassGemm, ev);
        return ZR_OK;
    }
    if (swiglu_fused(m, epilogue) && (!c_bf16 || c_f32 || n % 64 != 0))
        return set_err(ctx, ZR_E_INVARIANT, "fused SwiGLU writes the bf16 operand only (N=%d)", n);
    const bool fused = swiglu_fused(m, epilogue);
    const bool direct = (p.direct && c_f32 && !c_bf16 && epilogue == kEpiStore) || fused;
    const size_t split_stride = (size_t)m * n;
    if (!direct && (size_t)p.splits * split_stride > ctx->splitk_ws_floats)
        return set_err(ctx, ZR_E_OOM, "split-K workspace too small (%d x %d x %d)", p.splits, m, n);
    float* dst = direct ? c_f32 : ctx->splitk_ws;
    timing_mark_begin(ctx, kClassGemm, &ev);
    bool launched = false;
    if (p.few_rows) {
        if (split_act)
            few_rows_launch<4, 4, 2, 0>(p, ctx->stream, a, m, w_packed, dst, n, split_stride, nullptr);
        else
            few_rows_launch<4, 4, 1, 0>(p, ctx->stream, a, m, w_packed, dst, n, split_stride, nullptr);
        launched = true;
    }
#define ZR_GEMM_FUSED_CASE(WMV, WNV, WAM, WAN, ST)                                                     \
    if (fused && !launched && p.wm == WMV && p.wn == WNV && p.waves_m == WAM && p.waves_n == WAN &&    \
        p.stages == ST) {                                                                              \
        if (split_act)                                                                                 \
            gemm_launch<WMV, WNV, WAM, WAN, ST, 2, 1>(p, ctx->stream, a, m, k, w_packed, nullptr, n, 0, c_bf16, 1); \
        else                                                                                           \
            gemm_launch<WMV, WNV, WAM, WAN, ST, 1, 1>(p, ctx->stream, a, m, k, w_packed, nullptr, n, 0, c_bf16, 0); \
        launched = true;                                                                               \
    }
    ZR_GEMM_FUSED_CASE(2, 4, 2, 4, 3)
    ZR_GEMM_FUSED_CASE(2, 2, 2, 4, 3)
    ZR_GEMM_FUSED_CASE(2, 2, 1, 4, 3)
    ZR_GEMM_FUSED_CASE(1, 2, 4, 4, 3)
    ZR_GEMM_FUSED_CASE(2, 2, 3, 4, 3)
    ZR_GEMM_FUSED_CASE(2, 2, 4, 4, 3)
#undef ZR_GEMM_FUSED_CASE
#define ZR_GEMM_CASE(WMV, WNV, WAM, WAN, ST)                                                           \
    if (!fused && !launched && p.wm == WMV && p.wn == WNV && p.waves_m == WAM && p.waves_n == WAN &&   \
        p.stages == ST) {                                                                              \
        if (split_act)                                                                                 \
            gemm_launch<WMV, WNV, WAM, WAN, ST, 2>(p, ctx->stream, a, m, k, w_packed, dst, n, split_stride); \
        else                                                                                           \
            gemm_launch<WMV, WNV, WAM, WAN, ST, 1>(p, ctx->stream, a, m, k, w_packed, dst, n, split_stride); \
        launched = true;                                                                               \
    }
    ZR_GEMM_CASE(1, 1, 1, 4, 4)
    ZR_GEMM_CASE(2, 1, 1, 4, 4)
    ZR_GEMM_CASE(2, 2, 1, 4, 3)
    ZR_GEMM_CASE(2, 2, 3, 4, 3)
    ZR_GEMM_CASE(2, 2, 4, 4, 3)
    ZR_GEMM_CASE(2, 4, 4, 2, 3)
    ZR_GEMM_CASE(2, 4, 2, 4, 3)
    ZR_GEMM_CASE(2, 2, 2, 4, 3)
#undef ZR_GEMM_CASE
    if (!launched) return set_err(ctx, ZR_E_INVARIANT, "no GEMM kernel for the selected tile configuration");
    ZR_LAUNCH_CHECK(ctx);
    timing_mark_end(ctx, kClassGemm, ev);
    if (deferred) {
        *deferred = direct ? Slabs(c_f32) : Slabs(ctx->splitk_ws, p.splits, split_stride);
        return ZR_OK;
    }
    if (!direct) {
        timing_mark_begin(ctx, kClassOther, &ev);
        const size_t n_out = epilogue == kEpiSwiGLU ? (size_t)n / 2 : (size_t)n;
        const size_t total = (size_t)m * n_out;
        const unsigned blocks = (unsigned)std::min<size_t>((total + 255) / 256, 65535);
        hipLaunchKernelGGL(splitk_reduce_kernel, dim3(blocks), dim3(256), 0, ctx->stream, ctx->splitk_ws, p.splits,
                           m, n, split_stride, epilogue, c_f32, c_bf16, split_act ? 1 : 0);
        ZR_LAUNCH_CHECK(ctx);
        timing_mark_end(ctx, kClassOther, ev);
    }
    return ZR_OK;
}

}  // namespace zr
