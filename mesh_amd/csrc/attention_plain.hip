// Paged attention over plain-layout pools (tiles row-major [16 rows][D]) whose
// head_dim is a multiple of 4: every head_dim but 64 / 128, and any number of
// q heads per kv head.
//
// Reference semantics as in attention.hip (forward_pass.rs:2764-2895,
// 1317-1372): query row r of a sequence with `prefix` cached rows sees keys
// [0, prefix + r].
//
// Work decomposition.  The (row, q head) pairs of one kv head and sequence are
// columns, row-major; a tile is up to 16 CT of them, and a workgroup of nw
// waves owns one (tile, kv head).  Wave w walks pages w, w + nw, ... of the
// tile's visible window, so a page is read once per 16 CT columns, and the
// waves' (m, l, O) meet in LDS at the end: no partials in memory, no merge
// launch.  Tiles with the most pages are dispatched first; with kv_heads a
// multiple of 8 the tiles that share pages run on one XCD.
//
// Arithmetic is f32 throughout (v_mfma_f32_16x16x4_f32; bf16 pages are
// widened exactly), as the scalar kernel's: the bf16 units' hi + lo halves
// would keep 16 of the operands' 24 bits.  With lane l, column c = l % 16,
// quad q4 = l / 16, a page's 16 keys take
//   S[key][c] += K[key][d] Q[c][d]: step (j, e) sums dims 16 j + 4 q4 + e, so a
//     lane's K operand is 4 consecutive dims of key l % 16;
//   O[d][c] += V[key][d] P[key][c]: step i sums keys 4 q4 + i, which are the
//     lane's own scores; block b of a group of R 16-dim blocks holds dims
//     base + R (l % 16) + b, so a lane's V operand is R consecutive dims.
//
// Bound by the f32 matrix rate (157 TFLOP/s) for chunks and by HBM for decode
// rows.  Measured (32 heads of 80, bf16 pool, a 333-row chunk on a 700-row
// prefix beside 15 decode rows of ~900 keys, RoPE + append + attention with
// both calls' synchronisation): 111 us against 1781 us with the scalar kernel
// (one wave per row and q head, every K / V row read once per q head).
#include "zr_internal.h"

namespace zr {

struct PlainAttnArgs {
    const float* q;            // [T, q_cols]
    int q_cols;
    const void* pool;          // layer base of the pool
    size_t page_elems;
    const int* block_tables;
    int stride;
    const int* first_offset;
    const int* kv_before;
    const int* cu_q;
    const int4* tiles;         // {seq, first column, columns, pages}
    int D, G, kv_heads;
    float scale_log2;          // log2(e) / sqrt(D)
    float* out_f32;
    uint16_t* out_bf16;
    size_t out_lo_offset;
};

template <typename KV> struct Quad;
template <> struct Quad<float> {
    f32x4 v;
    __device__ inline void load(const float* p) { v = *(const f32x4*)p; }
    __device__ inline void clear() { v = f32x4{0.f, 0.f, 0.f, 0.f}; }
    __device__ inline float get(int i) const { return v[i]; }
};
template <> struct Quad<uint16_t> {
    uint2 v;
    __device__ inline void load(const uint16_t* p) { v = *(const uint2*)p; }
    __device__ inline void clear() { v = make_uint2(0, 0); }
    __device__ inline float get(int i) const {
        const uint32_t w = i < 2 ? v.x : v.y;
        return __uint_as_float(i & 1 ? w & 0xffff0000u : w << 16);
    }
};

__device__ inline float widen(float x) { return x; }
__device__ inline float widen(uint16_t x) { return bf16_bits_to_f32(x); }

// max over the lanes {l, l ^ 16, l ^ 32, l ^ 48} (the quads of one column)
__device__ inline float column_max(float x) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// One page's V operand: NB / 4 groups of 4 blocks (one 4-element load per key
// and lane each), then a group of R = NB % 4 blocks.
template <typename KV, int NB> struct PageV {
    static constexpr int NG = NB / 4, R = NB % 4;
    Quad<KV> g[4][NG > 0 ? NG : 1];
    KV r[4][R > 0 ? R : 1];
    __device__ inline float get(int i, int b) const {
        return b < 4 * NG ? g[i][b / 4].get(b % 4) : widen(r[i][b - 4 * NG]);
    }
};

template <typename KV, int NB> struct PageK {
    Quad<KV> k[NB];
};

// Registers: 8 waves (256 each) up to 128 dims, 4 waves (512) above.
constexpr int plain_max_waves(int nb) { return nb > 8 ? 4 : 8; }

template <typename KV, int NB, int CT>
__global__ __launch_bounds__(plain_max_waves(NB) * 64) void paged_attention_plain_kernel(
    PlainAttnArgs a, const int* __restrict__ block_tables) {
    extern __shared__ float comb[];  // [nw / 2][CT][NB + 1][4][64]: the waves' O, then (m, l)
    constexpr int NG = NB / 4, R = NB % 4;
    const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tile = blockIdx.x / a.kv_heads, kvh = blockIdx.x - tile * a.kv_heads;
    const int4 tl = a.tiles[tile];
    const int seq = __builtin_amdgcn_readfirstlane(tl.x), c0 = __builtin_amdgcn_readfirstlane(tl.y);
    const int ncols = __builtin_amdgcn_readfirstlane(tl.z), npages = __builtin_amdgcn_readfirstlane(tl.w);
    const int D = a.D, G = a.G;
    const int c = lane & 15, q4 = lane >> 4;
    const int kvb = __builtin_amdgcn_readfirstlane(a.kv_before[seq]);
    const int fo = __builtin_amdgcn_readfirstlane(a.first_offset[seq]);
    const int row0 = __builtin_amdgcn_readfirstlane(a.cu_q[seq]);
    const int* bt = block_tables + (size_t)seq * a.stride;
    const KV* pool = (const KV*)a.pool + (size_t)kvh * kPageRows * D;
    const size_t v_block = (size_t)a.kv_heads * kPageRows * D;
    const bool two = CT == 2 && ncols > 16;  // (uniform) the second column tile is live

    // Q, scaled into log2 units, and each column's last visible key
    float qf[CT][NB * 4];
    int jmax[CT], row[CT], head[CT];
    bool live[CT];
#pragma unroll
    for (int t = 0; t < CT; ++t) {
        const int col = t * 16 + c;
        live[t] = col < ncols;
        const int cc = c0 + (live[t] ? col : 0);
        const int r = cc / G;
        row[t] = row0 + r;
        head[t] = kvh * G + (cc - r * G);
        jmax[t] = kvb + r;
        const float* qp = a.q + (size_t)row[t] * a.q_cols + (size_t)head[t] * D + 4 * q4;
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            // heads of D % 4 == 0 floats in rows of q_cols (a multiple of 32): 16-byte aligned
            const f32x4 x = 16 * j + 4 * q4 < D ? *(const f32x4*)(qp + 16 * j) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < 4; ++e) qf[t][4 * j + e] = x[e] * a.scale_log2;
        }
    }

    auto load_k = [&](PageK<KV, NB>& k, int page) {
        const KV* p = pool + (size_t)page * a.page_elems + (size_t)c * D + 4 * q4;
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            if (16 * j + 4 * q4 < D)
                k.k[j].load(p + 16 * j);
            else
                k.k[j].clear();
        }
    };
    auto load_v = [&](PageV<KV, NB>& v, int page) {
        const KV* p = pool + (size_t)page * a.page_elems + v_block + (size_t)(4 * q4) * D;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                if (64 * g + 4 * c < D)
                    v.g[i][g].load(p + (size_t)i * D + 64 * g + 4 * c);
                else
                    v.g[i][g].clear();
            }
#pragma unroll
            for (int b = 0; b < R; ++b) {
                const int d = 64 * NG + R * c + b;
                v.r[i][b] = d < D ? p[(size_t)i * D + d] : KV(0);
            }
        }
    };

    f32x4 o[CT][NB];
    float m[CT], l[CT];
#pragma unroll
    for (int t = 0; t < CT; ++t) {
        m[t] = -INFINITY;
        l[t] = 0.0f;
#pragma unroll
        for (int b = 0; b < NB; ++b) o[t][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // The next page's loads are issued before this page's arithmetic where
    // both fit the registers of 8 waves per CU (4 above 128 dims), by the
    // compiler's report, and the columns of a page with values that are not
    // finite (below) go block by block of dims where a column's whole row of V,
    // widened at once, would not.  The 32-column forms of 81-128 dims spilled
    // 180-440 bytes, in the page loop for bf16, and those above 192 dims 112; now
    // none does, but 88 bytes with 81-96 bf16 dims (reading ahead still gains
    // there: 1047 us against 1205) and 68 with 113-128 bf16 ones, 184 with f32
    // ones, both off the loop's straight path.  Two 1000-row chunks on 3000 rows,
    // us before / now: 32 heads of 96, bf16 1092 / 1047, f32 1572 / 1106; 40 heads
    // of 128 on 8, bf16 3925 / 1664; 32 heads of 112, bf16 2810 / 1340.
    constexpr bool kAhead = NB > 8    ? NB < 16
                            : CT == 2 ? NB < 6 || (NB == 6 && sizeof(KV) == 2)
                                      : NB < 8 || sizeof(KV) == 2;
    constexpr bool kByBlock = NB >= 6 && !(NB == 8 && sizeof(KV) == 4);

    // keys below `free_end` are visible to every column of the tile
    const int free_end = kvb + c0 / G + 1;
    auto page_step = [&](const PageK<KV, NB>& k, const PageV<KV, NB>& v, int p) {
        const int j0 = p * kPageRows - fo;  // logical key of the page's first row
        const bool edge = j0 < 0 || j0 + kPageRows > free_end;
        float pr[CT][4];
#pragma unroll
        for (int t = 0; t < CT; ++t) {
            if (t == 1 && !two) continue;
            f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (e & 1)
                        s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k.k[j].get(e), qf[t][4 * j + e], s1, 0, 0, 0);
                    else
                        s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k.k[j].get(e), qf[t][4 * j + e], s0, 0, 0, 0);
                }
            float s[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[i] = s0[i] + s1[i];
                const int key = j0 + 4 * q4 + i;
                if (edge && (key < 0 || key > jmax[t])) s[i] = -INFINITY;
            }
            const float mn = fmaxf(m[t], column_max(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))));
            const float mu = mn == -INFINITY ? 0.0f : mn;  // no visible key yet
            const float alpha = exp2f(m[t] - mu);
            m[t] = mn;
            float ps = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                pr[t][i] = exp2f(s[i] - mu);
                ps += pr[t][i];
            }
            l[t] = l[t] * alpha + ps;
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int i = 0; i < 4; ++i) o[t][b][i] *= alpha;
        }
        // Rows that a column does not see have weight 0, but 0 x inf is NaN:
        // an edge page (rows of an earlier owner before or after the window,
        // keys of later rows of the chunk) with a V value that is not finite
        // takes its columns one at a time, with unseen rows cleared.
        if (edge) {
            bool bad = false;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int b = 0; b < NB; ++b) bad |= !(fabsf(v.get(i, b)) < INFINITY);
            if (__any(bad)) {
#pragma unroll
                for (int t = 0; t < CT; ++t) {
                    if (t == 1 && !two) continue;
                    if constexpr (kByBlock) {
#pragma unroll
                        for (int b = 0; b < NB; ++b)
#pragma clang loop unroll(disable)
                            for (int cs = 0; cs < 16; ++cs) {
                                const int jm = __shfl(jmax[t], cs, 64);
                                f32x4 x = o[t][b];
#pragma unroll
                                for (int i = 0; i < 4; ++i) {
                                    const int key = j0 + 4 * q4 + i;
                                    const float vv = key >= 0 && key <= jm ? v.get(i, b) : 0.0f;
                                    x = __builtin_amdgcn_mfma_f32_16x16x4f32(vv, pr[t][i], x, 0, 0, 0);
                                }
                                if (c == cs) o[t][b] = x;
                            }
                    } else {
                        for (int cs = 0; cs < 16; ++cs) {
                            const int jm = __shfl(jmax[t], cs, 64);
#pragma unroll
                            for (int b = 0; b < NB; ++b) {
                                f32x4 x = o[t][b];
#pragma unroll
                                for (int i = 0; i < 4; ++i) {
                                    const int key = j0 + 4 * q4 + i;
                                    const float vv = key >= 0 && key <= jm ? v.get(i, b) : 0.0f;
                                    x = __builtin_amdgcn_mfma_f32_16x16x4f32(vv, pr[t][i], x, 0, 0, 0);
                                }
                                if (c == cs) o[t][b] = x;
                            }
                        }
                    }
                }
                return;
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const float vv = v.get(i, b);
                o[0][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv, pr[0][i], o[0][b], 0, 0, 0);
                if constexpr (CT == 2)
                    if (two) o[1][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv, pr[1][i], o[1][b], 0, 0, 0);
            }
    };

    if constexpr (kAhead) {
        PageK<KV, NB> k[2];
        PageV<KV, NB> v[2];
        if (wave < npages) {
            const int pg = __builtin_amdgcn_readfirstlane(bt[wave]);
            load_k(k[0], pg);
            load_v(v[0], pg);
        }
        for (int p = wave; p < npages; p += 2 * nw) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int pp = p + u * nw;
                if (pp >= npages) break;
                if (pp + nw < npages) {
                    const int pg = __builtin_amdgcn_readfirstlane(bt[pp + nw]);
                    load_k(k[1 - u], pg);
                    load_v(v[1 - u], pg);
                }
                page_step(k[u], v[u], pp);
            }
        }
    } else {
        for (int p = wave; p < npages; p += nw) {
            PageK<KV, NB> k;
            PageV<KV, NB> v;
            const int pg = __builtin_amdgcn_readfirstlane(bt[p]);
            load_k(k, pg);
            load_v(v, pg);
            page_step(k, v, p);
        }
    }
#pragma unroll
    for (int t = 0; t < CT; ++t) {
        l[t] += __shfl_xor(l[t], 16, 64);
        l[t] += __shfl_xor(l[t], 32, 64);
    }

    // The waves' halves meet pairwise in LDS until wave 0 holds the tile (a
    // wave without a visible key has m = -inf, l = 0, O = 0 and weight 0).
    for (int n = nw; n > 1; n >>= 1) {
        const int h = n >> 1;
        __syncthreads();
        if (wave >= h && wave < n) {
            float* w = comb + (size_t)(wave - h) * CT * (NB + 1) * 256 + lane;
#pragma unroll
            for (int t = 0; t < CT; ++t) {
                float* wt = w + t * (NB + 1) * 256;
#pragma unroll
                for (int b = 0; b < NB; ++b)
#pragma unroll
                    for (int i = 0; i < 4; ++i) wt[(b * 4 + i) * 64] = o[t][b][i];
                wt[NB * 256] = m[t];
                wt[NB * 256 + 64] = l[t];
            }
        }
        __syncthreads();
        if (wave < h) {
            const float* w = comb + (size_t)wave * CT * (NB + 1) * 256 + lane;
#pragma unroll
            for (int t = 0; t < CT; ++t) {
                const float* wt = w + t * (NB + 1) * 256;
                const float m1 = wt[NB * 256], l1 = wt[NB * 256 + 64];
                const float mm = fmaxf(m[t], m1);
                const float f0 = m[t] == -INFINITY ? 0.0f : exp2f(m[t] - mm);
                const float f1 = m1 == -INFINITY ? 0.0f : exp2f(m1 - mm);
                m[t] = mm;
                l[t] = l[t] * f0 + l1 * f1;
#pragma unroll
                for (int b = 0; b < NB; ++b)
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[t][b][i] = o[t][b][i] * f0 + wt[(b * 4 + i) * 64] * f1;
            }
        }
    }
    if (wave != 0) return;
#pragma unroll
    for (int t = 0; t < CT; ++t) {
        if (!live[t]) continue;
        const float inv = 1.0f / l[t];
        const int col0 = head[t] * D;
        auto put4 = [&](int d, const float* y) {  // 4 consecutive dims, d % 4 == 0
            if (d >= D) return;
            if (a.out_bf16) {
                ushort4 hi, lo;
                split_bf16(y[0], hi.x, lo.x);
                split_bf16(y[1], hi.y, lo.y);
                split_bf16(y[2], hi.z, lo.z);
                split_bf16(y[3], hi.w, lo.w);
                const size_t idx = a_pack_index(row[t], col0 + d, a.q_cols);
                *(ushort4*)(a.out_bf16 + idx) = hi;
                if (a.out_lo_offset) *(ushort4*)(a.out_bf16 + a.out_lo_offset + idx) = lo;
            } else {
                *(f32x4*)(a.out_f32 + (size_t)row[t] * a.q_cols + col0 + d) = f32x4{y[0], y[1], y[2], y[3]};
            }
        };
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float y[4] = {o[t][4 * g][i] * inv, o[t][4 * g + 1][i] * inv, o[t][4 * g + 2][i] * inv,
                                    o[t][4 * g + 3][i] * inv};
                put4(64 * g + 4 * (4 * q4 + i), y);
            }
        // the last R blocks: the lane's 4 rows of each are the 4 R consecutive dims 64 NG + 4 R q4 + [0, 4 R)
#pragma unroll
        for (int w = 0; w < R; ++w) {
            float y[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) y[x] = o[t][4 * NG + (4 * w + x) % R][(4 * w + x) / R] * inv;
            put4(64 * NG + 4 * R * q4 + 4 * w, y);
        }
    }
}

template <typename KV, int NB>
static void launch_plain(const PlainAttnArgs& a, int n_tiles, int ct, int nw, hipStream_t stream,
                         const int* block_tables) {
    const dim3 grid((unsigned)n_tiles * a.kv_heads), block(nw * 64);
    const size_t lds = (size_t)(nw / 2) * ct * (NB + 1) * 256 * sizeof(float);
    if constexpr (NB <= 8) {
        if (ct == 2) {
            hipLaunchKernelGGL((paged_attention_plain_kernel<KV, NB, 2>), grid, block, lds, stream, a, block_tables);
            return;
        }
    }
    hipLaunchKernelGGL((paged_attention_plain_kernel<KV, NB, 1>), grid, block, lds, stream, a, block_tables);
}

template <typename KV>
static bool launch_plain_dims(const PlainAttnArgs& a, int n_tiles, int ct, int nw, hipStream_t s, const int* bt) {
    const int nb = (a.D + 15) / 16;
    if (nb <= 1) launch_plain<KV, 1>(a, n_tiles, ct, nw, s, bt);
    else if (nb == 2) launch_plain<KV, 2>(a, n_tiles, ct, nw, s, bt);
    else if (nb == 3) launch_plain<KV, 3>(a, n_tiles, ct, nw, s, bt);
    else if (nb == 4) launch_plain<KV, 4>(a, n_tiles, ct, nw, s, bt);
    else if (nb == 5) launch_plain<KV, 5>(a, n_tiles, ct, nw, s, bt);
    else if (nb == 6) launch_plain<KV, 6>(a, n_tiles, ct, nw, s, bt);
    else if (nb == 7) launch_plain<KV, 7>(a, n_tiles, ct, nw, s, bt);
    else if (nb == 8) launch_plain<KV, 8>(a, n_tiles, ct, nw, s, bt);
    else if (nb <= 10) launch_plain<KV, 10>(a, n_tiles, ct, nw, s, bt);
    else if (nb <= 12) launch_plain<KV, 12>(a, n_tiles, ct, nw, s, bt);
    else if (nb <= 16) launch_plain<KV, 16>(a, n_tiles, ct, nw, s, bt);
    else return false;
    return true;
}

// Tiles of 32 columns share each page among twice the columns but halve the
// workgroups; 8 waves per tile instead of 4 halve a tile's chain of pages.
// Both follow the fill: about 4 waves per SIMD's worth of workgroups first.
PlainAttnPlan plain_attention_plan(int head_dim, int kv_heads, int G, const int* q_len, int n) {
    PlainAttnPlan p;
    const bool wide_ok = head_dim <= 128;
    long t16 = 0, t32 = 0;
    bool wide = false;
    for (int s = 0; s < n; ++s) {
        const long cols = (long)q_len[s] * G;
        t16 += (cols + 15) / 16;
        t32 += (cols + 31) / 32;
        wide |= cols > 16;
    }
    p.ct = wide_ok && wide && t32 * kv_heads >= 256 ? 2 : 1;
    const long wgs = (p.ct == 2 ? t32 : t16) * kv_heads;
    // (8 waves where their exchange fits 64 KiB of LDS)
    p.waves = head_dim <= 128 && wgs < 512 && 4 * p.ct * ((head_dim + 15) / 16 + 1) <= 64 ? 8 : 4;
    return p;
}

zr_status launch_attention_plain(zr_context* ctx, StagedMeta* st, int layer, const float* q, float* out,
                                 uint16_t* out_bf16) {
    PlainAttnArgs a;
    a.q = q;
    a.q_cols = ctx->q_cols;
    a.page_elems = (size_t)2 * ctx->kv_cols * kPageRows;
    const size_t esz = ctx->desc.kv_dtype == ZR_DTYPE_BF16 ? 2 : 4;
    a.pool = (const char*)ctx->kv_pool + (size_t)layer * ctx->n_pages * a.page_elems * esz;
    a.block_tables = st->block_tables;
    a.stride = st->stride;
    a.first_offset = st->first_offset;
    a.kv_before = st->kv_before;
    a.cu_q = st->cu_q;
    a.tiles = st->pblocks;
    a.D = ctx->head_dim;
    a.G = ctx->q_per_kv;
    a.kv_heads = ctx->local_kv_heads;
    a.scale_log2 = 1.4426950408889634f / sqrtf((float)ctx->head_dim);
    a.out_f32 = out;
    a.out_bf16 = out_bf16;
    a.out_lo_offset = (ctx->desc.flags & ZR_FLAG_SPLIT_ACTIVATIONS) ? a_plane(st->total_q, ctx->q_cols) : 0;
    hipEvent_t ev;
    timing_mark_begin(ctx, kClassAttention, &ev);
    const bool ok = esz == 2 ? launch_plain_dims<uint16_t>(a, st->n_pblocks, st->plain.ct, st->plain.waves, ctx->stream,
                                                           st->block_tables)
                             : launch_plain_dims<float>(a, st->n_pblocks, st->plain.ct, st->plain.waves, ctx->stream,
                                                        st->block_tables);
    if (!ok) return set_err(ctx, ZR_E_UNSUPPORTED, "head_dim %d above 256", ctx->head_dim);
    ZR_LAUNCH_CHECK(ctx);
    timing_mark_end(ctx, kClassAttention, ev);
    return ZR_OK;
}

}  // namespace zr
