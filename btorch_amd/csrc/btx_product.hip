// The sparse product as a layer of its own and its backward, y = x W.
//
// Layouts as in btx_spmv.hip: CSR by source (row_ptr, col; destinations
// ascending) and the same edges destination-major (csc_ptr, csc_src; sources
// ascending).  Weights come in the destination-major order, the layer's own
// parameter order; perm[k] is the position there of CSR edge k.
//
// Every destination sums its terms in ascending source order from +0.0f with
// one fmaf per source with x != 0, so y equals torch.sparse.mm on the CPU bit
// for bit (btorch/models/linear.py:474-483).  Three forms, none of which
// stores a term:
//   rows     a workgroup takes one row of x and a tile of destinations held in
//            LDS, and streams the rows of W of the row's nonzero sources in
//            ascending order: a source's destinations are distinct, so its
//            terms need no atomics, and a barrier between sources keeps the
//            order.  Costs the active sources, whatever the edges.
//   columns  a quarter wavefront takes a destination and 64 rows of x
//            (transposed, so that a source's 64 values are one 256-byte read)
//            and walks the destination's edges.  Costs every edge, whatever the activity.
//   few      a wavefront takes a destination and four rows of x and gathers: one
//            launch, for products of few edges.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "../../include/btorch_amd.h"
#include "btx_common.h"

namespace btx {

constexpr int kRowTile = 16384;      // destinations of a `rows` workgroup, at most (64 KB of LDS)
constexpr int kSegment = 1024;       // values of a row that are counted and listed together
constexpr int kGroup = 64;           // rows of x per wavefront of the `columns` form
constexpr int64_t kFewRows = 4;      // rows of x of a wavefront of k_product_few

struct ProductArgs {
    const int64_t* row_ptr;
    const int32_t* col;
    const int64_t* perm;
    const int64_t* csc_ptr;
    const int32_t* csc_src;
    const float* w;       // destination-major order
    int64_t n_src;
    int64_t n_dst;
    int64_t nnz;
    const float* x;       // (rows, n_src), row stride x_stride
    int64_t x_stride;
    int64_t rows;
    float* y;             // (rows, n_dst)
    float* xt;            // [groups][n_src][64]
    int32_t* counts;      // nonzeros of each listed row
    int32_t* seg_counts;  // [segments][rows] nonzeros of every kSegment values
    int segments;
    int32_t* by_columns;  // [groups] 1 = left to the columns; NULL = the `rows` form takes all
    int most;             // nonzeros a row, on average of a group, up to which the `rows`
                          // form takes the group
};

// Whether the `rows` form takes the 64 rows of group g (decided for the group: a
// form's cost is the same for one of its rows as for all); every thread of the
// wavefront calls it.
__device__ __forceinline__ bool group_by_rows(const ProductArgs& a, int64_t g) {
    const int64_t row = g * kGroup + (threadIdx.x & 63);
    int64_t c = 0;
    if (row < a.rows)
#pragma unroll 8
        for (int s = 0; s < a.segments; ++s) c += a.seg_counts[s * a.rows + row];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    const int64_t here = a.rows - g * kGroup < kGroup ? a.rows - g * kGroup : kGroup;
    return c <= a.most * here;
}

// Nonzeros of every segment of every row, a wavefront each (a workgroup a row
// would take 30 us for 12,800 rows of 200 values).
__global__ __launch_bounds__(256) void k_row_counts(ProductArgs a) {
    const int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (item >= a.rows * a.segments) return;
    const int64_t row = item % a.rows, i0 = item / a.rows * kSegment;
    const int64_t i1 = i0 + kSegment < a.n_src ? i0 + kSegment : a.n_src;
    const float* xr = a.x + row * a.x_stride;
    int c = 0;
#pragma unroll 16
    for (int64_t i = i0 + (threadIdx.x & 63); i < i1; i += 64) c += xr[i] != 0.f;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    if ((threadIdx.x & 63) == 0) a.seg_counts[item] = c;
}

__device__ inline int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ inline int64_t uniform(int64_t v) {
    return (int64_t)((uint64_t)(uint32_t)uniform((int)(v >> 32)) << 32 | (uint32_t)uniform((int)v));
}
__device__ inline float uniform(float v) { return __int_as_float(uniform(__float_as_int(v))); }

// One row of x, destinations [d0, d0 + tile): the row's nonzero sources go through
// LDS in ascending order, L at a time, each with its row of W.  Bound by the
// instructions and the latency of a source's few edges per thread, whose weights
// perm scatters over the array, and with several wavefronts by the barrier per
// source: U sources are requested together, the next U before the current ones
// are added, without a branch per load (which waited for each: 0.18 against 0.13
// us a source of 20 edges), and a few rows are split into tiles over the CUs.  T
// threads by the edges of a source; one wavefront alone needs no barrier.  0.13
// to 0.17 us a source of 10 to 40 edges by 64 threads, 0.25 us of 163 by 256, 0.4
// us of 819 by 1024.  8000 x 1000, 20 edges a source, 4000 rows, 0.5 % active: 94
// us (1024 threads for every net, which scanned x in every workgroup: 332); 200 x
// 16384, 819 edges a source, 12,800 rows, 2.5 % active: 341 us with its lists (402).
// Taken back: three requests in flight (no faster by 64 or 256 threads; by 1024 one
// workgroup per CU).  Edge: an integer that holds the edges' positions.
template <typename Edge, int T>
__global__ __launch_bounds__(T, T == 1024 && sizeof(Edge) == 4 ? 8 : 1) void k_product_rows(
    ProductArgs a, int tile) {
    constexpr int U = T == 64 ? 16 : 8;
    constexpr int L = T == 64 ? 256 : T;   // sources a list in LDS holds
    using UEdge = std::conditional_t<sizeof(Edge) == 4, uint32_t, uint64_t>;
    extern __shared__ __align__(16) float s_y[];
    __shared__ Edge s_beg[L];
    __shared__ int s_len[L];
    __shared__ float s_x[L];
    const int tid = threadIdx.x;
    const int64_t row = blockIdx.x, d0 = (int64_t)blockIdx.y * tile;
    const int nd = (int)(a.n_dst - d0 < tile ? a.n_dst - d0 : tile);
    const float* xr = a.x + row * a.x_stride;
    if (a.by_columns != nullptr && a.by_columns[row / kGroup]) return;  // uniform
    const int spare = tile + 3;  // s_y is filled by four
    for (int q = tid; q < (nd + 3) / 4; q += T)
        reinterpret_cast<float4*>(s_y)[q] = make_float4(0.f, 0.f, 0.f, 0.f);
    // adds the `total` listed sources; every load is made, of edge 0 by threads
    // without one, and what is not this tile's goes to a value that is not kept
    // (a branch per load would wait for each)
    auto add = [&](int total) {
        if (a.nnz == 0) return;  // uniform
        const unsigned from = (unsigned)d0, many = (unsigned)nd;
        auto slot = [&](bool in, int col) {
            const unsigned q = (unsigned)col - from;
            return in && q < many ? (int)q : spare;
        };
        // this thread's first edge of U sources, with what the sources share
        auto ask = [&](int k0, int* d, Edge* pm, int* len, float* xk) {
            Edge beg[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                beg[u] = uniform(s_beg[k0 + u]);
                len[u] = uniform(s_len[k0 + u]);
                xk[u] = uniform(s_x[k0 + u]);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const unsigned t = tid < len[u] ? tid : 0;
                d[u] = (a.col + beg[u])[t];
                pm[u] = (Edge)(a.perm + beg[u])[t];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) d[u] = slot(tid < len[u], d[u]);
        };
        auto weights = [&](const int* d, const Edge* pm, float* w) {
#pragma unroll
            for (int u = 0; u < U; ++u) w[u] = a.w[(UEdge)(d[u] != spare ? pm[u] : 0)];
        };
        int d[U], d1[U], len[U], len1[U];
        Edge pm[U];
        float w[U], w1[U], xk[U], xk1[U];
        ask(0, d, pm, len, xk);
        weights(d, pm, w);
        for (int k0 = 0; k0 < total; k0 += U) {
            if (k0 + U < total) {
                ask(k0 + U, d1, pm, len1, xk1);
                weights(d1, pm, w1);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (T > 64 && k0 + u >= total) break;  // uniform
                s_y[d[u]] = fmaf(w[u], xk[u], s_y[d[u]]);
                // a longer source's other edges, four at a time
                if (len[u] > T) {  // uniform
                    const Edge beg = uniform(s_beg[k0 + u]);
                    for (unsigned t0 = T; t0 < (unsigned)len[u]; t0 += 4 * T) {
                        unsigned t[4];
                        int q4[4];
                        Edge p4[4];
                        float w4[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            t[i] = t0 + tid + i * T;
                            const unsigned e = t[i] < (unsigned)len[u] ? t[i] : 0;
                            q4[i] = (a.col + beg)[e];
                            p4[i] = (Edge)(a.perm + beg)[e];
                        }
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            q4[i] = slot(t[i] < (unsigned)len[u], q4[i]);
                            w4[i] = a.w[(UEdge)(q4[i] != spare ? p4[i] : 0)];
                        }
#pragma unroll
                        for (int i = 0; i < 4; ++i) s_y[q4[i]] = fmaf(w4[i], xk[u], s_y[q4[i]]);
                    }
                }
                // one wavefront's LDS accesses are done in order
                if (T == 64) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                else __syncthreads();
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                d[u] = d1[u];
                w[u] = w1[u];
                len[u] = len1[u];
                xk[u] = xk1[u];
            }
        }
        __syncthreads();  // the list is rewritten
    };
    const int32_t* src = reinterpret_cast<const int32_t*>(a.xt) + row * a.n_src;
    const int nonzero = a.counts[row];
    for (int base = 0; base < nonzero; base += L) {
#pragma unroll
        for (int p = tid; p < L; p += T) {
            if (base + p < nonzero) {
                const int s = src[base + p];
                const int64_t beg = a.row_ptr[s];
                const int len = (int)(a.row_ptr[s + 1] - beg);
                s_beg[p] = len > 0 ? (Edge)beg : 0;  // (every thread reads an edge)
                s_len[p] = len;
                s_x[p] = xr[s];
            } else {
                s_beg[p] = 0;
                s_len[p] = 0;
            }
        }
        __syncthreads();
        add(nonzero - base < L ? nonzero - base : L);
    }
    __syncthreads();
    float* yr = a.y + row * a.n_dst + d0;
    if (a.n_dst % 4 == 0 && tile % 4 == 0 && (reinterpret_cast<uintptr_t>(a.y) & 15) == 0)
        for (int q = tid; q < nd / 4; q += T)
            reinterpret_cast<float4*>(yr)[q] = reinterpret_cast<const float4*>(s_y)[q];
    else
        for (int q = tid; q < nd; q += T) yr[q] = s_y[q];
}

template <typename Edge>
static void launch_rows(const ProductArgs& a, int threads, int tile, hipStream_t s) {
    const dim3 grid((unsigned)a.rows, (unsigned)((a.n_dst + tile - 1) / tile));
    const auto kernel = threads == 64    ? &k_product_rows<Edge, 64>
                        : threads == 256 ? &k_product_rows<Edge, 256>
                                         : &k_product_rows<Edge, 1024>;
    hipLaunchKernelGGL(kernel, grid, dim3(threads), 4 * (size_t)(tile + 4), s, a, tile);
}

// out[g][i][b] = in[64 g + b][i] for the 64 values from i0; rows past `rows` are 0.
__device__ __forceinline__ void group_rows(const float* __restrict__ in, int64_t n, int64_t stride,
                                           int64_t rows, float* __restrict__ out, int64_t g,
                                           int64_t i0) {
    __shared__ float t[64][65];
    const int ln = threadIdx.x & 63;
    for (int b = threadIdx.x >> 6; b < 64; b += 4) {
        const int64_t row = g * kGroup + b, i = i0 + ln;
        t[b][ln] = row < rows && i < n ? in[row * stride + i] : 0.f;
    }
    __syncthreads();
    for (int k = threadIdx.x >> 6; k < 64; k += 4)
        if (i0 + k < n) out[(g * n + i0 + k) * kGroup + ln] = t[ln][k];
}

__global__ __launch_bounds__(256) void k_group_rows(const float* __restrict__ in, int64_t n,
                                                    int64_t stride, int64_t rows,
                                                    float* __restrict__ out) {
    group_rows(in, n, stride, rows, out, blockIdx.y, (int64_t)blockIdx.x * 64);
}

// Shares the groups out: the rows of one that takes the columns are transposed,
// rows of one that does not are listed, a wavefront per segment, where its
// transposed rows would go (xt: both take n_src values a row).
__global__ __launch_bounds__(256) void k_share_rows(ProductArgs a) {
    const int64_t g = blockIdx.y;
    if (a.by_columns != nullptr) {
        const bool taken = !group_by_rows(a, g);
        if (blockIdx.x == 0 && threadIdx.x == 0) a.by_columns[g] = taken;
        if (taken) {
            const int64_t i0 = (int64_t)blockIdx.x * 64;
            if (i0 < a.n_src) group_rows(a.x, a.n_src, a.x_stride, a.rows, a.xt, g, i0);
            return;
        }
    }
    const int wv = threadIdx.x >> 6, ln = threadIdx.x & 63;
    const int64_t item = (int64_t)blockIdx.x * 4 + wv, row = g * kGroup + item % kGroup;
    const int64_t seg = item / kGroup;
    if (row >= a.rows || seg >= a.segments) return;
    int p = 0;
    for (int64_t s = ln; s < seg; s += 64) p += a.seg_counts[s * a.rows + row];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) p += __shfl_xor(p, o, 64);
    if (seg == a.segments - 1 && ln == 0) a.counts[row] = p + a.seg_counts[seg * a.rows + row];
    const int64_t end = (seg + 1) * kSegment < a.n_src ? (seg + 1) * kSegment : a.n_src;
    const float* xr = a.x + row * a.x_stride;
    int32_t* list = reinterpret_cast<int32_t*>(a.xt) + row * a.n_src;
    for (int64_t i = seg * kSegment + ln; i - ln < end; i += 512) {
        bool on[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) on[u] = i + 64 * u < end && xr[i + 64 * u] != 0.f;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const uint64_t m = __ballot(on[u]);
            const int q = p + __popcll((unsigned long long)(m & ((1ull << ln) - 1ull)));
            if (on[u]) list[q] = (int32_t)(i + 64 * u);
            p += __popcll((unsigned long long)m);
        }
    }
}

// The inverse: out[64 g + b][i] = in[g][i][b].
__global__ __launch_bounds__(256) void k_ungroup_rows(const float* __restrict__ in, int64_t n,
                                                      int64_t rows, float* __restrict__ out) {
    __shared__ float t[64][65];
    const int64_t g = blockIdx.y, i0 = (int64_t)blockIdx.x * 64;
    const int ln = threadIdx.x & 63;
    for (int k = threadIdx.x >> 6; k < 64; k += 4)
        t[k][ln] = i0 + k < n ? in[(g * n + i0 + k) * kGroup + ln] : 0.f;
    __syncthreads();
    for (int b = threadIdx.x >> 6; b < 64; b += 4) {
        const int64_t row = g * kGroup + b;
        if (row < rows && i0 + ln < n) out[row * n + i0 + ln] = t[ln][b];
    }
}

// A quarter wavefront per (destination, group of 64 rows), four rows a thread;
// 16 destinations at a time per workgroup, so that y is written in runs.  Bound
// by the gathered rows of x out of L2: 183 us for 13.4M edges and 64 rows,
// 19 TB/s (a wavefront per destination, a row a thread: four times the
// requests and their scalar address work, 264 us; without the bound of four
// wavefronts per SIMD 135 registers leave three: 223 us).  Tiles and groups are
// shared out together: 100 destinations of 16,384 sources, 1000 rows 2.8 -> 0.23
// ms (a group at a time left all but seven workgroups idle), by when an edge
// takes its quarter 0.1 us (32 requests in flight instead of eight: 10% less).
__global__ __launch_bounds__(256, 4) void k_product_columns(ProductArgs a) {
    __shared__ float s_out[16][65];
    const int tid = threadIdx.x, ln = tid & 63, c16 = ln & 15;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t groups = (a.rows + kGroup - 1) / kGroup;
    const int64_t tiles = (a.n_dst + 15) / 16;
    int64_t first = blockIdx.x;  // this workgroup's first tile of the next group it is to take
    for (int64_t g0 = 0; g0 < groups; g0 += 64) {
        uint64_t todo = __ballot(g0 + ln < groups && a.by_columns[g0 + ln] != 0);
        while (todo) {
            const int64_t g = g0 + __ffsll((unsigned long long)todo) - 1;
            todo &= todo - 1ull;
            const float* xg = a.xt + g * a.n_src * kGroup;
            int64_t tl = first;
            for (; tl < tiles; tl += gridDim.x) {
                // a quarter of the wavefront per destination, four rows per thread
                const int q = wv * 4 + (ln >> 4);
                const int64_t d = tl * 16 + q;
                const int64_t e0 = d < a.n_dst ? a.csc_ptr[d] : 0;
                const int len = d < a.n_dst ? (int)(a.csc_ptr[d + 1] - e0) : 0;
                int most = len;
#pragma unroll
                for (int o = 16; o < 64; o <<= 1) {
                    const int other = __shfl_xor(most, o, 64);
                    most = other > most ? other : most;
                }
                most = __builtin_amdgcn_readfirstlane(most);
                float acc[4] = {0.f, 0.f, 0.f, 0.f};
                int my_s = c16 < len ? a.csc_src[e0 + c16] : 0;
                float my_w = c16 < len ? a.w[e0 + c16] : 0.f;
                for (int c = 0; c < most; c += 16) {
                    // the destination's next 16 edges
                    const int nx = c + 16 + c16;
                    const int next_s = nx < len ? a.csc_src[e0 + nx] : 0;
                    const float next_w = nx < len ? a.w[e0 + nx] : 0.f;
#pragma unroll
                    for (int h = 0; h < 16; h += 8) {
                        float4 x8[8];
#pragma unroll
                        for (int u = 0; u < 8; ++u) {
                            const int src = __shfl(my_s, (ln & 48) + h + u, 64);
                            x8[u] = make_float4(0.f, 0.f, 0.f, 0.f);
                            if (c + h + u < len)
                                x8[u] = *reinterpret_cast<const float4*>(xg + ((int64_t)src * kGroup + 4 * c16));
                        }
#pragma unroll
                        for (int u = 0; u < 8; ++u) {
                            const float wk = __shfl(my_w, (ln & 48) + h + u, 64);
                            const float x4[4] = {x8[u].x, x8[u].y, x8[u].z, x8[u].w};
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                const float t = fmaf(wk, x4[i], acc[i]);
                                acc[i] = x4[i] != 0.f ? t : acc[i];
                            }
                        }
                    }
                    my_s = next_s;
                    my_w = next_w;
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) s_out[q][4 * c16 + i] = acc[i];
                __syncthreads();
                // 16 destinations of 64 rows: a 64-byte run per row
                for (int k = tid; k < 16 * kGroup; k += 256) {
                    const int b = k >> 4, q = k & 15;
                    const int64_t row = g * kGroup + b, d = tl * 16 + q;
                    if (row < a.rows && d < a.n_dst) a.y[row * a.n_dst + d] = s_out[q][b];
                }
                __syncthreads();
            }
            first = tl - tiles;
        }
    }
}

// ROWS rows of x: a wavefront per destination reads 64 edges at a time, a lane
// each, and gathers their x out of L2; the nonzero ones, found by a ballot, are
// added in ascending source order.  One launch, whatever the activity: 21,739 x
// 21,739 of 3.5M edges 14 us a row in a replayed graph (counts, lists and the two
// forms above 25 to 85 us).
template <int ROWS>
__global__ __launch_bounds__(256) void k_product_few(ProductArgs a) {
    const int ln = threadIdx.x & 63;
    const int64_t r0 = (int64_t)blockIdx.y * ROWS;
    const int here = (int)(a.rows - r0 < ROWS ? a.rows - r0 : ROWS);
    const float* x = a.x + r0 * a.x_stride;
    float* y = a.y + r0 * a.n_dst;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    for (int64_t d = (int64_t)blockIdx.x * 4 + wv; d < a.n_dst; d += (int64_t)gridDim.x * 4) {
        const int64_t e0 = a.csc_ptr[d];
        const int len = (int)(a.csc_ptr[d + 1] - e0);
        float acc[ROWS] = {};
        for (int c = 0; c < len; c += 64) {
            const bool in = c + ln < len;
            const int src = in ? a.csc_src[e0 + c + ln] : 0;
            const int w = in ? __float_as_int(a.w[e0 + c + ln]) : 0;
            float xv[ROWS];
#pragma unroll
            for (int r = 0; r < ROWS; ++r)
                xv[r] = in && r < here ? x[r * a.x_stride + src] : 0.f;
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                uint64_t m = __ballot(xv[r] != 0.f);
                while (m) {
                    const int b = __ffsll((unsigned long long)m) - 1;
                    m &= m - 1;
                    acc[r] = fmaf(__int_as_float(__builtin_amdgcn_readlane(w, b)),
                                  __int_as_float(__builtin_amdgcn_readlane(__float_as_int(xv[r]), b)),
                                  acc[r]);
                }
            }
        }
        if (ln == 0)
#pragma unroll
            for (int r = 0; r < ROWS; ++r)
                if (r < here) y[r * a.n_dst + d] = acc[r];
    }
}

// gx of the layer: gxt[g][s][b] = sum over edges e of row s of w[e] *
// gt[g][col[e]][b]; one wavefront per (row, group), 32 gathered rows in flight.
// Bound by the weights, which perm scatters (0.8 GB fetched for 13.4M edges),
// and the gathered rows out of L2: 273 us at 64 rows (a row of the 64 per
// thread and an edge per instruction: 292; five wavefronts per SIMD spill: 407;
// the row pass of btx_spmv.hip that the layer's backward used before: 3.9 ms
// with its copies).
__global__ __launch_bounds__(256) void k_product_grad_x(const int64_t* __restrict__ rp,
                                                        const int32_t* __restrict__ col,
                                                        const int64_t* __restrict__ perm,
                                                        const float* __restrict__ w, int64_t n_src,
                                                        int64_t n_dst,
                                                        const float* __restrict__ gt,
                                                        float* __restrict__ gxt) {
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int64_t s = (int64_t)blockIdx.x * 4 + wv;
    const int64_t g = blockIdx.y;
    const int ln = threadIdx.x & 63;
    if (s >= n_src) return;
    const int q = ln >> 4, c16 = ln & 15;
    const float* gg = gt + g * n_dst * kGroup;
    const int64_t e0 = rp[s];
    const int len = (int)(rp[s + 1] - e0);
    // a quarter of the wavefront per edge, four of the rows per thread; the
    // terms of 64 edges in two partial sums each and the 64-edge sums in
    // float64: 7e-8 of the result against float64 throughout (sixteen float
    // sums over all edges 1.4e-7, two 3.6e-7)
    double sum[4] = {0.0, 0.0, 0.0, 0.0};
    int my_d = ln < len ? col[e0 + ln] : 0;
    float my_w = ln < len ? w[perm[e0 + ln]] : 0.f;
    for (int c = 0; c < len; c += 64) {
        const int m = len - c < 64 ? len - c : 64;
        // the next 64 edges; their weights lie scattered
        const int nx = c + 64 + ln;
        const int next_d = nx < len ? col[e0 + nx] : 0;
        const float next_w = nx < len ? w[perm[e0 + nx]] : 0.f;
        float acc[2][4] = {};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (32 * h >= m) break;  // uniform
            float4 g8[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int k = 32 * h + 4 * u + q;
                const int d = __shfl(my_d, k, 64);
                g8[u] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (k < m) g8[u] = *reinterpret_cast<const float4*>(gg + ((int64_t)d * kGroup + 4 * c16));
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const float wk = __shfl(my_w, 32 * h + 4 * u + q, 64);
                acc[h][0] = fmaf(wk, g8[u].x, acc[h][0]);
                acc[h][1] = fmaf(wk, g8[u].y, acc[h][1]);
                acc[h][2] = fmaf(wk, g8[u].z, acc[h][2]);
                acc[h][3] = fmaf(wk, g8[u].w, acc[h][3]);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[i] += (double)acc[0][i] + (double)acc[1][i];
        my_d = next_d;
        my_w = next_w;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        sum[i] += __shfl_xor(sum[i], 16, 64);
        sum[i] += __shfl_xor(sum[i], 32, 64);
    }
    if (q == 0)
        *reinterpret_cast<float4*>(gxt + (g * n_src + s) * kGroup + 4 * c16) =
            make_float4((float)sum[0], (float)sum[1], (float)sum[2], (float)sum[3]);
}

// gw of the layer, destination-major: gw[e] = sum over rows b of x[b, src[e]] *
// gy[b, dst].  A wavefront takes every gridDim.y-th 64 edges of a destination,
// whose gradients over 64 rows sit in LDS, and a thread an edge whose source's
// row bits it reads: only rows with x != 0 are added, in ascending order, group
// by group (a wavefront a destination: 16,384 x 100, 5000 rows, 30 % active, the
// whole backward 22 ms; so: 3.2).
__global__ __launch_bounds__(256) void k_product_grad_w(const int64_t* __restrict__ csc_ptr,
                                                        const int32_t* __restrict__ csc_src,
                                                        int64_t n_src, int64_t n_dst, int64_t rows,
                                                        const float* __restrict__ x,
                                                        int64_t x_stride,
                                                        const uint64_t* __restrict__ bits,
                                                        const float* __restrict__ gt,
                                                        float* __restrict__ gw) {
    __shared__ float s_g[4][kGroup];
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int64_t d = (int64_t)blockIdx.x * 4 + wv;
    const int ln = threadIdx.x & 63;
    if (d >= n_dst) return;
    const int64_t e0 = csc_ptr[d] + 64 * (int64_t)blockIdx.y, e1 = csc_ptr[d + 1];
    if (e0 >= e1) return;
    const int64_t groups = (rows + kGroup - 1) / kGroup, step = 64 * (int64_t)gridDim.y;
    for (int64_t g = 0; g < groups; ++g) {
        s_g[wv][ln] = gt[(g * n_dst + d) * kGroup + ln];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        for (int64_t e = e0 + ln; e < e1; e += step) {
            const int s = csc_src[e];
            uint64_t m = bits[g * n_src + s];
            float acc = 0.f;
            while (m) {
                const int b = __ffsll((unsigned long long)m) - 1;
                acc = fmaf(x[(g * kGroup + b) * x_stride + s], s_g[wv][b], acc);
                m &= m - 1ull;
            }
            gw[e] = g == 0 ? acc : gw[e] + acc;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// bits[g][s]: bit b = x[64 g + b, s] != 0.
__global__ __launch_bounds__(256) void k_row_bits(const float* __restrict__ x, int64_t n,
                                                  int64_t stride, int64_t rows,
                                                  uint64_t* __restrict__ bits) {
    const int64_t s = (int64_t)blockIdx.x * 256 + threadIdx.x, g = blockIdx.y;
    if (s >= n) return;
    uint64_t m = 0ull;
    const int64_t here = rows - g * kGroup < kGroup ? rows - g * kGroup : kGroup;
    const float* xg = x + g * kGroup * stride + s;
#pragma unroll 8
    for (int b = 0; b < here; ++b) m |= (uint64_t)(xg[b * stride] != 0.f) << b;
    bits[g * n + s] = m;
}

static size_t product_scratch(int64_t rows, int64_t n_src) {
    const int64_t groups = (rows + kGroup - 1) / kGroup;
    const int64_t segments = (n_src + kSegment - 1) / kSegment;
    return align256(4 * (size_t)(rows + groups + rows * segments)) +
           4 * (size_t)(groups * n_src * kGroup);
}

static size_t grad_scratch(int64_t rows, int64_t n_src, int64_t n_dst) {
    const size_t groups = (size_t)((rows + kGroup - 1) / kGroup);
    // gy and gx by groups, row bits
    return groups * kGroup * 4 * (size_t)(n_dst + n_src) + groups * 8 * (size_t)n_src + 256;
}

// Destinations of a `rows` workgroup: as few tiles as occupy every CU, of at
// least 1024 destinations.
static int row_tile(int64_t rows, int64_t n_dst) {
    const int64_t want = rows < 256 ? 256 / rows : 1;
    int64_t tile = ((n_dst + want - 1) / want + 63) / 64 * 64;
    tile = tile < 1024 ? 1024 : tile > kRowTile ? kRowTile : tile;
    return (int)(tile < n_dst ? tile : n_dst);
}

// Threads of a `rows` workgroup, by the edges of a source.  us by 64 / 256 / 1024
// threads:
//   1100 x 3000, 40 edges a source, 64 rows, 10 % active        35 / 40 / 48
//   3000 x 3000, 60 edges a source, 64 rows, 10 % active        65 / 79 / 100
//   3000 x 3000, 100 edges a source, 64 rows, 10 % active      212 / 81 / 108
//   4000 x 8000, 250 edges a source, 64 rows, 2 % active        95 / 47 / 53
//   1000 x 4000, 300 edges a source, 64 rows, 2 % active        32 / 35 / 24
//   16384 x 16384, 819 edges a source, 8 rows, 0.5 % active    198 / 104 / 57
static int row_threads(int64_t n_src, int64_t nnz) {
    const int64_t len = nnz / (n_src > 0 ? n_src : 1);
    return len <= 64 ? 64 : len <= 256 ? 256 : 1024;
}

// Nonzeros of a row up to which the `rows` form takes it, from what either form
// takes here in us (fitted to 15 nets of 64 to 100,000 sources, 40 to 40,000
// destinations and 10 to 2000 edges a source, 4 to 4000 rows, 0.1 to 10 % active:
// 0.2 % from the faster form on average, 20 % at most).  A source costs the rows
// form a chain of LDS accesses and loads or, with many workgroups, their edges or
// the weights' lines; the columns cost the transpose, the outputs and every edge,
// more once the rows of x leave an XCD's L2, or the chain of the edges of one
// destination.  Measured by rows / columns, us:
//   16384 x 16384, 819 edges a source, 64 rows, 328 active    257 / 164
//   16384 x 16384, 819 edges a source, 8 rows, 328 active     143 / 172
//   16384 x 100, 10 edges a source, 1000 rows, 16 active       60 / 240
//   1000 x 1000, 50 edges a source, 1000 rows, 20 active       27 / 38
//   1000 x 1000, 50 edges a source, 1000 rows, 100 active      46 / 38
//   100000 x 5000, 20 edges a source, 200 rows, 500 active    157 / 287
//   100000 x 5000, 20 edges a source, 200 rows, 2000 active   399 / 285
static int rows_limit(int64_t rows, int64_t n_src, int64_t n_dst, int64_t nnz) {
    const double groups = (double)((rows + kGroup - 1) / kGroup);
    const double len = (double)nnz / (double)n_src;
    const int tile = row_tile(rows, n_dst), threads = row_threads(n_src, nnz);
    const double wgs = (double)rows * (double)((n_dst + tile - 1) / tile);
    const double chain = threads == 64    ? 0.19
                         : threads == 256 ? 0.34 + 0.4e-3 * len
                                          : 0.24 + 0.25e-3 * len;
    // 4M weights and more leave the caches
    const double lines = nnz < 4000000 ? 0.0 : 7e-6 * (double)rows * len;
    const double source_us = std::max({chain, 3.6e-6 * wgs * len, lines});
    const double spread = std::min(3.5, std::max(1.0, 1.3 * (double)n_src / 16384.0));
    const double cols_us = 6.0 + groups * (0.2e-3 * (double)n_src + 32e-6 * (double)n_dst) +
                           std::max(0.1 * (double)nnz / (double)n_dst,
                                    8e-6 * spread * (double)nnz * groups);
    const double most = cols_us / source_us;
    return most >= (double)n_src ? (int)n_src : (int)most;
}

static int check_product(const char* who, int64_t n_src, int64_t n_dst, int64_t rows,
                         const void* scratch) {
    if (n_src >= (int64_t)1 << 31 || n_dst >= (int64_t)1 << 31)
        return fail(std::string(who) + ": sources and destinations must fit int32");
    if (rows > 65535) return fail(std::string(who) + ": rows exceeds 65535");
    if (((uintptr_t)scratch & 15) != 0) return fail(std::string(who) + ": scratch is not 16-byte aligned");
    return 0;
}

}  // namespace btx

using namespace btx;

BTX_API size_t btx_product_scratch_bytes(int64_t rows, int64_t n_src) {
    return rows > 0 && n_src > 0 ? product_scratch(rows, n_src) : 0;
}

BTX_API int btx_product(const int64_t* row_ptr, const int32_t* col, const int64_t* perm,
                        const int64_t* csc_ptr, const int32_t* csc_src, const float* w,
                        int64_t n_src, int64_t n_dst, int64_t nnz, const float* x,
                        int64_t x_row_stride, int64_t rows, float* y, void* scratch,
                        size_t scratch_bytes, void* stream) {
    if (rows <= 0 || n_dst <= 0) return 0;
    if (int rc = check_product("btx_product", n_src, n_dst, rows, scratch)) return rc;
    if (scratch_bytes < btx_product_scratch_bytes(rows, n_src) ||
        (scratch == nullptr && scratch_bytes > 0))
        return fail("btx_product: scratch too small");
    const hipStream_t s = (hipStream_t)stream;
    ProductArgs a{row_ptr, col, perm, csc_ptr, csc_src, w, n_src, n_dst, nnz, x, x_row_stride, rows,
                  y, nullptr, nullptr, nullptr, 0, nullptr, 0};
    // by destination while the edges, times the rows, stay few.  One row always
    // (13.4M edges: 28 us against 31 by rows at 16 active sources and 170 by
    // columns); up to four as far as 8M (27 us; 14M 52 us, by when the rows form is
    // as fast at low activity); more rows, which read the edges again for every
    // four, as far as 2M: 0.4 to 0.7 of the time of the faster other form from
    // 0.1 to 10 % active, 1.2 of it where all are (1000 x 1000, 50 edges a source,
    // 32 rows: 6 / 8 / 27 us at 0.5, 10 and 100 % against 15 / 22 / 22); at 5M
    // 28 us against 15 (200 x 16384, 819 edges a source, 32 rows)
    const int64_t few_edges = (int64_t)(rows <= kFewRows ? 8 : 2) << 20;
    if ((rows == 1 || rows * nnz <= few_edges) && nnz <= 8192 * n_dst) {
        const int64_t wgs = (n_dst + 3) / 4;
        const dim3 few((unsigned)(wgs < 8192 ? wgs : 8192), (unsigned)((rows + kFewRows - 1) / kFewRows));
        hipLaunchKernelGGL(rows == 1 ? k_product_few<1> : rows == 2 ? k_product_few<2>
                           : rows == 3 ? k_product_few<3> : k_product_few<4>,
                           few, dim3(256), 0, s, a);
        return check_launch("btx_product");
    }
    a.most = n_src > 0 ? rows_limit(rows, n_src, n_dst, nnz) : 0;
    const bool columns = a.most < n_src;  // some row may be left to them
    const int64_t groups = (rows + kGroup - 1) / kGroup;
    a.segments = (int)((n_src + kSegment - 1) / kSegment);
    a.counts = (int32_t*)scratch;
    a.by_columns = columns ? a.counts + rows : nullptr;
    a.seg_counts = a.counts + rows + groups;
    a.xt = (float*)((char*)scratch + align256(4 * (size_t)(rows + groups + rows * a.segments)));
    hipLaunchKernelGGL(k_row_counts, dim3((unsigned)((rows * a.segments + 3) / 4)), dim3(256), 0, s, a);
    const int64_t lists = (int64_t)a.segments * (kGroup / 4);
    const int64_t blocks = columns ? std::max(lists, (n_src + 63) / 64) : lists;
    hipLaunchKernelGGL(k_share_rows, dim3((unsigned)blocks, (unsigned)groups), dim3(256), 0, s, a);
    const int tile = row_tile(rows, n_dst), threads = row_threads(n_src, nnz);
    if (nnz < (int64_t)1 << 31) launch_rows<int>(a, threads, tile, s);
    else launch_rows<int64_t>(a, threads, tile, s);
    if (columns) {
        const int64_t items = (n_dst + 15) / 16 * groups;
        hipLaunchKernelGGL(k_product_columns, dim3((unsigned)(items < 2048 ? items : 2048)),
                           dim3(256), 0, s, a);
    }
    return check_launch("btx_product");
}

BTX_API size_t btx_product_grad_scratch_bytes(int64_t rows, int64_t n_src, int64_t n_dst) {
    return rows > 0 ? grad_scratch(rows, n_src, n_dst) : 0;
}

BTX_API int btx_product_grad(const int64_t* row_ptr, const int32_t* col, const int64_t* perm,
                             const int64_t* csc_ptr, const int32_t* csc_src, const float* w,
                             int64_t n_src, int64_t n_dst, int64_t nnz, const float* x,
                             int64_t x_row_stride, int64_t rows, const float* gy, float* gx,
                             float* gw, void* scratch, size_t scratch_bytes, void* stream) {
    if (rows <= 0 || n_src <= 0 || n_dst <= 0) return 0;
    if (int rc = check_product("btx_product_grad", n_src, n_dst, rows, scratch)) return rc;
    if (scratch == nullptr || scratch_bytes < grad_scratch(rows, n_src, n_dst))
        return fail("btx_product_grad: scratch too small");
    const hipStream_t s = (hipStream_t)stream;
    const int64_t groups = (rows + kGroup - 1) / kGroup;
    float* gt = (float*)scratch;
    float* gxt = gt + groups * n_dst * kGroup;
    uint64_t* bits = (uint64_t*)(gxt + groups * n_src * kGroup);
    hipLaunchKernelGGL(k_group_rows, dim3((unsigned)((n_dst + 63) / 64), (unsigned)groups),
                       dim3(256), 0, s, gy, n_dst, n_dst, rows, gt);
    if (gx != nullptr) {
        hipLaunchKernelGGL(k_product_grad_x, dim3((unsigned)((n_src + 3) / 4), (unsigned)groups),
                           dim3(256), 0, s, row_ptr, col, perm, w, n_src, n_dst, gt, gxt);
        hipLaunchKernelGGL(k_ungroup_rows, dim3((unsigned)((n_src + 63) / 64), (unsigned)groups),
                           dim3(256), 0, s, gxt, n_src, rows, gx);
    }
    if (gw != nullptr) {
        hipLaunchKernelGGL(k_row_bits, dim3((unsigned)((n_src + 255) / 256), (unsigned)groups),
                           dim3(256), 0, s, x, n_src, x_row_stride, rows, bits);
        // as many wavefronts per destination as fill the chip with 8192
        const int64_t len64 = (nnz / n_dst + 63) / 64, want = (8192 + n_dst - 1) / n_dst;
        const int64_t split = len64 < want ? len64 : want;
        hipLaunchKernelGGL(k_product_grad_w,
                           dim3((unsigned)((n_dst + 3) / 4), (unsigned)(split > 0 ? split : 1)),
                           dim3(256), 0, s, csc_ptr, csc_src, n_src, n_dst, rows, x, x_row_stride, bits, gt, gw);
    }
    return check_launch("btx_product_grad");
}
