// The sparse product as a layer of its own and its backward, y = x W.
//
// Layouts as in btx_spmv.hip: CSR by source (row_ptr, col; destinations
// ascending) and the same edges destination-major (csc_ptr, csc_src; sources
// ascending).  Weights come in the destination-major order, the layer's own
// parameter order; perm[k] is the position there of CSR edge k.
//
// Every destination sums its terms in ascending source order from +0.0f with
// one fmaf per source with x != 0, so y equals torch.sparse.mm on the CPU bit
// for bit (btorch/models/linear.py:474-483).  Two forms, neither of which
// stores a term:
//   rows     a workgroup takes one row of x and a tile of destinations held in
//            LDS, and streams the rows of W of the row's nonzero sources in
//            ascending order: a source's destinations are distinct, so its
//            terms need no atomics, and a barrier between sources keeps the
//            order.  Costs the active sources, whatever the edges.
//   columns  a quarter wavefront takes a destination and 64 rows of x
//            (transposed, so that a source's 64 values are one 256-byte read)
//            and walks the destination's edges.  Costs every edge, whatever the activity.

#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/btorch_amd.h"
#include "btx_common.h"

namespace btx {

constexpr int kRowTile = 16384;      // destinations of a `rows` workgroup, at most (64 KB of LDS)
constexpr int kRowThreads = 1024;
constexpr int kGroup = 64;           // rows of x per wavefront of the `columns` form
constexpr int64_t kFewRows = 4;      // up to which k_product_few takes them

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
    int32_t* counts;      // nonzeros of each row
    int32_t* by_columns;  // [groups] 1 = left to the columns; NULL = the `rows` form takes all
    int most;             // nonzeros a row, on average of a group, up to which the `rows`
                          // form takes the group
};

// Whether the `rows` form takes the 64 rows of group g (decided for the group: a
// form's cost is the same for one of its rows as for all); every thread of the
// wavefront calls it.
__device__ __forceinline__ bool group_by_rows(const ProductArgs& a, int64_t g) {
    const int64_t row = g * kGroup + (threadIdx.x & 63);
    int64_t c = row < a.rows ? a.counts[row] : 0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    const int64_t here = a.rows - g * kGroup < kGroup ? a.rows - g * kGroup : kGroup;
    return c <= a.most * here;
}

// Nonzeros of every row: THREADS threads a row, of a workgroup of 256 or 1024.
template <int THREADS>
__global__ __launch_bounds__(THREADS < 256 ? 256 : THREADS) void k_row_counts(
    const float* __restrict__ x, int64_t n, int64_t stride, int64_t rows,
    int32_t* __restrict__ counts) {
    constexpr int BLOCK = THREADS < 256 ? 256 : THREADS;
    const int64_t row = (int64_t)blockIdx.x * (BLOCK / THREADS) + threadIdx.x / THREADS;
    if (THREADS == 64 && row >= rows) return;
    const float* xr = x + row * stride;
    int c = 0;
#pragma unroll 8
    for (int64_t i = threadIdx.x % THREADS; i < n; i += THREADS) c += xr[i] != 0.f;
    int total;
    if (THREADS == 64) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
        total = c;
    } else {
        block_excl_scan<BLOCK / 64>(c, total);
    }
    if (threadIdx.x % THREADS == 0) counts[row] = total;
}

// One row of x, destinations [d0, d0 + tile): 1024 V of the row's values are
// read at a time and their nonzeros listed in LDS in ascending order, each
// with its row of W.  Bound by the misses one CU can have in flight on a
// source's weights, which perm scatters over the array, and by the barrier per
// source: eight sources are requested together, the next eight before the
// current ones are added, and a few rows are split into tiles over the CUs.
// 0.4 to 0.65 us a source of 163 to 819 edges (one source ahead, 1024 values at
// a time and whole rows: 0.8 to 1.9 us).  Taken back: three requests in flight
// (74 VGPRs, one workgroup per CU: 512 rows 15% slower), 256 threads.  Edge:
// an integer that holds the edges' positions (64 bits leave room for one
// workgroup per CU where 16,384 destinations are tiled).  V = 1 where a row has
// no more than 1024 values: 200 x 16,384, 12,800 rows, 5 active sources each,
// 0.383 ms; 0.411 with seven of eight reads and ballots per thread wasted.
template <typename Edge, int V>
__global__ __launch_bounds__(kRowThreads) void k_product_rows(ProductArgs a, int tile) {
    constexpr int T = kRowThreads;
    extern __shared__ __align__(16) float s_y[];
    __shared__ Edge s_beg[T];
    __shared__ int s_len[T];
    __shared__ float s_x[T];
    __shared__ int s_cnt[T / 64];
    constexpr int U = 8;
    const int tid = threadIdx.x, wv = tid >> 6, ln = tid & 63;
    const int64_t row = blockIdx.x, d0 = (int64_t)blockIdx.y * tile;
    const int nd = (int)(a.n_dst - d0 < tile ? a.n_dst - d0 : tile);
    const float* xr = a.x + row * a.x_stride;
    const int left = a.by_columns != nullptr ? a.by_columns[row / kGroup] : 0;
    for (int q = tid; q < (nd + 3) / 4; q += T)
        reinterpret_cast<float4*>(s_y)[q] = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int64_t s0 = 0; s0 < a.n_src; s0 += T * V) {
      // a wavefront reads 64 V consecutive values
      const int64_t s1 = s0 + wv * 64 * V + ln;
      float xv[V];
#pragma unroll
      for (int u = 0; u < V; ++u) xv[u] = s1 + 64 * u < a.n_src ? xr[s1 + 64 * u] : 0.f;
      if (left) return;  // uniform; asked for beside the first values
      int mine = 0;
#pragma unroll
      for (int u = 0; u < V; ++u) mine += __popcll((unsigned long long)__ballot(xv[u] != 0.f));
      if (ln == 0) s_cnt[wv] = mine;
      __syncthreads();
      int first = 0, nonzero = 0;
#pragma unroll
      for (int k = 0; k < T / 64; ++k) {
          first += k < wv ? s_cnt[k] : 0;
          nonzero += s_cnt[k];
      }
      // the nonzeros, 1024 at a time
      for (int base = 0; base < nonzero; base += T) {
        const int total = nonzero - base < T ? nonzero - base : T;
        int off = first - base;
#pragma unroll
        for (int u = 0; u < V; ++u) {
            const bool on = xv[u] != 0.f;
            const uint64_t m = __ballot(on);
            const int p = off + __popcll((unsigned long long)(m & ((1ull << ln) - 1ull)));
            off += __popcll((unsigned long long)m);
            if (on && p >= 0 && p < T) {
                const int64_t beg = a.row_ptr[s1 + 64 * u];
                s_beg[p] = (Edge)beg;
                s_len[p] = (int)(a.row_ptr[s1 + 64 * u + 1] - beg);
                s_x[p] = xv[u];
            }
        }
        __syncthreads();
        // this thread's first edge of eight sources: destination within the
        // tile (-1 = none), weight
        auto request = [&](int k0, int* d, float* w) {
            int64_t pm[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const bool in = k0 + u < total && tid < s_len[k0 + u];
                const Edge e = in ? s_beg[k0 + u] + tid : 0;
                d[u] = in ? a.col[e] : -1;
                pm[u] = in ? a.perm[e] : 0;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t q = d[u] - d0;
                d[u] = d[u] >= 0 && q >= 0 && q < nd ? (int)q : -1;
                w[u] = d[u] >= 0 ? a.w[pm[u]] : 0.f;
            }
        };
        int d[U], dn[U];
        float w[U], wn[U];
        if (total > 0) request(0, d, w);
        for (int k0 = 0; k0 < total; k0 += U) {
            if (k0 + U < total) request(k0 + U, dn, wn);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (k0 + u >= total) break;  // uniform
                const float xk = s_x[k0 + u];
                const int len = s_len[k0 + u];
                if (d[u] >= 0) s_y[d[u]] = fmaf(w[u], xk, s_y[d[u]]);
                for (int t = tid + T; t < len; t += T) {
                    const Edge e = s_beg[k0 + u] + t;
                    const int64_t q = a.col[e] - d0;
                    if (q >= 0 && q < nd) s_y[q] = fmaf(a.w[a.perm[e]], xk, s_y[q]);
                }
                __syncthreads();
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                d[u] = dn[u];
                w[u] = wn[u];
            }
        }
        __syncthreads();  // the list is rewritten
      }
      __syncthreads();  // and s_cnt
    }
    __syncthreads();
    float* yr = a.y + row * a.n_dst + d0;
    if (a.n_dst % 4 == 0 && tile % 4 == 0 && (reinterpret_cast<uintptr_t>(a.y) & 15) == 0)
        for (int q = tid; q < nd / 4; q += T)
            reinterpret_cast<float4*>(yr)[q] = reinterpret_cast<const float4*>(s_y)[q];
    else
        for (int q = tid; q < nd; q += T) yr[q] = s_y[q];
}

// out[g][i][b] = in[64 g + b][i] in tiles of 64 x 64; rows past `rows` are 0.
// `a` non-null: only the groups that take the columns.
__global__ __launch_bounds__(256) void k_group_rows(ProductArgs a, const float* __restrict__ in,
                                                    int64_t n, int64_t stride, int64_t rows,
                                                    float* __restrict__ out) {
    __shared__ float t[64][65];
    const int64_t g = blockIdx.y, i0 = (int64_t)blockIdx.x * 64;
    if (a.by_columns != nullptr) {
        const bool taken = !group_by_rows(a, g);
        if (blockIdx.x == 0 && threadIdx.x == 0) a.by_columns[g] = taken;
        if (!taken) return;
    }
    const int ln = threadIdx.x & 63;
    for (int b = threadIdx.x >> 6; b < 64; b += 4) {
        const int64_t row = g * kGroup + b, i = i0 + ln;
        t[b][ln] = row < rows && i < n ? in[row * stride + i] : 0.f;
    }
    __syncthreads();
    for (int k = threadIdx.x >> 6; k < 64; k += 4)
        if (i0 + k < n) out[(g * n + i0 + k) * kGroup + ln] = t[ln][k];
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

// A few rows of x: a wavefront per destination reads 64 edges at a time, a lane
// each, and gathers their x out of L2; the nonzero ones, found by a ballot, are
// added in ascending source order.  One launch, whatever the activity: 21,739 x
// 21,739 of 3.5M edges 14 us a row in a replayed graph (counting, the transpose
// and the two forms above 55 to 75 us).
template <int ROWS>
__global__ __launch_bounds__(256) void k_product_few(ProductArgs a) {
    const int ln = threadIdx.x & 63;
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
            for (int r = 0; r < ROWS; ++r) xv[r] = in ? a.x[r * a.x_stride + src] : 0.f;
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
            for (int r = 0; r < ROWS; ++r) a.y[r * a.n_dst + d] = acc[r];
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
    return align256(4 * (size_t)(rows + groups)) + 4 * (size_t)(groups * n_src * kGroup);
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

// Nonzeros of a row up to which the `rows` form takes it, from what either form
// takes here in us (fitted to 15 nets of 64 to 100,000 sources, 40 to 40,000
// destinations and 10 to 2000 edges a source, 1 to 4000 rows, 0.1 to 100 % active:
// 0.7 % from the faster form on average).  A source costs the rows form a
// barrier and a chain of loads, or, with many workgroups, its share of a CU or of
// the weights' lines; the columns cost the transpose and every edge, more once
// the rows of x leave an XCD's L2, or the chain of the edges of one destination.
// Measured by rows / columns, us:
//   16384 x 16384, 819 edges a source, 64 rows, 328 active    236 / 155
//   16384 x 16384, 819 edges a source, 64 rows, 82 active      91 / 155
//   16384 x 100, 10 edges a source, 64 rows, 328 active       134 / 206
//   16384 x 100, 10 edges a source, 1000 rows, 16 active       72 / 229
//   1000 x 1000, 50 edges a source, 64 rows, 20 active         19 / 20
//   1000 x 1000, 50 edges a source, 64 rows, all active       330 / 20
//   100000 x 5000, 20 edges a source, 200 rows, 100 active    106 / 272
static int rows_limit(int64_t rows, int64_t n_src, int64_t n_dst, int64_t nnz) {
    const double groups = (double)((rows + kGroup - 1) / kGroup);
    const double len = (double)nnz / (double)n_src;
    const int tile = row_tile(rows, n_dst);
    const double wgs = (double)rows * (double)((n_dst + tile - 1) / tile);
    const double per_cu = wgs > 256.0 ? wgs / 256.0 : 1.0;
    // us per edge: the weights in L2, in the caches beyond, past them
    const double edge = nnz < 1000000 ? 4e-6 : nnz < 4000000 ? 7e-6 : 10e-6;
    const double source_us = std::max({0.4 + 0.2e-3 * len, 1.4e-3 * wgs, edge * (double)rows * len});
    const double spread = std::min(3.5, std::max(1.0, 1.3 * (double)n_src / 16384.0));
    const double cols_us = 6.0 + 0.114e-3 * groups * (double)n_src +
                           std::max(0.1 * (double)nnz / (double)n_dst,
                                    10e-6 * spread * (double)nnz * groups);
    const double most = (cols_us - 0.14e-3 * (double)n_src * per_cu) / source_us;
    return most < 0.0 ? 0 : most >= (double)n_src ? (int)n_src : (int)most;
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
                  y, nullptr, nullptr, nullptr, 0};
    // one row always (13.4M edges: 28 us against 31 by rows at 16 active sources
    // and 170 by columns); up to four while their gathers stay few: 8M in all
    // take 27 us, 14M 52 us, by when the rows form is as fast at low activity
    if (rows <= kFewRows && (rows == 1 || rows * nnz <= ((int64_t)8 << 20)) && nnz <= 8192 * n_dst) {
        const int64_t wgs = (n_dst + 3) / 4;
        const dim3 few((unsigned)(wgs < 8192 ? wgs : 8192));
        hipLaunchKernelGGL(rows == 1 ? k_product_few<1> : rows == 2 ? k_product_few<2>
                           : rows == 3 ? k_product_few<3> : k_product_few<4>,
                           few, dim3(256), 0, s, a);
        return check_launch("btx_product");
    }
    a.most = n_src > 0 ? rows_limit(rows, n_src, n_dst, nnz) : 0;
    const bool columns = a.most < n_src;  // some row may be left to them
    const int64_t groups = (rows + kGroup - 1) / kGroup;
    if (columns) {
        a.counts = (int32_t*)scratch;
        a.by_columns = a.counts + rows;
        a.xt = (float*)((char*)scratch + align256(4 * (size_t)(rows + groups)));
        // a wavefront per short row: 12,800 rows of 200 values would take a
        // workgroup each 30 us
        if (n_src <= 4096)
            hipLaunchKernelGGL(k_row_counts<64>, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s, x,
                               n_src, x_row_stride, rows, a.counts);
        else
            hipLaunchKernelGGL(k_row_counts<1024>, dim3((unsigned)rows), dim3(1024), 0, s, x, n_src,
                               x_row_stride, rows, a.counts);
        hipLaunchKernelGGL(k_group_rows, dim3((unsigned)((n_src + 63) / 64), (unsigned)groups),
                           dim3(256), 0, s, a, x, n_src, x_row_stride, rows, a.xt);
    }
    const int tile = row_tile(rows, n_dst);
    const dim3 grid((unsigned)rows, (unsigned)((n_dst + tile - 1) / tile));
    const bool narrow = nnz < (int64_t)1 << 31, one = n_src <= kRowThreads;
    hipLaunchKernelGGL(narrow ? (one ? k_product_rows<int, 1> : k_product_rows<int, 8>)
                              : (one ? k_product_rows<int64_t, 1> : k_product_rows<int64_t, 8>),
                       grid, dim3(kRowThreads), 4 * (size_t)(tile + 3), s, a, tile);
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
                       dim3(256), 0, s, ProductArgs{}, gy, n_dst, n_dst, rows, gt);
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
