// Surrogate-gradient adjoint (BPTT) of the fused LIF + exponential-synapse
// + sparse-recurrent step, run backward in time one step per call.
//
// Layout: neuron-major (n, lanes) -- element (j, b) at j*lanes + b -- so the
// lanes of one neuron are contiguous and a wavefront reads one destination's
// 64 lanes with a single 256-byte access.
//
// Forward step (btorch/models/rnn.py:517-528, lif.py:144-187, synapse.py:171-178):
//   v1  = v + dt*((-(v - vr))/tau + (psc + x)/cm)
//   s   = H((v1 - vth)/(vth - vr)) * (ref == 0)
//   v'  = v1 - (vth - vr)*s            (hard: v1 - (v1 - vr)*s)
//   psc' = psc*(1 - k/tau_s) + W^T s
// Reverse step, given dL/dv', dL/dpsc', dL/dz:
//   gs   = gz + (W gpsc')[j] + gv' * d(v')/ds        (reset term unless detached)
//   gv1  = gv' * d(v')/dv1 + gs * mask * g(u) / (vth - vr)
//   gv   = gv1 * (1 - dt/tau),  gx = gv1 * dt/cm,  gpsc = gx + gpsc' * (1 - k/tau_s)
//   gtau += gv1 * dt * (v - vr)/tau^2,  gW[e] += s[src] * gpsc'[dst]
// with g the surrogate derivative (surrogate/sigmoid.py:22-29,
// superspike.py:25-31, erf.py:22-28) and the refractory mask detached as in
// lif.py:165-167.

#include <hip/hip_runtime.h>

#include "../../include/btorch_amd.h"
#include "btx_common.h"

namespace btx {

struct AdjArgs {
    int64_t n;
    int64_t lanes;
    float dt;
    int hard_reset;
    int detach_reset;
    int surrogate;
    float alpha;
    float damping;
    const float* tau;   int64_t tau_s;
    const float* vth;   int64_t vth_s;
    const float* vr;    int64_t vr_s;
    const float* cm;    int64_t cm_s;
    const float* tsyn;  int64_t tsyn_s;
    const float* ksyn;  int64_t ksyn_s;
    const float* v_prev;
    const float* v_pre;
    const float* z;
    const float* ref_prev;
    const float* gz;
    const float* gsyn;
    float* gv;
    float* gpsc;
    float* gx;
    float* gtau;
    float* gpsc_out;
};

__device__ __forceinline__ float surrogate_grad(int kind, float u, float alpha, float damping) {
    if (kind == BTX_SURR_SIGMOID) {
        const float k = 1.7627471740390860f;  // 2*ln(sqrt(2)+1)
        const float sg = 1.f / (1.f + expf(-k * alpha * u));
        return damping * 4.f * sg * (1.f - sg);
    }
    if (kind == BTX_SURR_SUPERSPIKE) {
        const float k = 0.41421356237309515f;  // sqrt(2)-1
        const float d = 1.f + k * alpha * fabsf(u);
        return damping / (d * d);
    }
    const float au = alpha * u;  // BTX_SURR_ERF
    return damping * expf(-0.6931471805599453f * au * au);
}

__global__ __launch_bounds__(256) void k_adj_lif(AdjArgs a) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t m = a.n * a.lanes;
    if (i >= m) return;
    const int64_t j = i / a.lanes;
    const float tau = a.tau[a.tau_s * j];
    const float vth = a.vth[a.vth_s * j];
    const float vr = a.vr[a.vr_s * j];
    const float cm = a.cm[a.cm_s * j];
    const float v = a.v_prev[i];
    const float v1 = a.v_pre[i];
    const float s = a.z[i];
    const float mask = a.ref_prev ? (a.ref_prev[i] == 0.f ? 1.f : 0.f) : 1.f;
    const float gvn = a.gv[i];
    const float gpn = a.gpsc[i];
    float gs = a.gz[i] + a.gsyn[i];
    float dvdv1 = 1.f;
    if (a.hard_reset) {
        dvdv1 = 1.f - s;
        if (!a.detach_reset) gs += gvn * (-(v1 - vr));
    } else if (!a.detach_reset) {
        gs += gvn * (-(vth - vr));
    }
    const float u = (v1 - vth) / (vth - vr);
    const float gu = gs * mask * surrogate_grad(a.surrogate, u, a.alpha, a.damping);
    const float gv1 = gvn * dvdv1 + gu / (vth - vr);
    a.gv[i] = gv1 * (1.f - a.dt / tau);
    const float gI = gv1 * (a.dt / cm);
    a.gx[i] = gI;
    const float k = a.ksyn[a.ksyn_s * j];
    const float ts = a.tsyn[a.tsyn_s * j];
    a.gpsc_out[i] = gI + gpn * (1.f - k / ts);
    if (a.gtau) {
        const float gt = gv1 * a.dt * (v - vr) / (tau * tau);
        atomicAdd(&a.gtau[a.tau_s * j], gt);
    }
}

// The reverse step where everything but gsyn and gpsc, which the products
// read and write, is lane-major (lanes, n), as the forward run left it: no
// array is transposed ahead of the sweep.  A workgroup takes 32 neurons of all
// lanes; gsyn and gpsc pass through LDS.  Bound by its eleven arrays (46 MB a
// step at 16k neurons x 64 lanes).  dL/dtau is summed over the lanes in the
// workgroup (an atomic per element, 64 to one address, took 140 us a step).
constexpr int kAdjTile = 32;

__global__ __launch_bounds__(256) void k_adj_lif_lanes(AdjArgs a) {
    __shared__ float s_syn[kAdjTile * 65], s_psc[kAdjTile * 65], s_tau[256];
    const int tid = threadIdx.x, lanes = (int)a.lanes;
    const int pad = lanes | 1;
    const int64_t j0 = (int64_t)blockIdx.x * kAdjTile;
    const int rows = (int)(a.n - j0 < kAdjTile ? a.n - j0 : kAdjTile);
    const int64_t base = j0 * lanes;
    for (int k = tid; k < rows * lanes; k += 256) {
        const int j = k / lanes, b = k - j * lanes;
        s_syn[j * pad + b] = a.gsyn[base + k];
        s_psc[j * pad + b] = a.gpsc[base + k];
    }
    __syncthreads();
    const int j = tid & (kAdjTile - 1);
    float gt = 0.f;
    if (j < rows) {
        const int64_t jn = j0 + j;
        const float tau = a.tau[a.tau_s * jn], vth = a.vth[a.vth_s * jn];
        const float vr = a.vr[a.vr_s * jn], cm = a.cm[a.cm_s * jn];
        const float dpsc = 1.f - a.ksyn[a.ksyn_s * jn] / a.tsyn[a.tsyn_s * jn];
        for (int b = tid / kAdjTile; b < lanes; b += 256 / kAdjTile) {
            const int64_t i = (int64_t)b * a.n + jn;
            const float v = a.v_prev[i], v1 = a.v_pre[i], s = a.z[i];
            const float mask = a.ref_prev ? (a.ref_prev[i] == 0.f ? 1.f : 0.f) : 1.f;
            const float gvn = a.gv[i], gpn = s_psc[j * pad + b];
            float gs = (a.gz ? a.gz[i] : 0.f) + s_syn[j * pad + b];
            float dvdv1 = 1.f;
            if (a.hard_reset) {
                dvdv1 = 1.f - s;
                if (!a.detach_reset) gs += gvn * (-(v1 - vr));
            } else if (!a.detach_reset) {
                gs += gvn * (-(vth - vr));
            }
            const float u = (v1 - vth) / (vth - vr);
            const float gu = gs * mask * surrogate_grad(a.surrogate, u, a.alpha, a.damping);
            const float gv1 = gvn * dvdv1 + gu / (vth - vr);
            a.gv[i] = gv1 * (1.f - a.dt / tau);
            const float gI = gv1 * (a.dt / cm);
            a.gx[i] = gI;
            s_psc[j * pad + b] = gI + gpn * dpsc;
            gt += gv1 * a.dt * (v - vr) / (tau * tau);
        }
    }
    s_tau[tid] = gt;
    __syncthreads();
    for (int k = tid; k < rows * lanes; k += 256) {
        const int jj = k / lanes;
        a.gpsc_out[base + k] = s_psc[jj * pad + (k - jj * lanes)];
    }
    if (a.gtau && tid < kAdjTile) {
        float t = 0.f;
#pragma unroll
        for (int k = 0; k < 256 / kAdjTile; ++k) t += s_tau[k * kAdjTile + tid];
        if (a.tau_s) {
            if (tid < rows) a.gtau[j0 + tid] += t;  // this workgroup's neuron alone
        } else {
#pragma unroll
            for (int o = kAdjTile / 2; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
            if (tid == 0) atomicAdd(a.gtau, t);
        }
    }
}

// Lane masks of K steps from their spike words [K][lanes][nwords] (lanes <=
// 64): masks[K][n], one wavefront per word.
__global__ __launch_bounds__(64) void k_lane_masks(const uint64_t* __restrict__ words,
                                                   int64_t lanes, int64_t n,
                                                   uint64_t* __restrict__ masks) {
    const int64_t t = blockIdx.y, nwords = (n + 63) >> 6;
    transpose_lane_bits(words + t * lanes * nwords, masks + t * n, lanes, nwords, n, 1,
                        blockIdx.x, 0);
}

// g_src[j, b] = sum over edges e of row j of w[e] * g_dst[col[e], b]; one
// wavefront per row, lane = batch lane (rows of more than 64 lanes loop).
// The row's edges are read 64 at a time, lane k holding edge c + k, and
// handed to every lane by readlane, so the g_dst loads of a chunk do not wait
// on an index load each.  Sums: even edge offsets of the row into acc0, odd
// ones into acc1, each in edge order, then acc0 + acc1.
__global__ __launch_bounds__(256) void k_adj_transpose(const int64_t* __restrict__ rp,
                                                       const int32_t* __restrict__ col,
                                                       const float* __restrict__ w,
                                                       int64_t n_rows, int64_t lanes,
                                                       const float* __restrict__ g_dst,
                                                       float* __restrict__ g_src) {
    // uniform across the wavefront (four rows per workgroup)
    const int64_t row =
        __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4u + (threadIdx.x >> 6)));
    const int ln = threadIdx.x & 63;
    if (row >= n_rows) return;
    const int64_t e0 = rp[row], e1 = rp[row + 1];
    for (int64_t b0 = 0; b0 < lanes; b0 += 64) {
        const int64_t b = b0 + ln;
        const bool on = b < lanes;
        // lanes past `lanes` read column 0 of the row (never stored)
        const float* gb = g_dst + (on ? b : 0);
        float acc0 = 0.f, acc1 = 0.f;
        for (int64_t c = e0; c < e1; c += 64) {
            const int m = (int)(e1 - c < 64 ? e1 - c : 64);
            const int my_d = ln < m ? col[c + ln] : 0;
            const int my_w = ln < m ? __float_as_int(w[c + ln]) : 0;
            int k = 0;
            for (; k + 8 <= m; k += 8) {
                // eight loads in flight, then the sums in edge order
                float g8[8], w8[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int64_t d = __builtin_amdgcn_readlane(my_d, k + j);
                    w8[j] = __int_as_float(__builtin_amdgcn_readlane(my_w, k + j));
                    g8[j] = gb[d * lanes];
                }
#pragma unroll
                for (int j = 0; j < 8; j += 2) {
                    acc0 += w8[j] * g8[j];
                    acc1 += w8[j + 1] * g8[j + 1];
                }
            }
            for (; k + 2 <= m; k += 2) {
                const int64_t d0 = __builtin_amdgcn_readlane(my_d, k);
                const int64_t d1 = __builtin_amdgcn_readlane(my_d, k + 1);
                const float w0 = __int_as_float(__builtin_amdgcn_readlane(my_w, k));
                const float w1 = __int_as_float(__builtin_amdgcn_readlane(my_w, k + 1));
                const float g0 = gb[d0 * lanes], g1 = gb[d1 * lanes];
                acc0 += w0 * g0;
                acc1 += w1 * g1;
            }
            if (k < m) {
                const int64_t d0 = __builtin_amdgcn_readlane(my_d, k);
                const float w0 = __int_as_float(__builtin_amdgcn_readlane(my_w, k));
                acc0 += w0 * gb[d0 * lanes];
            }
        }
        if (on) g_src[row * lanes + b] = acc0 + acc1;
    }
}

// gw[e] += sum over lanes b spiking at neuron j of g_dst[col[e], b], for
// every edge of every neuron with a nonzero spike mask (lanes <= 64, mask
// bit b = lane b), the lanes taken in ascending order.  One wavefront per
// neuron.  A neuron that spiked in a few lanes: lane k of the wavefront
// takes edge c + k and gathers its destinations' values lane by lane.  In
// more lanes: the g_dst rows of 32 edges are staged in the wavefront's LDS
// tile with 256-byte loads (lane = batch lane), and lane k then sums row k
// of the tile over the set bits.
constexpr int kWgradTile = 32;
constexpr int kWgradFew = 2;  // set bits up to which a lane gathers directly

__global__ __launch_bounds__(256) void k_adj_wgrad(const int64_t* __restrict__ rp,
                                                   const int32_t* __restrict__ col,
                                                   int64_t n_rows, int64_t lanes,
                                                   const uint64_t* __restrict__ masks,
                                                   const float* __restrict__ g_dst,
                                                   float* __restrict__ gw) {
    __shared__ float tile[4][kWgradTile * 65];
    const int wv = threadIdx.x >> 6;
    // uniform across the wavefront (four rows per workgroup)
    const int64_t row = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4u + (unsigned)wv));
    const int ln = threadIdx.x & 63;
    if (row >= n_rows) return;
    const uint64_t mk = masks[row];
    if (mk == 0) return;
    const int64_t e0 = rp[row], e1 = rp[row + 1];
    if (__popcll((unsigned long long)mk) <= kWgradFew) {
        for (int64_t e = e0 + ln; e < e1; e += 64) {
            const int64_t d = col[e];
            float acc = 0.f;
            uint64_t q = mk;
            while (q) {
                const int b = __ffsll((unsigned long long)q) - 1;
                acc += g_dst[d * lanes + b];
                q &= q - 1;
            }
            gw[e] += acc;
        }
        return;
    }
    float* t = tile[wv];
    const bool on = ln < lanes;
    for (int64_t c = e0; c < e1; c += kWgradTile) {
        const int m = (int)(e1 - c < kWgradTile ? e1 - c : kWgradTile);
        const int my_d = ln < m ? col[c + ln] : 0;
        int k = 0;
        for (; k + 8 <= m; k += 8) {
            float g8[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int64_t d = __builtin_amdgcn_readlane(my_d, k + j);
                g8[j] = on ? g_dst[d * lanes + ln] : 0.f;
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) t[(k + j) * 65 + ln] = g8[j];
        }
        for (; k < m; ++k) {
            const int64_t d = __builtin_amdgcn_readlane(my_d, k);
            t[k * 65 + ln] = on ? g_dst[d * lanes + ln] : 0.f;
        }
        // the tile is the wavefront's own: its LDS writes land before its
        // reads, the fences keep the compiler from moving them across
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (ln < m) {
            float acc = 0.f;
            uint64_t q = mk;
            while (q) {
                const int b = __ffsll((unsigned long long)q) - 1;
                acc += t[ln * 65 + b];
                q &= q - 1;
            }
            gw[c + ln] += acc;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// k_adj_transpose and k_adj_wgrad of one reverse step in one pass (33 to 64
// lanes): each destination row of g_dst is loaded once per edge, feeds the
// transposed sum of its lane and, when the neuron spiked in some lane, the
// wavefront's LDS tile for the weight gradient.  Bound by the latency of the
// gathered rows (4 MB of g_dst at 16k neurons x 64 lanes, from L2): the 32
// rows of a tile are requested together, those of the next tile before the
// current one is summed, and gw's old values before either (eight rows at a
// time, gw last: 512 us a step at 13.4M edges; so: 392).
__global__ __launch_bounds__(256) void k_adj_transpose_wgrad(
    const int64_t* __restrict__ rp, const int32_t* __restrict__ col,
    const float* __restrict__ w, int64_t n_rows, int64_t lanes,
    const uint64_t* __restrict__ masks, const float* __restrict__ g_dst,
    float* __restrict__ g_src, float* __restrict__ gw) {
    __shared__ float tile[4][kWgradTile * 65];
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int64_t row = (int64_t)blockIdx.x * 4 + wv;
    const int ln = threadIdx.x & 63;
    if (row >= n_rows) return;
    const uint64_t mk = masks[row];
    const int64_t e0 = rp[row];
    const int len = (int)(rp[row + 1] - e0);
    const bool on = ln < lanes;
    // lanes past `lanes` read column 0 (never stored, never summed)
    const float* gb = g_dst + (on ? ln : 0);
    const int32_t* cs = col + e0;
    const float* ws = w + e0;
    float* gws = gw + e0;
    float* t = tile[wv];
    float acc0 = 0.f, acc1 = 0.f;
    float g[kWgradTile];
    if (ln < kWgradTile) t[ln * 65 + 64] = 0.f;  // the column an odd set bit is missing from
    int my_d = ln < len ? cs[ln] : 0;
    auto request = [&](int m) {
        if (m >= kWgradTile) {
#pragma unroll
            for (int k = 0; k < kWgradTile; ++k)
                g[k] = gb[(int64_t)__builtin_amdgcn_readlane(my_d, k) * lanes];
        } else {
#pragma unroll
            for (int k = 0; k < kWgradTile; ++k)
                g[k] = k < m ? gb[(int64_t)__builtin_amdgcn_readlane(my_d, k) * lanes] : 0.f;
        }
    };
    if (len > 0) request(len);
    for (int c = 0; c < len; c += kWgradTile) {
        const int m = len - c < kWgradTile ? len - c : kWgradTile;
        const bool mine = ln < m;
        const int my_w = mine ? __float_as_int(ws[c + ln]) : 0;
        const float old = mk && mine ? gws[c + ln] : 0.f;
        // the next tile's destinations
        const int nc = c + kWgradTile + ln;
        my_d = ln < kWgradTile && nc < len ? cs[nc] : 0;
        if (m == kWgradTile) {
#pragma unroll
            for (int k = 0; k < kWgradTile; k += 2) {
                acc0 = fmaf(__int_as_float(__builtin_amdgcn_readlane(my_w, k)), g[k], acc0);
                acc1 = fmaf(__int_as_float(__builtin_amdgcn_readlane(my_w, k + 1)), g[k + 1], acc1);
            }
        } else {
#pragma unroll
            for (int k = 0; k < kWgradTile; ++k) {
                if (k < m) {
                    const float wk = __int_as_float(__builtin_amdgcn_readlane(my_w, k));
                    if (k & 1) acc1 = fmaf(wk, g[k], acc1);
                    else acc0 = fmaf(wk, g[k], acc0);
                }
            }
        }
        if (mk) {
            // rows past m hold zeros or stale values nobody sums
#pragma unroll
            for (int k = 0; k < kWgradTile; ++k) t[k * 65 + ln] = g[k];
        }
        if (c + kWgradTile < len) request(len - c - kWgradTile);
        if (mk) {
            // the tile is the wavefront's own: its LDS writes land before its
            // reads, the fences keep the compiler from moving them across
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            // thread ln sums row ln & 31 over half the set lanes: threads
            // below 32 the even ones of mk, in order, the others the odd ones
            const float* tr = t + (ln & (kWgradTile - 1)) * 65;
            float acc = 0.f;
            uint64_t q = mk;
            while (q) {
                const int b0 = __ffsll((unsigned long long)q) - 1;
                q &= q - 1;
                const int b1 = q ? __ffsll((unsigned long long)q) - 1 : 64;  // 64: a zero column
                q &= q - 1;
                acc += tr[ln < kWgradTile ? b0 : b1];
            }
            acc += __shfl_xor(acc, 32, 64);
            if (mine) gws[c + ln] = old + acc;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }
    if (on) g_src[row * lanes + ln] = acc0 + acc1;
}

// The same with lanes a multiple of 4, rows of g_dst 16-byte aligned and 32-bit
// byte offsets into it: a
// quarter of the wavefront per edge, four lanes per thread, so that a tile is
// eight requests instead of 32 and one instruction sums four edges (13.4M edges,
// 64 lanes: 392 -> 285 us a step, 285 -> 183 us where no neuron spiked, the
// latter 19 TB/s out of L2).
__global__ __launch_bounds__(256) void k_adj_transpose_wgrad4(
    const int64_t* __restrict__ rp, const int32_t* __restrict__ col,
    const float* __restrict__ w, int64_t n_rows, int64_t lanes,
    const uint64_t* __restrict__ masks, const float* __restrict__ g_dst,
    float* __restrict__ g_src, float* __restrict__ gw) {
    constexpr int kRow = 68;  // 64 lanes, a zero column, whole float4s
    __shared__ __align__(16) float tile[4][kWgradTile * kRow];
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int64_t row = (int64_t)blockIdx.x * 4 + wv;
    const int ln = threadIdx.x & 63;
    if (row >= n_rows) return;
    const uint64_t mk = masks[row];
    const int64_t e0 = rp[row];
    const int len = (int)(rp[row + 1] - e0);
    const int q = ln >> 4, c = (ln & 15) * 4;
    const bool on = c < lanes;
    // lanes past `lanes` read column 0 (never stored, never summed)
    const uint32_t c_in = on ? c : 0;
    const int32_t* cs = col + e0;
    const float* ws = w + e0;
    float* gws = gw + e0;
    float* t = tile[wv];
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 g[8];
    if (ln < kWgradTile) t[ln * kRow + 64] = 0.f;  // the column an odd set bit is missing from
    int my_d = ln < len ? cs[ln] : 0;
    auto request = [&](int m) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int d = __shfl(my_d, 4 * j + q, 64);
            g[j] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (4 * j + q < m)
                g[j] = *reinterpret_cast<const float4*>(g_dst + ((uint32_t)d * (uint32_t)lanes + c_in));
        }
    };
    if (len > 0) request(len);
    for (int k0 = 0; k0 < len; k0 += kWgradTile) {
        const bool mine = ln < kWgradTile && k0 + ln < len;
        const float my_w = mine ? ws[k0 + ln] : 0.f;
        const float old = mk && mine ? gws[k0 + ln] : 0.f;
        // the next tile's destinations
        const int nx = k0 + kWgradTile + ln;
        my_d = ln < kWgradTile && nx < len ? cs[nx] : 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float wk = __shfl(my_w, 4 * j + q, 64);
            acc.x = fmaf(wk, g[j].x, acc.x);
            acc.y = fmaf(wk, g[j].y, acc.y);
            acc.z = fmaf(wk, g[j].z, acc.z);
            acc.w = fmaf(wk, g[j].w, acc.w);
        }
        if (mk) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                *reinterpret_cast<float4*>(t + (4 * j + q) * kRow + c) = g[j];
        }
        if (k0 + kWgradTile < len) request(len - k0 - kWgradTile);
        if (mk) {
            // the tile is the wavefront's own: its LDS writes land before its
            // reads, the fences keep the compiler from moving them across
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            // thread ln sums row ln & 31 over half the set lanes: threads
            // below 32 the even ones of mk, in order, the others the odd ones
            const float* tr = t + (ln & (kWgradTile - 1)) * kRow;
            float sum = 0.f;
            uint64_t bits = mk;
            while (bits) {
                const int b0 = __ffsll((unsigned long long)bits) - 1;
                bits &= bits - 1;
                const int b1 = bits ? __ffsll((unsigned long long)bits) - 1 : 64;  // a zero column
                bits &= bits - 1;
                sum += tr[ln < kWgradTile ? b0 : b1];
            }
            sum += __shfl_xor(sum, 32, 64);
            if (mine) gws[k0 + ln] = old + sum;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) {
        acc.x += __shfl_xor(acc.x, o, 64);
        acc.y += __shfl_xor(acc.y, o, 64);
        acc.z += __shfl_xor(acc.z, o, 64);
        acc.w += __shfl_xor(acc.w, o, 64);
    }
    if (q == 0 && on) *reinterpret_cast<float4*>(g_src + row * lanes + c) = acc;
}

// Delayed synapses (HeterSynapsePSC / DelayedPSC): psc_s receives
// W_sub^T z_{s - age(sub)} through the virtual rows j*csr_d + sub, so the
// spike z_t of neuron j collects sum over sub of W_sub dL/dpsc_{t + age(sub)}
// -- the reverse delay ring.  G holds dL/dpsc of the K steps of a window,
// [K][n][lanes]; step tau of the window reads G[tau + age] when that index
// lies in [0, K) (later steps belong to another window).
//
// One wavefront per neuron, 64 of whose edges are read at a time, a lane each
// with the step its virtual row reads; PER = 64 / (lanes rounded up to a
// power of two) edges are then summed side by side, eight of each in flight,
// and the PER partial sums added at the end (an edge at a time, one wavefront
// for 16 lanes: 36 us a step at 4096 neurons, 0.41M edges).  Also the
// undelayed product of at most 32 lanes (csr_d = 1, age 0, K = 1).  Row: an
// integer that holds the rows of G, K*n of them.
template <int PER, typename Row>
__global__ __launch_bounds__(256) void k_adj_transpose_rows(
    const int64_t* __restrict__ rp, const int32_t* __restrict__ col,
    const float* __restrict__ w, int64_t n, int csr_d, int64_t lanes,
    const float* __restrict__ G, int64_t K, int64_t tau, const int* __restrict__ ages,
    float* __restrict__ g_src, int accumulate) {
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int64_t j = (int64_t)blockIdx.x * 4 + wv;
    const int ln = threadIdx.x & 63;
    if (j >= n) return;
    constexpr int W = 64 / PER;  // threads per edge
    const int grp = ln / W;
    const int64_t e0 = rp[j * csr_d];
    const int len = (int)(rp[(j + 1) * csr_d] - e0);
    // thread s: where virtual row s ends, and the step it reads (-1 = none)
    int ends = 0x7fffffff, step = -1;
    if (ln < csr_d) {
        ends = (int)(rp[j * csr_d + ln + 1] - e0);
        const int age = ages ? ages[ln] : 0;
        const int64_t st = tau + age;
        step = age >= 0 && st >= 0 && st < K ? (int)st : -1;
    }
    for (int64_t b0 = 0; b0 < lanes; b0 += W) {
        const int64_t b = b0 + ln % W;
        const bool on = b < lanes;
        const float* gb = G + (on ? b : 0);
        float acc = 0.f;
        for (int c = 0; c < len; c += 64) {
            const int e = c + ln;
            int sub = 0;
            for (int s = 0; s + 1 < csr_d; ++s) sub += e >= __builtin_amdgcn_readlane(ends, s);
            const int st = __shfl(step, sub, 64);
            const bool in = e < len && st >= 0;
            // row of G the edge reads, -1 = none
            const Row my_r = in ? (Row)(st * n) + col[e0 + e] : -1;
            const float my_w = in ? w[e0 + e] : 0.f;
            if (__ballot(in) == 0ull) continue;
            const int m = len - c < 64 ? len - c : 64;
            for (int k = 0; k < m; k += 8 * PER) {
                float g8[8], w8[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int src = k + u * PER + grp;
                    const Row r = __shfl(my_r, src & 63, 64);
                    w8[u] = __shfl(my_w, src & 63, 64);
                    const bool use = src < m && r >= 0;
                    g8[u] = use ? gb[(int64_t)r * lanes] : 0.f;
                    w8[u] = use ? w8[u] : 0.f;
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) acc = fmaf(w8[u], g8[u], acc);
            }
        }
#pragma unroll
        for (int o = W; o < 64; o <<= 1) acc += __shfl_xor(acc, o, 64);
        if (on && grp == 0) g_src[j * lanes + b] = accumulate ? g_src[j * lanes + b] + acc : acc;
    }
}

template <typename Row>
static void launch_transpose_rows_of(const int64_t* rp, const int32_t* col, const float* w,
                                     int64_t n, int csr_d, int64_t lanes, const float* G, int64_t K,
                                     int64_t tau, const int* ages, float* g_src, int accumulate,
                                     hipStream_t s) {
    const dim3 grid((unsigned)((n + 3) / 4)), block(256);
    if (lanes > 32)
        hipLaunchKernelGGL((k_adj_transpose_rows<1, Row>), grid, block, 0, s, rp, col, w, n, csr_d,
                           lanes, G, K, tau, ages, g_src, accumulate);
    else if (lanes > 16)
        hipLaunchKernelGGL((k_adj_transpose_rows<2, Row>), grid, block, 0, s, rp, col, w, n, csr_d,
                           lanes, G, K, tau, ages, g_src, accumulate);
    else if (lanes > 8)
        hipLaunchKernelGGL((k_adj_transpose_rows<4, Row>), grid, block, 0, s, rp, col, w, n, csr_d,
                           lanes, G, K, tau, ages, g_src, accumulate);
    else
        hipLaunchKernelGGL((k_adj_transpose_rows<8, Row>), grid, block, 0, s, rp, col, w, n, csr_d,
                           lanes, G, K, tau, ages, g_src, accumulate);
}

static void launch_transpose_rows(const int64_t* rp, const int32_t* col, const float* w, int64_t n,
                                  int csr_d, int64_t lanes, const float* G, int64_t K, int64_t tau,
                                  const int* ages, float* g_src, int accumulate, hipStream_t s) {
    if (K * n < (int64_t)1 << 31)
        launch_transpose_rows_of<int>(rp, col, w, n, csr_d, lanes, G, K, tau, ages, g_src,
                                      accumulate, s);
    else
        launch_transpose_rows_of<int64_t>(rp, col, w, n, csr_d, lanes, G, K, tau, ages, g_src,
                                          accumulate, s);
}

// gw[e] += sum over lanes b spiking at neuron j (mask bit b) of
// G[tau + age(sub)][col[e], b], for every virtual row j*csr_d + sub whose
// step lies in the window.  One wavefront per neuron; lanes stride the edges.
__global__ __launch_bounds__(256) void k_adj_wgrad_delayed(
    const int64_t* __restrict__ rp, const int32_t* __restrict__ col, int64_t n, int csr_d,
    int64_t lanes, const uint64_t* __restrict__ masks, const float* __restrict__ G, int64_t K,
    int64_t tau, const int* __restrict__ ages, float* __restrict__ gw) {
    const int64_t j = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int ln = threadIdx.x & 63;
    if (j >= n) return;
    const uint64_t mk = masks[j];
    if (mk == 0) return;
    for (int sub = 0; sub < csr_d; ++sub) {
        const int age = ages[sub];
        const int64_t st = tau + age;
        if (age < 0 || st < 0 || st >= K) continue;
        const float* g = G + st * n * lanes;
        const int64_t r = j * csr_d + sub;
        for (int64_t e = rp[r] + ln; e < rp[r + 1]; e += 64) {
            const int64_t d = col[e];
            float acc = 0.f;
            uint64_t q = mk;
            while (q) {
                const int b = __ffsll((unsigned long long)q) - 1;
                acc += g[d * lanes + b];
                q &= q - 1;
            }
            gw[e] += acc;
        }
    }
}

}  // namespace btx

using namespace btx;

BTX_API int btx_adj_lif_step(const btx_adj_lif_args* p, void* stream) {
    if (p == nullptr) return fail("btx_adj_lif_step: null args");
    const int64_t m = p->n * p->lanes;
    if (m <= 0) return 0;
    if (p->surrogate < BTX_SURR_SIGMOID || p->surrogate > BTX_SURR_ERF)
        return fail("btx_adj_lif_step: unknown surrogate");
    AdjArgs a{};
    a.n = p->n;
    a.lanes = p->lanes;
    a.dt = p->dt;
    a.hard_reset = p->hard_reset;
    a.detach_reset = p->detach_reset;
    a.surrogate = p->surrogate;
    a.alpha = p->alpha;
    a.damping = p->damping;
    a.tau = p->tau; a.tau_s = p->tau_stride;
    a.vth = p->v_th; a.vth_s = p->v_th_stride;
    a.vr = p->v_reset; a.vr_s = p->v_reset_stride;
    a.cm = p->c_m; a.cm_s = p->c_m_stride;
    a.tsyn = p->tau_syn; a.tsyn_s = p->tau_syn_stride;
    a.ksyn = p->k_syn; a.ksyn_s = p->k_syn_stride;
    a.v_prev = p->v_prev;
    a.v_pre = p->v_pre;
    a.z = p->z;
    a.ref_prev = p->ref_prev;
    a.gz = p->gz;
    a.gsyn = p->gsyn;
    a.gv = p->gv;
    a.gpsc = p->gpsc;
    a.gx = p->gx;
    a.gtau = p->gtau;
    a.gpsc_out = p->gpsc_out ? p->gpsc_out : p->gpsc;
    if (p->lane_major) {
        if (p->lanes > 64) return fail("btx_adj_lif_step: at most 64 lanes lane-major");
        hipLaunchKernelGGL(k_adj_lif_lanes, dim3((unsigned)((p->n + kAdjTile - 1) / kAdjTile)),
                           dim3(256), 0, (hipStream_t)stream, a);
        return check_launch("btx_adj_lif_step");
    }
    if (p->gz == nullptr) return fail("btx_adj_lif_step: gz is required neuron-major");
    hipLaunchKernelGGL(k_adj_lif, dim3((unsigned)((m + 255) / 256)), dim3(256), 0,
                       (hipStream_t)stream, a);
    return check_launch("btx_adj_lif_step");
}

BTX_API int btx_adj_transpose(const int64_t* row_ptr, const int32_t* col, const float* w,
                              int64_t n_rows, int64_t lanes, const float* g_dst, float* g_src,
                              void* stream) {
    if (n_rows <= 0 || lanes <= 0) return 0;
    hipLaunchKernelGGL(k_adj_transpose, dim3((unsigned)((n_rows + 3) / 4)), dim3(256), 0,
                       (hipStream_t)stream, row_ptr, col, w, n_rows, lanes, g_dst, g_src);
    return check_launch("btx_adj_transpose");
}

BTX_API int btx_adj_wgrad(const int64_t* row_ptr, const int32_t* col, int64_t n_rows,
                          int64_t lanes, const uint64_t* masks, const float* g_dst, float* gw,
                          void* stream) {
    if (n_rows <= 0 || lanes <= 0) return 0;
    if (lanes > 64) return fail("btx_adj_wgrad: at most 64 lanes per mask word");
    hipLaunchKernelGGL(k_adj_wgrad, dim3((unsigned)((n_rows + 3) / 4)), dim3(256), 0,
                       (hipStream_t)stream, row_ptr, col, n_rows, lanes, masks, g_dst, gw);
    return check_launch("btx_adj_wgrad");
}

BTX_API int btx_adj_lif_chunk(const btx_adj_lif_args* p, int64_t K, const int64_t* row_ptr,
                              const int32_t* col, const float* w, const uint64_t* masks,
                              float* gw, void* stream) {
    if (p == nullptr) return fail("btx_adj_lif_chunk: null args");
    return btx_adj_lif_sweep(p, K, p->n * p->lanes, nullptr, row_ptr, col, w, 1, nullptr, nullptr,
                             masks, gw, stream);
}

BTX_API int btx_adj_lif_sweep(const btx_adj_lif_args* p, int64_t K, int64_t gz_stride,
                              const float* ref_entry, const int64_t* row_ptr, const int32_t* col,
                              const float* w, int csr_d, const int* ages, float* G,
                              const uint64_t* masks, float* gw, void* stream) {
    if (p == nullptr) return fail("btx_adj_lif_sweep: null args");
    if (K <= 0 || p->n <= 0 || p->lanes <= 0) return 0;
    if (p->lanes > 64) return fail("btx_adj_lif_sweep: at most 64 lanes per mask word");
    if (p->gsyn == nullptr || p->gpsc == nullptr || masks == nullptr || gw == nullptr)
        return fail("btx_adj_lif_sweep: gsyn, gpsc, masks and gw are required");
    const bool delayed = ages != nullptr;
    if (delayed && (G == nullptr || csr_d < 1 || csr_d > BTX_MAX_BINS))
        return fail("btx_adj_lif_sweep: delays need G and 1 <= csr_d <= 64");
    const int64_t m = p->n * p->lanes;
    const hipStream_t st = (hipStream_t)stream;
    const dim3 rows((unsigned)((p->n + 3) / 4));
    btx_adj_lif_args s = *p;
    for (int64_t t = K - 1; t >= 0; --t) {
        // dL/dpsc after step t through the transposed product and the weight
        // gradient of step t's spikes (33 to 64 lanes without delays: one
        // pass), then the elementwise reverse step
        const uint64_t* mk = masks + t * p->n;
        float* gsyn = (float*)p->gsyn;
        if (delayed) {
            launch_transpose_rows(row_ptr, col, w, p->n, csr_d, p->lanes, G, K, t, ages, gsyn, 0, st);
            hipLaunchKernelGGL(k_adj_wgrad_delayed, rows, dim3(256), 0, st, row_ptr, col, p->n,
                               csr_d, p->lanes, mk, G, K, t, ages, gw);
            s.gpsc = G + t * m;
            s.gpsc_out = t > 0 ? G + (t - 1) * m : p->gpsc;
        } else if (p->lanes > 32) {
            const bool vec = p->lanes % 4 == 0 && m * 4 < (int64_t)1 << 32 && ((uintptr_t)p->gpsc & 15) == 0 &&
                             ((uintptr_t)gsyn & 15) == 0;
            hipLaunchKernelGGL(vec ? k_adj_transpose_wgrad4 : k_adj_transpose_wgrad, rows,
                               dim3(256), 0, st, row_ptr, col, w, p->n, p->lanes, mk, p->gpsc,
                               gsyn, gw);
        } else {
            launch_transpose_rows(row_ptr, col, w, p->n, 1, p->lanes, p->gpsc, 1, 0, nullptr, gsyn,
                                  0, st);
            hipLaunchKernelGGL(k_adj_wgrad, rows, dim3(256), 0, st, row_ptr, col, p->n, p->lanes,
                               mk, p->gpsc, gw);
        }
        if (int rc = check_launch("btx_adj_lif_sweep")) return rc;
        s.v_prev = p->v_prev + t * m;
        s.v_pre = p->v_pre + t * m;
        s.z = p->z + t * m;
        if (p->ref_prev)
            s.ref_prev = ref_entry == nullptr ? p->ref_prev + t * m
                         : t == 0             ? ref_entry
                                              : p->ref_prev + (t - 1) * m;
        s.gz = p->gz ? p->gz + t * gz_stride : nullptr;
        s.gx = p->gx + t * m;
        if (int rc = btx_adj_lif_step(&s, stream)) return rc;
    }
    return 0;
}

BTX_API int btx_lane_masks(const uint64_t* words, int64_t steps, int64_t lanes, int64_t n,
                           uint64_t* masks, void* stream) {
    if (steps <= 0 || lanes <= 0 || n <= 0) return 0;
    if (lanes > 64) return fail("btx_lane_masks: at most 64 lanes per mask word");
    const int64_t nwords = (n + 63) / 64;
    for (int64_t t0 = 0; t0 < steps; t0 += 65535) {
        const int64_t t = steps - t0 < 65535 ? steps - t0 : 65535;
        hipLaunchKernelGGL(k_lane_masks, dim3((unsigned)nwords, (unsigned)t), dim3(64), 0,
                           (hipStream_t)stream, words + t0 * lanes * nwords, lanes, n,
                           masks + t0 * n);
    }
    return check_launch("btx_lane_masks");
}

BTX_API int btx_adj_transpose_delayed(const int64_t* row_ptr, const int32_t* col, const float* w,
                                      int64_t n, int csr_d, int64_t lanes, const float* G,
                                      int64_t K, int64_t tau, const int* ages, float* g_src,
                                      int accumulate, void* stream) {
    if (n <= 0 || lanes <= 0) return 0;
    if (csr_d < 1 || csr_d > BTX_MAX_BINS) return fail("btx_adj_transpose_delayed: bad csr_d");
    launch_transpose_rows(row_ptr, col, w, n, csr_d, lanes, G, K, tau, ages, g_src, accumulate,
                          (hipStream_t)stream);
    return check_launch("btx_adj_transpose_delayed");
}

BTX_API int btx_adj_wgrad_delayed(const int64_t* row_ptr, const int32_t* col, int64_t n,
                                  int csr_d, int64_t lanes, const uint64_t* masks,
                                  const float* G, int64_t K, int64_t tau, const int* ages,
                                  float* gw, void* stream) {
    if (n <= 0 || lanes <= 0) return 0;
    if (lanes > 64) return fail("btx_adj_wgrad_delayed: at most 64 lanes per mask word");
    if (csr_d < 1 || csr_d > BTX_MAX_BINS) return fail("btx_adj_wgrad_delayed: bad csr_d");
    hipLaunchKernelGGL(k_adj_wgrad_delayed, dim3((unsigned)((n + 3) / 4)), dim3(256), 0,
                       (hipStream_t)stream, row_ptr, col, n, csr_d, lanes, masks, G, K, tau,
                       ages, gw);
    return check_launch("btx_adj_wgrad_delayed");
}
