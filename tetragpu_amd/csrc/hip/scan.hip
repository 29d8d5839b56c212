// Device-wide exclusive scan and fill kernels.  Up to 16384 items: one
// workgroup, one launch.  Up to SCAN_SUMMED tiles of 4096 items: two launches,
// per-tile sums, then the downsweep, in which every workgroup adds up the sums
// before its tile itself (at most 8 a thread; launches are what a scan of this
// size costs: Kuhn 24^3's three scans took 20 us in nine launches).  More
// tiles: the sums are scanned by a launch in between.  Every tile is read
// twice and written once.
#include "common.h"

namespace {

constexpr int SCAN_BLOCK = 256;
constexpr int SCAN_ITEMS = 16;
constexpr int SCAN_TILE = SCAN_BLOCK * SCAN_ITEMS;
constexpr int SCAN_ONE = 1024;       // threads of the single-workgroup scan
constexpr int64_t SCAN_SUMMED = 2048;  // tiles whose sums each workgroup adds up itself
// What k_scan_down finds in partials: nothing (one workgroup), the tiles'
// sums, or their exclusive scan.
enum Partials { ALONE, SUMS, PREFIXES };

template <typename TIn, typename TAcc>
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_reduce(
    const TIn *__restrict__ in, int64_t n, TAcc *__restrict__ partials) {
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE;
    TAcc sum = 0;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; k++) {
        int64_t g = base + k * SCAN_BLOCK + threadIdx.x;
        if (g < n) sum += (TAcc)in[g];
    }
    sum = tgd::wave_sum(sum);
    __shared__ TAcc ws[SCAN_BLOCK / 64];
    if (__lane_id() == 0) ws[threadIdx.x / 64] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        TAcc t = 0;
#pragma unroll
        for (int w = 0; w < SCAN_BLOCK / 64; w++) t += ws[w];
        partials[blockIdx.x] = t;
    }
}

// Single workgroup: exclusive scan of the per-tile sums, total to *total.
template <typename TAcc, typename TOut>
__global__ __launch_bounds__(1024) void k_scan_partials(
    TAcc *__restrict__ partials, int64_t nb, TOut *__restrict__ total) {
    __shared__ TAcc wsum[16];
    const int lane = __lane_id(), wid = threadIdx.x / 64;
    TAcc carry = 0;
    for (int64_t c = 0; c < nb; c += 1024) {
        const int64_t i = c + threadIdx.x;
        const TAcc x = i < nb ? partials[i] : (TAcc)0;
        const TAcc inc = tgd::wave_inclusive_sum(x);
        if (lane == 63) wsum[wid] = inc;
        __syncthreads();
        if (wid == 0) {
            TAcc w = lane < 16 ? wsum[lane] : (TAcc)0;
            w = tgd::wave_inclusive_sum(w);
            if (lane < 16) wsum[lane] = w;
        }
        __syncthreads();
        const TAcc before = wid > 0 ? wsum[wid - 1] : (TAcc)0;
        if (i < nb) partials[i] = carry + before + inc - x;
        const TAcc tile_total = wsum[15];
        __syncthreads();
        carry += tile_total;
    }
    if (threadIdx.x == 0) *total = (TOut)carry;
}

__device__ __forceinline__ int pad(int i) { return i + (i >> 5); }

template <typename TIn, typename TOut, typename TAcc, int BLOCK, Partials HAVE>
__global__ __launch_bounds__(BLOCK) void k_scan_down(
    const TIn *in, TOut *out, int64_t n, const TAcc *__restrict__ partials) {
    constexpr int TILE = BLOCK * SCAN_ITEMS;
    __shared__ TAcc lds[TILE + TILE / 32];
    __shared__ TAcc wsum[BLOCK / 64], wbase[BLOCK / 64];
    const int64_t base = (int64_t)blockIdx.x * TILE;
    const int t = threadIdx.x, lane = __lane_id(), wid = t / 64;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; k++) {
        const int i = k * BLOCK + t;
        const int64_t g = base + i;
        lds[pad(i)] = g < n ? (TAcc)in[g] : (TAcc)0;
    }
    if (HAVE == SUMS) {
        TAcc before = 0;
        for (int64_t i = t; i < (int64_t)blockIdx.x; i += BLOCK) before += partials[i];
        before = tgd::wave_sum(before);
        if (lane == 0) wbase[wid] = before;
    }
    __syncthreads();
    TAcc v[SCAN_ITEMS];
    TAcc s = 0;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; k++) {
        v[k] = lds[pad(t * SCAN_ITEMS + k)];
        s += v[k];
    }
    const TAcc inc = tgd::wave_inclusive_sum(s);
    if (lane == 63) wsum[wid] = inc;
    __syncthreads();
    TAcc run = inc - s;
    if (HAVE == PREFIXES) run += partials[blockIdx.x];
#pragma unroll
    for (int w = 0; w < BLOCK / 64; w++) {
        if (HAVE == SUMS) run += wbase[w];
        if (w < wid) run += wsum[w];
    }
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; k++) {
        lds[pad(t * SCAN_ITEMS + k)] = run;
        run += v[k];
    }
    if (HAVE != PREFIXES && blockIdx.x == gridDim.x - 1 && t == BLOCK - 1) out[n] = (TOut)run;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; k++) {
        const int i = k * BLOCK + t;
        const int64_t g = base + i;
        if (g < n) out[g] = (TOut)lds[pad(i)];
    }
}

template <typename T>
__global__ void k_fill(T *__restrict__ p, T value, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = value;
}

__global__ void k_zero3(int32_t *a, int64_t na, int32_t *b, int64_t nb, int32_t *c, int64_t nc) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < na + nb + nc;
         i += (int64_t)gridDim.x * blockDim.x) {
        if (i < na) a[i] = 0;
        else if (i < na + nb) b[i - na] = 0;
        else c[i - na - nb] = 0;
    }
}

template <typename TIn, typename TOut, typename TAcc>
int scan_impl(const TIn *in, TOut *out, int64_t n, void *tmp, hipStream_t s) {
    if (n < 0) return tg::ERR_ARG;
    if (n == 0) {
        hipLaunchKernelGGL((k_fill<TOut>), dim3(1), dim3(64), 0, s, out, (TOut)0, (int64_t)1);
        TG_LAUNCH_CHECK("k_fill");
        return tg::OK;
    }
    const int64_t nb = (n + SCAN_TILE - 1) / SCAN_TILE;
    TAcc *partials = (TAcc *)tmp;
    if (n <= SCAN_ONE * SCAN_ITEMS) {
        hipLaunchKernelGGL((k_scan_down<TIn, TOut, TAcc, SCAN_ONE, ALONE>), dim3(1),
                           dim3(SCAN_ONE), 0, s, in, out, n, partials);
        TG_LAUNCH_CHECK("k_scan_down");
        return tg::OK;
    }
    hipLaunchKernelGGL((k_scan_reduce<TIn, TAcc>), dim3((unsigned)nb), dim3(SCAN_BLOCK), 0, s,
                       in, n, partials);
    TG_LAUNCH_CHECK("k_scan_reduce");
    if (nb <= SCAN_SUMMED) {
        hipLaunchKernelGGL((k_scan_down<TIn, TOut, TAcc, SCAN_BLOCK, SUMS>), dim3((unsigned)nb),
                           dim3(SCAN_BLOCK), 0, s, in, out, n, partials);
    } else {
        hipLaunchKernelGGL((k_scan_partials<TAcc, TOut>), dim3(1), dim3(1024), 0, s, partials, nb,
                           out + n);
        TG_LAUNCH_CHECK("k_scan_partials");
        hipLaunchKernelGGL((k_scan_down<TIn, TOut, TAcc, SCAN_BLOCK, PREFIXES>),
                           dim3((unsigned)nb), dim3(SCAN_BLOCK), 0, s, in, out, n, partials);
    }
    TG_LAUNCH_CHECK("k_scan_down");
    return tg::OK;
}

}  // namespace

namespace tg {

size_t scan_tmp_bytes(int64_t n) {
    int64_t nb = (n + SCAN_TILE - 1) / SCAN_TILE;
    return (size_t)(nb < 1 ? 1 : nb) * sizeof(int64_t) + 256;
}

int scan_exclusive_i32(const int32_t *in, int32_t *out, int64_t n, void *tmp,
                       hipStream_t s) {
    return scan_impl<int32_t, int32_t, int32_t>(in, out, n, tmp, s);
}

int fill_i32(int32_t *p, int32_t value, int64_t n, hipStream_t s) {
    if (n <= 0) return OK;
    unsigned g = grid_for(n, 256);
    if (g > 4096) g = 4096;
    hipLaunchKernelGGL((k_fill<int32_t>), dim3(g), dim3(256), 0, s, p, value, n);
    TG_LAUNCH_CHECK("k_fill<i32>");
    return OK;
}
int zero_i32(int32_t *a, int64_t na, int32_t *b, int64_t nb, int32_t *c, int64_t nc,
             hipStream_t s) {
    if (!a) na = 0;
    if (!b) nb = 0;
    if (!c) nc = 0;
    if (na + nb + nc <= 0) return OK;
    unsigned g = grid_for(na + nb + nc, 256);
    if (g > 4096) g = 4096;
    hipLaunchKernelGGL(k_zero3, dim3(g), dim3(256), 0, s, a, na, b, nb, c, nc);
    TG_LAUNCH_CHECK("k_zero3");
    return OK;
}
int fill_u8(uint8_t *p, uint8_t value, int64_t n, hipStream_t s) {
    if (n <= 0) return OK;
    unsigned g = grid_for(n, 256);
    if (g > 4096) g = 4096;
    hipLaunchKernelGGL((k_fill<uint8_t>), dim3(g), dim3(256), 0, s, p, value, n);
    TG_LAUNCH_CHECK("k_fill<u8>");
    return OK;
}

}  // namespace tg
