// Itemized risk of a Europeans product on Dupire (mcBase.h:858-989 for vanilla
// calls): the adjoint of call k of one maturity is, along a path, the path's
// own chain times S 1{S > K_k} at the maturity, so the calls of a maturity
// share one reverse sweep per path.  A path whose spot at the maturity passes
// exactly the first b strikes carries the adjoint of calls 1 .. b: it is swept
// once, into the local-vol grid of list b, and the risk of call k is the sum of
// the grids of lists k, k + 1, ...
//
// After a forward-only launch (ck_mode 1) that keeps every block of 64 paths'
// checkpoints and end states:
//   item_classify_kernel  lists each maturity's paths by b (paths under the
//                         lowest strike are in no list);
//   item_reverse_kernel   sweeps the lists, one block per chunk of a list, the
//                         block's grid in LDS as in the path kernels, added to
//                         the list's grid at the end;
//   item_finish_kernel    adds the lists above, and maps the sums onto the
//                         local-vol nodes (sqrt(dt) and the time interpolation
//                         of Dupire::init).
//
// What bounds it: the sweeps' vector instructions and LDS atomics.  The lanes
// of a wave gather their checkpoints from different blocks of 64 paths, a
// 32-byte (FP64) or 16-byte (FP32) word and a bracket word per four steps,
// which the caches hold up to some 2^17 paths (the engine leaves few calls on
// many paths to the sweep per payoff).  30 calls over six maturities
// on 2^16 paths, 156 steps, 30 x 36 grid, FP64: one launch per call took 3.2 ms
// (17.5 sweeps of all paths over the 156 steps, a synchronisation each); the
// lists are 2.6 sweeps, 0.14 ms of reverse.  (A grid per chunk, summed by the
// finish, and two copies: 0.27 ms.)
#include <hip/hip_runtime.h>

#include <algorithm>

#include "cf_path_kernel.h"

namespace cfk {

namespace {

// Checkpoint slot of path p (0-based in the call) and its lane there: the
// block of 64 Sobol indices the forward kept it in (sobol_block).
struct Where {
    size_t slot;
    int lane;
};
__device__ __forceinline__ Where locate(const ItemParams& P, int64_t p)
{
    const int64_t sidx = P.first_path + 1 + p, q = sidx >> 6;
    const int64_t q0 = (P.first_path + 1) >> 6, q1 = (P.first_path + P.n_path) >> 6;
    return {size_t(P.merge_tail && q == q1 ? 0 : q - q0), int(sidx & 63)};
}

template <typename R>
struct Slot {
    const R* x;          // states
    const uint8_t* b;    // bracket bytes
    int lane, n4;
    // element of step i (ckpt_rows)
    __device__ __forceinline__ int el(int i) const
    {
        return sizeof(R) == 4 || i < n4 ? ((i >> 2) << 8) + (lane << 2) + (i & 3) : i * kWave + lane;
    }
};
template <typename R>
__device__ __forceinline__ Slot<R> slot_of(const ItemParams& P, const Where& w)
{
    Slot<R> s;
    s.x = static_cast<const R*>(P.ckpt) + (w.slot * P.ck_rows + kCkptGuardRows) * kWave;
    s.b = reinterpret_cast<const uint8_t*>(s.x + size_t(ckpt_steps(P.n_steps, int(sizeof(R)))) * kWave);
    s.lane = w.lane;
    s.n4 = P.n_steps & ~3;
    return s;
}
// state at timeline point i
template <typename R>
__device__ __forceinline__ R state_at(const ItemParams& P, const Where& w, const Slot<R>& s, int i)
{
    if (i < P.n_steps) return s.x[s.el(i)];
    return static_cast<const R*>(P.state)[w.slot * P.state_rows * kWave + w.lane];
}

// Blocks of 1024 paths (x) by maturity (y).
template <typename R>
__global__ void __launch_bounds__(1024) item_classify_kernel(const ItemParams P)
{
    __shared__ uint32_t cnt[kMaxItemStrikes], base[kMaxItemStrikes];
    const int s = blockIdx.y, lo = P.first[s], nb = P.first[s + 1] - lo, lane = threadIdx.x & 63;
    if (int(threadIdx.x) < nb) cnt[threadIdx.x] = 0;
    __syncthreads();
    const int64_t p = int64_t(blockIdx.x) * 1024 + threadIdx.x;
    int b = 0;
    if (p < P.n_path) {
        const Where w = locate(P, p);
        const R F = state_spot(state_at<R>(P, w, slot_of<R>(P, w), P.points[s]), P.spot);
        // (a path out of the type's range passes all: its chain shows in every risk)
        for (int k = 0; k < nb; ++k) b += F <= R(P.strikes[lo + k]) ? 0 : 1;
    }
    // ranks within the block, then the block's places in the lists
    uint32_t rank = 0;
    for (int j = 1; j <= nb; ++j) {
        const uint64_t m = __builtin_amdgcn_ballot_w64(b == j);
        if (m == 0) continue;
        uint32_t r = 0;
        if (lane == __builtin_ctzll(m)) r = atomicAdd(&cnt[j - 1], uint32_t(__builtin_popcountll(m)));
        r = __builtin_amdgcn_readlane(r, __builtin_ctzll(m));
        if (b == j) rank = r + __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u));
    }
    __syncthreads();
    if (int(threadIdx.x) < nb && cnt[threadIdx.x] > 0)
        base[threadIdx.x] = atomicAdd(&P.counts[lo + threadIdx.x], cnt[threadIdx.x]);
    __syncthreads();
    if (b > 0) P.ids[size_t(lo + b - 1) * size_t(P.n_path) + base[b - 1] + rank] = uint32_t(p);
}

// Zeroes the lists' counts and sums (a launch rather than a memset: the call
// may be captured).
__global__ void __launch_bounds__(256) item_clear_kernel(const ItemParams P)
{
    const size_t i = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (i < size_t(P.n_cols)) {
        P.counts[i] = 0;
        P.deltas[i] = 0.0;
    }
    if (i < size_t(P.n_cols) * size_t(P.n_steps) * size_t(P.n_spots)) P.grids[i] = 0.0;
}

// Blocks: the first chunks of the lists, then their second ones, and so on (the
// lists' lengths are known on the device only: the blocks past their ends come
// last and leave at once), the longest sweeps first.  GIV: the local-vol table
// through L1, where it and a grid do not both fit LDS.  The paths of a list
// end within one strike interval, so their lanes meet on few nodes: the block
// takes as many copies of its grid as LDS holds at the list's steps, up to
// eight.
template <typename R, bool GIV>
__global__ void __launch_bounds__(1024) item_reverse_kernel(const ItemParams P)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int c = P.order[int(blockIdx.x) % P.n_cols], chunk = int(blockIdx.x) / P.n_cols;
    const uint32_t begin = uint32_t(chunk) * uint32_t(P.per_block), count = P.counts[c];
    if (begin >= count) return;
    const uint32_t end = min(begin + uint32_t(P.per_block), count);
    const int n = P.n_steps, m = P.n_spots, mp = lv_cols(m), pt = P.col_point[c];
    const int waves = blockDim.x >> 6, tid = threadIdx.x, nthr = blockDim.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const ItemSmem L = item_smem(pt, m, waves, int(sizeof(R)), GIV);
    const int stride = ivbar_copy_stride(pt, m);
    const int copies = max(1, min(kMaxItemCopies, int((size_t(P.lds) - L.grid) / (size_t(stride) * 8))));
    R* kxi = reinterpret_cast<R*>(smem + L.knots);
    R* iv_lds = reinterpret_cast<R*>(smem + L.iv);
    double* acc = reinterpret_cast<double*>(smem + L.acc);
    double* grid = reinterpret_cast<double*>(smem + L.grid);
    const R* gk = static_cast<const R*>(P.knots);
    const R* gi = static_cast<const R*>(P.inv_dx);
    const R* gv = static_cast<const R*>(P.iv);
    for (int e = tid; e <= m; e += nthr) { kxi[2 * e] = gk[e]; kxi[2 * e + 1] = gi[e]; }
    if constexpr (!GIV)
        for (int e = tid; e < pt * mp; e += nthr) iv_lds[e] = gv[e];
    for (int e = tid; e < copies * stride; e += nthr) grid[e] = 0.0;
    __syncthreads();
    const R* iv;
    if constexpr (GIV) iv = gv; else iv = iv_lds;
    double* gl = grid + (lane % copies) * stride;
    const uint32_t* ids = P.ids + size_t(c) * size_t(P.n_path);

    double delta = 0.0;
    for (uint32_t t = begin + uint32_t(wave) * kWave; t < end; t += uint32_t(waves) * kWave) {
        const bool active = t + uint32_t(lane) < end;
        const Where w = locate(P, ids[active ? t + uint32_t(lane) : begin]);
        const Slot<R> sl = slot_of<R>(P, w);
        R xnext = state_at<R>(P, w, sl, pt);
        R abar = state_spot(xnext, P.spot);   // S x d payoff / d S, the call in the money
        // one step of the reverse sweep as the path kernels take it
        auto step = [&](int i, R xi, int lo) {
            const Bracket<R> b = local_vol_at(kxi, iv + i * mp, xi, lo);
            const R ws = recip_mul(xnext - xi, b.vol) - R(0.5) * b.vol;
            const R vb = abar * ws;
            abar = abar + vb * b.slope;
            if (active) {
                double* row = gl + i * mp;
                atomicAdd(row + b.j, double(vb * b.wa));
                atomicAdd(row + b.j + 1, double(vb * b.wb));
            }
            xnext = xi;
        };
        R x[4];
        uint32_t bw = 0;
        auto load = [&](int g) {   // (below step 0: the slot's guard rows, never used)
            const int e = (g << 8) + (sl.lane << 2);
            if constexpr (sizeof(R) == 4) {
                const float4 v = *reinterpret_cast<const float4*>(sl.x + e);
                x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
            } else {
                const double2* d = reinterpret_cast<const double2*>(sl.x + e);
                const double2 a = d[0], b = d[1];
                x[0] = a.x; x[1] = a.y; x[2] = b.x; x[3] = b.y;
            }
            bw = *reinterpret_cast<const uint32_t*>(sl.b + e);
        };
        int top = pt - 1;
        if constexpr (sizeof(R) == 8)
            for (; top >= sl.n4; --top) step(top, sl.x[sl.el(top)], int(sl.b[sl.el(top)]));
        if (top >= 0) {
            load(top >> 2);
            for (int g = top >> 2; g >= 0; --g) {
                const R y[4] = {x[0], x[1], x[2], x[3]};
                const uint32_t w4 = bw;
                load(g - 1);
#pragma unroll
                for (int k = 3; k >= 0; --k)
                    if (4 * g + k <= top) step(4 * g + k, y[k], int((w4 >> (8 * k)) & 0xffu));
            }
        }
        if (active) delta += double(abar) / P.spot;
    }
    const double ds = wave_sum(delta);
    if (lane == kSumLane) acc[wave] = ds;
    __syncthreads();
    if (tid == 0) {
        double d = 0.0;
        for (int k = 0; k < waves; ++k) d += acc[k];
        unsafeAtomicAdd(P.deltas + c, d);
    }
    double* dst = P.grids + size_t(c) * size_t(n) * size_t(m);
    for (int e = tid; e < pt * m; e += nthr) {
        const int i = e / m, j = e - i * m;
        double v = 0.0;
        for (int k = 0; k < copies; ++k) {
            const double* r = grid + size_t(k) * stride + size_t(i) * mp;
            v += r[j + 1];
            if (j == 0) v += r[0];
            if (j == m - 1) v += r[m + 1];
        }
        if (v != 0.0) unsafeAtomicAdd(dst + e, v);
    }
}

// Blocks: local-vol spot j (x) by maturity (y).  The lists of a maturity from
// the highest strike down: their grids join the running sums of column j,
// which are the adjoints of the list's own call.
__global__ void __launch_bounds__(256) item_finish_kernel(const ItemParams P)
{
    extern __shared__ __align__(16) unsigned char smem[];
    double* a = reinterpret_cast<double*>(smem);   // [n_steps] sqrt(dt)-scaled running sums
    const int j = blockIdx.x, s = blockIdx.y, n = P.n_steps, m = P.n_spots, nT = P.n_times, pt = P.points[s];
    const int tid = threadIdx.x;
    const double np = double(P.n_path);
    for (int i = tid; i < pt; i += 256) a[i] = 0.0;
    double delta = 0.0;
    for (int c = P.first[s + 1] - 1; c >= P.first[s]; --c) {
        for (int i = tid; i < pt; i += 256)
            a[i] += P.grids[(size_t(c) * size_t(n) + size_t(i)) * size_t(m) + j] * P.sqrtdt[i];
        __syncthreads();
        const int out = P.out_col[c];
        for (int t = tid; t < nT; t += 256) {
            double r = 0.0;
            for (int i = P.t_lo[t]; i < min(P.t_hi[t], pt); ++i) {
                if (P.tj0[i] == t) r += a[i] * P.tw0[i];
                if (P.tj1[i] == t && P.tw1[i] != 0.0) r += a[i] * P.tw1[i];
            }
            P.risks[(size_t(1) + size_t(j) * nT + t) * size_t(P.n_cols) + out] = r / np;
        }
        if (j == 0 && tid == 0) {
            delta += P.deltas[c];
            P.risks[out] = delta / np;
        }
        __syncthreads();
    }
}

}  // namespace

int launch_item_reverse(const ItemParams& P, int n_samples, int real_bytes, bool giv, void* stream)
{
    hipStream_t st = static_cast<hipStream_t>(stream);
    const size_t cells = size_t(P.n_cols) * std::max<size_t>(1, size_t(P.n_steps) * size_t(P.n_spots));
    hipLaunchKernelGGL(item_clear_kernel, dim3(unsigned((cells + 255) / 256)), dim3(256), 0, st, P);
    const dim3 cg(unsigned((P.n_path + 1023) / 1024), unsigned(n_samples));
    if (real_bytes == 4) hipLaunchKernelGGL((item_classify_kernel<float>), cg, dim3(1024), 0, st, P);
    else hipLaunchKernelGGL((item_classify_kernel<double>), cg, dim3(1024), 0, st, P);
    const void* f = real_bytes == 4 ? (giv ? reinterpret_cast<const void*>(&item_reverse_kernel<float, true>)
                                           : reinterpret_cast<const void*>(&item_reverse_kernel<float, false>))
                                    : (giv ? reinterpret_cast<const void*>(&item_reverse_kernel<double, true>)
                                           : reinterpret_cast<const void*>(&item_reverse_kernel<double, false>));
    const size_t smem = size_t(P.lds);
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, int(smem));
    if (e != hipSuccess) return int(e);
    void* args[] = {const_cast<ItemParams*>(&P)};
    e = hipLaunchKernel(f, dim3(unsigned(P.n_cols * P.chunks)), dim3(1024), args, smem, st);
    if (e != hipSuccess) return int(e);
    hipLaunchKernelGGL(item_finish_kernel, dim3(unsigned(P.n_spots), unsigned(n_samples)), dim3(256),
                       size_t(P.n_steps > 0 ? P.n_steps : 1) * 8, st, P);
    return int(hipGetLastError());
}

}  // namespace cfk
