// Candidate (nearest-neighbour) lists of many instances on the GPU:
// compute_nn_lists (vrpHelper.cpp:188-236), one wave per row, the row
// sorted in LDS (k_nn_lists), or, for the entry point that allocates
// nothing, one thread per row in a global scratch array.
//
// Each row is sorted with the reference's own steps, sort2
// (utilities.cpp:246-267): the middle element is swapped to the front as
// pivot, smaller elements are swapped forward one by one, the pivot is
// swapped to the boundary, and the two parts [left, last] and
// [last + 1, right] are sorted in turn.  The parts are disjoint, so the
// order they are sorted in does not change the result: here the smaller
// part goes next and the larger waits on a stack of at most log2(n) + 1
// entries.  Rows with equal distances therefore come out in the
// reference's order (tie 0), or in index order when the index breaks ties
// (tie 1), exactly as the host builder aco_compute_nn_lists.
#include <mutex>
#include <string>
#include <vector>

#include "aco_device.h"
#include "aco_internal.h"

namespace cvrp {

struct NnJob {
    const float *dist;   // n rows of pitch dpitch, row-major
    int *out;            // n x width
    int n, width, first_row, dpitch;
};

constexpr int kNnStack = 32;   // > log2(n) + 1 for every n the library accepts

__device__ __forceinline__ bool nn_less(float a, int ia, float b, int ib, int tie)
{
    return a < b || (tie != 0 && a == b && ia < ib);
}

// Sorts keys v[0..n) with node ids ix[0..n) (global or LDS arrays).
template <typename I>
__device__ void nn_sort_row(float *v, I *ix, int n, int tie)
{
    int sl[kNnStack], sr[kNnStack];
    int sp = 0, l = 0, r = n - 1;
    for (;;) {
        if (l >= r) {
            if (sp == 0) return;
            --sp;
            l = sl[sp];
            r = sr[sp];
            continue;
        }
        const int mid = (l + r) / 2;
        const float pv = v[mid];
        const int pi = ix[mid];
        v[mid] = v[l];
        ix[mid] = ix[l];
        v[l] = pv;
        ix[l] = (I)pi;
        int last = l;
        for (int k = l + 1; k <= r; ++k) {
            const float vk = v[k];
            const int ik = ix[k];
            if (nn_less(vk, ik, pv, pi, tie)) {
                ++last;
                v[k] = v[last];
                ix[k] = ix[last];
                v[last] = vk;
                ix[last] = (I)ik;
            }
        }
        v[l] = v[last];
        ix[l] = ix[last];
        v[last] = pv;
        ix[last] = (I)pi;
        if (last - l + 1 < r - last) {
            sl[sp] = last + 1;
            sr[sp] = r;
            r = last;
        } else {
            sl[sp] = l;
            sr[sp] = last;
            l = last + 1;
        }
        ++sp;
    }
}

// ---- one row per wave, in LDS ----
//
// A pass over [l, r] with its pivot in front swaps the j-th smaller element
// (position s_j) with position l + j.  All its swaps are made at once:
// smaller element j ends at l + j, and what stands at l + j moves to s_j, so
// another element at p moves to s_(p-l) for as long as p <= l + m (m smaller
// elements), each hop further right.  The hops of all elements together are
// at most m, and about log(r - l) for one element unless nearly all are
// smaller.  Every element lands where the sequential swaps put it, equal
// distances included.
//
// Parts of more than kNnSmall elements are split this way, 64 elements at a
// time; smaller ones are handed to the lanes, which sort 64 of them side by
// side with the sequential steps.  One thread per row, as before, is a chain
// of n log2(n) LDS round trips: 1001 rows of 1001 nodes 3.58 ms, now 0.28 ms,
// bound by the latency of about 2n/kNnSmall passes per wave.
constexpr int kNnSmall = 32;
constexpr int kNnRowBytes = 4 + 2 + 4 + 2 + 2;   // keys, ids, a second copy of both, s_j

__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// sort2 on at most kNnSmall elements; parts waiting are packed in a word, 10
// bits each (at most log2(kNnSmall) + 1 = 6 of them).
__device__ __forceinline__ void nn_sort_small(float *v, unsigned short *ix, int n, int tie)
{
    static_assert(kNnSmall == 32, "two 5-bit bounds per waiting part");
    unsigned long long waiting = 0;
    int count = 0, l = 0, r = n - 1;
    for (;;) {
        if (l >= r) {
            if (count == 0) return;
            --count;
            l = (int)(waiting >> 5) & 31;
            r = (int)waiting & 31;
            waiting >>= 10;
            continue;
        }
        const int mid = (l + r) / 2;
        const float pv = v[mid];
        const unsigned short pi = ix[mid];
        v[mid] = v[l];
        ix[mid] = ix[l];
        int last = l;
        for (int k = l + 1; k <= r; ++k) {
            const float vk = v[k];
            const unsigned short ik = ix[k];
            if (nn_less(vk, ik, pv, pi, tie)) {
                ++last;
                v[k] = v[last];
                ix[k] = ix[last];
                v[last] = vk;
                ix[last] = ik;
            }
        }
        v[l] = v[last];
        ix[l] = ix[last];
        v[last] = pv;
        ix[last] = pi;
        int wl = l, wr = last;
        if (last - l + 1 < r - last) {
            wl = last + 1;
            wr = r;
            r = last;
        } else {
            l = last + 1;
        }
        waiting = waiting << 10 | (unsigned long long)(wl << 5 | wr);
        ++count;
    }
}

__global__ __launch_bounds__(64) void k_nn_lists(const NnJob *jobs, int njobs, int tie, int nmax)
{
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int stack[2 * kNnStack];
    const int row = blockIdx.x, lane = threadIdx.x;
    int lo = 0, hi = njobs - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (jobs[mid].first_row <= row) lo = mid;
        else hi = mid - 1;
    }
    const NnJob J = jobs[lo];
    const int node = row - J.first_row, n = J.n;
    const float *d = J.dist + (size_t)node * J.dpitch;
    float *v = reinterpret_cast<float *>(smem), *v2 = v + nmax;
    unsigned short *ix = reinterpret_cast<unsigned short *>(v2 + nmax), *ix2 = ix + nmax, *sp = ix2 + nmax;
    for (int i = lane; i < n; i += 64) {
        // a node is not its own neighbour, nor is the depot anyone's
        v[i] = i == node || i == 0 ? INFINITY : d[i];
        ix[i] = (unsigned short)i;
    }
    wave_lds_sync();
    int waiting = 0, l = 0, r = n - 1;   // uniform
    int small = 0, sl = 0, sn = 0;       // lane q < small: the part of sn elements at sl
    for (;;) {
        if (r - l + 1 <= kNnSmall) {
            if (r > l) {
                if (lane == small) {
                    sl = l;
                    sn = r - l + 1;
                }
                ++small;
            }
            if (small == 64 || waiting == 0) {
                if (lane < small) nn_sort_small(v + sl, ix + sl, sn, tie);
                wave_lds_sync();
                small = 0;
            }
            if (waiting == 0) break;
            --waiting;
            l = __builtin_amdgcn_readfirstlane(stack[2 * waiting]);
            r = __builtin_amdgcn_readfirstlane(stack[2 * waiting + 1]);
            continue;
        }
        const int mid = (l + r) / 2;
        const float pv = v[mid], fv = v[l];
        const unsigned short pi = ix[mid], fi = ix[l];
        wave_lds_sync();
        if (lane == 0) {
            v[mid] = fv;
            ix[mid] = fi;
        }
        wave_lds_sync();
        // s_1 .. s_m, relative to l
        int m = 0;
        for (int k0 = l + 1; k0 <= r; k0 += 64) {
            const int k = k0 + lane;
            const bool less = k <= r && nn_less(v[k <= r ? k : r], ix[k <= r ? k : r], pv, pi, tie);
            const unsigned long long b = __ballot(less);
            if (less) sp[m + __popcll(b & ((1ull << lane) - 1ull)) + 1] = (unsigned short)(k - l);
            m += __popcll(b);
        }
        wave_lds_sync();
        // every element but the pivot to its place (the m-th smaller one and
        // the pivot change places at the end: l and l + m)
        int before = 0;
        for (int k0 = l + 1; k0 <= r; k0 += 64) {
            const int k = k0 + lane, kk = k <= r ? k : r;
            const float vk = v[kk];
            const unsigned short ik = ix[kk];
            const bool less = k <= r && nn_less(vk, ik, pv, pi, tie);
            const unsigned long long b = __ballot(less);
            if (k <= r) {
                int q = k - l;
                if (less) {
                    q = before + __popcll(b & ((1ull << lane) - 1ull)) + 1;
                    if (q == m) q = 0;
                } else {
                    while (q <= m) q = sp[q];
                }
                v2[l + q] = vk;
                ix2[l + q] = ik;
            }
            before += __popcll(b);
        }
        if (lane == 0) {
            v2[l + m] = pv;
            ix2[l + m] = pi;
        }
        wave_lds_sync();
        for (int k = l + lane; k <= r; k += 64) {
            v[k] = v2[k];
            ix[k] = ix2[k];
        }
        const int last = l + m;
        int wl = l, wr = last;
        if (last - l + 1 < r - last) {
            wl = last + 1;
            wr = r;
            r = last;
        } else {
            l = last + 1;
        }
        if (lane == 0) {
            stack[2 * waiting] = wl;
            stack[2 * waiting + 1] = wr;
        }
        ++waiting;
        wave_lds_sync();
    }
    for (int h = lane; h < J.width; h += 64) J.out[(size_t)node * J.width + h] = ix[h];
}

static hipError_t launch_nn_lists(const NnJob *djobs, int nj, int rows, int tie, int nmax, hipStream_t st)
{
    static_assert(kMaxNodes * kNnRowBytes + 8 * kNnStack <= (64 << 10), "a row fits a block's LDS");
    hipLaunchKernelGGL(k_nn_lists, dim3(rows), dim3(64), (size_t)nmax * kNnRowBytes, st, djobs, nj, tie, nmax);
    return hipGetLastError();
}

// ---- the same lists without device allocation ----
//
// aco_compute_nn_lists_batch_noalloc sorts in `scratch`, a file-scope device
// array of kNnScratchBytes that every call on a GPU shares (each GPU holds
// its own copy until the process ends).  A launch takes up to kNnRowJobs
// row ranges, passed by value, so nothing is copied to the device first;
// each row of an n-node instance uses 8n bytes of scratch (sort keys and
// node ids).  Every scratch word a row reads is written by that row first,
// so nothing has to start at zero.  Calls that overlap on one GPU race on
// the array.
constexpr size_t kNnScratchBytes = size_t(64) << 20;
constexpr int kNnRowJobs = 32;

static __device__ __align__(256) unsigned char scratch[kNnScratchBytes];

struct NnRowJob {
    const float *dist;   // n x n device array
    int *out;            // n x width device array
    float *v;            // rows x n scratch keys
    int *ix;             // rows x n scratch ids
    int n, width, row0, first;   // first: first thread of this job in the launch
};

struct NnRowJobs {
    NnRowJob j[kNnRowJobs];
    int count, threads;
};

__global__ __launch_bounds__(256) void k_nn_rows(NnRowJobs J, int tie)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= J.threads) return;
    int q = 0;
    while (q + 1 < J.count && J.j[q + 1].first <= t) ++q;
    const NnRowJob R = J.j[q];
    const int r = t - R.first, node = R.row0 + r, n = R.n;
    const float *d = R.dist + (size_t)node * n;
    float *v = R.v + (size_t)r * n;
    int *ix = R.ix + (size_t)r * n;
    for (int i = 0; i < n; ++i) {
        v[i] = d[i];
        ix[i] = i;
    }
    v[node] = INFINITY;
    v[0] = INFINITY;
    nn_sort_row(v, ix, n, tie);
    for (int h = 0; h < R.width; ++h) R.out[(size_t)node * R.width + h] = ix[h];
}

// Per-device address of `scratch` (the array's name is a host-side stand-in,
// not a device address), looked up once per device with that device current.
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[64];

static int scratch_address(void **ptr)
{
    int dev = 0;
    const hipError_t ed = hipGetDevice(&dev);
    if (ed != hipSuccess || dev < 0 || dev >= 64)
        return set_error(ACO_ERR_NODEV, std::string("aco_compute_nn_lists_batch_noalloc: no current device: ") +
                                            hipGetErrorString(ed));
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return set_error(ACO_ERR_HIP, std::string("aco_compute_nn_lists_batch_noalloc: hipGetSymbolAddress: ") +
                                              hipGetErrorString(e));
        g_scratch_ptr[dev] = p;
    }
    *ptr = g_scratch_ptr[dev];
    return ACO_OK;
}

// Instances are processed in chunks of at most this many matrix elements
// (the host path stages the distance matrices on the device).
constexpr size_t kNnChunkElems = size_t(1) << 26;

int gpu_nn_lists(hipStream_t st, int count, const int *n, const float *const *dist, const int *width,
                 int tie, int *const *out)
{
    for (int b = 0; b < count; ++b)
        if (n[b] < 3 || n[b] > kMaxNodes || width[b] < 1 || width[b] > n[b] - 2)
            return set_error(ACO_ERR_ARG, "nn lists: need 3 <= n <= 4096 and 1 <= width <= n-2");
    int b0 = 0;
    while (b0 < count) {
        // one chunk: instances b0 .. b1-1
        size_t elems = 0, outs = 0;
        int b1 = b0, rows = 0, nmax = 0;
        while (b1 < count && (b1 == b0 || elems + (size_t)n[b1] * n[b1] <= kNnChunkElems)) {
            elems += (size_t)n[b1] * n[b1];
            outs += (size_t)n[b1] * width[b1];
            rows += n[b1];
            nmax = n[b1] > nmax ? n[b1] : nmax;
            ++b1;
        }
        const int nj = b1 - b0;
        const size_t bytes = elems * 4 + outs * 4 + (size_t)nj * sizeof(NnJob) + 1024;
        unsigned char *buf = nullptr;
        if (hipMalloc(&buf, bytes) != hipSuccess)
            return set_error(ACO_ERR_HIP, "nn lists: device allocation of " + std::to_string(bytes) + " bytes failed");
        float *ddist = reinterpret_cast<float *>(buf);
        int *dout = reinterpret_cast<int *>(ddist + elems);
        NnJob *djobs = reinterpret_cast<NnJob *>(
            (reinterpret_cast<uintptr_t>(dout + outs) + 255) & ~uintptr_t(255));
        std::vector<NnJob> jobs(nj);
        size_t eo = 0, oo = 0;
        int ro = 0;
        hipError_t err = hipSuccess;
        for (int j = 0; j < nj && err == hipSuccess; ++j) {
            const int b = b0 + j;
            jobs[j] = NnJob{ddist + eo, dout + oo, n[b], width[b], ro, n[b]};
            err = hipMemcpyAsync(ddist + eo, dist[b], (size_t)n[b] * n[b] * 4, hipMemcpyHostToDevice, st);
            eo += (size_t)n[b] * n[b];
            oo += (size_t)n[b] * width[b];
            ro += n[b];
        }
        if (err == hipSuccess)
            err = hipMemcpyAsync(djobs, jobs.data(), sizeof(NnJob) * nj, hipMemcpyHostToDevice, st);
        if (err == hipSuccess) err = launch_nn_lists(djobs, nj, rows, tie, nmax, st);
        oo = 0;
        for (int j = 0; j < nj && err == hipSuccess; ++j) {
            const int b = b0 + j;
            err = hipMemcpyAsync(out[b], dout + oo, (size_t)n[b] * width[b] * 4, hipMemcpyDeviceToHost, st);
            oo += (size_t)n[b] * width[b];
        }
        const hipError_t es = hipStreamSynchronize(st);
        if (err == hipSuccess) err = es;
        (void)hipFree(buf);
        if (err != hipSuccess) return set_error(ACO_ERR_HIP, std::string("nn lists: ") + hipGetErrorString(err));
        b0 = b1;
    }
    return ACO_OK;
}

// The same lists from distance matrices already on the device (n[b] rows
// of pitch pitch[b]) into device arrays out[b] (n[b] x width[b]).  Enqueued
// on st and waited for.
int gpu_nn_lists_dev(hipStream_t st, int count, const int *n, const float *const *dist, const int *pitch,
                     const int *width, int tie, int *const *out)
{
    if (count == 0) return ACO_OK;
    int rows = 0, nmax = 0;
    std::vector<NnJob> jobs(count);
    for (int b = 0; b < count; ++b) {
        jobs[b] = NnJob{dist[b], out[b], n[b], width[b], rows, pitch[b]};
        rows += n[b];
        nmax = n[b] > nmax ? n[b] : nmax;
    }
    NnJob *djobs = nullptr;
    if (hipMalloc(&djobs, sizeof(NnJob) * count) != hipSuccess)
        return set_error(ACO_ERR_HIP, "nn lists: device allocation failed");
    hipError_t err = hipMemcpyAsync(djobs, jobs.data(), sizeof(NnJob) * count, hipMemcpyHostToDevice, st);
    if (err == hipSuccess) err = launch_nn_lists(djobs, count, rows, tie, nmax, st);
    const hipError_t es = hipStreamSynchronize(st);
    if (err == hipSuccess) err = es;
    (void)hipFree(djobs);
    if (err != hipSuccess) return set_error(ACO_ERR_HIP, std::string("nn lists: ") + hipGetErrorString(err));
    return ACO_OK;
}

}  // namespace cvrp

extern "C" int aco_compute_nn_lists_batch(int32_t count, const int32_t *n, const float *const *dist,
                                          const int32_t *nn, int32_t tie, int32_t *const *out)
{
    using namespace cvrp;
    if (count < 0 || (count > 0 && (!n || !dist || !nn || !out)) || (tie != 0 && tie != 1))
        return set_error(ACO_ERR_ARG, "aco_compute_nn_lists_batch: bad argument");
    for (int b = 0; b < count; ++b) {
        if (n[b] < 3 || n[b] > kMaxNodes || nn[b] < 1 || nn[b] > n[b] - 2 || !dist[b] || !out[b])
            return set_error(ACO_ERR_ARG, "aco_compute_nn_lists_batch: instance " + std::to_string(b) +
                                              " needs 3 <= n <= 4096 and 1 <= nn <= n-2");
    }
    if (count == 0) return ACO_OK;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return set_error(ACO_ERR_NODEV, "no HIP device");
    hipStream_t st = nullptr;
    if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess)
        return set_error(ACO_ERR_HIP, "aco_compute_nn_lists_batch: stream creation failed");
    const int rc = gpu_nn_lists(st, count, n, dist, nn, tie, out);
    (void)hipStreamDestroy(st);
    return rc;
}

extern "C" int aco_compute_nn_lists_batch_noalloc(int32_t count, const int32_t *n, const float *const *dist,
                                                  const int32_t *nn, int32_t tie, int32_t *const *out, void *stream)
{
    using namespace cvrp;
    if (count < 0 || (count > 0 && (!n || !dist || !nn || !out)) || (tie != 0 && tie != 1))
        return set_error(ACO_ERR_ARG, "aco_compute_nn_lists_batch_noalloc: bad argument");
    for (int b = 0; b < count; ++b) {
        if (n[b] < 3 || n[b] > kMaxNodes || nn[b] < 1 || nn[b] > n[b] - 2 || !dist[b] || !out[b])
            return set_error(ACO_ERR_ARG, "aco_compute_nn_lists_batch_noalloc: instance " + std::to_string(b) +
                                              " needs 3 <= n <= 4096 and 1 <= nn <= n-2");
        if ((size_t)n[b] * 8 > kNnScratchBytes)
            return set_error(ACO_ERR_ARG, "aco_compute_nn_lists_batch_noalloc: a row of instance " +
                                              std::to_string(b) + " exceeds the " +
                                              std::to_string(kNnScratchBytes) + "-byte scratch");
    }
    if (count == 0) return ACO_OK;
    void *base = nullptr;
    int rc = scratch_address(&base);
    if (rc) return rc;
    const hipStream_t st = static_cast<hipStream_t>(stream);
    unsigned char *const sbase = static_cast<unsigned char *>(base);
    // fill launches: row ranges of consecutive instances while scratch and
    // the job table last
    NnRowJobs J;
    size_t used = 0;
    J.count = 0;
    J.threads = 0;
    auto flush = [&]() -> int {
        if (J.count == 0) return ACO_OK;
        hipLaunchKernelGGL(k_nn_rows, dim3((J.threads + 255) / 256), dim3(256), 0, st, J, (int)tie);
        const hipError_t e = hipGetLastError();
        J.count = 0;
        J.threads = 0;
        used = 0;
        if (e != hipSuccess)
            return set_error(ACO_ERR_HIP, std::string("aco_compute_nn_lists_batch_noalloc: ") + hipGetErrorString(e));
        return ACO_OK;
    };
    for (int b = 0; b < count; ++b) {
        const size_t row_bytes = (size_t)n[b] * 8;
        int row = 0;
        while (row < n[b]) {
            if (J.count == kNnRowJobs || used + row_bytes > kNnScratchBytes) {
                if ((rc = flush())) return rc;
            }
            const int rows = (int)std::min<size_t>((size_t)(n[b] - row), (kNnScratchBytes - used) / row_bytes);
            NnRowJob &R = J.j[J.count++];
            R.dist = dist[b];
            R.out = out[b];
            R.v = reinterpret_cast<float *>(sbase + used);
            R.ix = reinterpret_cast<int *>(sbase + used + (size_t)rows * n[b] * 4);
            R.n = n[b];
            R.width = nn[b];
            R.row0 = row;
            R.first = J.threads;
            J.threads += rows;
            used += (size_t)rows * row_bytes;
            used = (used + 255) & ~size_t(255);
            row += rows;
        }
    }
    return flush();
}
