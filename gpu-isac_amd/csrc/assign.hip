// Equal-size group assignment of particles to classes from the alignment
// scores d[n][p] (the consumer of multi_ref_align's d, bin/sp_isac2_gpu.py:1119-1144,
// where EMAN2's Util.assign_groups does it on the host).
//
// Contract (restated from the reference's call site and its comment there):
// pairs (class n, particle p) are taken in descending score order (ties: lower
// class, then lower particle) and a particle joins its pair's class when it has
// no class yet and the class holds fewer than cap = n_img / n_ref particles.
// With one strict order on the pairs, that greedy result is the unique stable
// assignment, and particle-proposing deferred acceptance finds it in parallel:
// every free particle proposes to its best class not yet tried; every class
// keeps its cap best proposers (score descending, particle ascending) and
// releases the rest; repeat until no free particle has a class left.  The order of
// the proposals does not change the result, so a few rounds over all particles place
// most of them and one workgroup then follows the chains of the last (k_chains).
//
// Output (n_img + 1 ints): class k's particles (ascending) at [k*cap, (k+1)*cap),
// then the r = n_img - n_ref*cap particles no class took (ascending), then one
// class id for those r particles, the class of the highest remaining pair
// (0 when r = 0).  NaN scores count as -infinity.
#include "isac_internal.h"
#include "../../include/gpu_aln_pack.h"

#include <cfloat>
#include <climits>
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <vector>

namespace isac {
namespace {

constexpr int kWave = 64;
constexpr int kSortN = 4096;          // LDS sort capacity of one class step
constexpr int kMaxCap = 2048;         // largest class size supported
constexpr int kChainFree = 1024;      // most free particles k_chains starts from
constexpr int kChainSteps = 4096;     // most proposals of one of its wavefronts
constexpr int kRounds = 8;            // rounds before k_chains (4: 0.1 ms slower, 20000 x 100)

__device__ __forceinline__ float score(const float *d, int pitch, int n, int p) {
    const float v = d[(size_t)n * pitch + p];
    return v == v ? v : -INFINITY;
}

// (v1, a1) before (v2, a2): larger value first, then smaller index.
__device__ __forceinline__ bool before(float v1, int a1, float v2, int a2) {
    return v1 > v2 || (v1 == v2 && a1 < a2);
}

// The wavefront's best class for particle p strictly after (lv, ln) in the order (value
// desc, class asc), or (.., INT_MAX) if every class has been tried; in all lanes.
__device__ __forceinline__ void next_class(const float *d, int pitch, int N, int p, int ln, float lv, int lane,
                                           float &bv, int &bn) {
    bv = -INFINITY;
    bn = INT_MAX;
    for (int n0 = lane; n0 < N; n0 += 4 * kWave) {   // four loads in flight
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = score(d, pitch, min(n0 + r * kWave, N - 1), p);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int n = n0 + r * kWave;
            const bool after = n < N && (ln < 0 || before(lv, ln, v[r], n));   // strictly after the last try
            if (after && (bn == INT_MAX || before(v[r], n, bv, bn))) {
                bv = v[r];
                bn = n;
            }
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const float ov = __shfl_xor(bv, off, kWave);
        const int on = __shfl_xor(bn, off, kWave);
        if (on != INT_MAX && (bn == INT_MAX || before(ov, on, bv, bn))) {
            bv = ov;
            bn = on;
        }
    }
}

// One wavefront per particle: a free particle proposes to its best class after
// the last one it tried.
__global__ __launch_bounds__(256) void k_propose(const float *__restrict__ d, int pitch, int N,
                                                 int P, int *__restrict__ status,
                                                 int *__restrict__ last_n, float *__restrict__ last_v,
                                                 int *__restrict__ cnt, int *__restrict__ props) {
    const int lane = threadIdx.x & 63;
    const int p = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (p >= P) return;
    if (status[p] != 0) return;   // held or exhausted (uniform over the wavefront)
    float bv;
    int bn;
    next_class(d, pitch, N, p, last_n[p], last_v[p], lane, bv, bn);
    if (lane != 0) return;
    if (bn == INT_MAX) {
        status[p] = 2;   // every class has been tried
        return;
    }
    last_n[p] = bn;
    last_v[p] = bv;
    status[p] = 1;
    const int slot = atomicAdd(&cnt[bn], 1);
    props[(size_t)bn * P + slot] = p;
}

// Smallest power of two >= x (x >= 1).
__device__ __forceinline__ int pow2_at_least(int x) {
    int n = 1;
    while (n < x) n <<= 1;
    return n;
}

// Bitonic sort of the first n (a power of two <= kSortN) (value, index) pairs in
// LDS, order `before`.
__device__ void lds_sort(float *v, int *a, int n, int tid, int nthreads) {
    for (int k = 2; k <= n; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int i = tid; i < n; i += nthreads) {
                const int l = i ^ j;
                if (l > i) {
                    const bool up = (i & k) == 0;
                    const bool swap = up ? before(v[l], a[l], v[i], a[i]) : before(v[i], a[i], v[l], a[l]);
                    if (swap) {
                        const float tv = v[i];
                        v[i] = v[l];
                        v[l] = tv;
                        const int ta = a[i];
                        a[i] = a[l];
                        a[l] = ta;
                    }
                }
            }
            __syncthreads();
        }
    }
}

// One workgroup per class: merge the holders (LDS [0, h)) with this round's
// proposers in chunks (LDS [cap, kSortN)), keep the cap best, release the rest.
__global__ __launch_bounds__(256) void k_accept(const float *__restrict__ d, int pitch, int P,
                                                int cap, int *__restrict__ cnt,
                                                const int *__restrict__ props,
                                                int *__restrict__ holders, float *__restrict__ hold_v,
                                                int *__restrict__ hold_cnt, int *__restrict__ status) {
    __shared__ float sv[kSortN];
    __shared__ int sa[kSortN];
    const int c = blockIdx.x, tid = threadIdx.x;
    const int m = cnt[c];
    if (m == 0) return;   // uniform
    int h = hold_cnt[c];
    for (int i = tid; i < cap; i += 256) {
        const int p = i < h ? holders[(size_t)c * cap + i] : -1;
        sv[i] = p >= 0 ? score(d, pitch, c, p) : -INFINITY;
        sa[i] = p >= 0 ? p : INT_MAX;
    }
    const int chunk = kSortN - cap;
    for (int q0 = 0; q0 < m; q0 += chunk) {
        const int q1 = min(m, q0 + chunk);
        const int n = pow2_at_least(cap + (q1 - q0));   // <= kSortN
        for (int i = cap + tid; i < n; i += 256) {
            const int q = q0 + (i - cap);
            const int p = q < q1 ? props[(size_t)c * P + q] : -1;
            sv[i] = p >= 0 ? score(d, pitch, c, p) : -INFINITY;
            sa[i] = p >= 0 ? p : INT_MAX;
        }
        __syncthreads();
        lds_sort(sv, sa, n, tid, 256);
        // valid entries now lead; those past cap are released
        for (int i = cap + tid; i < n; i += 256)
            if (sa[i] != INT_MAX) status[sa[i]] = 0;
        h = min(cap, h + (q1 - q0));
        __syncthreads();
    }
    for (int i = tid; i < h; i += 256) {
        holders[(size_t)c * cap + i] = sa[i];
        hold_v[(size_t)c * cap + i] = sv[i];
    }
    if (tid == 0) {
        hold_cnt[c] = h;
        cnt[c] = 0;
    }
}

// The last rounds, one workgroup: each wavefront takes a free particle, proposes for it,
// goes on with the particle that its class releases, and so on until one finds room, then
// takes the next free one.  A class is locked while its holders change; a wavefront holds
// one lock at a time and never waits with it, so every wait ends.  More than kChainFree
// free particles: nothing is done.  A wavefront that has made kChainSteps proposals frees
// its particle and ends.  left[0] = 1 if free particles may be left.
// A round of the two kernels above costs 19 us however few propose, and there are as many
// as the longest chain has proposals: of 20000 particles and 100 classes 112 rounds, the last
// 95 with 2300 proposals in all.  Here those take 0.53 ms, 2 us of latency a proposal and 16
// proposals at once; as rounds, with a read-back every eighth, the whole took 3.4 ms, now 0.77.
__global__ __launch_bounds__(1024) void k_chains(const float *__restrict__ d, int pitch, int N, int P, int cap,
                                                 int *__restrict__ last_n, float *__restrict__ last_v,
                                                 int *holders, float *hold_v, int *hold_cnt, int *status, int *left) {
    __shared__ int list[kChainFree], lock[1024];
    __shared__ int n_free, head, more;
    const int tid = threadIdx.x, lane = tid & 63;
    if (tid == 0) n_free = head = more = 0;
    lock[tid] = 0;
    __syncthreads();
    for (int p = tid; p < P; p += 1024)
        if (status[p] == 0) {
            const int i = atomicAdd(&n_free, 1);
            if (i < kChainFree) list[i] = p;
        }
    __syncthreads();
    const int nf = n_free;
    if (nf > kChainFree) {   // uniform
        if (tid == 0) left[0] = 1;
        return;
    }
    int steps = 0;
    while (steps < kChainSteps) {
        int q = 0;
        if (lane == 0) q = atomicAdd(&head, 1);
        q = __shfl(q, 0, kWave);
        if (q >= nf) break;
        int p = list[q];
        for (; p >= 0 && steps < kChainSteps; ++steps) {   // p is free and this wavefront's own
            float bv;
            int bn;
            next_class(d, pitch, N, p, last_n[p], last_v[p], lane, bv, bn);
            if (bn == INT_MAX) {
                if (lane == 0) status[p] = 2;
                p = -1;
                break;
            }
            if (lane == 0) {
                last_n[p] = bn;
                last_v[p] = bv;
                while (atomicCAS(&lock[bn & 1023], 0, 1) != 0) __builtin_amdgcn_s_sleep(1);
            }
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
            int *hp = holders + (size_t)bn * cap;
            float *hv = hold_v + (size_t)bn * cap;
            const int h = hold_cnt[bn];
            int slot = h, out = -1;   // a free place, nobody released
            if (h >= cap) {           // the last of the holders in the class's order
                float wv = INFINITY;
                int wp = -1, ws = 0;
                for (int i0 = lane; i0 < cap; i0 += 4 * kWave) {
                    float v[4];
                    int a[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int i = min(i0 + r * kWave, cap - 1);   // a repeated entry changes nothing
                        v[r] = hv[i];
                        a[r] = hp[i];
                    }
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (wp < 0 || before(wv, wp, v[r], a[r])) {
                            wv = v[r];
                            wp = a[r];
                            ws = min(i0 + r * kWave, cap - 1);
                        }
                }
#pragma unroll
                for (int off = 32; off >= 1; off >>= 1) {
                    const float ov = __shfl_xor(wv, off, kWave);
                    const int op = __shfl_xor(wp, off, kWave), os = __shfl_xor(ws, off, kWave);
                    if (op >= 0 && (wp < 0 || before(wv, wp, ov, op))) {
                        wv = ov;
                        wp = op;
                        ws = os;
                    }
                }
                const bool in = before(bv, p, wv, wp);
                slot = in ? ws : -1;
                out = in ? wp : p;
            }
            if (lane == 0 && slot >= 0) {
                hp[slot] = p;
                hv[slot] = bv;
                status[p] = 1;
                if (out >= 0)
                    status[out] = 0;
                else
                    hold_cnt[bn] = h + 1;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            __builtin_amdgcn_wave_barrier();
            if (lane == 0) atomicExch(&lock[bn & 1023], 0);
            p = out;
        }
        if (p >= 0 && lane == 0) more = 1;   // out of steps
    }
    if (lane == 0 && steps >= kChainSteps) more = 1;
    __syncthreads();
    if (tid == 0) left[0] = more;
}

// Output, part 1: block c writes class c's holders ascending at out[c*cap ...].
__global__ __launch_bounds__(256) void k_class_out(int cap, const int *__restrict__ holders,
                                                   const int *__restrict__ hold_cnt,
                                                   int *__restrict__ out) {
    __shared__ float sv[kSortN];
    __shared__ int sa[kSortN];
    const int c = blockIdx.x, tid = threadIdx.x;
    const int h = hold_cnt[c];
    const int n = pow2_at_least(cap);   // cap <= kMaxCap <= kSortN
    for (int i = tid; i < n; i += 256) {
        // sort by particle ascending: value = -particle, index = particle
        const int p = i < h ? holders[(size_t)c * cap + i] : INT_MAX;
        sv[i] = p == INT_MAX ? -INFINITY : -(float)p;
        sa[i] = p;
    }
    __syncthreads();
    lds_sort(sv, sa, n, tid, 256);
    for (int i = tid; i < cap; i += 256) out[(size_t)c * cap + i] = i < h ? sa[i] : -1;
}

// Output, part 2 (one workgroup): the unplaced particles ascending after the
// classes, then the class of the highest remaining pair.
__global__ __launch_bounds__(1024) void k_assign_output(const float *__restrict__ d, int pitch, int N,
                                                       int P, int cap, const int *__restrict__ status,
                                                       int *__restrict__ out) {
    __shared__ int wsum[16];
    __shared__ float rv[1024];
    __shared__ int rn[1024], rp[1024];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    // unplaced particles, ascending (ordered scan over chunks of 1024)
    int base = N * cap;
    float bestv = -INFINITY;
    int bestn = INT_MAX, bestp = INT_MAX;
    for (int p0 = 0; p0 < P; p0 += 1024) {
        const int p = p0 + tid;
        const bool f = p < P && status[p] != 1;
        const unsigned long long m = __ballot(f);
        if (lane == 0) wsum[w] = __popcll(m);
        __syncthreads();
        int ahead = __popcll(m & ((1ull << lane) - 1)), total = 0;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            ahead += v < w ? wsum[v] : 0;
            total += wsum[v];
        }
        if (f) {
            out[base + ahead] = p;
            for (int n = 0; n < N; ++n) {
                const float v = score(d, pitch, n, p);
                if (bestn == INT_MAX || before(v, n, bestv, bestn) ||
                    (v == bestv && n == bestn && p < bestp)) {
                    bestv = v;
                    bestn = n;
                    bestp = p;
                }
            }
        }
        base += total;
        __syncthreads();
    }
    // highest remaining pair (value desc, class asc, particle asc)
    rv[tid] = bestv;
    rn[tid] = bestn;
    rp[tid] = bestp;
    __syncthreads();
    for (int off = 512; off >= 1; off >>= 1) {
        if (tid < off) {
            const float ov = rv[tid + off];
            const int on = rn[tid + off], op = rp[tid + off];
            const bool better = on != INT_MAX &&
                                (rn[tid] == INT_MAX || ov > rv[tid] ||
                                 (ov == rv[tid] && (on < rn[tid] || (on == rn[tid] && op < rp[tid]))));
            if (better) {
                rv[tid] = ov;
                rn[tid] = on;
                rp[tid] = op;
            }
        }
        __syncthreads();
    }
    if (tid == 0) out[P] = rn[0] == INT_MAX ? 0 : rn[0];
}

__global__ void k_assign_init(int *status, int *last_n, float *last_v, int P, int *hold_cnt,
                              int *cnt, int N) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < P) {
        status[i] = 0;
        last_n[i] = -1;
        last_v[i] = INFINITY;
    }
    if (i < N) {
        hold_cnt[i] = 0;
        cnt[i] = 0;
    }
}

// One device allocation cut into arrays (256-byte aligned).
struct Buf {
    void *p = nullptr;
    size_t bytes = 0;
    template <class T>
    T *as() { return static_cast<T *>(p); }
};
struct Arena {
    std::vector<Buf *> parts;
    void *base = nullptr;
    ~Arena() {
        if (base) (void)hipFree(base);
    }
    void add(Buf &b, size_t bytes) {
        b.bytes = (std::max<size_t>(bytes, 4) + 255) & ~(size_t)255;
        parts.push_back(&b);
    }
    hipError_t allocate() {
        size_t total = 0;
        for (Buf *b : parts) total += b->bytes;
        const hipError_t e = hipMalloc(&base, total);
        char *at = static_cast<char *>(base);
        for (Buf *b : parts) {
            b->p = at;
            at += b->bytes;
        }
        return e;
    }
};

int err(int code, const char *msg) {
    report_error(code, msg);
    return code;
}

}  // namespace

int assign_groups(const float *d_d, int N, int P, int pitch, int *d_out, hipStream_t st) {
    if (N < 1 || P < N || pitch < P || !d_d || !d_out)
        return err(2, "assign_groups: need 1 <= n_ref <= n_img <= d_pitch and device buffers");
    const int cap = P / N;
    if (cap > kMaxCap)
        return err(4, "assign_groups: classes of more than 2048 particles are not supported");
    Buf status, last_n, last_v, cnt, props, holders, hold_v, hold_cnt, left;
    Arena arena;
    arena.add(status, (size_t)P * 4);
    arena.add(last_n, (size_t)P * 4);
    arena.add(last_v, (size_t)P * 4);
    arena.add(cnt, (size_t)N * 4);
    arena.add(props, (size_t)N * P * 4);
    arena.add(holders, (size_t)N * cap * 4);
    arena.add(hold_cnt, (size_t)N * 4);
    arena.add(hold_v, (size_t)N * cap * 4);
    arena.add(left, 4);
    if (arena.allocate() != hipSuccess) return err(1, "assign_groups: device allocation failed");
    const int mx = P > N ? P : N;
    hipLaunchKernelGGL(k_assign_init, dim3((mx + 255) / 256), dim3(256), 0, st, status.as<int>(),
                       last_n.as<int>(), last_v.as<float>(), P, hold_cnt.as<int>(), cnt.as<int>(), N);
    // every pass makes at least one proposal until no particle is free; a particle
    // proposes to each class at most once, so N * P + 1 passes bound the loop.
    const long long max_passes = (long long)N * P + 1;
    for (long long pass = 0; pass < max_passes; ++pass) {
        for (int r = 0; r < kRounds; ++r) {
            hipLaunchKernelGGL(k_propose, dim3((P + 3) / 4), dim3(256), 0, st, d_d, pitch, N, P,
                               status.as<int>(), last_n.as<int>(), last_v.as<float>(),
                               cnt.as<int>(), props.as<int>());
            hipLaunchKernelGGL(k_accept, dim3(N), dim3(256), 0, st, d_d, pitch, P, cap,
                               cnt.as<int>(), props.as<int>(), holders.as<int>(), hold_v.as<float>(),
                               hold_cnt.as<int>(), status.as<int>());
        }
        hipLaunchKernelGGL(k_chains, dim3(1), dim3(1024), 0, st, d_d, pitch, N, P, cap, last_n.as<int>(),
                           last_v.as<float>(), holders.as<int>(), hold_v.as<float>(), hold_cnt.as<int>(),
                           status.as<int>(), left.as<int>());
        int more = 0;
        if (hipMemcpyAsync(&more, left.p, 4, hipMemcpyDeviceToHost, st) != hipSuccess ||
            hipStreamSynchronize(st) != hipSuccess)
            return err(1, "assign_groups: proposal round failed");
        if (more == 0) break;
    }
    hipLaunchKernelGGL(k_class_out, dim3(N), dim3(256), 0, st, cap, holders.as<int>(),
                       hold_cnt.as<int>(), d_out);
    hipLaunchKernelGGL(k_assign_output, dim3(1), dim3(1024), 0, st, d_d, pitch, N, P, cap,
                       status.as<int>(), d_out);
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess)
        return err(1, "assign_groups: launch failed");
    return 0;
}

}  // namespace isac

extern "C" {

int isac_assign_groups_device(const float *d_d, unsigned int n_ref, unsigned int n_img,
                              unsigned int d_pitch, int *d_out, void *stream) {
    return isac::assign_groups(d_d, (int)n_ref, (int)n_img, (int)d_pitch, d_out,
                               (hipStream_t)stream);
}

int isac_assign_groups(const float *h_d, unsigned int n_ref, unsigned int n_img, int *h_out) {
    if (!h_d || !h_out || n_ref < 1 || n_img < n_ref) {
        isac::report_error(2, "isac_assign_groups: need host buffers and 1 <= n_ref <= n_img");
        return 2;
    }
    void *dd = nullptr, *dout = nullptr;
    const size_t nd = (size_t)n_ref * n_img * sizeof(float), no = ((size_t)n_img + 1) * sizeof(int);
    if (hipMalloc(&dd, nd) != hipSuccess || hipMalloc(&dout, no) != hipSuccess ||
        hipMemcpy(dd, h_d, nd, hipMemcpyHostToDevice) != hipSuccess) {
        if (dd) (void)hipFree(dd);
        if (dout) (void)hipFree(dout);
        isac::report_error(1, "isac_assign_groups: device buffers failed");
        return 1;
    }
    int rc = isac::assign_groups(static_cast<const float *>(dd), (int)n_ref, (int)n_img, (int)n_img,
                                 static_cast<int *>(dout), nullptr);
    if (rc == 0 && hipMemcpy(h_out, dout, no, hipMemcpyDeviceToHost) != hipSuccess) {
        isac::report_error(1, "isac_assign_groups: copy back failed");
        rc = 1;
    }
    (void)hipFree(dd);
    (void)hipFree(dout);
    return rc;
}

}  // extern "C"
