// Counting plans of pattern size 3 in closed form.
//
// Reference path replaced: EmbeddingExplorationEngine::extend_embeddings
// (src/engine.cc:914-1118) on schedules such as kautomine/three_motif.cc
// apply(): every edge (v0, v1) is an embedding of size 2 and its step list
// counts elements of N(v0), N(v1), their intersection or a difference that
// pass a position-class predicate.
//
// Level by level that streams, for every edge, one of the two lists against
// the other: sum of d(v)^2 ids (7 G on 4.84 M vertices / 42.9 M edges, 207 of
// 225 ms in plan_level_kernel).  The sum over all edges needs none of it:
//   * an element of N(v0) & N(v1) is the third corner of a triangle, and every
//     triangle is met once per order of its corners, i.e. once for each order
//     code of (v0, v1) and each class of the third (below, between, above):
//     its contribution is T, the number of triangles, per (code, class) pair
//     that the predicate holds -- in a degree-oriented graph only v0 < v1 < x;
//   * elements of N(v0) or N(v1) alone fall into classes by their position in
//     the sorted list, and the sums over a vertex's neighbours are polynomials
//     in s (neighbours below it) and f (above it):
//     A = sum C(s, 2), B = sum C(f, 2), X = sum s f, S = sum s, F = sum f.
//     N(v0), v0 < v1:  below X, between B, equal to v1 F, above B;
//     N(v0), v1 < v0:  below A, equal to v1 S, between A, above X;
//     N(v1) mirrors them, since a symmetric graph has every edge both ways:
//     N(v1), v0 < v1:  below A, equal to v0 S, between A, above X;
//     N(v1), v1 < v0:  below X, between B, equal to v0 F, above B.
// T comes from the persistent clique kernels, the five sums from one pass over
// the vertices (10 ms in all on that graph).  The rule: size 1 has one list
// that scatters or counts N(v0); every order code its scatters reach has a
// list of operations on N(v0) and N(v1) that only counts; the lists are
// strictly increasing without self-loops, and the graph is oriented (then
// N(v1) may not be counted by itself) or has every edge both ways, which is
// checked on the device once per graph.  Anything else runs level by level,
// and so do graphs whose forward degrees the clique kernels do not take.

#include <cstdlib>
#include <cstring>
#include <mutex>

#include "kz_device.h"
#include "kz_kernels.h"
#include "kz_plan.h"

namespace kz {

namespace {

enum { kSumA, kSumB, kSumX, kSumS, kSumF, kBad, kSums };

// The five sums over all vertices; kBad counts vertices whose own id is in
// their list or that have neighbours below them in an oriented graph.
__global__ __launch_bounds__(256) void split_sums_kernel(const uint64_t* __restrict__ rowptr,
                                                         const uint32_t* __restrict__ col, uint32_t n, int oriented,
                                                         unsigned long long* __restrict__ sums) {
    unsigned long long t[kSums] = {0, 0, 0, 0, 0, 0};
    for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) {
        const uint64_t b = rowptr[v];
        const uint32_t d = uint32_t(rowptr[v + 1] - b);
        const uint64_t s = lower_bound_global(col + b, d, v), f = d - s;
        t[kSumA] += s * (s - 1) / 2;  // (0 for s = 0: the product wraps to 0)
        t[kSumB] += f * (f - 1) / 2;
        t[kSumX] += s * f;
        t[kSumS] += s;
        t[kSumF] += f;
        if ((s < d && col[b + s] == v) || (oriented && s)) t[kBad] += 1;
    }
#pragma unroll
    for (int i = 0; i < kSums; ++i) {
        const unsigned long long x = wave_sum_u64(t[i]);
        if ((threadIdx.x & 63) == 0 && x) atomicAdd(&sums[i], x);
    }
}

// Forward entries u -> v (v > u) without the reverse entry v -> u; with as
// many entries below as above their vertex, none means a symmetric graph.
// One wave per vertex.
__global__ __launch_bounds__(256) void reverse_check_kernel(const uint64_t* __restrict__ rowptr,
                                                            const uint32_t* __restrict__ col, uint32_t n,
                                                            unsigned long long* __restrict__ missing) {
    const uint32_t lane = threadIdx.x & 63;
    unsigned long long bad = 0;
    for (uint32_t u = blockIdx.x * 4 + (threadIdx.x >> 6); u < n; u += gridDim.x * 4) {
        const uint64_t b = rowptr[u], e = rowptr[u + 1];
        for (uint64_t p = b + lane; p < e; p += 64) {
            const uint32_t v = col[p];
            if (v <= u) continue;
            if (v >= n) {
                ++bad;
                continue;
            }
            const uint64_t vb = rowptr[v];
            if (!bsearch_global(col + vb, uint32_t(rowptr[v + 1] - vb), u)) ++bad;
        }
    }
    bad = wave_sum_u64(bad);
    if (lane == 0 && bad) atomicAdd(missing, bad);
}

struct DeviceWords {
    unsigned long long* p = nullptr;
    ~DeviceWords() { (void)hipFree(p); }
};

// What one predicate counts, as multiples of T and of the five sums.
struct Weights {
    uint64_t t = 0, s[kSums] = {0, 0, 0, 0, 0, 0};
};

// code 1: v1 < v0, code 2: v0 < v1; set 0: N(v0), 1: N(v1)
void add_runs(Weights& w, uint32_t pred, int code, int set, uint64_t times) {
    const bool low = (code == 1) == (set == 0);  // the list's own vertex is the higher of the two
    const int k[5] = {low ? kSumA : kSumX, low ? kSumS : -1, low ? kSumA : kSumB, low ? -1 : kSumF, low ? kSumX : kSumB};
    for (int c = 0; c < 5; ++c)
        if (((pred >> c) & 1u) && k[c] >= 0) w.s[k[c]] += times;
}
void add_members(Weights& w, uint32_t pred, int code, bool oriented, uint64_t times) {
    for (int c = 0; c < 5; c += 2)
        if (((pred >> c) & 1u) && (!oriented || (code == 2 && c == 4))) w.t += times;
}

}  // namespace

// Runs plan p in closed form: KZ_OK with *taken set, or KZ_OK with *taken
// clear when the level-by-level executor has to run it.
int plan3_execute(DeviceGraph& g, const PlanDesc& p, uint64_t* raw, kz_run_stats* st, bool* taken) {
    *taken = false;
    const char* env = std::getenv("KZ_PLAN_FLAT");  // =0: the general path (for comparisons)
    if (p.pattern_size != 3 || (env && env[0] == '0') || g.n == 0 || plan_validate(p) != KZ_OK) return KZ_OK;
    auto nbr = [](const kz_set_ref& r) { return r.kind == KZ_SET_NBR; };
    Weights w[KZ_MAX_AGGREGATORS];
    // size 1: order code 0
    if (p.type_table[1][0] == 0xFF) return KZ_OK;
    const kz_step_list& R = p.lists[p.type_table[1][0]];
    uint64_t times[3] = {0, 0, 0};  // embeddings per edge of order code 1 and 2
    if (R.num_ops) return KZ_OK;
    for (int o = 0; o < R.num_outs; ++o) {
        const kz_out& out = R.outs[o];
        if (!nbr(out.src)) return KZ_OK;
        if (out.kind == KZ_OUT_SCATTER) {
            times[1] += out.pred & 1u;
            times[2] += (out.pred >> 2) & 1u;
        } else {
            if (out.pred & 1u) w[out.aggregator].s[kSumS] += 1;
            if (out.pred & 4u) w[out.aggregator].s[kSumF] += 1;
        }
    }
    if (g.oriented) times[1] = 0;
    bool members = false;
    for (int code = 1; code <= 2; ++code) {
        if (!times[code]) continue;
        if (p.type_table[2][code] == 0xFF) return KZ_OK;  // an error, if reached: the executor reports it
        const kz_step_list& L = p.lists[p.type_table[2][code]];
        for (int j = 0; j < L.num_ops; ++j)
            if (!nbr(L.ops[j].lhs) || !nbr(L.ops[j].rhs)) return KZ_OK;
        for (int o = 0; o < L.num_outs; ++o) {
            const kz_out& out = L.outs[o];
            if (out.kind != KZ_OUT_COUNT) return KZ_OK;
            Weights& a = w[out.aggregator];
            int whole = -1;  // the list counted by itself, if any
            uint64_t shared = 0;
            if (nbr(out.src)) {
                whole = out.src.a;
            } else if (out.src.a == 2) {
                const kz_op& op = L.ops[out.src.b];
                const bool same = op.lhs.a == op.rhs.a;
                if (op.op == KZ_OP_INTERSECT) {
                    if (same) whole = op.lhs.a;
                    else shared = 1;
                } else if (!same) {
                    whole = op.lhs.a;
                    shared = ~uint64_t(0);  // minus the common ones
                }
            } else {
                return KZ_OK;
            }
            if (whole == 1 && g.oriented) return KZ_OK;
            if (whole >= 0) add_runs(a, out.pred, code, whole, times[code]);
            if (shared) {
                add_members(a, out.pred, code, g.oriented != 0, shared * times[code]);
                members |= a.t != 0;
            }
        }
    }
    // several threads may run plans on one graph: one at a time takes the
    // closed form, which shares the graph's prepared execution (the executor,
    // which shares nothing, runs without the lock)
    std::lock_guard<std::mutex> lk(g.exec_mu);
    if (g.plan3 == 2) return KZ_OK;
    if (members && (g.plan3 == 3 || (g.oriented && g.max_degree > kMaxBitmapDegree))) return KZ_OK;
    hipStream_t s = rt().stream;
    DeviceWords dev;
    if (hipMalloc(&dev.p, 8 * (kSums + 1)) != hipSuccess) {
        (void)hipGetLastError();
        return KZ_OK;
    }
    unsigned long long h[kSums + 1] = {0};
    hipEvent_t e0, e1;
    KZ_HIP(hipEventCreate(&e0));
    KZ_HIP(hipEventCreate(&e1));
    const uint32_t grid = std::min<uint32_t>((g.n + 255) / 256, uint32_t(rt().num_cus) * 8);
    float ms = 0;
    auto sums = [&]() -> int {
        KZ_HIP(hipEventRecord(e0, s));
        KZ_HIP(hipMemcpyAsync(dev.p, h, sizeof(h), hipMemcpyHostToDevice, s));
        hipLaunchKernelGGL(split_sums_kernel, dim3(grid), dim3(256), 0, s, g.rowptr, g.col, g.n, g.oriented, dev.p);
        if (!g.oriented && !g.plan3)
            hipLaunchKernelGGL(reverse_check_kernel, dim3(uint32_t(rt().num_cus) * 8), dim3(256), 0, s, g.rowptr, g.col,
                               g.n, dev.p + kSums);
        KZ_HIP(hipGetLastError());
        KZ_HIP(hipEventRecord(e1, s));
        KZ_HIP(hipMemcpyAsync(h, dev.p, sizeof(h), hipMemcpyDeviceToHost, s));
        KZ_HIP(hipStreamSynchronize(s));
        KZ_HIP(hipEventElapsedTime(&ms, e0, e1));
        return KZ_OK;
    };
    const int e = sums();
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (e) return e;
    if (!g.plan3) g.plan3 = !h[kBad] && !h[kSums] && (g.oriented || h[kSumS] == h[kSumF]) ? 1 : 2;
    if (g.plan3 == 2) return KZ_OK;
    uint64_t T = 0;
    double t_ms = 0;
    if (members) {
        CliqueJob* job = nullptr;
        const bool kept = g.fwd_ready;
        if (ensure_forward(g) != KZ_OK || g.fwd_max > kMaxBitmapDegree || graph_job(g, 3, &job) != KZ_OK) {
            // not tried again on every call; a copy built for nothing is freed
            g.plan3 = 3;
            if (!kept) release_forward(g);
            return KZ_OK;
        }
        if (int err = clique_job_run(*job, &T, &t_ms)) return err;
    }
    for (uint32_t a = 0; a < p.num_aggregators; ++a) {
        uint64_t v = w[a].t * T;
        for (int i = 0; i < kBad; ++i) v += w[a].s[i] * h[i];
        raw[a] = v;
    }
    if (st) {
        st->device_ms = double(ms) + t_ms;
        st->launches = members ? 2 : 1;
        st->chunks = 1;
        st->embeddings[1] = g.n;
        st->embeddings[2] = times[1] * h[kSumS] + times[2] * h[kSumF];
        st->peak_bytes = 8 * (kSums + 1);
    }
    *taken = true;
    return KZ_OK;
}

}  // namespace kz
