// Transfer kernels: the polarized transport of every (pixel, time, frequency) item as per-slice
// 4x4 transfer maps from marched samples, their composition along each ray, and thin (Stokes I) images.
// Reference: transport.jl:99-316, polarized.jl:41-198, Splats.jl:58-147, populations.jl:13-104,
// trajectories.jl:80-128, step.jl:342-398.
#include "ks_kernels.hpp"
#include "ks_dsample.hpp"
#include <rocprim/device/device_radix_sort.hpp>

namespace ksd {

// ---- polarized transport from stored samples (transport.jl:263-290) ----------------------------------------
// Work items (slice m, item), item = j + npix (it + nt inu) fastest: samples m chunk + 1 .. of the
// item's ray, composed into the slice's map seg[(20 m + f) nitems + item]. With rec != nullptr the
// adjoint records (RecField) of every step-taking sample are written, and aflg[(k - 1) nitems + item]
// = 1 when the sample takes a step. A task is one workgroup's 128 consecutive slots (slot = item slot +
// nitems m); the item slots run over the cache's wavefront patches (slot_item).
struct TransferArgs {
    double a, thetao;
    const double* soa;
    int64_t npix;
    int N, chunk, nch;
    Samples smp;
    int ns, nknots;
    const double* times; int nt;
    const double* nus; int nnu;
    double L;
    const int* kstop;
    uint8_t* aflg;
};
KS_DEV int64_t npix_items(const TransferArgs& A) { return A.npix * A.nt * A.nnu; }
// A wavefront's workspace in LDS, field-major over its 64 lanes: the geometry of its rays' current sample, the sums of
// the sample's contributions and whether it has any, the rays' screen coordinates and frequency, the pair queue (lane |
// splat << 6), the slice's candidate splats. 8.9 KB in FP32 and 16.4 KB in FP64: in FP32 as many wavefronts as the
// registers allow fit a compute unit (160 KB), in FP64 nine (a workgroup's two: eight).
constexpr int QCAP = 256;              // the queue holds < 64 pending pairs and up to 64 pushes of each of two splats
template <class S>
struct WaveWork {
    S geo[GEO_FIELDS * 64], sum[11 * 64], alpha[64], beta[64], nu[64];
    uint64_t mask[CAND_MAX / 64];
    int q[QCAP], act[64];
};
static_assert(sizeof(WaveWork<f32>) == 9088 && sizeof(WaveWork<double>) == 16768, "the figures above");
// Values written by some lanes of the wavefront are read by others: the LDS operations of a wavefront run in order, and
// the compiler keeps theirs across this.
KS_DEV void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
KS_DEV uint64_t uniform64(uint64_t x) {
    return ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(x >> 32)) << 32) | (uint32_t)__builtin_amdgcn_readfirstlane((int)x);
}
// The prefilter's fields of two splats at wave-uniform addresses, held in scalar registers: four scalar loads in flight at
// once. Left to the compiler, each field is loaded where it is used, and a splat's test waits for its loads one after
// another (as vector loads, before the pointer said that nothing writes them: 56 % of the FP64 transfer's wavefront cycles
// were such waits). MI355X, transfer of one pass: FP64, 32 thermal splats at 128^2 x 1024 4.9 -> 3.7 ms, 48 power-law splats
// 2.04 -> 1.65, 1024 kappa splats on knots (112 x 96 x 512) 61 -> 50; FP32, the same at 256^2 x 1024 165 -> 121, 64 thermal
// splats (4 frames of 128^2 x 1024) 12.4 -> 10.4, 128 mixed splats (36,864 points x 512 x 12) 69 -> 57.
typedef int sgpr16 __attribute__((ext_vector_type(16), aligned(4)));
typedef int sgpr8 __attribute__((ext_vector_type(8), aligned(4)));
struct SplatTests {
    sgpr16 p, r;
    sgpr8 q, s;
    __device__ __forceinline__ SplatTests(const SplatCf* __restrict__ u, const SplatCf* __restrict__ v) {
        p = *(const sgpr16*)u; q = *(const sgpr8*)((const int*)u + 16);
        r = *(const sgpr16*)v; s = *(const sgpr8*)((const int*)v + 16);
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile("" : "+s"(p), "+s"(q), "+s"(r), "+s"(s));
#endif
    }
    __device__ __forceinline__ static SplatTest of(sgpr16 p, sgpr8 q) {
        SplatTest t;
        int w[24];
        for (int i = 0; i < 16; ++i) w[i] = p[i];
        for (int i = 0; i < 8; ++i) w[16 + i] = q[i];
        __builtin_memcpy(&t, w, sizeof t);
        return t;
    }
    __device__ __forceinline__ SplatTest a() const { return of(p, q); }
    __device__ __forceinline__ SplatTest b() const { return of(r, s); }
};
// The slice of the q-th of n rows of tasks: the middle of the rays first, then outwards. A ray is nearest the hole around
// its middle, where the splats crowd: in this order the tasks' costs fall (by five from the first sixteenth to the last),
// and the queue's last ones are cheap.
KS_DEV int slice_order(int q, int n) { return (q & 1) ? (n - 1) / 2 + (q + 1) / 2 : (n - 1) / 2 - q / 2; }
// One wavefront: 64 items x one slice. Sample by sample, the lanes test their ray's sample against the candidate splats
// (may_weigh) and queue the pairs that pass; whenever 64 are queued, or the candidates are through, the queued pairs'
// weights, frames and coefficients run one pair a lane (splat_contribution), and each adds its 11 values to its
// sample's sums in LDS, the pairs of one splat at a time: a sample's contributions are added in ascending splat order,
// whatever wavefront it sits in. Then every lane takes its sample's step. Before, each lane visited its own sample's
// splats, with 43 to 71% of the lanes in a splat's support, over slices four times as long, and 5 to 40% of the vector
// issue slots used. MI355X, whole call, before and after: FP64 image of 6 thermal splats (50 x 37 x 301) 1.17 -> 0.37 ms,
// FP64 march and image of 32 thermal splats (128^2 x 1024) 13.9 -> 9.2 ms, FP64 gradient of 48 power-law splats
// (102 x 67 x 333, 2 frames) 28.4 -> 14.0 ms, FP64 fit iteration of 1024 kappa splats (112 x 96 x 512) 780 -> 351 ms, mixed
// (256^2 x 1024) 1084 -> 953 ms, mixed movie of 128 splats (36,864 points x 512 x 12 frames) 113 -> 76 ms.
// The queue, not the lanes, decides what runs: all lanes take part in every collective, and each loop exit is uniform.
template <int KIND, class S, bool CULL>
__device__ __forceinline__ void transfer_task(const TransferArgs& A, const SplatCT<S>* __restrict__ sp, const S* __restrict__ knots,
                                    const S* __restrict__ ktimes, S* __restrict__ seg, S* __restrict__ rec, const SplatCf* __restrict__ spf, const f32* __restrict__ knots_f,
                                    int64_t task, WaveWork<S>& W) {
    const int64_t npix = A.npix;
    const int N = A.N;
    const int64_t nitems = npix * A.nt * A.nnu;
    const int64_t tid = task * 128 + threadIdx.x;
    const bool live = tid < nitems * A.nch;     // the tail's lanes take slot 0 and write nothing
    const int64_t slot = live ? tid : 0;
    const Samples& smp = A.smp;
    const int64_t item = slot_item(smp, slot % nitems, npix);     // wavefronts over compact patches of sky
    const int m = slice_order((int)(slot / nitems), A.nch);
    const int64_t j = item % npix;
    const int64_t fr = item / npix;
    const int it = (int)(fr % A.nt), inu = (int)(fr / A.nt);
    const double a = A.a;
    const Spin Sp = make_spin(a);
    const double dtau = A.soa[(int64_t)PF_TAUTOT * npix + j] / (double)(N + 1);
    const S aS = S(a), tos = S(sin(A.thetao));
    const double t_obs = A.times[it], nu = A.nus[inu];
    const int ks = A.kstop ? A.kstop[j] : N + 1;
    const double hor = Sp.rp * (1.0 + 1e-3);
    const int kbeg = m * A.chunk + 1, kend = kbeg + A.chunk - 1 < N ? kbeg + A.chunk - 1 : N;
    const int64_t st = (int64_t)N * nitems;
    const int lane = (int)(threadIdx.x % 64);
    W.alpha[lane] = S(A.soa[(int64_t)PF_ALPHA * npix + j]);
    W.beta[lane] = S(A.soa[(int64_t)PF_BETA * npix + j]);
    W.nu[lane] = S(nu);
    // the per-tile cull: the splats that can reach the wavefront's samples of this slice, a bit each (the rest add exact
    // zeros to every sample of the tile); every splat without it
    const int nblk = (A.ns + 63) / 64;
    if constexpr (CULL) {     // the launcher picks CULL for CULL_MIN_NS <= ns <= CAND_MAX
        double lo[4] = {INFINITY, INFINITY, INFINITY, INFINITY}, hi[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
        if (live)
            for (int k = kbeg; k <= kend; ++k) {
                const int64_t o = (int64_t)(k - 1) * npix + j;
                if ((smp.fl[o] & 1) && smp.r[o] > hor && k < ks) {
                    const double v[4] = {smp.x[o], smp.y[o], smp.z[o], t_obs - smp.t[o]};
                    for (int q = 0; q < 4; ++q) { lo[q] = fmin(lo[q], v[q]); hi[q] = fmax(hi[q], v[q]); }
                }
            }
        double px = 0.0, py = 0.0, pz = 0.0, R = 0.0, tmin = 0.0, tmax = 0.0;
        const bool any = wave_region(lo, hi, px, py, pz, R, tmin, tmax);
        for (int b = 0; b < nblk; ++b) {
            const int i = b * 64 + lane;
            const uint64_t mk = __ballot(any && i < A.ns && splat_may_reach(sp[i], px, py, pz, R, tmin, tmax, knots, ktimes));
            if (lane == 0) W.mask[b] = mk;
        }
    }
    wave_sync();
    SegMapT<S> sm;
    sm.init();
    for (int s = 0; s < A.chunk; ++s) {
        const int k = kbeg + s;
        const bool in = live && k <= kend;
        const int64_t o = (int64_t)((in ? k : 1) - 1) * npix + j;
        const uint8_t fl = smp.fl[o];
        const double r = smp.r[o];
        const bool valid = in && (fl & 1) && r > hor && k < ks;
        bool step = false, ready = false;
        if (__ballot(valid)) {
            const S t = S(t_obs - smp.t[o]), x = S(smp.x[o]), y = S(smp.y[o]), z = S(smp.z[o]);
            const float tf = (float)val(t), xf = (float)val(x), yf = (float)val(y), zf = (float)val(z);
            S D(0.0);
            int qh = 0, qn = 0, b = -1;
            uint64_t mk = 0;
            bool more = true;
            // the sample among the knot times (of part kt_c of the model's), and its interval where the lanes share one
            int kt_c = -1, nk_c = 0, kk_u = -1;
            KnotAt<S> at{0, S(0.0)};
            auto may = [&](const SplatTest& c) {
                float e3[3];
                if (KIND == MODEL_KNOT || c.nk > 0) {
                    if (c.kt0 != kt_c || c.nk != nk_c) {
                        kt_c = c.kt0; nk_c = c.nk;
                        at = knot_at(ktimes + kt_c, nk_c, t);
                        const uint64_t vm = __ballot(valid);
                        const int k0 = __builtin_amdgcn_readlane(at.kk, __builtin_ctzll(vm));
                        kk_u = (__ballot(at.kk != k0) & vm) == 0 ? k0 : -1;
                    }
                    const float w = (float)val(at.w);
                    if (kk_u >= 0) knot_offset(knots_f + 3 * ((int64_t)c.knot0 + kk_u), c.nk < 2, w, xf, yf, zf, e3);
                    else knot_offset(knots_f + 3 * ((int64_t)c.knot0 + at.kk), c.nk < 2, w, xf, yf, zf, e3);
                } else {
                    pattern_offset(c, tf, xf, yf, zf, e3);
                }
                return valid && offset_may_weigh(c, tf, e3);
            };
            auto push = [&](bool hit, int i) {
                const uint64_t hm = __ballot(hit);
                if (hit) W.q[(qh + qn + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(hm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)hm, 0u))) & (QCAP - 1)] = lane | (i << 6);
                qn += __popcll(hm);
            };
            for (;;) {
                while (qn < 64) {
                    while (mk == 0 && more) {
                        if (++b >= nblk) more = false;
                        else if constexpr (CULL) mk = uniform64(W.mask[b]);
                        else mk = A.ns - 64 * b >= 64 ? ~0ull : (1ull << (A.ns - 64 * b)) - 1;
                    }
                    if (!more) break;
                    // two splats at a time (the last one of an odd count twice, its second test not counted)
                    const int i = b * 64 + __builtin_ctzll(mk);
                    mk &= mk - 1;
                    const bool two = mk != 0;
                    const int i2 = two ? b * 64 + __builtin_ctzll(mk) : i;
                    mk &= mk - 1;
                    const SplatTests tests(spf + i, spf + i2);
                    const bool h1 = may(tests.a()), h2 = may(tests.b());
                    push(h1, i);
                    push(two && h2, i2);
                }
                if (qn == 0) break;
                if (!ready) {            // the sample's geometry, in FP64, for its first queued pairs
                    ready = true;
                    for (int q = 0; q < 11; ++q) W.sum[64 * q + lane] = S(0.0);
                    W.act[lane] = 0;
                    if (valid) {
                        Geo Gd;
                        make_geo(a, r, smp.th[o], A.soa[(int64_t)PF_ETA * npix + j], A.soa[(int64_t)PF_LAM * npix + j], (fl & 2) != 0, (fl & 4) != 0, Gd);
                        geo_store(geo_as<S>(Gd), W.geo + lane, 64);
                        D = S(A.L / (nu * (1.0 / NU0)) * Gd.S * dtau);       // path_weight
                    }
                }
                wave_sync();
                const int cnt = qn < 64 ? qn : 64;
                const bool on = lane < cnt;
                const int e = W.q[(qh + lane) & (QCAP - 1)];
                const int l = on ? e & 63 : lane, i = on ? e >> 6 : 0;
                const KnotAt<S> al{__shfl(at.kk, l, 64), lane_value(at.w, l)};
                const S tt = lane_value(t, l), xx = lane_value(x, l), yy = lane_value(y, l), zz = lane_value(z, l);
                bool act = false;
                S c[11];
                for (int q = 0; q < 11; ++q) c[q] = S(0.0);
                if (on) {
                    const SplatCT<S>& sc = sp[i];
                    const bool have = (KIND == MODEL_KNOT || sc.nk > 0) && sc.kt0 == kt_c && sc.nk == nk_c;
                    const S G_ = splat_weight<KIND>(sc, knots, ktimes, tt, xx, yy, zz, have ? &al : nullptr);
                    if (G_ > 0.0) {
                        GeoT<S> G;
                        geo_load(W.geo + l, 64, G);
                        act = splat_contribution<KIND>(sc, G, aS, W.alpha[l], W.beta[l], tos, W.nu[l], G_, c);
                    }
                }
                uint64_t todo = __ballot(act);
                while (todo) {
                    const int si = __builtin_amdgcn_readlane(i, __builtin_ctzll(todo));
                    const bool mine = act && i == si;
                    if (mine) {
                        for (int q = 0; q < 11; ++q) W.sum[64 * q + l] += c[q];
                        W.act[l] = 1;
                    }
                    wave_sync();
                    todo &= ~__ballot(mine);
                }
                qh += cnt;
                qn -= cnt;
                if (!more && qn == 0) break;
            }
            wave_sync();
            step = ready && W.act[lane] != 0;
            if (step) {
                S j4[4], a4[4], r3[3];
                for (int q = 0; q < 4; ++q) { j4[q] = W.sum[64 * q + lane]; a4[q] = W.sum[64 * (4 + q) + lane]; }
                for (int q = 0; q < 3; ++q) r3[q] = W.sum[64 * (8 + q) + lane];
                map_step(sm, j4, a4, r3, D);
                if (rec) {
                    S* w = rec + (int64_t)(k - 1) * nitems + item;
                    for (int q = 0; q < 4; ++q) { w[(REC_J + q) * st] = j4[q]; w[(REC_A + q) * st] = a4[q]; }
                    for (int q = 0; q < 3; ++q) w[(REC_RHO + q) * st] = r3[q];
                    w[REC_D * st] = D;
                    for (int f = 0; f < GEO_FIELDS; ++f) w[(REC_GEO + f) * st] = W.geo[64 * f + lane];
                }
            }
            wave_sync();
        }
        if (rec && in) A.aflg[(int64_t)(k - 1) * nitems + item] = step ? 1 : 0;
    }
    if (live) sm.store(seg, m, nitems, item);
}

// The launch: a persistent grid of the resident workgroups, each taking the next ticket q from the queue head until
// ntasks are taken; task q is tasks[q] when a task list is given (a cost-descending order from an earlier launch's
// per-task times, or the autotuner's sample of the work), else q (ntasks < 2^31). With cost != nullptr the wall-clock
// ticks each task took go to cost[task] (zeroed by the launcher). The tasks are heavy-tailed (1024 kappa splats, 256^2 x
// 1024: median 0.6 ms, 99th percentile 31 ms), and dispatched one workgroup a task the hardware kept 1.7 of 4 wavefronts
// a SIMD in flight: 340 ms, against 190 from the queue in index order and 166 in cost order (64 thermal splats,
// 128^2 x 1024 x 4 frames: 21.2, 13.3, 12.7; FP64, 32 splats, 128^2 x 1024: 7.7, 5.8, 5.2). The loop holds
// no lane-dependent branch outside the task: all 64 lanes of wavefront 0 execute the pop (lane 0 adds one, the others
// zero), the first lane's ticket is shared through LDS, and every exit and back edge of the loop is a
// wavefront-uniform (scalar) branch, so all lanes of the workgroup iterate together and each pass through the
// barriers is a pass through the pop.
template <int KIND, class S, bool CULL>
__global__ void __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu((transfer_waves<KIND, S>))))
ks_chunk_transfer(TransferArgs A, const SplatCT<S>* __restrict__ sp, const S* __restrict__ knots, const S* __restrict__ ktimes,
                  S* __restrict__ seg, S* __restrict__ rec, const SplatCf* __restrict__ spf, const f32* __restrict__ knots_f,
                  const int* __restrict__ tasks, int64_t ntasks, unsigned* __restrict__ head, uint32_t* __restrict__ cost) {
    __shared__ WaveWork<S> s_w[2];
    __shared__ unsigned s_q;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / 64));
    for (;;) {
        if (wave == 0) {
            const unsigned ticket = atomicAdd(head, threadIdx.x == 0 ? 1u : 0u);
            s_q = __builtin_amdgcn_readfirstlane(ticket);
        }
        __syncthreads();
        const int64_t q = (int64_t)__builtin_amdgcn_readfirstlane(s_q);
        __syncthreads();             // every wavefront has read s_q before the next pop overwrites it
        if (q >= ntasks) break;
        const int64_t task = tasks ? (int64_t)tasks[q] : q;
        const uint64_t t0 = cost ? wall_clock64() : 0;
        transfer_task<KIND, S, CULL>(A, sp, knots, ktimes, seg, rec, spf, knots_f, task, s_w[wave]);
        if (cost) {
            __syncthreads();
            atomicMax(cost + task, (uint32_t)min<uint64_t>(wall_clock64() - t0, 0xffffffffull));
        }
    }
}

// ---- thin splats: sums over chunks of the samples --------------------------------------------------------------------
// part[m npix + j] = the thin sum (Splats.jl:113-128: sum_i j_i g^2 Sigma dtau with the ZAMO redshift g) of samples
// m THIN_CHUNK + 1 .. of pixel j. A thread holds its samples in registers and takes the splats in turn, their constants
// once for all of them; bound by the FP64 sine, cosine and exponential of every (sample, splat). Folded into the march
// (one thread a 64-sample segment, one wavefront a SIMD for its registers) the sums ran at a fifth of the issue rate:
// 300 splats, 96 x 72 x 400, fused march 12.5 -> 3.8 ms; 40 splats over stored samples 1.38 -> 0.51 ms.
constexpr int THIN_CHUNK = 4;
__global__ void __launch_bounds__(128) ks_thin_parts(double a, const double* __restrict__ soa, int64_t npix, int N, Samples smp,
                                                     const SplatC* __restrict__ sp, int ns, double t_obs, double* __restrict__ part) {
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int nch = (N + THIN_CHUNK - 1) / THIN_CHUNK;
    if (tid >= npix * nch) return;
    const int64_t j = tid % npix;
    const int m = (int)(tid / npix);
    const double lam = soa[(int64_t)PF_LAM * npix + j];
    const double dtau = soa[(int64_t)PF_TAUTOT * npix + j] / (double)(N + 1);
    const double guard = make_spin(a).rp * (1.0 + 1e-3);
    double t[THIN_CHUNK], x[THIN_CHUNK], y[THIN_CHUNK], z[THIN_CHUNK], w[THIN_CHUNK], jt[THIN_CHUNK];
    bool any = false;
    for (int u = 0; u < THIN_CHUNK; ++u) {
        const int k = m * THIN_CHUNK + 1 + u;
        const int64_t o = (int64_t)((k <= N ? k : N) - 1) * npix + j;
        const double r = smp.r[o];
        const bool ok = k <= N && (smp.fl[o] & 1) && guard < r && r < 1e3;
        t[u] = t_obs - smp.t[o]; x[u] = smp.x[o]; y[u] = smp.y[o]; z[u] = smp.z[o];
        jt[u] = w[u] = 0.0;
        if (ok) { w[u] = thin_weight(a, lam, r, smp.th[o], dtau); any = true; }
        else { t[u] = x[u] = y[u] = z[u] = 0.0; }
    }
    double acc = 0.0;
    if (any) {
        for (int i = 0; i < ns; ++i) {
            const SplatC& c = sp[i];
#pragma unroll
            for (int u = 0; u < THIN_CHUNK; ++u) {
                double sph, cph;
                phase_sincos(c.omega * (t[u] - c.t0), &sph, &cph);
                jt[u] += exp(c.lnA - 0.5 * gauss_exponent(c, t[u], x[u], y[u], z[u], sph, cph));
            }
        }
        for (int u = 0; u < THIN_CHUNK; ++u) acc += w[u] > 0.0 ? w[u] * jt[u] : 0.0;
    }
    part[(int64_t)m * npix + j] = acc;
}
// The same sums fused with the march, a thread an anchor segment, for the few splats (THIN_MARCH_TILE) whose sums the march's idle
// issue slots take: part[m npix + j] = the sum over segment m of pixel j (0 past its last segment), res its anchor residuals.
struct ThinF {
    const SplatC* sp; int ns; double a, rp, rm, t_obs, lam, acc;
    KS_DEV void operator()(int, const Samp& s, double dtau) {
        if (!(s.ok && rp * (1.0 + 1e-3) < s.r && s.r < 1e3)) return;
        double x, y, z, jt = 0.0;
        quasi_cartesian_ks(a, rp, rm, s.r, s.th, s.ph, x, y, z);
        for (int i = 0; i < ns; ++i) {
            const SplatC& c = sp[i];
            double sph, cph;
            phase_sincos(c.omega * (t_obs - s.t - c.t0), &sph, &cph);
            jt += exp(c.lnA - 0.5 * gauss_exponent(c, t_obs - s.t, x, y, z, sph, cph));
        }
        acc += thin_weight(a, lam, s.r, s.th, dtau) * jt;
    }
};
__global__ void __launch_bounds__(128) ks_thin_march(double a, double thetao, const double* __restrict__ soa, int64_t npix, int N, int M,
                                                     const SplatC* __restrict__ sp, int ns, double t_obs, int nseg_max, double* __restrict__ part,
                                                     double* __restrict__ res) {
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= npix * nseg_max) return;
    const int64_t j = tid % npix;
    const int m = (int)(tid / npix);
    const Spin S = make_spin(a);
    const PixC p = load_pixel(soa, npix, j);
    double acc = 0.0, r1 = 0.0, r2 = 0.0;
    const int Lseg = segment_length(M, 1.0 - p.k);
    const int kbeg = m * Lseg + 1;
    if (kbeg <= N && kbeg * (p.tau_total / (double)(N + 1)) <= p.tau_h) {
        const int kend = kbeg + Lseg - 1 < N ? kbeg + Lseg - 1 : N;
        ThinF f{sp, ns, a, S.rp, S.rm, t_obs, p.lam, 0.0};
        march_range(p, S, thetao, N, M, kbeg, kend, f, r1, r2);
        acc = f.acc;
    }
    res[2 * (m * npix + j)] = r1; res[2 * (m * npix + j) + 1] = r2;
    part[m * npix + j] = acc;
}
__global__ void ks_thin_combine(int64_t npix, int nseg_max, const double* __restrict__ part, double* __restrict__ out) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= npix) return;
    // one thread a pixel: COMBINE_GROUP loads in flight, added in order (one at a time, 8192 pixels of 256 chunks took 76 us)
    constexpr int COMBINE_GROUP = 16;
    double s = 0.0;
    int m = 0;
    for (; m + COMBINE_GROUP <= nseg_max; m += COMBINE_GROUP) {
        double v[COMBINE_GROUP];
#pragma unroll
        for (int u = 0; u < COMBINE_GROUP; ++u) v[u] = part[(int64_t)(m + u) * npix + j];
#pragma unroll
        for (int u = 0; u < COMBINE_GROUP; ++u) s += v[u];
    }
    for (; m < nseg_max; ++m) s += part[(int64_t)m * npix + j];
    out[j] = s;
}

// ---- composition of the segment maps ---------------------------------------------------------------------------
// S = sum_m P_0 ... P_{m-1} S_m, the observed Stokes vector nu-hat^3 S (observed_stokes, transport.jl:311-316). A
// workgroup takes 64 items, each of its COMBINE_WAVES wavefronts a run of their segments; the runs' maps are composed
// in order through LDS (one wavefront over all segments left most of the chip idle: 65 us for 128^2 items of 32
// segments, 256 wavefronts).
template <class G>
__global__ void __launch_bounds__(64 * COMBINE_WAVES)
ks_seg_combine(int64_t npix, int N, int chunk, int nt, const double* __restrict__ nus, int nnu, const G* __restrict__ seg, double* __restrict__ out) {
    __shared__ double s_map[COMBINE_WAVES][SEG_FIELDS][64];
    const int64_t nitems = npix * nt * nnu;
    const int lane = (int)(threadIdx.x % 64), wv = (int)(threadIdx.x / 64);
    const int64_t item = (int64_t)blockIdx.x * 64 + lane;
    double P[16], Sv[4] = {0, 0, 0, 0};
    for (int i = 0; i < 16; ++i) P[i] = (i % 5 == 0) ? 1.0 : 0.0;
    if (item < nitems) {
        const int nseg = (N + chunk - 1) / chunk;
        const int per = (nseg + COMBINE_WAVES - 1) / COMBINE_WAVES;
        const int m1 = (wv + 1) * per < nseg ? (wv + 1) * per : nseg;
        for (int m = wv * per; m < m1; ++m) {
            double Pm[16], Sm[4];
            seg_load(seg, m, nitems, item, Pm, Sm);
            seg_append(P, Sv, Pm, Sm);
        }
    }
    for (int q = 0; q < 16; ++q) s_map[wv][q][lane] = P[q];
    for (int q = 0; q < 4; ++q) s_map[wv][16 + q][lane] = Sv[q];
    __syncthreads();
    if (wv != 0 || item >= nitems) return;
    for (int w = 1; w < COMBINE_WAVES; ++w) {
        double Pm[16], Sm[4];
        for (int q = 0; q < 16; ++q) Pm[q] = s_map[w][q][lane];
        for (int q = 0; q < 4; ++q) Sm[q] = s_map[w][16 + q][lane];
        seg_append(P, Sv, Pm, Sm);
    }
    const double nh = nus[(item / npix) / nt] * (1.0 / NU0);
    const double s3 = nh * nh * nh;
    for (int q = 0; q < 4; ++q) out[4 * item + q] = Sv[q] * s3;
}

// ---- launchers ----
__global__ void ks_fill_i32(int* __restrict__ p, int64_t n, int v) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}
hipError_t launch_fill_i32(hipStream_t s, int* p, int64_t n, int v) {
    hipLaunchKernelGGL(ks_fill_i32, dim3(grid_for(n, 256)), dim3(256), 0, s, p, n, v);
    return hipGetLastError();
}
template <int KIND, class S, bool CULL>
static hipError_t chunk_transfer_c(hipStream_t s, const TransferArgs& A, const SplatCT<S>* sp, const S* knots, const S* ktimes, S* seg, S* rec,
                                   const SplatCf* spf, const f32* knots_f, const TransferLaunch& tl) {
    const int64_t all = (npix_items(A) * A.nch + 127) / 128;
    const int64_t ntasks = tl.tasks ? tl.ntasks : all;
    if (ntasks <= 0) return hipSuccess;
    if (ntasks >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
    if (!tl.head) return hipErrorInvalidValue;
    static int groups = 0;       // per instantiation
    if (!groups) groups = resident_groups(ks_chunk_transfer<KIND, S, CULL>, 128);
    if (!groups) return hipErrorInvalidValue;
    // the head and the per-task costs start at zero (fill kernels: no memset nodes in a captured graph)
    hipLaunchKernelGGL(ks_fill_i32, dim3(1), dim3(64), 0, s, tl.head, (int64_t)1, 0);
    if (tl.cost) hipLaunchKernelGGL(ks_fill_i32, dim3(grid_for(ntasks, 256)), dim3(256), 0, s, (int*)tl.cost, ntasks, 0);
    const int64_t grid = std::min<int64_t>(ntasks, (int64_t)groups);
    hipLaunchKernelGGL((ks_chunk_transfer<KIND, S, CULL>), dim3((unsigned)grid), dim3(128), 0, s, A, sp, knots, ktimes, seg, rec, spf, knots_f, tl.tasks,
                       ntasks, (unsigned*)tl.head, tl.cost);
    return hipGetLastError();
}
template <int KIND, class S>
static hipError_t chunk_transfer_k(hipStream_t s, const TransferArgs& A, const SplatCT<S>* sp, const S* knots, const S* ktimes, S* seg, S* rec,
                                   const SplatCf* spf, const f32* knots_f, const TransferLaunch& tl) {
    // the per-tile cull bounds pattern-rotating splats by their arc and knot splats by the sphere holding their knots
    if (A.ns >= CULL_MIN_NS && A.ns <= CAND_MAX) return chunk_transfer_c<KIND, S, true>(s, A, sp, knots, ktimes, seg, rec, spf, knots_f, tl);
    return chunk_transfer_c<KIND, S, false>(s, A, sp, knots, ktimes, seg, rec, spf, knots_f, tl);
}
template <class S>
static hipError_t chunk_transfer_s(hipStream_t s, int kind, const TransferArgs& A, const SplatCT<S>* sp, const S* knots, const S* ktimes, S* seg,
                                   S* rec, const SplatCf* spf, const f32* knots_f, const TransferLaunch& tl) {
    if (tl.chunk < 1) return hipErrorInvalidValue;
    switch (kind) {
        case MODEL_THERMAL: return chunk_transfer_k<MODEL_THERMAL, S>(s, A, sp, knots, ktimes, seg, rec, spf, knots_f, tl);
        case MODEL_POWERLAW: return chunk_transfer_k<MODEL_POWERLAW, S>(s, A, sp, knots, ktimes, seg, rec, spf, knots_f, tl);
        case MODEL_KAPPA: return chunk_transfer_k<MODEL_KAPPA, S>(s, A, sp, knots, ktimes, seg, rec, spf, knots_f, tl);
        case MODEL_COMPOSITE: return chunk_transfer_k<MODEL_COMPOSITE, S>(s, A, sp, knots, ktimes, seg, rec, spf, knots_f, tl);
        default: return chunk_transfer_k<MODEL_KNOT, S>(s, A, sp, knots, ktimes, seg, rec, spf, knots_f, tl);
    }
}
hipError_t launch_chunk_transfer(hipStream_t s, int kind, double a, double thetao, const double* soa, int64_t npix, int N, Samples smp,
                                 const SplatC* sp, int ns, const double* knots, const double* ktimes, int nknots, const SplatCf* spf,
                                 const f32* knots_f, const double* times, int nt, const double* nus, int nnu, double L,
                                 const int* kstop, double* seg, double* rec, uint8_t* aflg, const TransferLaunch& tl) {
    const TransferArgs A{a, thetao, soa, npix, N, tl.chunk, (N + tl.chunk - 1) / tl.chunk, smp, ns, nknots, times, nt, nus, nnu, L, kstop, aflg};
    return chunk_transfer_s<double>(s, kind, A, sp, knots, ktimes, seg, rec, spf, knots_f, tl);
}
hipError_t launch_chunk_transfer_f32(hipStream_t s, int kind, double a, double thetao, const double* soa, int64_t npix, int N, Samples smp,
                                     const SplatCf* sp, int ns, const f32* knots, const f32* ktimes, int nknots,
                                     const double* times, int nt, const double* nus, int nnu, double L, const int* kstop,
                                     f32* seg, f32* rec, uint8_t* aflg, const TransferLaunch& tl) {
    const TransferArgs A{a, thetao, soa, npix, N, tl.chunk, (N + tl.chunk - 1) / tl.chunk, smp, ns, nknots, times, nt, nus, nnu, L, kstop, aflg};
    return chunk_transfer_s<f32>(s, kind, A, sp, knots, ktimes, seg, rec, sp, knots, tl);
}
__global__ void ks_iota_i32(int* __restrict__ p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = (int)i;
}
// The tasks in descending order of their recorded costs (ticks): order[0 ..n) from cost[0 ..n); keys and ids are
// n-long work arrays. Called with tmp = nullptr it sets tmp_bytes to the workspace the sort needs.
hipError_t launch_order_tasks(hipStream_t s, const uint32_t* cost, int64_t n, uint32_t* keys, int* ids, int* order, void* tmp, size_t& tmp_bytes) {
    if (tmp) hipLaunchKernelGGL(ks_iota_i32, dim3(grid_for(n, 256)), dim3(256), 0, s, ids, n);
    return rocprim::radix_sort_pairs_desc(tmp, tmp_bytes, cost, keys, ids, order, (unsigned)n, 0, 32, s);
}
int64_t transfer_tasks(int64_t npix, int nt, int nnu, int N, int chunk) {
    return (npix * nt * nnu * ((N + chunk - 1) / chunk) + 127) / 128;
}
int thin_chunks(int N) { return (N + THIN_CHUNK - 1) / THIN_CHUNK; }
hipError_t launch_thin_parts(hipStream_t s, double a, const double* soa, int64_t npix, int N, Samples smp, const SplatC* sp, int ns, double t_obs,
                             double* part) {
    hipLaunchKernelGGL(ks_thin_parts, dim3(grid_for(npix * thin_chunks(N), 128)), dim3(128), 0, s, a, soa, npix, N, smp, sp, ns, t_obs, part);
    return hipGetLastError();
}
hipError_t launch_thin_march(hipStream_t s, double a, double thetao, const double* soa, int64_t npix, int N, int M, const SplatC* sp, int ns,
                             double t_obs, int nseg_max, double* part, double* res) {
    hipLaunchKernelGGL(ks_thin_march, dim3(grid_for(npix * nseg_max, 128)), dim3(128), 0, s, a, thetao, soa, npix, N, M, sp, ns, t_obs, nseg_max, part,
                       res);
    return hipGetLastError();
}
hipError_t launch_thin_combine(hipStream_t s, int64_t npix, int nseg_max, const double* part, double* out) {
    hipLaunchKernelGGL(ks_thin_combine, dim3(grid_for(npix, 256)), dim3(256), 0, s, npix, nseg_max, part, out);
    return hipGetLastError();
}
hipError_t launch_seg_combine(hipStream_t s, int64_t npix, int N, int chunk, int nt, const double* nus, int nnu, const void* seg, int seg32,
                              double* out) {
    const dim3 grid(grid_for(npix * nt * nnu, 64)), block(64 * COMBINE_WAVES);
    if (seg32) hipLaunchKernelGGL(ks_seg_combine<f32>, grid, block, 0, s, npix, N, chunk, nt, nus, nnu, (const f32*)seg, out);
    else hipLaunchKernelGGL(ks_seg_combine<double>, grid, block, 0, s, npix, N, chunk, nt, nus, nnu, (const double*)seg, out);
    return hipGetLastError();
}

// ---- per-ray splat lists (ray_lists, dual_gradient.jl:283-359) ----------------------------------------------
// One thread per (ray j in sorted order, frame f): hits[i + ns (j + npix f)] = 1 when a sample of ray j before its
// half-orbit cutoff kstop[j] (none when kstop is null) that takes a step (ok, outside the horizon guard) lies inside
// splat i's support sphere at the frame's time (outside_support), else 0; cnt[j + npix f] = the number of hits.
// Splats outer: a splat's test stops at the ray's first samples inside its sphere, and each byte is written once. Bound by the
// latency of the samples' loads, HIT_GROUP samples of which are in flight together (5 splats, 128 x 128 x 512: one at a time
// 7.0 ms, 6.5 before the sine had its present form; 3.1 so. Leaving samples out first by their distance to the circle of the
// splat's centre gained nothing.)
constexpr int HIT_GROUP = 4;
__global__ void __launch_bounds__(64) ks_ray_hits(double rp, int64_t npix, int N, Samples smp, const SplatC* __restrict__ sp, int ns,
                                                  const double* __restrict__ times, int nt, const int* __restrict__ kstop,
                                                  uint8_t* __restrict__ hits, int* __restrict__ cnt) {
    const int64_t item = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (item >= npix * nt) return;
    const int64_t j = item % npix;
    const double t_obs = times[item / npix];
    const int kend = kstop ? (kstop[j] - 1 < N ? kstop[j] - 1 : N) : N;
    const double hor = rp * (1.0 + 1e-3);
    int n = 0;
    for (int i = 0; i < ns; ++i) {
        const SplatC& c = sp[i];
        uint8_t hit = 0;
        for (int k0 = 1; k0 <= kend && !hit; k0 += HIT_GROUP) {
            double r[HIT_GROUP], t[HIT_GROUP], x[HIT_GROUP], y[HIT_GROUP], z[HIT_GROUP];
            uint8_t fl[HIT_GROUP];
#pragma unroll
            for (int u = 0; u < HIT_GROUP; ++u) {
                const int64_t o = (int64_t)((k0 + u <= kend ? k0 + u : kend) - 1) * npix + j;
                fl[u] = smp.fl[o]; r[u] = smp.r[o]; t[u] = smp.t[o]; x[u] = smp.x[o]; y[u] = smp.y[o]; z[u] = smp.z[o];
            }
#pragma unroll
            for (int u = 0; u < HIT_GROUP; ++u) {
                if (hit || !(fl[u] & 1) || !(r[u] > hor)) continue;
                double sph, cph;
                hit = outside_support(c, t_obs - t[u], x[u], y[u], z[u], sph, cph) ? 0 : 1;
            }
        }
        hits[(int64_t)i + (int64_t)ns * item] = hit;
        n += hit;
    }
    cnt[item] = n;
}
// ids[s + cap t] = the (s+1)-th hit splat of output item t in ascending order (0-based), -1 past its count. Output
// item t = p + npix f reads item iperm[p] + npix f of hits (the screen pixel p's sorted slot), or t itself when
// iperm is null.
__global__ void ks_ray_fill(int64_t items, int64_t npix, int ns, int cap, const uint8_t* __restrict__ hits, const int* __restrict__ iperm,
                            int32_t* __restrict__ ids) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= items) return;
    const int64_t it = iperm ? iperm[t % npix] + npix * (t / npix) : t;
    int n = 0;
    for (int i = 0; i < ns; ++i)
        if (hits[(int64_t)i + (int64_t)ns * it] && n < cap) ids[(int64_t)cap * t + n++] = i;
    for (; n < cap; ++n) ids[(int64_t)cap * t + n] = -1;
}

hipError_t launch_ray_hits(hipStream_t s, double rp, int64_t npix, int N, Samples smp, const SplatC* sp, int ns, const double* times, int nt,
                           const int* kstop, uint8_t* hits, int* cnt) {
    hipLaunchKernelGGL(ks_ray_hits, dim3(grid_for(npix * nt, 64)), dim3(64), 0, s, rp, npix, N, smp, sp, ns, times, nt, kstop, hits, cnt);
    return hipGetLastError();
}
hipError_t launch_ray_fill(hipStream_t s, int64_t items, int64_t npix, int ns, int cap, const uint8_t* hits, const int* iperm, int32_t* ids) {
    hipLaunchKernelGGL(ks_ray_fill, dim3(grid_for(items, 128)), dim3(128), 0, s, items, npix, ns, cap, hits, iperm, ids);
    return hipGetLastError();
}

}  // namespace ksd
