// Adjoint kernels: the dual sweep over stored samples (polarized_tails!, polarized_dual_sweep!,
// dual_gradient.jl:125-249): tails and adjoints at the chunk boundaries from the chunk maps, the
// per-sample adjoints inside each chunk, the per-splat element adjoints with a wavefront sum, and a
// deterministic reduction over the item blocks.
#include "ks_kernels.hpp"
#include "ks_dsample.hpp"

namespace ksd {

// ---- the dual-sweep adjoint (dual_gradient.jl:125-249) over stored samples -------------------------------------
// Per item: from the chunk maps (P_m, S_m), the tail behind each chunk T_out[m] = S_{m+1} + P_{m+1} T_out[m+1]
// (T_out[last] = 0), and the adjoint in front of each chunk w_in[m] = (P_0 ... P_{m-1})^T w_1 with w_1 = nu-hat^3
// dstokes (dual_gradient.jl:162). wT[(8 m + q) nitems + item] = w_in, wT[(8 m + 4 + q) nitems + item] = T_out.
// A workgroup takes 64 items, each of its wavefronts a run of their chunks: first the run's own map, then through LDS
// the tail behind the run and the adjoint in front of it, then the run's chunks (ks_seg_combine has the same split).
template <class G>
__global__ void __launch_bounds__(64 * COMBINE_WAVES)
ks_adj_combine(int64_t npix, int N, int chunk, int nt, const double* __restrict__ nus, int nnu, const G* __restrict__ seg,
               const double* __restrict__ dstokes, double* __restrict__ wT) {
    __shared__ double s_map[COMBINE_WAVES][SEG_FIELDS][64];
    const int64_t nitems = npix * nt * nnu;
    const int lane = (int)(threadIdx.x % 64), wv = (int)(threadIdx.x / 64);
    const int64_t item = (int64_t)blockIdx.x * 64 + lane;
    const int nseg = (N + chunk - 1) / chunk;
    const int per = (nseg + COMBINE_WAVES - 1) / COMBINE_WAVES;
    const int m0 = wv * per, m1 = m0 + per < nseg ? m0 + per : nseg;
    {
        double P[16], Sv[4] = {0, 0, 0, 0};
        for (int i = 0; i < 16; ++i) P[i] = (i % 5 == 0) ? 1.0 : 0.0;
        if (item < nitems)
            for (int m = m0; m < m1; ++m) {
                double Pm[16], Sm[4];
                seg_load(seg, m, nitems, item, Pm, Sm);
                seg_append(P, Sv, Pm, Sm);
            }
        for (int q = 0; q < 16; ++q) s_map[wv][q][lane] = P[q];
        for (int q = 0; q < 4; ++q) s_map[wv][16 + q][lane] = Sv[q];
    }
    __syncthreads();
    if (item >= nitems) return;
    double T[4] = {0, 0, 0, 0};
    for (int w = COMBINE_WAVES - 1; w > wv; --w) {
        double Tn[4];
        for (int i = 0; i < 4; ++i) {
            double v = s_map[w][16 + i][lane];
            for (int q = 0; q < 4; ++q) v += s_map[w][4 * i + q][lane] * T[q];
            Tn[i] = v;
        }
        for (int i = 0; i < 4; ++i) T[i] = Tn[i];
    }
    const double nh = nus[(item / npix) / nt] * (1.0 / NU0);
    const double s3 = nh * nh * nh;
    double w[4];
    for (int q = 0; q < 4; ++q) w[q] = dstokes[4 * item + q] * s3;
    for (int v = 0; v < wv; ++v) {
        double wn[4];
        for (int c = 0; c < 4; ++c) {
            double acc = 0.0;
            for (int i = 0; i < 4; ++i) acc += s_map[v][4 * i + c][lane] * w[i];
            wn[c] = acc;
        }
        for (int q = 0; q < 4; ++q) w[q] = wn[q];
    }
    for (int m = m1 - 1; m >= m0; --m) {
        double Pm[16], Sm[4];
        seg_load(seg, m, nitems, item, Pm, Sm);
        for (int q = 0; q < 4; ++q) wT[(8 * (int64_t)m + 4 + q) * nitems + item] = T[q];
        double Tn[4];
        for (int i = 0; i < 4; ++i) {
            double v = Sm[i];
            for (int q = 0; q < 4; ++q) v += Pm[4 * i + q] * T[q];
            Tn[i] = v;
        }
        for (int i = 0; i < 4; ++i) T[i] = Tn[i];
    }
    for (int m = m0; m < m1; ++m) {
        double Pm[16], Sm[4];
        seg_load(seg, m, nitems, item, Pm, Sm);
        for (int q = 0; q < 4; ++q) wT[(8 * (int64_t)m + q) * nitems + item] = w[q];
        double wn[4];
        for (int c = 0; c < 4; ++c) {
            double v = 0.0;
            for (int i = 0; i < 4; ++i) v += Pm[4 * i + c] * w[i];
            wn[c] = v;
        }
        for (int q = 0; q < 4; ++q) w[q] = wn[q];
    }
}

// The FP64 step and step adjoint of an FP32 sample, out of line (the rare samples with a Faraday depth
// |rho| Delta above FARADAY_FP64, where the forward pass takes the FP64 step too).
// (inputs and outputs by value, as step_f64_for_f32's: the callers' arrays stay in registers)
struct Vec4_32 { f32 v[4]; };
struct Seeds32 { f32 w[4], R[4]; };
struct StepAdj32 { f32 Otw[4], jb[4], ab[4], rb[3]; };
KS_COLD StepAdj32 step_adjoint_f64_for_f32(const Step32 s, const Seeds32 z) {
    double jd[4], ad[4], rd[3], wd[4], Rd[4], Od[4], jbd[4], abd[4], rbd[3];
    for (int i = 0; i < 4; ++i) { jd[i] = val(s.j[i]); ad[i] = val(s.a[i]); wd[i] = val(z.w[i]); Rd[i] = val(z.R[i]); }
    for (int i = 0; i < 3; ++i) rd[i] = val(s.r[i]);
    sample_adjoint(jd, ad, rd, val(s.D), wd, Rd, Od, jbd, abd, rbd);
    StepAdj32 o;
    for (int i = 0; i < 4; ++i) { o.Otw[i] = f32(Od[i]); o.jb[i] = f32(jbd[i]); o.ab[i] = f32(abd[i]); }
    for (int i = 0; i < 3; ++i) o.rb[i] = f32(rbd[i]);
    return o;
}
KS_COLD Vec4_32 step_apply_f64_for_f32(const Step32 s, const Vec4_32 Tin) {
    double jd[4], ad[4], rd[3], Ti[4], To[4];
    for (int i = 0; i < 4; ++i) { jd[i] = val(s.j[i]); ad[i] = val(s.a[i]); Ti[i] = val(Tin.v[i]); }
    for (int i = 0; i < 3; ++i) rd[i] = val(s.r[i]);
    step_apply(jd, ad, rd, val(s.D), Ti, To);
    Vec4_32 o;
    for (int i = 0; i < 4; ++i) o.v[i] = f32(To[i]);
    return o;
}

// The adjoint of one sample's step, and the step applied to a tail, in the transfer's scalar; in FP32
// the samples with a Faraday depth |rho| Delta above FARADAY_FP64 take the FP64 step and its adjoint.
template <class S>
KS_DEV void step_adjoint_s(const S j4[4], const S a4[4], const S r3[3], S D, const S w[4], const S R[4], S Otw[4], S jb[4], S ab[4], S rb[3]) {
    if constexpr (!std::is_same<S, double>::value) {
        const S fd = sqrt(r3[0] * r3[0] + r3[1] * r3[1] + r3[2] * r3[2]) * D;
        if (fd > FARADAY_FP64) {
            Seeds32 z;
            for (int i = 0; i < 4; ++i) { z.w[i] = w[i]; z.R[i] = R[i]; }
            const StepAdj32 o = step_adjoint_f64_for_f32(step32_of(j4, a4, r3, D), z);
            for (int i = 0; i < 4; ++i) { Otw[i] = o.Otw[i]; jb[i] = o.jb[i]; ab[i] = o.ab[i]; }
            for (int i = 0; i < 3; ++i) rb[i] = o.rb[i];
            return;
        }
    }
    sample_adjoint(j4, a4, r3, D, w, R, Otw, jb, ab, rb);
}
template <class S>
KS_DEV void step_apply_s(const S j4[4], const S a4[4], const S r3[3], S D, const S Tin[4], S Tout[4]) {
    if constexpr (!std::is_same<S, double>::value) {
        const S fd = sqrt(r3[0] * r3[0] + r3[1] * r3[1] + r3[2] * r3[2]) * D;
        if (fd > FARADAY_FP64) {
            Vec4_32 ti;
            for (int i = 0; i < 4; ++i) ti.v[i] = Tin[i];
            const Vec4_32 o = step_apply_f64_for_f32(step32_of(j4, a4, r3, D), ti);
            for (int i = 0; i < 4; ++i) Tout[i] = o.v[i];
            return;
        }
    }
    step_apply(j4, a4, r3, D, Tin, Tout);
}

// Per (chunk, item): the tails T_{k+1} of the chunk's samples back to front from T_out[m], then the
// adjoint front to back from w_in[m]: per sample the adjoints of its j, alpha, rho (into bar, beside the
// records, which stay intact so that the reverse pass can run again on the same forward pass) and
// w <- O^T w (polarized_dual_kernel!'s ray loop, dual_gradient.jl:151-178).
template <class S>
__global__ void __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(Waves<S>::adjstep))) ks_adj_segment(int N, int chunk, int64_t nitems, int nch, const double* __restrict__ wT, const S* __restrict__ rec,
                                                      S* __restrict__ bar, const uint8_t* __restrict__ aflg, S* __restrict__ tails, Samples smp,
                                                      int64_t npix) {
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= nitems * nch) return;
    const int64_t item = slot_item(smp, tid % nitems, npix);     // wavefronts over compact patches of sky
    const int m = (int)(tid / nitems);
    const int kbeg = m * chunk + 1, kend = kbeg + chunk - 1 < N ? kbeg + chunk - 1 : N;
    const int64_t st = (int64_t)N * nitems;
    S T[4], w[4];
    for (int q = 0; q < 4; ++q) { w[q] = S(wT[(8 * (int64_t)m + q) * nitems + item]); T[q] = S(wT[(8 * (int64_t)m + 4 + q) * nitems + item]); }
    for (int k = kend; k >= kbeg; --k) {
        const int64_t fo = (int64_t)(k - 1) * nitems + item;
        if (!aflg[fo]) continue;
        const S* o = rec + fo;
        S j4[4], a4[4], r3[3];
        for (int i = 0; i < 4; ++i) { j4[i] = o[(REC_J + i) * st]; a4[i] = o[(REC_A + i) * st]; }
        for (int i = 0; i < 3; ++i) r3[i] = o[(REC_RHO + i) * st];
        for (int q = 0; q < 4; ++q) tails[(int64_t)q * st + fo] = T[q];
        S Tn[4];
        step_apply_s(j4, a4, r3, o[REC_D * st], T, Tn);
        for (int q = 0; q < 4; ++q) T[q] = Tn[q];
    }
    for (int k = kbeg; k <= kend; ++k) {
        const int64_t fo = (int64_t)(k - 1) * nitems + item;
        if (!aflg[fo]) continue;
        const S* o = rec + fo;
        S j4[4], a4[4], r3[3], R[4];
        for (int i = 0; i < 4; ++i) { j4[i] = o[(REC_J + i) * st]; a4[i] = o[(REC_A + i) * st]; R[i] = tails[(int64_t)i * st + fo]; }
        for (int i = 0; i < 3; ++i) r3[i] = o[(REC_RHO + i) * st];
        S Otw[4], jb[4], ab[4], rb[3];
        step_adjoint_s(j4, a4, r3, o[REC_D * st], w, R, Otw, jb, ab, rb);
        S* b = bar + fo;
        for (int i = 0; i < 4; ++i) { b[i * st] = jb[i]; b[(4 + i) * st] = ab[i]; }
        for (int i = 0; i < 3; ++i) b[(8 + i) * st] = rb[i];
        for (int q = 0; q < 4; ++q) w[q] = Otw[q];
    }
}

// The work list of the element adjoints: a unit is 64 items x ADJ_SLICE samples, a block one (unit, splat) whose splat
// can reach a step-taking sample of the unit (the bounding sphere of those samples and their emission times,
// splat_may_reach). One wavefront per unit writes a bit per splat and their count; one workgroup gives every unit the
// list position of its first block; one wavefront per unit then writes the list, and each mask word's position. The
// units of a batch are listed XCD by XCD (unit u on XCD u % 8), so that all blocks of a unit run beside one L2, which
// reads the unit's samples once. Blocks that are culled cost nothing further: before, each was a workgroup that
// stored 22 zeros for the reduction to read (four in five of the 24 million of 1024 kappa splats at 256^2 x 1024).
__global__ void __launch_bounds__(64) ks_unit_mask(int64_t npix, int N, Samples smp, const double* __restrict__ times, int nt,
                                                   int64_t nitems, const uint8_t* __restrict__ aflg, const SplatC* __restrict__ sp, int ns,
                                                   const double* __restrict__ knots, const double* __restrict__ ktimes, int64_t unit0,
                                                   uint64_t* __restrict__ mask, int* __restrict__ count) {
    const int64_t unit = unit0 + blockIdx.x;
    const int nslice = (N + ADJ_SLICE - 1) / ADJ_SLICE;
    const int64_t ib = unit / nslice;
    const int kfirst = (int)(unit % nslice) * ADJ_SLICE + 1;
    const int klast = kfirst + ADJ_SLICE - 1 < N ? kfirst + ADJ_SLICE - 1 : N;
    const int lane = (int)threadIdx.x;
    const int64_t item = ib * 64 + lane;
    double lo[4] = {INFINITY, INFINITY, INFINITY, INFINITY}, hi[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    if (item < nitems) {
        const int64_t j = item % npix;
        const double t_obs = times[(item / npix) % nt];
        for (int k = kfirst; k <= klast; ++k) {
            if (!aflg[(int64_t)(k - 1) * nitems + item]) continue;
            const int64_t so = (int64_t)(k - 1) * npix + j;
            const double v[4] = {smp.x[so], smp.y[so], smp.z[so], t_obs - smp.t[so]};
            for (int q = 0; q < 4; ++q) { lo[q] = fmin(lo[q], v[q]); hi[q] = fmax(hi[q], v[q]); }
        }
    }
    double px = 0.0, py = 0.0, pz = 0.0, R = 0.0, tmin = 0.0, tmax = 0.0;
    const bool any = wave_region(lo, hi, px, py, pz, R, tmin, tmax);
    const int nw = (ns + 63) / 64;
    int n = 0;
    for (int b = 0; b < nw; ++b) {
        const int i = 64 * b + lane;
        const uint64_t m = __ballot(any && i < ns && splat_may_reach(sp[i], px, py, pz, R, tmin, tmax, knots, ktimes));
        if (lane == 0) mask[(int64_t)blockIdx.x * nw + b] = m;
        n += __popcll(m);
    }
    if (lane == 0) count[blockIdx.x] = n;
}
// the unit at position p of the list's order: XCD p / per, its units in ascending order (per = ceil(nb / 8); >= nb: none)
KS_DEV int64_t listed_unit(int64_t p, int64_t per) { return (p % per) * 8 + p / per; }
constexpr int LIST_THREADS = 1024;
// first[u]: the list position of unit u's first block; xcd[0..8]: the ranges of the XCDs. Each thread sums a run of the
// order, the runs' sums are scanned in LDS, and each thread then walks its run again.
__global__ void __launch_bounds__(LIST_THREADS) ks_unit_first(int64_t nb, const int* __restrict__ count, int* __restrict__ first, int* __restrict__ xcd) {
    __shared__ int s_sum[LIST_THREADS];
    const int64_t per = (nb + 7) / 8, all = 8 * per, run = (all + LIST_THREADS - 1) / LIST_THREADS;
    const int t = (int)threadIdx.x;
    const int64_t p0 = t * run, p1 = p0 + run < all ? p0 + run : all;
    int n = 0;
    for (int64_t p = p0; p < p1; ++p) {
        const int64_t u = listed_unit(p, per);
        if (u < nb) n += count[u];
    }
    s_sum[t] = n;
    __syncthreads();
    for (int d = 1; d < LIST_THREADS; d *= 2) {
        const int v = t >= d ? s_sum[t - d] : 0;
        __syncthreads();
        s_sum[t] += v;
        __syncthreads();
    }
    int pos = s_sum[t] - n;
    for (int64_t p = p0; p < p1; ++p) {
        const int64_t u = listed_unit(p, per);
        if (p % per == 0) xcd[p / per] = pos;
        if (u < nb) { first[u] = pos; pos += count[u]; }
    }
    if (t == LIST_THREADS - 1) xcd[8] = s_sum[t];
}
// list[e] = (unit of the batch, splat); at[u nw + b] = the position of the first block of mask word b
__global__ void __launch_bounds__(64) ks_unit_list(int ns, const uint64_t* __restrict__ mask, const int* __restrict__ first, int2* __restrict__ list,
                                                   int* __restrict__ at) {
    const int64_t u = blockIdx.x;
    const int nw = (ns + 63) / 64, lane = (int)threadIdx.x;
    int pos = first[u];
    for (int b = 0; b < nw; ++b) {
        const uint64_t m = mask[u * nw + b];
        if (lane == 0) at[u * nw + b] = pos;
        if ((m >> lane) & 1) list[pos + __popcll(m & ((1ull << lane) - 1))] = make_int2((int)u, 64 * b + lane);
        pos += __popcll(m);
    }
}

// Per block of the list (64 consecutive items, slice of ADJ_SLICE samples, splat): the element adjoints of every
// (item, sample) pair inside the splat's weight cutoff, 22 partial sums per lane, summed over the
// wavefront into part[22 e + r] for the block's list position e. The slices bound the work of
// one wavefront: the pairs of a splat crowd into a few item blocks and stretches of the rays, and
// whole-ray units left most of the chip idle behind the heaviest ones.
// The wavefront walks its items' samples with the FP32 prefilter (may_weigh), WALK samples at a time with
// their loads issued together, and queues the pairs that pass (ballot + mbcnt into an LDS ring); whenever 64 are queued,
// or the samples are through, it runs the element adjoint of up to 64 pairs, so that lanes outside the splat's support
// do not idle through it (one call site for both: a second inlined copy doubled the kernel's 60 KB of code).
// MI355X, element adjoints of one pass, before and after (list, one call site, prefilter): FP64, 32 thermal splats at
// 128^2 x 1024 9.4 -> 6.9 ms, 48 power-law splats 8.0 -> 6.0, 1024 kappa splats (112 x 96 x 512) 237 -> 167; mixed, 1024
// kappa splats (256^2 x 1024) 583 -> 451, 64 thermal splats (4 frames of 128^2 x 1024) 22.7 -> 19.3.
// Every pair of a wavefront belongs to
// splat i, so the sums stay per lane in registers; the queue order is fixed, so the result is
// deterministic.
// POPS: the populations the launch meets, POP_THERMAL (thermal and knot splats), POP_POWERLAW, POP_KAPPA, and
// POP_KNOTS (centres that follow knots); a launch of one population carries only its branch, whose registers would
// otherwise cost it occupancy; mixed populations take a runtime branch on the splat's kind.
// block-wide copy of a per-splat constant struct into LDS
template <class T> KS_DEV void copy_to_lds(T* dst, const T* __restrict__ src, int lane) {
    static_assert(sizeof(T) % 4 == 0, "copied in dwords");
    for (int q = lane; q < (int)(sizeof(T) / 4); q += 64) ((int*)dst)[q] = ((const int*)src)[q];
}
template <class S, int POPS>
__device__ __forceinline__ void adj_splats_block(int64_t e, int64_t unit, int i, double a, double thetao, const double* __restrict__ soa, int64_t npix, int N,
                                                 Samples smp, const SplatCT<S>* __restrict__ sp, const SplatAdjT<S>* __restrict__ sadj,
                                                 const SplatCf* __restrict__ spf, const f32* __restrict__ knots_f, const f32* __restrict__ ktimes_f,
                                                 const S* __restrict__ knots, const S* __restrict__ ktimes,
                                                 const double* __restrict__ times, int nt, const double* __restrict__ nus, int64_t nitems,
                                                 const S* __restrict__ rec, const S* __restrict__ bar, const uint8_t* __restrict__ aflg,
                                                 double* __restrict__ part) {
    constexpr int WALK = 8;                 // samples tested per group, their loads issued together
    constexpr int QCAP = 1024;              // ring capacity: < 64 pending + 64 per sample of a group
    static_assert(QCAP >= 64 * (WALK + 1) && (QCAP & (QCAP - 1)) == 0, "the ring must hold a group's pushes");
    __shared__ double s_alpha[64], s_beta[64], s_tobs[64], s_nu[64];
    __shared__ int64_t s_item[64];
    __shared__ int s_q[QCAP];   // entry = lane | k << 6
    const int nslice = (N + ADJ_SLICE - 1) / ADJ_SLICE;
    const int64_t ib = unit / nslice;
    const int kfirst = (int)(unit % nslice) * ADJ_SLICE + 1;
    const int klast = kfirst + ADJ_SLICE - 1 < N ? kfirst + ADJ_SLICE - 1 : N;
    const int lane = (int)threadIdx.x;
    const bool valid = ib * 64 + lane < nitems;
    const int64_t item = ib * 64 + lane;      // sorted order: the pair queue already packs the lanes
    // the splat's constants in LDS, read where they are used: held in registers for the whole kernel
    // they outgrow the scalar file and spill into vector lanes
    __shared__ SplatCT<S> s_c;
    __shared__ SplatAdjT<S> s_sa;
    __syncthreads();                          // the last block's reads are done
    copy_to_lds(&s_c, sp + i, lane);
    copy_to_lds(&s_sa, sadj + i, lane);
    const SplatTest test = splat_test(spf[i]);
    const SplatCT<S>& c = s_c;
    const SplatAdjT<S>& sa = s_sa;
    int64_t j = 0;
    double t_obs = 0.0;
    if (valid) {
        j = item % npix;
        const int64_t fr = item / npix;
        t_obs = times[fr % nt];
        s_alpha[lane] = soa[(int64_t)PF_ALPHA * npix + j];
        s_beta[lane] = soa[(int64_t)PF_BETA * npix + j];
        s_tobs[lane] = t_obs;
        s_nu[lane] = nus[fr / nt];
        s_item[lane] = item;
    }
    __syncthreads();
    const S tos = S(sin(thetao)), aS = S(a);
    const int64_t st = (int64_t)N * nitems;
    // the FP32 path reads the samples' FP32 copy (one 16-byte load per sample instead of four 8-byte loads; its
    // launcher requires it)
    constexpr bool use_p4 = std::is_same<S, f32>::value;
    S grad[ADJ_ROWS];
    for (int r = 0; r < ADJ_ROWS; ++r) grad[r] = S(0.0);
    int qhead = 0, qn = 0;   // wavefront-uniform ring state
    auto run_batch = [&](int cnt) {
        if (lane < cnt) {
            const int e = s_q[(qhead + lane) & (QCAP - 1)];
            const int l = e & 63, k = e >> 6;
            const int64_t it2 = s_item[l];
            const int64_t fo = (int64_t)(k - 1) * nitems + it2;
            const int64_t so = (int64_t)(k - 1) * npix + it2 % npix;
            S dl[13];
            S tt, xx, yy, zz;
            if constexpr (use_p4) {
                const float4 q = smp.p4[so];
                tt = S((float)s_tobs[l] - q.w); xx = S(q.x); yy = S(q.y); zz = S(q.z);
            } else {
                tt = S(s_tobs[l] - smp.t[so]); xx = S(smp.x[so]); yy = S(smp.y[so]); zz = S(smp.z[so]);
            }
            S Gw;
            if constexpr ((POPS & POP_KNOTS) != 0) Gw = c.nk > 0 ? weight_dlog_knot(c, sa, knots, ktimes, tt, xx, yy, zz, dl) : weight_dlog(c, sa, tt, xx, yy, zz, dl);
            else Gw = weight_dlog(c, sa, tt, xx, yy, zz, dl);
            if (Gw > 0.0) {
                const S* o = bar + fo;
                S bars[BAR_FIELDS];
                for (int q = 0; q < BAR_FIELDS; ++q) bars[q] = o[q * st];
                GeoT<S> G;
                geo_load(rec + fo + REC_GEO * st, st, G);        // written by the forward transfer
                constexpr int fl = POPS & POP_FLUIDS;
                if constexpr (fl == POP_THERMAL)
                    element_adjoint_thermal(c, sa, G, aS, S(s_alpha[l]), S(s_beta[l]), tos, S(s_nu[l]), bars, Gw, dl, grad);
                else if constexpr (fl == POP_POWERLAW)
                    element_adjoint_pop(c, sa, G, aS, S(s_alpha[l]), S(s_beta[l]), tos, S(s_nu[l]), bars, Gw, dl, grad);
                else if constexpr (fl == POP_KAPPA)
                    element_adjoint_kappa(c, sa, G, aS, S(s_alpha[l]), S(s_beta[l]), tos, S(s_nu[l]), bars, Gw, dl, grad);
                else if (c.kind == MODEL_KAPPA)
                    element_adjoint_kappa(c, sa, G, aS, S(s_alpha[l]), S(s_beta[l]), tos, S(s_nu[l]), bars, Gw, dl, grad);
                else if (c.kind == MODEL_POWERLAW)
                    element_adjoint_pop(c, sa, G, aS, S(s_alpha[l]), S(s_beta[l]), tos, S(s_nu[l]), bars, Gw, dl, grad);
                else
                    element_adjoint_thermal(c, sa, G, aS, S(s_alpha[l]), S(s_beta[l]), tos, S(s_nu[l]), bars, Gw, dl, grad);
            }
        }
        qhead = (qhead + cnt) & (QCAP - 1);
        qn -= cnt;
    };
    int k0 = kfirst;
    for (;;) {
        while (qn < 64 && k0 <= klast) {
            uint8_t fl[WALK];
            float tk[WALK], xk[WALK], yk[WALK], zk[WALK];     // t_obs - t~ and the position of each sample of the group
#pragma unroll
            for (int u = 0; u < WALK; ++u) {
                const int k = k0 + u;
                fl[u] = 0;
                tk[u] = xk[u] = yk[u] = zk[u] = 0.0f;
                if (valid && k <= klast) {
                    const int64_t so = (int64_t)(k - 1) * npix + j;
                    fl[u] = aflg[(int64_t)(k - 1) * nitems + item];
                    if constexpr (use_p4) {
                        const float4 q = smp.p4[so];
                        tk[u] = (float)t_obs - q.w; xk[u] = q.x; yk[u] = q.y; zk[u] = q.z;
                    } else {
                        tk[u] = (float)(t_obs - smp.t[so]); xk[u] = (float)smp.x[so]; yk[u] = (float)smp.y[so]; zk[u] = (float)smp.z[so];
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < WALK; ++u) {
                const bool act = fl[u] && may_weigh<MODEL_THERMAL>(test, knots_f, ktimes_f, tk[u], xk[u], yk[u], zk[u]);
                const uint64_t m = __ballot(act);
                if (act) {
                    const int rank = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                    s_q[(qhead + qn + rank) & (QCAP - 1)] = lane | ((k0 + u) << 6);
                }
                qn += __popcll(m);
            }
            k0 += WALK;
        }
        if (qn == 0) break;
        __syncthreads();
        run_batch(qn < 64 ? qn : 64);
        __syncthreads();
    }
    // wavefront sum (blockDim = 64 = one wavefront), in FP64
    double gsum[ADJ_ROWS];
    for (int r = 0; r < ADJ_ROWS; ++r) {
        double v = val(grad[r]);
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
        gsum[r] = v;
    }
    // lane r < ADJ_ROWS stores row r (the lanes past the rows repeat the last row): selects, no lane-dependent branch
    double mine = gsum[ADJ_ROWS - 1];
    for (int r = 0; r < ADJ_ROWS - 1; ++r) mine = lane == r ? gsum[r] : mine;
    part[e * ADJ_ROWS + min(lane, ADJ_ROWS - 1)] = mine;
}

// The launch: a persistent grid of the resident workgroups (a multiple of 8, so workgroup w runs on XCD w % 8), each
// taking tickets from its XCD's queue heads[w % 8] over the XCD's range of the list, and from the other XCDs' once that
// is through. The ticket is taken by all 64 lanes (lane 0 adds one) and made scalar, so the loop's exit and back edge
// are uniform branches.
template <class S, int POPS>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu((adjelem_waves<S, POPS>))))
ks_adj_splats(double a, double thetao, const double* __restrict__ soa, int64_t npix, int N, Samples smp, const SplatCT<S>* __restrict__ sp,
              const SplatAdjT<S>* __restrict__ sadj, const SplatCf* __restrict__ spf, const f32* __restrict__ knots_f,
              const f32* __restrict__ ktimes_f, const S* __restrict__ knots, const S* __restrict__ ktimes,
              const double* __restrict__ times, int nt, const double* __restrict__ nus, int64_t nitems, const S* __restrict__ rec,
              const S* __restrict__ bar, const uint8_t* __restrict__ aflg, int64_t unit0, const int2* __restrict__ list,
              const int* __restrict__ xcd, double* __restrict__ part, unsigned* __restrict__ heads) {
    int x = (int)(blockIdx.x % 8), tried = 0;
    for (;;) {
        const unsigned t = __builtin_amdgcn_readfirstlane(atomicAdd(heads + x, threadIdx.x == 0 ? 1u : 0u));
        const int64_t e = (int64_t)xcd[x] + t;
        if (e < xcd[x + 1]) {
            const int2 b = list[e];
            adj_splats_block<S, POPS>(e, unit0 + __builtin_amdgcn_readfirstlane(b.x), __builtin_amdgcn_readfirstlane(b.y), a, thetao, soa, npix, N, smp,
                                      sp, sadj, spf, knots_f, ktimes_f, knots, ktimes, times, nt, nus, nitems, rec, bar, aflg, part);
        } else {
            x = (x + 1) & 7;
            ++tried;
        }
        if (tried == 8) break;
    }
}

// dparams[r + ADJ_ROWS i] = the sum over a batch's blocks of splat i in a fixed order (deterministic): REDUCE_PARTS
// workgroups a splat, each over a run of the units, lane l of its four wavefronts taking the run's units l, l + 256, ...
// that hold a block of the splat; a fixed butterfly over the lanes, the wavefronts in order, then (ks_adj_reduce_parts)
// the runs in order, added to the sums of the earlier batches when accumulate (the batches in order)
constexpr int REDUCE_PARTS = 16;
__global__ void __launch_bounds__(256) ks_adj_reduce(const double* __restrict__ part, int64_t nunits, int ns, const uint64_t* __restrict__ mask,
                                                     const int* __restrict__ at, double* __restrict__ sums) {
    const int i = (int)(blockIdx.x / REDUCE_PARTS), y = (int)(blockIdx.x % REDUCE_PARTS);
    const int nw = (ns + 63) / 64, w = i / 64, bit = i % 64;
    const int64_t per = (nunits + REDUCE_PARTS - 1) / REDUCE_PARTS;
    const int64_t u1 = (y + 1) * per < nunits ? (y + 1) * per : nunits;
    double s[ADJ_ROWS];
    for (int r = 0; r < ADJ_ROWS; ++r) s[r] = 0.0;
    for (int64_t u = y * per + threadIdx.x; u < u1; u += 256) {
        const uint64_t m = mask[u * nw + w];
        if (!((m >> bit) & 1)) continue;
        const double* p = part + (int64_t)(at[u * nw + w] + __popcll(m & ((1ull << bit) - 1))) * ADJ_ROWS;
        for (int r = 0; r < ADJ_ROWS; ++r) s[r] += p[r];
    }
    __shared__ double s_w[4][ADJ_ROWS];
    for (int r = 0; r < ADJ_ROWS; ++r) {
        double v = s[r];
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
        if (threadIdx.x % 64 == 0) s_w[threadIdx.x / 64][r] = v;
    }
    __syncthreads();
    if (threadIdx.x < ADJ_ROWS) sums[(int64_t)blockIdx.x * ADJ_ROWS + threadIdx.x] = s_w[0][threadIdx.x] + s_w[1][threadIdx.x] + s_w[2][threadIdx.x] + s_w[3][threadIdx.x];
}
__global__ void ks_adj_reduce_parts(const double* __restrict__ sums, int ns, int accumulate, double* __restrict__ dparams) {
    const int t = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (t >= ns * ADJ_ROWS) return;
    const int i = t / ADJ_ROWS, r = t % ADJ_ROWS;
    double v = 0.0;
    for (int y = 0; y < REDUCE_PARTS; ++y) v += sums[((int64_t)i * REDUCE_PARTS + y) * ADJ_ROWS + r];
    dparams[t] = accumulate ? dparams[t] + v : v;
}

// ---- launchers ----
hipError_t launch_adj_combine(hipStream_t s, int64_t npix, int N, int chunk, int nt, const double* nus, int nnu, const void* seg, int seg32,
                              const double* dstokes, double* wT) {
    const dim3 grid(grid_for(npix * nt * nnu, 64)), block(64 * COMBINE_WAVES);
    if (seg32) hipLaunchKernelGGL(ks_adj_combine<f32>, grid, block, 0, s, npix, N, chunk, nt, nus, nnu, (const f32*)seg, dstokes, wT);
    else hipLaunchKernelGGL(ks_adj_combine<double>, grid, block, 0, s, npix, N, chunk, nt, nus, nnu, (const double*)seg, dstokes, wT);
    return hipGetLastError();
}
hipError_t launch_adj_segment(hipStream_t s, int N, int chunk, int64_t nitems, const double* wT, const double* rec, double* bar,
                              const uint8_t* aflg, double* tails, Samples smp, int64_t npix) {
    const int nch = (N + chunk - 1) / chunk;
    hipLaunchKernelGGL(ks_adj_segment<double>, dim3(grid_for(nitems * nch, 128)), dim3(128), 0, s, N, chunk, nitems, nch, wT, rec, bar, aflg,
                       tails, smp, npix);
    return hipGetLastError();
}
hipError_t launch_adj_segment_f32(hipStream_t s, int N, int chunk, int64_t nitems, const double* wT, const f32* rec, f32* bar,
                                  const uint8_t* aflg, f32* tails, Samples smp, int64_t npix) {
    const int nch = (N + chunk - 1) / chunk;
    hipLaunchKernelGGL(ks_adj_segment<f32>, dim3(grid_for(nitems * nch, 128)), dim3(128), 0, s, N, chunk, nitems, nch, wT, rec, bar, aflg,
                       tails, smp, npix);
    return hipGetLastError();
}
template <class S>
static hipError_t adj_splats_k(hipStream_t s, const AdjWork& w, int pops, double a, double thetao, const double* soa, int64_t npix, int N, Samples smp,
                               const SplatCT<S>* sp, const SplatAdjT<S>* sadj, const SplatCf* spf, const f32* knots_f, const f32* ktimes_f,
                               const S* knots, const S* ktimes, const double* times, int nt, const double* nus, int64_t nitems, const S* rec,
                               const S* bar, const uint8_t* aflg, int64_t unit0, int64_t nb, int ns) {
    if (hipError_t e = launch_fill_i32(s, w.heads, 8, 0)) return e;
    // the resident workgroups of the launch's instantiation, a multiple of 8
#define KS_ADJ_LAUNCH(P) do { static int groups = 0; \
        if (!groups) groups = resident_groups(ks_adj_splats<S, P>, 64) / 8 * 8; \
        if (groups < 8) return hipErrorInvalidValue; \
        hipLaunchKernelGGL((ks_adj_splats<S, P>), dim3((unsigned)std::min<int64_t>(groups, (nb * ns + 7) / 8 * 8)), dim3(64), 0, s, a, thetao, soa, npix, N, \
                           smp, sp, sadj, spf, knots_f, ktimes_f, knots, ktimes, times, nt, nus, nitems, rec, bar, aflg, unit0, (const int2*)w.list, w.xcd, \
                           w.part, (unsigned*)w.heads); } while (0)
    switch (pops) {
        case POP_THERMAL: KS_ADJ_LAUNCH(POP_THERMAL); break;
        case POP_THERMAL | POP_KNOTS: KS_ADJ_LAUNCH(POP_THERMAL | POP_KNOTS); break;
        case POP_POWERLAW: KS_ADJ_LAUNCH(POP_POWERLAW); break;
        case POP_POWERLAW | POP_KNOTS: KS_ADJ_LAUNCH(POP_POWERLAW | POP_KNOTS); break;
        case POP_KAPPA: KS_ADJ_LAUNCH(POP_KAPPA); break;
        case POP_KAPPA | POP_KNOTS: KS_ADJ_LAUNCH(POP_KAPPA | POP_KNOTS); break;
        default: KS_ADJ_LAUNCH(POP_FLUIDS | POP_KNOTS); break;        // more than one population
    }
#undef KS_ADJ_LAUNCH
    return hipGetLastError();
}
hipError_t launch_adj_splats(hipStream_t s, const AdjWork& w, int pops, double a, double thetao, const double* soa, int64_t npix, int N, Samples smp,
                             const SplatC* sp, const SplatAdj* sadj, const SplatCf* spf, const f32* knots_f, const f32* ktimes_f, int ns,
                             const double* knots, const double* ktimes, const double* times, int nt, const double* nus, int64_t nitems,
                             const double* rec, const double* bar, const uint8_t* aflg, int64_t unit0, int64_t nb) {
    return adj_splats_k<double>(s, w, pops, a, thetao, soa, npix, N, smp, sp, sadj, spf, knots_f, ktimes_f, knots, ktimes, times, nt, nus, nitems, rec,
                                bar, aflg, unit0, nb, ns);
}
hipError_t launch_adj_splats_f32(hipStream_t s, const AdjWork& w, int pops, double a, double thetao, const double* soa, int64_t npix, int N, Samples smp,
                                 const SplatCf* sp, const SplatAdjf* sadj, int ns, const f32* knots, const f32* ktimes,
                                 const double* times, int nt, const double* nus, int64_t nitems, const f32* rec, const f32* bar,
                                 const uint8_t* aflg, int64_t unit0, int64_t nb) {
    if (!smp.p4) return hipErrorInvalidValue;          // the FP32 element adjoints read the samples' FP32 copy
    return adj_splats_k<f32>(s, w, pops, a, thetao, soa, npix, N, smp, sp, sadj, sp, knots, ktimes, knots, ktimes, times, nt, nus, nitems, rec, bar,
                             aflg, unit0, nb, ns);
}
hipError_t launch_adj_list(hipStream_t s, const AdjWork& w, int64_t npix, int N, Samples smp, const double* times, int nt, int64_t nitems,
                           const uint8_t* aflg, const SplatC* sp, int ns, const double* knots, const double* ktimes, int64_t unit0, int64_t nb) {
    hipLaunchKernelGGL(ks_unit_mask, dim3((unsigned)nb), dim3(64), 0, s, npix, N, smp, times, nt, nitems, aflg, sp, ns, knots, ktimes, unit0, w.mask, w.count);
    hipLaunchKernelGGL(ks_unit_first, dim3(1), dim3(LIST_THREADS), 0, s, nb, w.count, w.first, w.xcd);
    hipLaunchKernelGGL(ks_unit_list, dim3((unsigned)nb), dim3(64), 0, s, ns, w.mask, w.first, (int2*)w.list, w.at);
    return hipGetLastError();
}
hipError_t launch_adj_reduce(hipStream_t s, const AdjWork& w, int64_t nunits, int ns, int accumulate, double* dparams) {
    hipLaunchKernelGGL(ks_adj_reduce, dim3((unsigned)(ns * REDUCE_PARTS)), dim3(256), 0, s, w.part, nunits, ns, w.mask, w.at, w.sums);
    hipLaunchKernelGGL(ks_adj_reduce_parts, dim3(grid_for((int64_t)ns * ADJ_ROWS, 256)), dim3(256), 0, s, w.sums, ns, accumulate, dparams);
    return hipGetLastError();
}
int adj_reduce_parts() { return REDUCE_PARTS; }

}  // namespace ksd
