// kernels_mlt.hip -- primary sample space MLT (PSSMLTIntegrator, Extensions/
// Integrator/PSSMLT.fs) as a wavefront over many chains.
//
// Every chain advances one mutation per round; a round is
//   mlt_start (StartIteration + camera samples) -> [trace_closest -> bin ->
//   shade_mlt -> trace_shadow] x max_depth -> mlt_accept
// reusing the path-tracing traversal kernels.  A chain's primary samples live
// in HBM, index-major (sample i of chain c at xs[i * cap + c]) so that a wave
// of consecutive chains touches consecutive 16-byte records.
#include "kernels.hpp"
#include "kernels_mlt.hpp"
#include "shading.hpp"
#include "traverse.hpp"
#include "wave.hpp"

namespace bnd {

__device__ __forceinline__ void wave_push_m(bool pred, uint32_t* ctr, uint32_t* arr, uint32_t val) {
    const uint64_t m = __ballot(pred);
    if (m == 0) return;
    const int leader = __ffsll((unsigned long long)m) - 1;
    uint32_t base = 0;
    if ((int)lane_id() == leader) base = atomicAdd(ctr, (uint32_t)__popcll(m));
    base = __shfl(base, leader);
    if (pred) arr[base + mbcnt(m)] = val;
}

// ErfInv of PSSMLT.fs:69-94 (Giles 2010 single-precision polynomial).
__device__ __forceinline__ float erf_inv(float x) {
    x = min_n(max_n(x, -0.99999f), 0.99999f);
    float w = -log_f(fmaf(x, -x, 1.0f));
    float p;
    if (w < 5.0f) {
        w = w - 2.5f;
        p = 2.81022636e-08f;
        p = fmaf(p, w, 3.43273939e-07f);
        p = fmaf(p, w, -3.5233877e-06f);
        p = fmaf(p, w, -4.39150654e-06f);
        p = fmaf(p, w, 0.00021858087f);
        p = fmaf(p, w, -0.00125372503f);
        p = fmaf(p, w, -0.00417768164f);
        p = fmaf(p, w, 0.246640727f);
        return fmaf(p, w, 1.50140941f) * x;
    }
    w = sqrtf(w) - 3.0f;
    p = -0.000200214257f;
    p = fmaf(p, w, 0.000100950558f);
    p = fmaf(p, w, 0.00134934322f);
    p = fmaf(p, w, -0.00367342844f);
    p = fmaf(p, w, 0.00573950773f);
    p = fmaf(p, w, -0.0076224613f);
    p = fmaf(p, w, 0.00943887047f);
    p = fmaf(p, w, 1.00167406f);
    return fmaf(p, w, 2.83297682f) * x;
}

// The catch-up mutation of a sample over n small steps (PSSMLT.fs:106-135):
// Gaussian in one draw, Kelemen one term per step.
__device__ __forceinline__ float gaussian_step(float u, float sigma, int n, float v) {
    const float ns = sqrtf(2.0f) * erf_inv(fmaf(2.0f, u, -1.0f));
    return fmaf(ns, sigma * sqrtf((float)n), v);
}
__device__ __forceinline__ float kelemen_term(float u, float a, float eps_max) {
    const float u1 = u - 0.5f;
    const float u2 = u1 < 0.0f ? 1.0f + 2.0f * u1 : 2.0f * u1;
    return copysignf(eps_max * exp_f(-a * u2), u1);
}

// MLTSampler of one chain (PSSMLT.fs:35-150), loaded into registers for one
// kernel and written back at the end.  FRESH: the first iteration of a new
// sampler (all samples are large-step draws in index order), which needs no
// sample storage.
template <bool FRESH>
struct ChainSampler {
    const MltBuf* M;
    uint32_t c;             // chain slot
    uint32_t inner;
    int cur, last_large, init;
    bool large;
    __device__ __forceinline__ void load(const MltBuf& m, uint32_t slot) {
        M = &m;
        c = slot;
        inner = m.inner[slot];
        if (!FRESH) {
            const int4 st = m.state[slot];
            cur = st.x; last_large = st.y; init = st.z; large = st.w != 0;
        }
    }
    __device__ __forceinline__ void store() const {
        M->inner[c] = inner;
        if (!FRESH) M->state[c] = make_int4(cur, last_large, init, large ? 1 : 0);
    }
    // StartIteration (PSSMLT.fs:58-61)
    __device__ __forceinline__ void start_iteration(float large_step_prob) {
        large = cur == 0 || lcg(inner) < large_step_prob;
        cur = cur + 1;
    }
    // The records of samples [i0, i0 + N), read together so that their loads
    // overlap: the initialised ones (below `init`; EnsureReady visits them in
    // index order, so `init` only grows past indices not read here).
    template <int N>
    __device__ __forceinline__ void fetch(int i0, float4 (&r)[N]) const {
#pragma unroll
        for (int j = 0; j < N; ++j)
            r[j] = !FRESH && i0 + j < init ? M->xs[(size_t)(i0 + j) * M->cap + c] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    // EnsureReady (PSSMLT.fs:68-136) of sample i, whose record `r` was fetched.
    __device__ __forceinline__ float ensure(int i, float4 r) {
        if (FRESH) return lcg(inner);
        float4* rec = M->xs + (size_t)i * M->cap + c;
        float v, vb;
        int lm, mb;
        if (init <= i) {
            v = 0.0f; vb = 0.0f; lm = 0; mb = 0;
            init = i + 1;
        } else {
            v = r.x; vb = r.y; lm = __float_as_int(r.z); mb = __float_as_int(r.w);
        }
        if (lm < last_large) { v = lcg(inner); lm = last_large; }
        vb = v; mb = lm;
        if (large) {
            v = lcg(inner);
        } else {
            float val;
            if (M->strategy == 0) {
                val = gaussian_step(lcg(inner), M->sigma, cur - lm, v);
            } else {
                val = v;
                const float a = log_f(M->eps_max / M->eps_min);
                for (int k = lm; k <= cur - 1; ++k) {
                    val = val + kelemen_term(lcg(inner), a, M->eps_max);
                }
            }
            v = val - floorf(val);
        }
        lm = cur;
        *rec = make_float4(v, vb, __int_as_float(lm), __int_as_float(mb));
        return v;
    }
};

// Chain set-up for chains [c0, c0+n): the outer sampler picks a bootstrap
// path through the alias table (PSSMLT.fs:286-290) whose seed starts a fresh
// MLTSampler.
__global__ void k_mlt_chain_init(MltBuf M, MltParamsDev p, const float* aprob, const int* aidx, int c0, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t chain = (uint32_t)(c0 + i);
    uint32_t outer = xxhash2((uint32_t)p.frame_id, chain);
    // AliasTable.Sample (AliasTable.fs:52-62), index clamped to the table.
    const int nb = p.n_bootstrap;
    float u = lcg(outer) * (float)nb;
    int k = sat_int(u);
    k = k < nb - 1 ? k : nb - 1;
    k = k < 0 ? 0 : k;
    u = u - (float)k;
    const int bid = u < aprob[k] ? k : aidx[k];
    M.outer[i] = outer;
    M.bid[i] = bid;
    M.inner[i] = xxhash2((uint32_t)p.frame_id, (uint32_t)bid);
    M.state[i] = make_int4(0, 0, 0, 0);
    M.rad[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    M.accepted[i] = 0;
}

// StartIteration and the camera ray of one MLT path (PSSMLT.fs:254-266,
// 292-304, 333-345).  Bootstrap (FRESH) paths seed their own sampler.
template <bool FRESH>
__global__ __launch_bounds__(256) void k_mlt_start(DevScene S, PathBuf P, MltBuf M, MltParamsDev p, Ctl* ctl,
                                                   uint32_t* queue, int id0, int n) {
    for (int base = blockIdx.x * blockDim.x; base < n; base += gridDim.x * blockDim.x) {
        const int i = base + threadIdx.x;
        const bool ok = i < n;
        if (ok) {
            ChainSampler<FRESH> smp;
            if (FRESH) {
                smp.M = &M;
                smp.c = (uint32_t)i;
                smp.inner = xxhash2((uint32_t)p.frame_id, (uint32_t)(id0 + i));
            } else {
                smp.load(M, (uint32_t)i);
                smp.start_iteration(p.large_step_prob);
            }
            float4 rs[4];
            smp.fetch(0, rs);
            const float u0 = smp.ensure(0, rs[0]), u1 = smp.ensure(1, rs[1]);
            const float upx = u0 * (float)p.width, upy = u1 * (float)p.height;
            const int ix = min(p.width - 1, sat_int(upx));
            const int iy = min(p.height - 1, sat_int(upy));
            V2 frac = {upx - (float)ix, upy - (float)iy};
            V2 uLens;
            uLens.x = smp.ensure(2, rs[2]);
            uLens.y = smp.ensure(3, rs[3]);
            const Ray r = camera_ray(S, ix, iy, frac, uLens);
            P.o[i] = f4(r.o, 0.0f);
            P.d[i] = f4(r.d, 0.0f);
            P.beta[i] = make_float4(1.0f, 1.0f, 1.0f, 0.0f);
            P.L[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            M.pix_new[i] = iy * p.width + ix;
            smp.store();
        }
        wave_push_m(ok, &ctl->q_count[0], queue, (uint32_t)i);
    }
}

// NEE set-up, BSDF sampling and Russian roulette of one vertex from its seven
// primary samples (PSSMLT.fs:199-243).
struct MltVertex {
    bool shadow, cont;                // casts a shadow ray / the path continues
    V3 sh_d, nee_a, nee_b;            // shadow ray from g.p, factors of its NEE term
    float sh_t;
    V3 d, beta;                       // continuing ray from g.p
    float pdf;
};
__device__ __forceinline__ void mlt_scatter(const DevScene& S, const Ray& r, const Geom& g, int mat, V3 beta,
                                            float uLight, V2 uEmit, float uLobe, V2 uBSDF, float uRR, int depth,
                                            int max_depth, int rr_depth, MltVertex& v) {
    const Mat m = load_mat(S, mat);
    const V3 wo_l = to_local(g, -r.d);
    const LightSample ls = light_sample(S, g.p, uLight, uEmit);
    v.shadow = false;
    v.cont = false;
    if (ls.pdf != 0.0f) {
        const BSDF e = mat_eval(m, wo_l, to_local(g, ls.wi));
        const float dist = length(ls.p - g.p);
        v.sh_t = dist - 1e-3f;
        v.sh_d = ls.wi;
        v.nee_a = beta * e.f;
        v.nee_b = ls.L * rcp_e(e.pdf + ls.pdf);
        v.shadow = true;
    }
    V3 wi_l;
    const BSDF bs = mat_sample(m, wo_l, uLobe, uBSDF, wi_l);
    if (bs.pdf != 0.0f) {
        v.d = to_world(g, wi_l);
        beta = beta * bs.f * rcp_e(bs.pdf);
        v.cont = true;
        if (depth >= rr_depth) {
            const float q = min_n(1.0f, max_n(beta.x, max_n(beta.y, beta.z)));
            if (uRR < q) beta = beta * rcp_e(q);
            else v.cont = false;
        }
        v.beta = beta;
        v.pdf = bs.pdf;
    }
    v.cont = v.cont && depth + 1 < max_depth;
}

// PSSMLTIntegrator.Li after a closest hit (PSSMLT.fs:184-243): emission with
// MIS, then seven primary samples drawn for every hit, then NEE set-up, BSDF
// sampling and Russian roulette.  The NEE term is applied by trace_shadow.
template <bool FRESH>
__global__ __launch_bounds__(256) void k_shade_mlt(DevScene S, PathBuf P, MltBuf M, Ctl* ctl, const uint32_t* bins,
                                                   uint32_t bin_cap, uint32_t* queue_next, int nxt, uint32_t* shq,
                                                   uint32_t* sh_ctr, int depth, int max_depth, int rr_depth) {
    uint32_t start[kBins + 1];
    start[0] = 0;
    for (int b = 0; b < kBins; ++b) start[b + 1] = start[b] + ctl->bin_count[b];
    const uint32_t total = start[kBins];
    for (uint32_t base = blockIdx.x * blockDim.x; base < total; base += gridDim.x * blockDim.x) {
        const uint32_t i = base + threadIdx.x;
        bool cont = false, shadow = false;
        uint32_t slot = 0;
        if (i < total) {
            int b = 0;
            while (i >= start[b + 1]) ++b;
            slot = bins[(size_t)b * bin_cap + (i - start[b])];
            const float4 o4 = P.o[slot], d4 = P.d[slot];
            const Ray r = {xyz(o4), xyz(d4)};
            const float prev_pdf = d4.w;
            const int4 h = P.hit[slot];
            const Geom g = hit_geometry(S, r, h.x, h.y, __int_as_float(h.z));
            const int4 info = S.insts[h.x].info;
            V3 L = xyz(P.L[slot]);
            V3 beta = xyz(P.beta[slot]);
            if (info.w >= 0) {
                V3 Le;
                float lpdf;
                light_eval(S, h.x, r.o, g, Le, lpdf);
                const float w = depth == 0 ? 1.0f : prev_pdf * rcp_e(lpdf + prev_pdf);
                L = fma3(beta, Le * w, L);
            }
            ChainSampler<FRESH> smp;
            smp.load(M, slot);
            const int s0 = 4 + 7 * depth;
            float4 rs[7];
            smp.fetch(s0, rs);
            const float uLight = smp.ensure(s0, rs[0]);
            V2 uEmit;
            uEmit.x = smp.ensure(s0 + 1, rs[1]);
            uEmit.y = smp.ensure(s0 + 2, rs[2]);
            const float uLobe = smp.ensure(s0 + 3, rs[3]);
            V2 uBSDF;
            uBSDF.x = smp.ensure(s0 + 4, rs[4]);
            uBSDF.y = smp.ensure(s0 + 5, rs[5]);
            const float uRR = smp.ensure(s0 + 6, rs[6]);
            smp.store();
            if (info.z >= 0) {
                MltVertex v;
                mlt_scatter(S, r, g, info.z, beta, uLight, uEmit, uLobe, uBSDF, uRR, depth, max_depth, rr_depth, v);
                shadow = v.shadow;
                cont = v.cont;
                if (shadow) {
                    P.sh_o[slot] = f4(g.p, v.sh_t);
                    P.sh_d[slot] = f4(v.sh_d, 0.0f);
                    P.nee_a[slot] = f4(v.nee_a, 0.0f);
                    P.nee_b[slot] = f4(v.nee_b, 0.0f);
                }
                if (cont) {
                    P.o[slot] = f4(g.p, 0.0f);
                    P.d[slot] = f4(v.d, v.pdf);
                    P.beta[slot] = f4(v.beta, 0.0f);
                }
            }
            P.L[slot] = f4(L, 0.0f);
        }
        wave_push_m(cont, &ctl->q_count[nxt], queue_next, slot);
        wave_push_m(shadow, sh_ctr, shq, slot);
    }
}

__device__ __forceinline__ float luminance(V3 L) { return dot(L, mk(0.2126f, 0.7152f, 0.0722f)); }

// Bootstrap weight y = luminance(L) (PSSMLT.fs:268-273).
__global__ void k_mlt_boot_done(PathBuf P, float* weights, int id0, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const V3 L = xyz(P.L[i]) * rcp_e(1.0f);
    weights[id0 + i] = luminance(L);
}

// End of the replayed bootstrap path of a chain (PSSMLT.fs:306-312): keep
// L, y and the pixel, Accept(), and re-seed the inner sampler.
__global__ void k_mlt_replay_done(PathBuf P, MltBuf M, MltParamsDev p, int c0, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const V3 L = xyz(P.L[i]) * rcp_e(1.0f);
    M.Lcur[i] = f4(L, luminance(L));
    M.pix_cur[i] = M.pix_new[i];
    int4 st = M.state[i];
    if (st.w) st.y = st.x;                                  // Accept(): LastLargeStepIteration
    M.state[i] = st;
    M.inner[i] = xxhash3((uint32_t)(c0 + i), (uint32_t)M.bid[i], (uint32_t)p.frame_id);
}

__device__ __forceinline__ void film_add(float* film, const MltParamsDev& p, int pix, V3 c) {
    const int x = pix % p.width, y = pix / p.width;
    float* f = film + 3 * ((size_t)(p.height - y - 1) * p.width + x);     // Film.fs:50
    atomicAdd(f, c.x);
    atomicAdd(f + 1, c.y);
    atomicAdd(f + 2, c.z);
}

// Metropolis acceptance of one mutation (PSSMLT.fs:347-373).
// PrimarySample.Restore (PSSMLT.fs:31-33): Value = ValueBackUp,
// LastModification = ModificationBackUp.
__device__ __forceinline__ void restore_sample(float4* rec, float4 r) {
    if (__float_as_uint(r.x) != __float_as_uint(r.y) || __float_as_uint(r.z) != __float_as_uint(r.w))
        *rec = make_float4(r.y, r.y, r.w, r.w);
}

__global__ void k_mlt_accept(PathBuf P, MltBuf M, MltParamsDev p, float* film, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const V3 Ln = xyz(P.L[i]) * rcp_e(1.0f);
    const float yn = luminance(Ln);
    const float4 lc = M.Lcur[i];
    const V3 Lc = xyz(lc);
    const float y = lc.w;
    int4 st = M.state[i];
    const bool large = st.w != 0;
    const float a = min_n(1.0f, yn / y);
    const float w_old = (1.0f - a) / fmaf(y, p.inv_b, p.large_step_prob);
    V3 rad = xyz(M.rad[i]) + w_old * Lc;
    const float w_new = (a + (large ? 1.0f : 0.0f)) / fmaf(yn, p.inv_b, p.large_step_prob);
    uint32_t outer = M.outer[i];
    if (lcg(outer) < a) {
        M.accepted[i] = M.accepted[i] + 1;
        film_add(film, p, M.pix_cur[i], rad * p.inv_eff);
        rad = w_new * Ln;
        M.pix_cur[i] = M.pix_new[i];
        M.Lcur[i] = f4(Ln, yn);
        if (large) st.y = st.x;                              // Accept()
    } else {
        if (a > 0.0f) film_add(film, p, M.pix_new[i], (w_new * p.inv_eff) * Ln);
        // Reject(): restore every initialised sample, step the iteration back.
        // Eight records in flight per lane; a record that already equals its
        // backup is left unwritten.
        float4* rec = M.xs + i;
        const size_t stride = M.cap;
        int k = 0;
        for (; k + 8 <= st.z; k += 8) {
            float4 r[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) r[j] = rec[(size_t)(k + j) * stride];
#pragma unroll
            for (int j = 0; j < 8; ++j) restore_sample(rec + (size_t)(k + j) * stride, r[j]);
        }
        for (; k < st.z; ++k) restore_sample(rec + (size_t)k * stride, rec[(size_t)k * stride]);
        st.x = st.x - 1;
    }
    M.outer[i] = outer;
    M.rad[i] = f4(rad, 0.0f);
    M.state[i] = st;
}

// ------------------------------------------------- one wave per chain
// Few chains leave the wavefront above latency-bound: each of a mutation's
// bounces is six launches for a handful of waves.  Here a wave owns a chain
// and runs its mutations one after the other without leaving the kernel.  All
// lanes hold the path (the same values: no divergence, one memory
// transaction); what a mutation does many times over is spread over them: the
// samples of a vertex are mutated side by side, eight lanes each, and a
// rejection restores 64 samples at a time.  The primary samples live in LDS
// for the launch.
//
// The draws of a sample depend on its own record only through their number, so
// every sample's first random state is known from a prefix sum, by skipping
// the LCG ahead; terms are added in the reference's order, so a chain's
// trajectory is that of the wavefront, bit for bit.
__device__ __forceinline__ uint32_t lcg_skip(uint32_t s, uint32_t n) {
    uint32_t a = 0x000343fdu, c = 0x00269ec3u;               // s -> a*s + c, squared step by step
    while (__ballot(n != 0) != 0) {
        if (n & 1) s = a * s + c;
        c = (a + 1u) * c;
        a = a * a;
        n >>= 1;
    }
    return s;
}
template <int LANE>
__device__ __forceinline__ float group_lane(float v) {       // lane LANE of each group of eight
    return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), (LANE << 5) | 0x18));
}
struct WaveChain {
    const MltBuf& M;
    float4* xs;             // LDS: the chain's records
    float log_ratio;        // ln(eps_max / eps_min)
    uint32_t inner;
    int cur, last_large, init;
    bool large;
    // EnsureReady of samples [s0, s0 + N), N <= 8, in order; group g of eight
    // lanes holds sample s0 + g.  Returns the lane's group's value.
    __device__ __forceinline__ float ensure(int s0, int N) {
        const int lane = (int)lane_id(), g = lane >> 3, q = lane & 7;
        const int i = s0 + g;
        const bool mine = g < N;
        float v = 0.0f;
        int lm = 0;
        if (mine && i < init) {
            const float4 r = xs[i];
            v = r.x; lm = __float_as_int(r.z);
        }
        const bool stale = lm < last_large;                  // catch up with the last large step first
        lm = stale ? last_large : lm;
        const int steps = large || M.strategy == 0 ? 1 : max(cur - lm, 0);
        const uint32_t draws = mine ? (uint32_t)((stale ? 1 : 0) + steps) : 0u;
        uint32_t before = 0, total = 0;
        for (int k = 0; k < N; ++k) {
            const uint32_t d = (uint32_t)__builtin_amdgcn_readlane((int)draws, 8 * k);
            if (k < g) before += d;
            total += d;
        }
        uint32_t rng = lcg_skip(inner, before);
        inner = lcg_skip(inner, total);
        if (mine && stale) v = lcg(rng);
        const float vb = v;
        const int mb = lm;
        if (large) {
            v = lcg(rng);
        } else {
            float val = v;
            if (M.strategy == 0) {
                val = gaussian_step(lcg(rng), M.sigma, cur - lm, v);
            } else {
                // lane q computes terms q, q + 8, ... of its group's sample
                for (int k = 0; k < q; ++k) (void)lcg(rng);
                for (int k = 0; __ballot(mine && k < steps) != 0; k += 8) {
                    uint32_t r = rng;
                    const float t = kelemen_term(lcg(r), log_ratio, M.eps_max);
                    for (int j = 0; j < 8; ++j) (void)lcg(rng);
                    const int left = steps - k;
                    float u;
                    u = group_lane<0>(t); val = left > 0 ? val + u : val;
                    u = group_lane<1>(t); val = left > 1 ? val + u : val;
                    u = group_lane<2>(t); val = left > 2 ? val + u : val;
                    u = group_lane<3>(t); val = left > 3 ? val + u : val;
                    u = group_lane<4>(t); val = left > 4 ? val + u : val;
                    u = group_lane<5>(t); val = left > 5 ? val + u : val;
                    u = group_lane<6>(t); val = left > 6 ? val + u : val;
                    u = group_lane<7>(t); val = left > 7 ? val + u : val;
                }
            }
            v = val - floorf(val);
        }
        if (mine && q == 0) xs[i] = make_float4(v, vb, __int_as_float(cur), __int_as_float(mb));
        wave_sync();
        init = max(init, s0 + N);
        return v;
    }
    __device__ __forceinline__ float of(float v, int g) const {     // group g's value, in every lane
        return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 8 * g));
    }
};

constexpr int kMltWaveK = 16;
// `mutations` mutations of each of the chains [0, n) (PSSMLT.fs:333-373).
// WAVES per SIMD: alone on its SIMD a wave may use every register; where there
// are more chains than SIMDs four waves share one, at 128 VGPRs, with spills
// (1024 chains: 63.5 ms alone, 67.9 ms with four; 16384: 47.1 and 36.6 ms).
template <int WAVES, int MODE>
__global__ __launch_bounds__(64, WAVES) void k_mlt_wave_chains(DevScene S, MltBuf M, MltParamsDev p, float* film,
                                                           uint32_t* spill, size_t spill_stride, int n,
                                                           int mutations, int nx, int max_depth, int rr_depth) {
    extern __shared__ float4 xs[];
    __shared__ uint32_t stk[kMltWaveK * 64];
    const int lane = (int)lane_id();
    Traversal<kMltWaveK, MODE, 64> tr;
    tr.st = LaneStack<kMltWaveK, 64>{stk + lane, spill, (uint32_t)spill_stride, blockIdx.x * 64u + (uint32_t)lane, 0};
    tr.clear();
    tr.G.set(S);
    __shared__ uint8_t order[MODE == kList ? sizeof(FlatScene::order) : 1];
    if (MODE == kList) {
        for (int k = lane; k < (int)sizeof order; k += 64) order[k] = S.flat->order[k / kFlatMax][k % kFlatMax];
        tr.order = order;
        wave_sync();
    }
    // a whole traversal of one ray, the same in every lane
    auto trace = [&](const Ray& r, float tmax, bool any) {
        tr.start(r, tmax, S.exact_only != 0);
        if (MODE == kList) tr.take_instances_wave(any);
        else tr.take_tlas_root();
        if (!(tmax == tmax)) tr.empty();
        if constexpr (MODE == kList)
            if (any) return tr.any_hit_wave(stk, kMltWaveK * 64);
        bool found = false;
        while (tr.step_fast(any, found)) {}
        if (any) tr.clear();
        return found;
    };
    for (int c = blockIdx.x; c < n; c += gridDim.x) {
        WaveChain smp{M, xs, log_f(M.eps_max / M.eps_min), M.inner[c]};
        int4 st = M.state[c];
        smp.cur = st.x; smp.last_large = st.y; smp.init = st.z; smp.large = st.w != 0;
        for (int k = lane; k < nx; k += 64)
            xs[k] = k < smp.init ? M.xs[(size_t)k * M.cap + c] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        wave_sync();
        uint32_t outer = M.outer[c];
        float4 lc = M.Lcur[c];
        V3 rad = xyz(M.rad[c]);
        int pix_cur = M.pix_cur[c], accepted = M.accepted[c];
        for (int m = 0; m < mutations; ++m) {
            // StartIteration and the camera ray (PSSMLT.fs:58-61, 333-345)
            smp.large = smp.cur == 0 || lcg(smp.inner) < p.large_step_prob;
            smp.cur = smp.cur + 1;
            const float u = smp.ensure(0, 4);
            const float upx = smp.of(u, 0) * (float)p.width, upy = smp.of(u, 1) * (float)p.height;
            const int ix = min(p.width - 1, sat_int(upx)), iy = min(p.height - 1, sat_int(upy));
            Ray r = camera_ray(S, ix, iy, V2{upx - (float)ix, upy - (float)iy}, V2{smp.of(u, 2), smp.of(u, 3)});
            const int pix_new = iy * p.width + ix;
            V3 L = mk(0, 0, 0), beta = mk(1, 1, 1);
            float prev_pdf = 0.0f;
            for (int depth = 0; depth < max_depth; ++depth) {
                trace(r, kInf, false);
                if (tr.hit_inst < 0) break;
                const Geom g = hit_geometry(S, r, tr.hit_inst, tr.prim_of(S.insts[tr.hit_inst].info), tr.t);
                const int4 info = S.insts[tr.hit_inst].info;
                if (info.w >= 0) {
                    V3 Le;
                    float lpdf;
                    light_eval(S, tr.hit_inst, r.o, g, Le, lpdf);
                    const float w = depth == 0 ? 1.0f : prev_pdf * rcp_e(lpdf + prev_pdf);
                    L = fma3(beta, Le * w, L);
                }
                const float s = smp.ensure(4 + 7 * depth, 7);
                if (info.z < 0) break;
                MltVertex v;
                mlt_scatter(S, r, g, info.z, beta, smp.of(s, 0), V2{smp.of(s, 1), smp.of(s, 2)}, smp.of(s, 3),
                            V2{smp.of(s, 4), smp.of(s, 5)}, smp.of(s, 6), depth, max_depth, rr_depth, v);
                if (v.shadow && !trace({g.p, v.sh_d}, v.sh_t, true)) L = fma3(v.nee_a, v.nee_b, L);
                if (!v.cont) break;
                r = {g.p, v.d};
                beta = v.beta;
                prev_pdf = v.pdf;
            }
            const V3 Ln = L * rcp_e(1.0f);
            const float yn = luminance(Ln), y = lc.w;
            const V3 Lc = xyz(lc);
            const float a = min_n(1.0f, yn / y);
            const float w_old = (1.0f - a) / fmaf(y, p.inv_b, p.large_step_prob);
            rad = rad + w_old * Lc;
            const float w_new = (a + (smp.large ? 1.0f : 0.0f)) / fmaf(yn, p.inv_b, p.large_step_prob);
            if (lcg(outer) < a) {
                ++accepted;
                if (lane == 0) film_add(film, p, pix_cur, rad * p.inv_eff);
                rad = w_new * Ln;
                pix_cur = pix_new;
                lc = f4(Ln, yn);
                if (smp.large) smp.last_large = smp.cur;         // Accept()
            } else {
                if (a > 0.0f && lane == 0) film_add(film, p, pix_new, (w_new * p.inv_eff) * Ln);
                for (int k = lane; k < smp.init; k += 64) {      // Reject()
                    const float4 q = xs[k];
                    xs[k] = make_float4(q.y, q.y, q.w, q.w);
                }
                wave_sync();
                smp.cur = smp.cur - 1;
            }
        }
        for (int k = lane; k < smp.init; k += 64) M.xs[(size_t)k * M.cap + c] = xs[k];
        if (lane == 0) {
            M.inner[c] = smp.inner;
            M.state[c] = make_int4(smp.cur, smp.last_large, smp.init, smp.large ? 1 : 0);
            M.outer[c] = outer;
            M.Lcur[c] = lc;
            M.rad[c] = f4(rad, 0.0f);
            M.pix_cur[c] = pix_cur;
            M.accepted[c] = accepted;
        }
    }
}

// Final Film.Accumulate of a chain (PSSMLT.fs:375).
__global__ void k_mlt_finish(MltBuf M, MltParamsDev p, float* film, int* accepted_out, int c0, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    film_add(film, p, M.pix_cur[i], xyz(M.rad[i]) * p.inv_eff);
    accepted_out[c0 + i] = M.accepted[i];
}

// ------------------------------------------------------------------ launch
static int blocks(int n) { return (n + 255) / 256; }
void launch_mlt_chain_init(const MltBuf& M, const MltParamsDev& p, const float* aprob, const int* aidx, int c0, int n,
                           hipStream_t st) {
    hipLaunchKernelGGL(k_mlt_chain_init, dim3(blocks(n)), dim3(256), 0, st, M, p, aprob, aidx, c0, n);
}
void launch_mlt_start(bool fresh, const DevScene& S, const PathBuf& P, const MltBuf& M, const MltParamsDev& p,
                      Ctl* ctl, uint32_t* queue, int id0, int n, int grid, hipStream_t st) {
    const int g = min(grid, blocks(n));
    if (fresh) hipLaunchKernelGGL(k_mlt_start<true>, dim3(g), dim3(256), 0, st, S, P, M, p, ctl, queue, id0, n);
    else hipLaunchKernelGGL(k_mlt_start<false>, dim3(g), dim3(256), 0, st, S, P, M, p, ctl, queue, id0, n);
}
void launch_shade_mlt(bool fresh, const DevScene& S, const PathBuf& P, const MltBuf& M, Ctl* ctl,
                      const uint32_t* bins, uint32_t bin_cap, uint32_t* queue_next, int nxt, uint32_t* shq,
                      int depth, int max_depth, int rr_depth, int grid, hipStream_t st, int par) {
    uint32_t* sh_ctr = par < 0 ? &ctl->sh_count : &ctl->shc[par];
    if (fresh)
        hipLaunchKernelGGL(k_shade_mlt<true>, dim3(grid), dim3(256), 0, st, S, P, M, ctl, bins, bin_cap, queue_next,
                           nxt, shq, sh_ctr, depth, max_depth, rr_depth);
    else
        hipLaunchKernelGGL(k_shade_mlt<false>, dim3(grid), dim3(256), 0, st, S, P, M, ctl, bins, bin_cap, queue_next,
                           nxt, shq, sh_ctr, depth, max_depth, rr_depth);
}
void launch_mlt_boot_done(const PathBuf& P, float* weights, int id0, int n, hipStream_t st) {
    hipLaunchKernelGGL(k_mlt_boot_done, dim3(blocks(n)), dim3(256), 0, st, P, weights, id0, n);
}
void launch_mlt_replay_done(const PathBuf& P, const MltBuf& M, const MltParamsDev& p, int c0, int n, hipStream_t st) {
    hipLaunchKernelGGL(k_mlt_replay_done, dim3(blocks(n)), dim3(256), 0, st, P, M, p, c0, n);
}
void launch_mlt_accept(const PathBuf& P, const MltBuf& M, const MltParamsDev& p, float* film, int n, hipStream_t st) {
    hipLaunchKernelGGL(k_mlt_accept, dim3(blocks(n)), dim3(256), 0, st, P, M, p, film, n);
}
void launch_mlt_finish(const MltBuf& M, const MltParamsDev& p, float* film, int* accepted, int c0, int n,
                       hipStream_t st) {
    hipLaunchKernelGGL(k_mlt_finish, dim3(blocks(n)), dim3(256), 0, st, M, p, film, accepted, c0, n);
}

void launch_mlt_wave_chains(const DevScene& S, const MltBuf& M, const MltParamsDev& p, float* film, const Buffers& B,
                            int n, int mutations, int max_depth, int rr_depth, int n_simd, int grid,
                            hipStream_t st) {
    const int nx = 4 + 7 * max_depth;
    const size_t lds = (size_t)nx * sizeof(float4);
    const bool alone = n <= n_simd;
    auto* run = alone ? k_mlt_wave_chains<1, kNodes> : k_mlt_wave_chains<4, kNodes>;
    if (S.mode == kRecs) run = alone ? k_mlt_wave_chains<1, kRecs> : k_mlt_wave_chains<4, kRecs>;
    if (S.mode == kList) run = alone ? k_mlt_wave_chains<1, kList> : k_mlt_wave_chains<4, kList>;
    hipLaunchKernelGGL(run, dim3(min(n, grid)), dim3(64), lds, st, S, M, p, film, B.spill, B.spill_stride, n, mutations,
                       nx, max_depth, rr_depth);
}

}  // namespace bnd
