// Monte Carlo collisions of a kinetic species with a background material on the device
// (collisions/MCC.java:167-297): constant cross-section (Sigma.SigmaConst), charge exchange
// (ModelCEX) or elastic (ModelMEX) scattering.  One pass visits every particle slot once; the
// random draws come from Philox4x32-10 keyed by the seed and indexed by (particle id, step), so a
// particle's fate does not depend on the order or the thread it is processed in.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "sf_particle_math.h"
#include "sf_rng.h"

namespace sf {

// Field2D.gather with the gather_safe fallback (Field2D.java:300-390) on an FP64 node field.
__device__ __forceinline__ double gather_node(const MeshP& m, const double* __restrict__ f, double fi, double fj) {
    int i = (int)fi, j = (int)fj;
    double di = fi - i, dj = fj - j;
    auto at = [&](int a, int b) { return f[(size_t)b * m.ni + a]; };
    if (i < 0 || j < 0 || i + 1 >= m.ni || j + 1 >= m.nj) {
        if (i < 0) { i = 0; di = 0; }
        if (j < 0) { j = 0; dj = 0; }
        if (i >= m.ni - 1) { i = m.ni - 1; di = 0; }
        if (j >= m.nj - 1) { j = m.nj - 1; dj = 0; }
        double v = (1 - di) * (1 - dj) * at(i, j);
        if (di > 0) v += di * (1 - dj) * at(i + 1, j);
        if (di > 0 && dj > 0) v += di * dj * at(i + 1, j + 1);
        if (dj > 0) v += (1 - di) * dj * at(i, j + 1);
        return v;
    }
    double v = (1 - di) * (1 - dj) * at(i, j);
    v += di * (1 - dj) * at(i + 1, j);
    v += di * dj * at(i + 1, j + 1);
    v += (1 - di) * dj * at(i, j + 1);
    return v;
}

struct MccTarget {
    const double *den, *u, *v, *w, *T;
};
struct MccParams {
    double sigma, dt, source_mass, target_mass, max_T, mpw;
    int model;   // 0 CEX, 1 MEX
    uint32_t k0, k1, step, tag;
};

// MCC.perform's body for one particle slot; returns the number of collisions (0 or 1).
__device__ __forceinline__ unsigned int mcc_particle(const MeshP& m, const PState& s, int64_t p, const MccTarget& tg,
                                                     const MccParams& pp, unsigned long long* __restrict__ count,
                                                     double* __restrict__ S) {
    const int32_t c = s.cell[p];
    if (c < 0) return 0;   // hole left by a dead particle
    const double lc0 = cell_i(c) + (double)s.fx[p], lc1 = cell_j(c) + (double)s.fy[p];
    const double den_a = gather_node(m, tg.den, lc0, lc1);
    if (den_a <= 0) return 0;
    // Material.sampleVelocity: the target's stream velocity at the particle
    const double t0 = gather_node(m, tg.u, lc0, lc1), t1 = gather_node(m, tg.v, lc0, lc1),
                 t2 = gather_node(m, tg.w, lc0, lc1);
    double v0 = s.vx[p], v1 = s.vy[p], v2 = s.vz[p];
    const double g0 = t0 - v0, g1 = t1 - v1, g2 = t2 - v2;
    const double g = sqrt(g0 * g0 + g1 * g1 + g2 * g2);
    const double P = 1 - exp(-pp.sigma * g * pp.dt * den_a);
    ParticleRng rng{pp.k0, pp.k1, (uint32_t)s.id[p], pp.step, pp.tag};
    if (P < rng.draw(0)) return 0;   // no collision
    // Material.sampleMaxwellianVelocity(mesh, lc, 0, max_T) with Utils.SampleMaxw3D
    double T = gather_node(m, tg.T, lc0, lc1);
    if (T < 0) T = 0;
    if (pp.max_T > 0 && T > pp.max_T) T = pp.max_T;
    const double vth = sqrt(2 * K_B * T / pp.target_mass);
    const double sh = sqrt(0.5);
    // draws 2..13, 14..25 and 26..37: one component each
    const double x0 = t0 + (vth * 1.2) * (sh * 1 * ((rng.sum12(2) - 0.5 * 12) * 1.0));
    const double x1 = t1 + (vth * 1.2) * (sh * 1 * ((rng.sum12(14) - 0.5 * 12) * 1.0));
    const double x2 = t2 + (vth * 1.2) * (sh * 1 * ((rng.sum12(26) - 0.5 * 12) * 1.0));
    const double E1 = 0.5 * pp.source_mass * sqrt(v0 * v0 + v1 * v1 + v2 * v2);
    if (pp.model == 0) {   // ModelCEX: the ion takes the neutral's velocity
        v0 = x0;
        v1 = x1;
        v2 = x2;
    } else {               // ModelMEX: isotropic scattering in the centre-of-mass frame
        const double rm1 = pp.source_mass / (pp.source_mass + pp.target_mass);
        const double rm2 = pp.target_mass / (pp.source_mass + pp.target_mass);
        const double h0 = v0 - x0, h1 = v1 - x1, h2 = v2 - x2;
        const double gm = sqrt(h0 * h0 + h1 * h1 + h2 * h2);
        const double c0 = rm1 * v0 + rm2 * x0, c1 = rm1 * v1 + rm2 * x1, c2 = rm1 * v2 + rm2 * x2;
        const double B = 2. * rng.draw(38) - 1.0;
        const double A = sqrt(1. - B * B);
        const double C = 2. * M_PI * rng.draw(39);
        v0 = c0 + (B * gm) * rm2;
        v1 = c1 + (A * cos(C) * gm) * rm2;
        v2 = c2 + (A * sin(C) * gm) * rm2;
    }
    const float f0 = (float)v0, f1 = (float)v1, f2 = (float)v2;
    s.vx[p] = f0;
    s.vy[p] = f1;
    s.vz[p] = f2;
    const double E2 = 0.5 * pp.source_mass * sqrt(v0 * v0 + v1 * v1 + v2 * v2);
    const double dS = pp.mpw * (E1 - E2) / (pp.dt * node_vol_at(m, lc0, lc1));
    // target.getS(mesh).scatter(lc, dS) (Field2D.scatter, Field2D.java:244-295)
    const int si = (int)lc0, sj = (int)lc1;
    if (!(si < 0 || sj < 0 || si >= m.ni - 1 || sj >= m.nj - 1)) {
        double w[4];
        scatter_weights(m, si, sj, lc0 - si, lc1 - sj, w);
        atomicAdd(S + (size_t)sj * m.ni + si, w[0] * dS);
        atomicAdd(S + (size_t)sj * m.ni + si + 1, w[1] * dS);
        atomicAdd(S + (size_t)(sj + 1) * m.ni + si + 1, w[2] * dS);
        atomicAdd(S + (size_t)(sj + 1) * m.ni + si, w[3] * dS);
    }
    atomicAdd(count + (size_t)sj * m.ni + si, 1ull);   // col-count-sum at node ((int)lc0, (int)lc1)
    return 1;
}

// Largest target density and largest |u|, |v|, |w| over the nodes, rounded up to FP32, as the bit
// patterns of non-negative floats (which order like the numbers).  A value that is not finite gives
// infinity.  Each workgroup leaves its maxima, the last one combines them and leaves the counter at zero
// for the next target (zero at first), so a target costs one launch.  Few workgroups with four nodes a
// thread in flight: a thousand would wait for their atomics on that counter (1024 x 512 nodes: 45 us
// with 1024 of them, 10 with these).
constexpr int MCC_BOUND_BLOCKS = 256;
constexpr int64_t MCC_BOUND_MIN = 1 << 18;   // particles (beyond a quarter of the nodes) for which a pass pays for the bound
struct MccBound {
    unsigned int bound[4], done;
    float part[MCC_BOUND_BLOCKS][4];
};
__global__ void __launch_bounds__(256) mcc_target_bounds(int64_t nn, MccTarget tg, MccBound* __restrict__ out) {
    __shared__ float red[4][4];
    __shared__ bool last;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    float b[4] = {0.f, 0.f, 0.f, 0.f};
    auto up = [](double x) {   // FP32 at least x
        const float f = (float)(x * (1.0 + 1e-6));
        return f <= 3e38f ? f : __int_as_float(0x7F800000);   // NaN and overflow: infinity
    };
    auto wave_max = [&]() {   // of b, each wave's into red
#pragma unroll
        for (int k = 0; k < 4; k++) {
            for (int o = 32; o > 0; o >>= 1) b[k] = fmaxf(b[k], __shfl_xor(b[k], o));
            if (lane == 0) red[k][wave] = b[k];
        }
        __syncthreads();
    };
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t u0 = blockIdx.x * (int64_t)256 + t; u0 < nn; u0 += 4 * stride) {
        double f[4][4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int64_t u = u0 + q * stride < nn ? u0 + q * stride : u0;
            f[q][0] = tg.den[u];
            f[q][1] = tg.u[u];
            f[q][2] = tg.v[u];
            f[q][3] = tg.w[u];
        }
#pragma unroll
        for (int q = 0; q < 4; q++) {
            b[0] = fmaxf(b[0], up(f[q][0] < 0 ? 0.0 : f[q][0]));
#pragma unroll
            for (int k = 1; k < 4; k++) b[k] = fmaxf(b[k], up(fabs(f[q][k])));
        }
    }
    wave_max();
    if (t < 4) out->part[blockIdx.x][t] = fmaxf(fmaxf(red[t][0], red[t][1]), fmaxf(red[t][2], red[t][3]));
    __threadfence();
    __syncthreads();
    if (t == 0) last = atomicAdd(&out->done, 1u) == gridDim.x - 1;
    __syncthreads();
    if (!last) return;
    __threadfence();   // the other workgroups' parts
    static_assert(MCC_BOUND_BLOCKS == 256, "one part a thread");
#pragma unroll
    for (int k = 0; k < 4; k++) b[k] = t < (int)gridDim.x ? out->part[t][k] : 0.f;
    wave_max();
    if (t < 4) out->bound[t] = __float_as_uint(fmaxf(fmaxf(red[t][0], red[t][1]), fmaxf(red[t][2], red[t][3])));
    if (t == 0) out->done = 0;
}

// Few particles collide in a pass (1e-5 to 1e-2 of them), and most are ruled out without the
// target's fields: P = 1 - exp(-x) <= x = sigma g dt n, n is at most the target's largest node
// density (a gather is a convex combination of nodes) and g at most |v| + |largest target
// velocity| by component, so a particle whose draw exceeds that bound does not collide.  Only the
// cell, the velocity and the id are read for it (20 B instead of 28 B and 16 FP64 node loads).  The
// bound is evaluated in FP32 with a margin (1e-4 relative, 1e-12 absolute) far above the rounding
// of either side, so no particle that the full test would collide is dropped.  The others are
// queued in LDS and take the full test (mcc_particle) together, so that its gathers run with full
// waves.  4e7 particles: 0.70 ms with the full test for every particle, 0.164 ms so: 4.9 TB/s
// of the 20 B.  (2e7 particles of which 2e-3, 2e-2 and 0.9 pass the bound: 1.43 -> 0.14, 3.2 -> 0.28 and
// 5.9 -> 4.7 ms; without the queue the collisions ran on a few lanes of each wave.)
// A workgroup tests SLOTS slots a thread at a time, 4 in 16-byte loads.  A population of at most a workgroup
// of 256 for every CU takes 1: the colliding particles of 1024 slots would take their workgroup four
// rounds while most CUs have none (1e4 particles that all collide: 42.0 us with 4, 26.6 with 1; 6.5e4 50
// and 41; 2e5, on more workgroups than CUs, 67 and 102).  So does a pass without a bound, which tests all
// of them (1024 x 512 nodes, 7e4 and 2.7e5 particles: 29 and 33 us, 42 with 4).
template <int SLOTS>
__global__ void __launch_bounds__(256) mcc_kernel(MeshP m, PState s, int64_t np, MccTarget tg, MccParams pp,
                                                  const MccBound* __restrict__ bounds, int bounded,
                                                  unsigned long long* __restrict__ count, double* __restrict__ S,
                                                  unsigned long long* __restrict__ ncol) {
    static_assert(SLOTS == 1 || SLOTS == 4, "slots of a thread");
    constexpr int CHUNK_SLOTS = 256 * SLOTS;
    __shared__ int64_t queue[CHUNK_SLOTS + 256];
    __shared__ int nq;
    const int t = threadIdx.x, lane = t & 63;
    const unsigned int* const bound = bounds->bound;
    const float inf = __int_as_float(0x7F800000);   // (rules out no particle)
    const float kx = bounded ? (float)(pp.sigma * pp.dt * 1.0001 * (double)__uint_as_float(bound[0])) : inf;
    const float tu = __uint_as_float(bound[1]), tv = __uint_as_float(bound[2]), tw = __uint_as_float(bound[3]);
    unsigned int ncol_local = 0;   // added to ncol once per wave
    if (t == 0) nq = 0;
    __syncthreads();
    for (int64_t c0 = (int64_t)blockIdx.x * CHUNK_SLOTS; c0 < np; c0 += (int64_t)gridDim.x * CHUNK_SLOTS) {
        // a chunk starts on a multiple of 1024 slots where a thread has 4, so those are 16-byte aligned
        const int64_t p0 = c0 + SLOTS * t;
        int4 c = make_int4(-1, -1, -1, -1), id = make_int4(0, 0, 0, 0);
        float4 vx = make_float4(0.f, 0.f, 0.f, 0.f), vy = vx, vz = vx;
        if (SLOTS == 1) {
            if (p0 < np) {
                c.x = s.cell[p0];
                id.x = s.id[p0];
                vx.x = s.vx[p0];
                vy.x = s.vy[p0];
                vz.x = s.vz[p0];
            }
        } else if (p0 + 3 < np) {
            c = *reinterpret_cast<const int4*>(s.cell + p0);
            id = *reinterpret_cast<const int4*>(s.id + p0);
            vx = *reinterpret_cast<const float4*>(s.vx + p0);
            vy = *reinterpret_cast<const float4*>(s.vy + p0);
            vz = *reinterpret_cast<const float4*>(s.vz + p0);
        } else if (p0 < np) {
            const int64_t p1 = min(p0 + 1, np - 1), p2 = min(p0 + 2, np - 1);
            c = make_int4(s.cell[p0], p0 + 1 < np ? s.cell[p1] : -1, p0 + 2 < np ? s.cell[p2] : -1, -1);
            id = make_int4(s.id[p0], s.id[p1], s.id[p2], 0);
            vx = make_float4(s.vx[p0], s.vx[p1], s.vx[p2], 0.f);
            vy = make_float4(s.vy[p0], s.vy[p1], s.vy[p2], 0.f);
            vz = make_float4(s.vz[p0], s.vz[p1], s.vz[p2], 0.f);
        }
        auto test = [&](int j, int32_t cj, int32_t idj, float ux, float uy, float uz) {
            // draw 0 is (o.y : o.x) >> 11 over 2^53, at least o.y / 2^32
            const uint4 o = philox4x32_10(make_uint4(0u, (uint32_t)idj, pp.step, pp.tag), pp.k0, pp.k1);
            const float gx = fabsf(ux) + tu, gy = fabsf(uy) + tv, gz = fabsf(uz) + tw;
            const float x = kx * sqrtf(gx * gx + gy * gy + gz * gz) + 1e-12f;
            const bool full = cj >= 0 && !((float)o.y * (0x1.0p-32f * 0.99999f) > x);
            const unsigned long long mk = __ballot(full);
            if (mk) {
                int base = 0;
                if (lane == 0) base = atomicAdd(&nq, __popcll(mk));
                base = __shfl(base, 0);
                if (full) queue[base + __popcll(mk & ((1ull << lane) - 1ull))] = p0 + j;
            }
        };
        test(0, c.x, id.x, vx.x, vy.x, vz.x);
        if (SLOTS > 1) {
            test(1, c.y, id.y, vx.y, vy.y, vz.y);
            test(2, c.z, id.z, vx.z, vy.z, vz.z);
            test(3, c.w, id.w, vx.w, vy.w, vz.w);
        }
        __syncthreads();
        // whole groups of 256 now, the rest with the next chunk's (or at the end)
        const bool last = c0 + (int64_t)gridDim.x * CHUNK_SLOTS >= np;
        const int n = nq;
        __syncthreads();   // every thread has n before the next chunk adds to nq
        if (n >= 256 || last) {
            const int done = last ? n : n / 256 * 256;
            for (int q = t; q < done; q += 256) ncol_local += mcc_particle(m, s, queue[q], tg, pp, count, S);
            const int rest = n - done;   // below 256
            const int64_t moved = t < rest ? queue[done + t] : 0;
            __syncthreads();
            if (t < rest) queue[t] = moved;
            if (t == 0) nq = rest;
            __syncthreads();
        }
    }
    for (int o = 32; o > 0; o >>= 1) ncol_local += __shfl_xor(ncol_local, o);
    if (lane == 0 && ncol_local) atomicAdd(ncol, (unsigned long long)ncol_local);
}

__global__ void mcc_fields_kernel(int64_t nn, int which, const unsigned long long* __restrict__ count,
                                  const double* __restrict__ S, const double* __restrict__ node_vol, double mpw,
                                  double inv_samples, double inv_time, double* __restrict__ out) {
    for (int64_t u = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; u < nn; u += (int64_t)gridDim.x * blockDim.x) {
        const double n = (double)count[u];
        double v;
        switch (which) {
            case 0: v = n; break;                                          // col-count-sum
            case 1: v = n * mpw; break;                                    // col-real-sum
            case 2: v = n * inv_samples; break;                            // col-count
            case 3: v = n * mpw * inv_time / node_vol[u]; break;           // nu
            default: v = S[u]; break;                                      // target S
        }
        out[u] = v;
    }
}

}  // namespace sf

using namespace sf;

struct sf_mcc {
    sf_ctx* ctx = nullptr;
    sf_mcc_desc desc{};
    double target_mass = 0;
    double* d_target = nullptr;          // [5][nn] den, u, v, w, T
    unsigned long long* d_count = nullptr;
    double* d_S = nullptr;
    unsigned long long* d_ncol = nullptr;
    unsigned long long* h_ncol = nullptr;   // pinned: the pass's count without a staged copy
    MccBound* d_bound = nullptr;         // bounds of the target's density and velocity (mcc_target_bounds)
    bool have_target = false;
    bool bounded = false;                // d_bound is the present target's
    int target_passes = 0;               // passes over the present target
    int num_samples = 0;
    double time_start = 0, time_last = 0;
    uint32_t stream_tag = 0;             // module-tagged counter word of the Philox streams
};

static MccTarget mcc_target(const sf_mcc* c, size_t nn) {
    return MccTarget{c->d_target, c->d_target + nn, c->d_target + 2 * nn, c->d_target + 3 * nn, c->d_target + 4 * nn};
}

static int grid_n(int64_t n, int max_blocks) {
    int64_t b = (n + 255) / 256;
    if (b < 1) b = 1;
    return (int)(b < max_blocks ? b : max_blocks);
}

// The bound of a target takes 6 to 10 us on a mesh up to 1024 x 512 and saves 13 ps a particle and pass: it
// is made with the target where a pass about pays for it, else at the target's second pass.  A host that
// sets the target before every pass waits for both (301 x 157 nodes, 7e4 and 2.7e5 particles: 137 and
// 140 us without the bound, 153 with); one that keeps it loses 1 to 4 us of the first pass.
static bool bound_pays(const sf_mcc* c) {
    return c->ctx->species[c->desc.source_species]->np >
           MCC_BOUND_MIN + (int64_t)c->ctx->mp.ni * c->ctx->mp.nj / 4;
}
static int make_bound(sf_mcc* c) {
    sf_ctx* ctx = c->ctx;
    const int64_t nn = (int64_t)ctx->mp.ni * ctx->mp.nj;
    hipLaunchKernelGGL(mcc_target_bounds, dim3(grid_n(nn, MCC_BOUND_BLOCKS)), dim3(256), 0, ctx->stream, nn,
                       mcc_target(c, (size_t)nn), c->d_bound);
    SF_HIP(ctx, hipGetLastError());
    c->bounded = true;
    return SF_OK;
}


extern "C" {

int sf_mcc_create(sf_ctx* ctx, const sf_mcc_desc* desc, sf_mcc** out) {
    SF_CHECK_CTX(ctx);
    if (!desc || !out) return sf_fail(ctx, SF_ERR_ARG, "sf_mcc_create: null argument");
    *out = nullptr;
    if (!ctx->mesh_ready) return sf_fail(ctx, SF_ERR_STATE, "sf_mcc_create: mesh not set up");
    if (desc->source_species < 0 || desc->source_species >= (int)ctx->species.size())
        return sf_fail(ctx, SF_ERR_ARG, "sf_mcc_create: no species %d", desc->source_species);
    if (!ctx->species[desc->source_species]->desc.track_ids)
        return sf_fail(ctx, SF_ERR_STATE, "sf_mcc_create: the source species must track particle ids");
    if (desc->model != SF_MCC_CEX && desc->model != SF_MCC_MEX)
        return sf_fail(ctx, SF_ERR_UNSUPPORTED, "sf_mcc_create: model %d is not supported", desc->model);
    if (!(desc->sigma >= 0) || !(desc->target_molwt > 0))
        return sf_fail(ctx, SF_ERR_ARG, "sf_mcc_create: sigma must be >= 0 and target_molwt > 0");
    uint32_t stream_tag = 0;
    {
        int rc = claim_stream(ctx, desc->seed, RNG_MODULE_MCC, desc->tag, &stream_tag);
        if (rc) return rc;
    }
    SF_HIP(ctx, hipSetDevice(ctx->device));
    const size_t nn = (size_t)ctx->mp.ni * ctx->mp.nj;
    sf_mcc* c = new sf_mcc();
    c->ctx = ctx;
    c->desc = *desc;
    c->stream_tag = stream_tag;
    if (c->desc.frequency < 1) c->desc.frequency = 1;
    c->target_mass = desc->target_molwt * AMU;
    hipError_t e = hipMalloc((void**)&c->d_target, 5 * nn * sizeof(double));
    if (e == hipSuccess) e = hipMalloc((void**)&c->d_count, nn * sizeof(unsigned long long));
    if (e == hipSuccess) e = hipMalloc((void**)&c->d_S, nn * sizeof(double));
    if (e == hipSuccess) e = hipMalloc((void**)&c->d_ncol, sizeof(unsigned long long));
    if (e == hipSuccess) e = hipHostMalloc((void**)&c->h_ncol, sizeof(unsigned long long));
    if (e == hipSuccess) e = hipMalloc((void**)&c->d_bound, sizeof(MccBound));
    if (e == hipSuccess) e = hipMemsetAsync(c->d_bound, 0, sizeof(MccBound), ctx->stream);
    if (e == hipSuccess) e = hipMemsetAsync(c->d_target, 0, 5 * nn * sizeof(double), ctx->stream);
    if (e == hipSuccess) e = hipMemsetAsync(c->d_count, 0, nn * sizeof(unsigned long long), ctx->stream);
    if (e == hipSuccess) e = hipMemsetAsync(c->d_S, 0, nn * sizeof(double), ctx->stream);
    if (e != hipSuccess) {
        hipFree(c->d_target);
        hipFree(c->d_count);
        hipFree(c->d_S);
        hipFree(c->d_ncol);
        hipHostFree(c->h_ncol);
        hipFree(c->d_bound);
        delete c;
        release_stream(ctx, desc->seed, stream_tag);
        return sf_fail(ctx, SF_ERR_HIP, "sf_mcc_create: %s", hipGetErrorString(e));
    }
    *out = c;
    return SF_OK;
}

int sf_mcc_destroy(sf_mcc* c) {
    if (!c) return SF_ERR_ARG;
    hipSetDevice(c->ctx->device);
    hipStreamSynchronize(c->ctx->stream);
    hipFree(c->d_target);
    hipFree(c->d_count);
    hipFree(c->d_S);
    hipFree(c->d_ncol);
    hipHostFree(c->h_ncol);
    hipFree(c->d_bound);
    release_stream(c->ctx, c->desc.seed, c->stream_tag);
    delete c;
    return SF_OK;
}

int sf_mcc_set_target(sf_mcc* c, const double* den, const double* u, const double* v, const double* w,
                      const double* temp) {
    if (!c) return SF_ERR_ARG;
    sf_ctx* ctx = c->ctx;
    if (!den) return sf_fail(ctx, SF_ERR_ARG, "sf_mcc_set_target: the target density is required");
    SF_HIP(ctx, hipSetDevice(ctx->device));
    const size_t nn = (size_t)ctx->mp.ni * ctx->mp.nj;
    SF_HIP(ctx, hipStreamSynchronize(ctx->stream));
    // (the copies wait for the device; the clears follow on the context's stream, which the bounds and the
    // next pass run on: a clear on the null stream would not be ordered before them)
    c->bounded = false;
    c->target_passes = 0;
    const double* src[5] = {den, u, v, w, temp};
    for (int k = 0; k < 5; k++) {
        if (src[k]) SF_HIP(ctx, hipMemcpy(c->d_target + k * nn, src[k], nn * sizeof(double), hipMemcpyHostToDevice));
        else SF_HIP(ctx, hipMemsetAsync(c->d_target + k * nn, 0, nn * sizeof(double), ctx->stream));
    }
    c->have_target = true;
    return bound_pays(c) ? make_bound(c) : SF_OK;
}

int sf_mcc_perform(sf_mcc* c, int it, double time, int64_t* collisions) {
    if (!c) return SF_ERR_ARG;
    sf_ctx* ctx = c->ctx;
    if (collisions) *collisions = 0;
    if (!c->have_target) return sf_fail(ctx, SF_ERR_STATE, "sf_mcc_perform: no target fields set");
    if (c->desc.stop_it > 0 && it > c->desc.stop_it) return SF_OK;
    if (it % c->desc.frequency != 0) return SF_OK;
    if (c->num_samples == 0) c->time_start = time;
    c->num_samples++;
    c->time_last = time;
    SF_HIP(ctx, hipSetDevice(ctx->device));
    Species* sp = ctx->species[c->desc.source_species];
    const size_t nn = (size_t)ctx->mp.ni * ctx->mp.nj;
    const MccTarget tg = mcc_target(c, nn);
    MccParams pp;
    pp.sigma = c->desc.sigma;
    pp.dt = c->desc.frequency * ctx->dt;
    pp.source_mass = sp->mass;
    pp.target_mass = c->target_mass;
    pp.max_T = c->desc.max_target_temp;
    pp.mpw = sp->desc.spwt;
    pp.model = c->desc.model;
    pp.k0 = (uint32_t)c->desc.seed;
    pp.k1 = (uint32_t)(c->desc.seed >> 32);
    pp.step = (uint32_t)it;
    pp.tag = c->stream_tag;
    SF_HIP(ctx, hipMemsetAsync(c->d_ncol, 0, sizeof(unsigned long long), ctx->stream));
    if (sp->np > 0) {
        if (!c->bounded && (c->target_passes > 0 || bound_pays(c))) {   // (the particles may have come later)
            const int rc = make_bound(c);
            if (rc) return rc;
        }
        c->target_passes++;
        auto pass = [&](auto kernel, int chunk) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)std::min<int64_t>((sp->np + chunk - 1) / chunk, 2048)), dim3(256), 0,
                               ctx->stream, ctx->mp, sp->buf[sp->cur], sp->np, tg, pp, (const MccBound*)c->d_bound,
                               (int)c->bounded, c->d_count, c->d_S, c->d_ncol);
        };
        if (!c->bounded || sp->np <= 256 * (int64_t)ctx->ncu) pass(mcc_kernel<1>, 256);
        else pass(mcc_kernel<4>, 1024);
        SF_HIP(ctx, hipGetLastError());
    }
    SF_HIP(ctx, hipMemcpyAsync(c->h_ncol, c->d_ncol, sizeof(unsigned long long), hipMemcpyDeviceToHost, ctx->stream));
    SF_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (collisions) *collisions = (int64_t)*c->h_ncol;
    return SF_OK;
}

int sf_mcc_field(sf_mcc* c, int which, double* out) {
    if (!c) return SF_ERR_ARG;
    sf_ctx* ctx = c->ctx;
    if (!out || which < 0 || which > 4) return sf_fail(ctx, SF_ERR_ARG, "sf_mcc_field: bad argument");
    SF_HIP(ctx, hipSetDevice(ctx->device));
    const int64_t nn = (int64_t)ctx->mp.ni * ctx->mp.nj;
    Species* sp = ctx->species[c->desc.source_species];
    double* d_out = nullptr;
    const int rc = field_workspace(ctx, &d_out);
    if (rc) return rc;
    // the reference divides by the sampling time without a guard (MCC.java:152-153)
    const double inv_samples = c->num_samples > 0 ? 1.0 / c->num_samples : 0.0;
    const double inv_time = 1.0 / (c->time_last - c->time_start);
    hipLaunchKernelGGL(mcc_fields_kernel, dim3(grid_n(nn, 8192)), dim3(256), 0, ctx->stream, nn, which,
                       (const unsigned long long*)c->d_count, (const double*)c->d_S, (const double*)ctx->d_node_vol,
                       sp->desc.spwt, inv_samples, inv_time, d_out);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(out, d_out, nn * sizeof(double), hipMemcpyDeviceToHost, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) return sf_fail(ctx, SF_ERR_HIP, "sf_mcc_field: %s", hipGetErrorString(e));
    return SF_OK;
}

int sf_mcc_clear_samples(sf_mcc* c, int clear_source) {
    if (!c) return SF_ERR_ARG;
    sf_ctx* ctx = c->ctx;
    SF_HIP(ctx, hipSetDevice(ctx->device));
    const size_t nn = (size_t)ctx->mp.ni * ctx->mp.nj;
    SF_HIP(ctx, hipMemsetAsync(c->d_count, 0, nn * sizeof(unsigned long long), ctx->stream));
    if (clear_source) SF_HIP(ctx, hipMemsetAsync(c->d_S, 0, nn * sizeof(double), ctx->stream));
    SF_HIP(ctx, hipStreamSynchronize(ctx->stream));
    c->num_samples = 0;
    return SF_OK;
}

}  // extern "C"
