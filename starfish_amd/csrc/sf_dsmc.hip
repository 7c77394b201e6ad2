// DSMC collisions on the device (collisions/DSMC.java:167-430): Bird's no-time-counter scheme
// per cell after the counting sort, with Boyd's weighting for two species, a constant or VHS
// (SigmaPlus.SigmaBird463) cross-section and the elastic VHS/VSS scattering of ModelElastic.
// A cell's particle list is the cell range of the sorted species, ordered by particle id
// (dsmc_order), so that the pair choice (an index into that list) and the cell's Philox
// stream give the same collisions on every run.  The pairs of a cell are processed in sequence, as
// in the reference, by one lane; a wave runs up to 64 cells (dsmc_collide).
#include <algorithm>
#include <cmath>
#include <vector>

#include "sf_particle_math.h"
#include "sf_rng.h"

namespace sf {

constexpr int DSMC_MAXP = 2048;   // binned particles of one species in one cell
// Ranges of at most DSMC_SMALL particles are ordered in the registers of one wave (8 keys a lane,
// 16 registers), longer ones by a workgroup in LDS: twice the keys would double the wave's registers
// and unrolled code for cells that few runs have.
constexpr int DSMC_SMALL = 512;

struct DsmcParams {
    int same, sigma_type;
    double c0, sigma0, ref_temp, vti, mr, gamma, vss_inv;
    double mass_a, mass_b, spwt_a, spwt_b, delta_t;
    uint32_t k0, k1, step, tag;
};

__device__ __forceinline__ double dsmc_sigma(const DsmcParams& pp, double g) {
    if (pp.sigma_type == 0) return pp.c0;
    return pp.sigma0 * pow(2. * K_B * pp.ref_temp / (pp.mr * g * g), pp.vti - 0.5) / pp.gamma;   // Bird eq. 4.63
}

// Particles of the cell that the reference bins into it: (int)lc inside the cells (a particle on
// the last node line has offset 1 in the last cell and is skipped, DSMC.java:206-214).
__device__ __forceinline__ bool dsmc_in_cell(const MeshP& m, const PState& s, int64_t p) {
    const int32_t c = s.cell[p];
    if (c < 0) return false;
    return cell_i(c) + (double)s.fx[p] < m.ni - 1 && cell_j(c) + (double)s.fy[p] < m.nj - 1;
}

// Number of binned particles in the cell range [a, b): the range length, except in the last
// cell row and column where particles may sit on the last node line.
__device__ int dsmc_count(const MeshP& m, const PState& s, int a, int b, bool edge) {
    if (!edge) return b - a;
    int n = 0;
    for (int p = a + (int)(threadIdx.x & 63); p < b; p += 64) n += dsmc_in_cell(m, s, p) ? 1 : 0;
    for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o);
    return n;
}

// What the collision loop of a cell needs from dsmc_order: the number of candidate pairs (0: none)
// and of binned particles of each species.
struct DsmcCell {
    int nsel, n1, n2;
};
// What a pass counts, zero before it: one clear and one readback (into pinned memory) for all three.
struct DsmcStatus {
    unsigned long long ncol;   // collisions
    int overflow;              // most particles of a cell that was refused (0: none)
    int nbig;                  // cells in the list that dsmc_order_big orders
};

// Slots of the binned particles of [a, b), ordered by id, into order[a ..), for ranges of at most
// 64 E particles: a bitonic sort of (id << 32 | slot) in registers.  Element i of the list is
// register i % E of lane i / E, so strides below E stay in a lane and the others are one 64-bit
// shuffle; padding is all-ones.
template <int E>
__device__ __forceinline__ void order_in_registers(const MeshP& m, const PState& s, int a, int b,
                                                   int32_t* __restrict__ order) {
    constexpr int LE = E == 1 ? 0 : (E == 2 ? 1 : (E == 4 ? 2 : 3));
    static_assert((1 << LE) == E, "E is 1, 2, 4 or 8");
    const int lane = threadIdx.x & 63;
    unsigned long long k[E];
    int n = 0;
#pragma unroll
    for (int j = 0; j < E; j++) {
        const int p = a + j * 64 + lane;
        const bool in = p < b && dsmc_in_cell(m, s, p);
        k[j] = in ? ((unsigned long long)(uint32_t)s.id[p] << 32) | (uint32_t)p : ~0ull;
        n += __popcll(__ballot(in));
    }
#pragma unroll
    for (int sz = 1; sz <= 6 + LE; sz++) {
#pragma unroll
        for (int st = sz - 1; st >= 0; st--) {
            if (st >= LE) {
                const int lx = 1 << (st - LE);
                const bool up = sz == 6 + LE || (lane & (1 << (sz - LE))) == 0;
                const bool keep_min = ((lane & lx) == 0) == up;
#pragma unroll
                for (int j = 0; j < E; j++) {
                    const unsigned long long o = __shfl_xor(k[j], lx);
                    k[j] = ((o < k[j]) == keep_min) ? o : k[j];
                }
            } else {
#pragma unroll
                for (int j = 0; j < E; j++) {
                    const int q = j ^ (1 << st);
                    if (q < j) continue;
                    const bool up = sz < LE ? (j & (1 << sz)) == 0
                                            : (sz == 6 + LE || (lane & (1 << (sz - LE))) == 0);
                    const unsigned long long x = k[j], y = k[q];
                    const bool sw = (x > y) == up;
                    k[j] = sw ? y : x;
                    k[q] = sw ? x : y;
                }
            }
        }
    }
#pragma unroll
    for (int j = 0; j < E; j++)
        if (lane * E + j < n) order[a + lane * E + j] = (int32_t)(uint32_t)k[j];
}

__device__ __forceinline__ void order_small(const MeshP& m, const PState& s, int a, int b, int32_t* order) {
    const int len = b - a;
    if (len <= 64) order_in_registers<1>(m, s, a, b, order);
    else if (len <= 128) order_in_registers<2>(m, s, a, b, order);
    else if (len <= 256) order_in_registers<4>(m, s, a, b, order);
    else order_in_registers<8>(m, s, a, b, order);
}

// The same for a longer range, by one workgroup of 256 threads in LDS (key[0 .. pow2), pow2 <=
// DSMC_MAXP: only binned particles enter it, and dsmc_order refuses more).
__device__ void order_in_lds(const MeshP& m, const PState& s, int a, int b, int32_t* order, unsigned long long* key,
                             int* count) {
    const int t = threadIdx.x, lane = t & 63;
    if (t == 0) *count = 0;
    __syncthreads();
    for (int p0 = a; p0 < b; p0 += 256) {
        const int p = p0 + t;
        const bool in = p < b && dsmc_in_cell(m, s, p);
        const unsigned long long mask = __ballot(in);
        int base = 0;
        if (lane == 0) base = atomicAdd(count, __popcll(mask));
        base = __shfl(base, 0);
        if (in)
            key[base + __popcll(mask & ((1ull << lane) - 1ull))] =
                ((unsigned long long)(uint32_t)s.id[p] << 32) | (uint32_t)p;
    }
    __syncthreads();
    const int n = *count;
    int np2 = 1;
    while (np2 < n) np2 <<= 1;
    for (int k = n + t; k < np2; k += 256) key[k] = ~0ull;
    __syncthreads();
    for (int size = 2; size <= np2; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int q = t; q < np2 / 2; q += 256) {
                const int k = 2 * q - (q & (stride - 1)), partner = k + stride;
                const bool up = (k & size) == 0;
                const unsigned long long x = key[k], y = key[partner];
                if ((x > y) == up) {
                    key[k] = y;
                    key[partner] = x;
                }
            }
            __syncthreads();
        }
    }
    for (int k = t; k < n; k += 256) order[a + k] = (int32_t)(uint32_t)key[k];
    __syncthreads();   // key and count are reused
}

// Pair count and particle order of every cell, one wave per cell.  The sort is what bounds it
// (about 45 compare-exchange steps for the 380 particles of a cell of the 512 x 256 gas); it
// stays in registers, so no LDS limits the waves in flight.  Cells with a range longer than
// DSMC_SMALL go to the list big (status->nbig counts it), whose order dsmc_order_big makes.
// 5e7 particles in 512 x 256 cells, at least one candidate pair in each: a pass of a step (order
// and collisions) takes 0.52 ms here, 0.02 in dsmc_order_big and 0.30 in dsmc_collide; it took 4.8 ms
// as one kernel with a bitonic sort in LDS and the pair loop on one lane of the cell's wave.
__global__ void __launch_bounds__(256) dsmc_order(MeshP m, PState sa, const int32_t* __restrict__ off_a, PState sb,
                                                  const int32_t* __restrict__ off_b, DsmcParams pp,
                                                  const double* __restrict__ sig_cr_max, double* __restrict__ rem,
                                                  int32_t* __restrict__ order_a, int32_t* __restrict__ order_b,
                                                  DsmcCell* __restrict__ cells, int* __restrict__ big,
                                                  DsmcStatus* __restrict__ status) {
    const int lane = threadIdx.x & 63;
    const int c = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (c >= m.nci * m.ncj) return;
    const int ci = c % m.nci, cj = c / m.nci;
    const bool edge = ci == m.nci - 1 || cj == m.ncj - 1;
    const int a0 = off_a[c], a1 = off_a[c + 1];
    int b0 = a0, b1 = a1;
    if (!pp.same) {
        b0 = off_b[c];
        b1 = off_b[c + 1];
    }
    const double np1 = dsmc_count(m, sa, a0, a1, edge);
    double np2 = np1;
    if (!pp.same) np2 = dsmc_count(m, sb, b0, b1, edge);
    // collideCell (DSMC.java:238-350): NTC pair count with Boyd's weights (eq. 5); evaluated
    // without fused multiply-adds, so that its integer part is the reference's
    const double scm0 = sig_cr_max[c];
    double nsel_f;
    {
#pragma clang fp contract(off)
        const double cell_volume = node_vol_at(m, ci + 0.5, cj + 0.5);
        double Pab = pp.spwt_b / pp.spwt_a, Pba = pp.spwt_a / pp.spwt_b;
        if (Pab > 1) Pab = 1;
        if (Pba > 1) Pba = 1;
        nsel_f = ((np1 * pp.spwt_a / cell_volume) * np2 * pp.delta_t * scm0) / (Pab + (pp.spwt_b / pp.spwt_a) * Pba);
        if (!pp.same) nsel_f *= 2.0;
        nsel_f += rem[c];
    }
    int nsel = (int)nsel_f;
    const bool pairs = !((pp.same && (np1 < 2 || np2 < 2)) || np1 < 1 || np2 < 1);
    double new_rem = nsel_f - nsel;   // an exact subtraction
    if (nsel > np1 * np2) {
        nsel = (int)(np1 * np2);
        new_rem = 0;
    }
    const bool over = pairs && nsel != 0 && (np1 > DSMC_MAXP || np2 > DSMC_MAXP);
    const bool go = pairs && nsel != 0 && !over;
    if (lane == 0) {
        if (pairs && !over) rem[c] = new_rem;
        if (over) atomicMax(&status->overflow, (int)fmax(np1, np2));
        cells[c] = DsmcCell{go ? nsel : 0, (int)np1, (int)np2};
    }
    if (!go) return;
    if (a1 - a0 > DSMC_SMALL || b1 - b0 > DSMC_SMALL) {
        if (lane == 0) big[atomicAdd(&status->nbig, 1)] = c;
        return;
    }
    order_small(m, sa, a0, a1, order_a);
    if (!pp.same) order_small(m, sb, b0, b1, order_b);
}

// A cell's range holds its binned particles and, in the last row and column, particles on the last
// node line: those of a range may exceed DSMC_MAXP, the binned ones that enter the LDS list not.
__global__ void __launch_bounds__(256) dsmc_order_big(MeshP m, PState sa, const int32_t* __restrict__ off_a, PState sb,
                                                      const int32_t* __restrict__ off_b, int same,
                                                      int32_t* __restrict__ order_a, int32_t* __restrict__ order_b,
                                                      const int* __restrict__ big,
                                                      const DsmcStatus* __restrict__ status) {
    __shared__ unsigned long long key[DSMC_MAXP];
    __shared__ int count;
    const int nbig = status->nbig;
    for (int q = blockIdx.x; q < nbig; q += gridDim.x) {
        const int c = big[q];
        order_in_lds(m, sa, off_a[c], off_a[c + 1], order_a, key, &count);
        if (!same) order_in_lds(m, sb, off_b[c], off_b[c + 1], order_b, key, &count);
    }
}

// The last Philox block a stream drew from: draws 2q and 2q + 1 are its two halves.
struct PairedRng {
    ParticleRng r;
    uint32_t block;
    double even, odd;
    __device__ __forceinline__ double draw(uint32_t k) {
        if ((k >> 1) != block) {
            block = k >> 1;
            const uint4 o = philox4x32_10(make_uint4(block, r.id, r.step, r.tag), r.k0, r.k1);
            even = (double)((((uint64_t)o.y << 32) | o.x) >> 11) * 0x1.0p-53;
            odd = (double)((((uint64_t)o.w << 32) | o.z) >> 11) * 0x1.0p-53;
        }
        return (k & 1) ? odd : even;
    }
};

// The collision loop of every cell, one LANE per cell.  A cell's pairs are sequential (a particle
// drawn twice must see its first collision's velocity, and a pair's draws follow the last one's),
// but the cells are independent: those of a wave share its instruction stream, where a loop on one
// lane of a wave per cell spent the same instructions (Philox, pow, sin, cos) on one cell.  Only where
// all cells together are a few waves do lanes wait more for each other's collisions than they share:
// a wave takes 2^cell_shift cells, 64 unless that leaves fewer than DSMC_WAVES waves.  A pass with
// many pairs a cell: 4 cells of 1500 particles 1.84 ms (64 cells a wave 2.11), 100 of 400 0.63 (0.78);
// but 3200 of 400 0.93 ms with 64 cells a wave, 1.05 with 32, 1.28 with 8 and 1.68 with 2.
constexpr int DSMC_WAVES = 32;
__global__ void __launch_bounds__(64) dsmc_collide(MeshP m, PState sa, const int32_t* __restrict__ off_a, PState sb,
                                                   const int32_t* __restrict__ off_b, DsmcParams pp, int cell_shift,
                                                   const int32_t* __restrict__ order_a,
                                                   const int32_t* __restrict__ order_b,
                                                   const DsmcCell* __restrict__ cells, double* __restrict__ sig_cr_max,
                                                   double* __restrict__ count_sum, double* __restrict__ real_sum,
                                                   DsmcStatus* __restrict__ status) {
    const int c = (blockIdx.x << cell_shift) + threadIdx.x;
    double sums0 = 0, sums1 = 0;
    if ((int)threadIdx.x < (1 << cell_shift) && c < m.nci * m.ncj && cells[c].nsel > 0) {
        const DsmcCell cell = cells[c];
        const int ci = c % m.nci, cj = c / m.nci;
        const double np1 = cell.n1, np2 = cell.n2, scm0 = sig_cr_max[c];
        const int32_t* la = order_a + off_a[c];
        const int32_t* lb = pp.same ? la : order_b + off_b[c];
        const PState& Sb = pp.same ? sa : sb;
        PairedRng rng{{pp.k0, pp.k1, (uint32_t)c, pp.step, pp.tag}, 0xFFFFFFFFu, 0.0, 0.0};
        uint32_t k = 0;
        double scm = 0;
        const double rm1 = pp.mass_a / (pp.mass_a + pp.mass_b), rm2 = pp.mass_b / (pp.mass_a + pp.mass_b);
        for (int q = 0; q < cell.nsel; q++) {
            const int p1 = (int)(rng.draw(k++) * np1);
            int p2;
            do {
                p2 = (int)(rng.draw(k++) * np2);
            } while (pp.same && p1 == p2);
            const int64_t ga = la[p1], gb = lb[p2];
            double va[3] = {sa.vx[ga], sa.vy[ga], sa.vz[ga]};
            double vb[3] = {Sb.vx[gb], Sb.vy[gb], Sb.vz[gb]};
            const double g0 = va[0] - vb[0], g1 = va[1] - vb[1], g2 = va[2] - vb[2];
            const double cr = sqrt(g0 * g0 + g1 * g1 + g2 * g2);
            const double sigma_cr = cr * dsmc_sigma(pp, cr);
            if (sigma_cr > scm) scm = sigma_cr;
            const double P = sigma_cr / scm0;
            if (rng.draw(k++) < P) {
                // ModelElastic (DSMC.java:360-430), Bird's DSMC0 scattering
                double vc[3], vr[3];
                for (int d = 0; d < 3; d++) vc[d] = rm1 * va[d] + rm2 * vb[d];
                if (fabs(pp.vss_inv - 1.) < 1.e-4) {
                    const double B = 2. * rng.draw(k++) - 1.0;
                    const double A = sqrt(1. - B * B);
                    vr[0] = B * cr;
                    const double C = 2. * M_PI * rng.draw(k++);
                    vr[1] = A * cos(C) * cr;
                    vr[2] = A * sin(C) * cr;
                } else {
                    const double B = 2. * (pow(rng.draw(k++), pp.vss_inv)) - 1.;
                    const double A = sqrt(1. - B * B);
                    const double C = 2. * M_PI * rng.draw(k++);
                    const double OC = cos(C), SC = sin(C);
                    const double D = sqrt(g1 * g1 + g2 * g2);
                    if (D > 1.e-6) {
                        vr[0] = B * g0 + A * SC * D;
                        vr[1] = B * g1 + A * (cr * g2 * OC - g0 * g1 * SC) / D;
                        vr[2] = B * g2 - A * (cr * g1 * OC + g0 * g2 * SC) / D;
                    } else {
                        vr[0] = B * g1;
                        vr[1] = A * OC * g1;
                        vr[2] = A * SC * g1;
                    }
                }
                bool wa = true, wb = true;
                if (pp.spwt_a != pp.spwt_b) {   // Boyd's probabilities for unequal weights
                    wa = rng.draw(k++) < pp.spwt_b / pp.spwt_a;
                    wb = rng.draw(k++) < pp.spwt_a / pp.spwt_b;
                }
                if (wa) {
                    sa.vx[ga] = (float)(vc[0] + vr[0] * rm2);
                    sa.vy[ga] = (float)(vc[1] + vr[1] * rm2);
                    sa.vz[ga] = (float)(vc[2] + vr[2] * rm2);
                }
                if (wb) {
                    Sb.vx[gb] = (float)(vc[0] - vr[0] * rm1);
                    Sb.vy[gb] = (float)(vc[1] - vr[1] * rm1);
                    Sb.vz[gb] = (float)(vc[2] - vr[2] * rm1);
                }
                sums0 += 1.0;
                sums1 += 0.5 * (pp.spwt_a + pp.spwt_b);
            }
        }
        if (scm > 0) sig_cr_max[c] = scm;
        const size_t u = (size_t)cj * m.ni + ci;
        count_sum[u] += sums0;
        real_sum[u] += sums1;
    }
    for (int o = 32; o > 0; o >>= 1) sums0 += __shfl_xor(sums0, o);
    if (threadIdx.x == 0 && sums0 > 0) atomicAdd(&status->ncol, (unsigned long long)sums0);
}

__global__ void dsmc_fields_kernel(int64_t nn, int which, const double* __restrict__ count_sum,
                                   const double* __restrict__ real_sum, double inv_samples, double inv_time,
                                   double* __restrict__ out) {
    for (int64_t u = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; u < nn; u += (int64_t)gridDim.x * blockDim.x) {
        double v;
        switch (which) {
            case 0: v = count_sum[u]; break;                // col-count-sum
            case 1: v = real_sum[u]; break;                 // col-real-sum
            case 2: v = count_sum[u] * inv_samples; break;  // col-count
            default: v = real_sum[u] * inv_time; break;     // nu
        }
        out[u] = v;
    }
}

// Utils.gamma (core/common/Utils.java:218-236): Bird's approximation of the Gamma function
static double bird_gamma(double X) {
    double A = 1., Y = X;
    if (Y < 1.0) {
        A = A / Y;
    } else {
        do {
            Y = Y - 1;
            if (Y >= 1.) A = A * Y;
        } while (Y >= 1.);
    }
    return A * (1. - 0.5748646 * Y + 0.9512363 * Y * Y - 0.6998588 * Y * Y * Y + 0.4245549 * Y * Y * Y * Y -
                0.1010678 * Y * Y * Y * Y * Y);
}

}  // namespace sf

using namespace sf;

struct sf_dsmc {
    sf_ctx* ctx = nullptr;
    sf_dsmc_desc desc{};
    DsmcParams pp{};
    double* d_scm = nullptr;      // [ncells] sig_cr_max
    double* d_rem = nullptr;      // [ncells]
    double* d_count = nullptr;    // [nn] col-count-sum
    double* d_real = nullptr;     // [nn] col-real-sum
    DsmcCell* d_cells = nullptr;  // [ncells] pair and particle counts of the running pass
    int* d_big = nullptr;         // [ncells] list of the cells that dsmc_order_big orders
    DsmcStatus* d_status = nullptr;
    DsmcStatus* h_status = nullptr;   // pinned
    int num_samples = 0;
};

extern "C" {

int sf_dsmc_create(sf_ctx* ctx, const sf_dsmc_desc* desc, sf_dsmc** out) {
    SF_CHECK_CTX(ctx);
    if (!desc || !out) return sf_fail(ctx, SF_ERR_ARG, "sf_dsmc_create: null argument");
    *out = nullptr;
    if (!ctx->mesh_ready) return sf_fail(ctx, SF_ERR_STATE, "sf_dsmc_create: mesh not set up");
    const int ns = (int)ctx->species.size();
    if (desc->species_a < 0 || desc->species_a >= ns || desc->species_b < 0 || desc->species_b >= ns)
        return sf_fail(ctx, SF_ERR_ARG, "sf_dsmc_create: bad species pair %d, %d", desc->species_a, desc->species_b);
    Species* A = ctx->species[desc->species_a];
    Species* B = ctx->species[desc->species_b];
    if (!A->desc.track_ids || !B->desc.track_ids)
        return sf_fail(ctx, SF_ERR_STATE, "sf_dsmc_create: both species must track particle ids");
    if (desc->sigma_type != SF_SIGMA_CONST && desc->sigma_type != SF_SIGMA_BIRD463)
        return sf_fail(ctx, SF_ERR_UNSUPPORTED, "sf_dsmc_create: sigma type %d is not supported", desc->sigma_type);
    if (!(desc->vss_alpha_a > 0) || !(desc->vss_alpha_b > 0))
        return sf_fail(ctx, SF_ERR_ARG, "sf_dsmc_create: vss_alpha must be > 0");
    DsmcParams pp{};
    pp.same = desc->species_a == desc->species_b;
    pp.sigma_type = desc->sigma_type;
    pp.c0 = desc->sigma_c0;
    const double d_ref = desc->diam_a + desc->diam_b;
    pp.sigma0 = 0.25 * M_PI * d_ref * d_ref;
    if (pp.sigma_type == SF_SIGMA_BIRD463 && !(pp.sigma0 > 0))
        return sf_fail(ctx, SF_ERR_ARG, "sf_dsmc_create: material diameter <diam> not defined");
    pp.ref_temp = 0.5 * (desc->ref_temp_a + desc->ref_temp_b);
    pp.vti = 0.5 * (desc->visc_temp_index_a + desc->visc_temp_index_b);
    pp.mass_a = A->mass;
    pp.mass_b = B->mass;
    pp.mr = A->mass * B->mass / (A->mass + B->mass);
    pp.gamma = bird_gamma(2.5 - pp.vti);
    pp.vss_inv = 0.5 * (1.0 / desc->vss_alpha_a + 1.0 / desc->vss_alpha_b);
    pp.spwt_a = A->desc.spwt;
    pp.spwt_b = B->desc.spwt;
    pp.k0 = (uint32_t)desc->seed;
    pp.k1 = (uint32_t)(desc->seed >> 32);
    {
        int rc = claim_stream(ctx, desc->seed, RNG_MODULE_DSMC, desc->tag, &pp.tag);
        if (rc) return rc;
    }
    SF_HIP(ctx, hipSetDevice(ctx->device));
    const size_t nn = (size_t)ctx->mp.ni * ctx->mp.nj, nc = (size_t)ctx->mp.nci * ctx->mp.ncj;
    sf_dsmc* d = new sf_dsmc();
    d->ctx = ctx;
    d->desc = *desc;
    if (d->desc.frequency < 1) d->desc.frequency = 1;
    d->pp = pp;
    std::vector<double> scm(nc, desc->sig_cr_max0 > 0 ? desc->sig_cr_max0 : 1e-16);
    hipError_t e = hipMalloc((void**)&d->d_scm, nc * 8);
    if (e == hipSuccess) e = hipMalloc((void**)&d->d_rem, nc * 8);
    if (e == hipSuccess) e = hipMalloc((void**)&d->d_count, nn * 8);
    if (e == hipSuccess) e = hipMalloc((void**)&d->d_real, nn * 8);
    if (e == hipSuccess) e = hipMalloc((void**)&d->d_cells, nc * sizeof(DsmcCell));
    if (e == hipSuccess) e = hipMalloc((void**)&d->d_big, nc * sizeof(int));
    if (e == hipSuccess) e = hipMalloc((void**)&d->d_status, sizeof(DsmcStatus));
    if (e == hipSuccess) e = hipHostMalloc((void**)&d->h_status, sizeof(DsmcStatus));
    if (e == hipSuccess) e = hipMemcpy(d->d_scm, scm.data(), nc * 8, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemsetAsync(d->d_rem, 0, nc * 8, ctx->stream);
    if (e == hipSuccess) e = hipMemsetAsync(d->d_count, 0, nn * 8, ctx->stream);
    if (e == hipSuccess) e = hipMemsetAsync(d->d_real, 0, nn * 8, ctx->stream);
    if (e != hipSuccess) {
        hipFree(d->d_scm);
        hipFree(d->d_rem);
        hipFree(d->d_count);
        hipFree(d->d_real);
        hipFree(d->d_cells);
        hipFree(d->d_big);
        hipFree(d->d_status);
        hipHostFree(d->h_status);
        delete d;
        release_stream(ctx, desc->seed, pp.tag);
        return sf_fail(ctx, SF_ERR_HIP, "sf_dsmc_create: %s", hipGetErrorString(e));
    }
    *out = d;
    return SF_OK;
}

int sf_dsmc_destroy(sf_dsmc* d) {
    if (!d) return SF_ERR_ARG;
    hipSetDevice(d->ctx->device);
    hipStreamSynchronize(d->ctx->stream);
    hipFree(d->d_scm);
    hipFree(d->d_rem);
    hipFree(d->d_count);
    hipFree(d->d_real);
    hipFree(d->d_cells);
    hipFree(d->d_big);
    hipFree(d->d_status);
    hipHostFree(d->h_status);
    release_stream(d->ctx, d->desc.seed, d->pp.tag);
    delete d;
    return SF_OK;
}

int sf_dsmc_perform(sf_dsmc* d, int it, int64_t* collisions) {
    if (!d) return SF_ERR_ARG;
    sf_ctx* ctx = d->ctx;
    if (collisions) *collisions = 0;
    if (it % d->desc.frequency != 0) return SF_OK;
    SF_HIP(ctx, hipSetDevice(ctx->device));
    d->num_samples++;
    Species* A = ctx->species[d->desc.species_a];
    Species* B = ctx->species[d->desc.species_b];
    // the cell lists are the cell ranges of freshly sorted, compacted species
    for (Species* sp : {A, B}) {
        if (sp->since_sort != 0 || sp->nsorted != sp->np) {
            int rc = sort_species(ctx, sp);
            if (rc) return rc;
        }
    }
    DsmcParams pp = d->pp;
    pp.delta_t = d->desc.frequency * ctx->dt;
    pp.step = (uint32_t)it;
    SF_HIP(ctx, hipMemsetAsync(d->d_status, 0, sizeof(DsmcStatus), ctx->stream));
    const int ncells = ctx->mp.nci * ctx->mp.ncj;
    // the species' key arrays hold nothing between pushes: the passes keep the cells' orders there
    const PState sa = A->buf[A->cur], sb = B->buf[B->cur];
    const int32_t *oa = A->offsets, *ob = B->offsets;
    hipLaunchKernelGGL(dsmc_order, dim3((ncells + 3) / 4), dim3(256), 0, ctx->stream, ctx->mp, sa, oa, sb, ob, pp,
                       (const double*)d->d_scm, d->d_rem, A->key, B->key, d->d_cells, d->d_big, d->d_status);
    hipLaunchKernelGGL(dsmc_order_big, dim3(std::min(ncells, 1024)), dim3(256), 0, ctx->stream, ctx->mp, sa, oa, sb, ob,
                       pp.same, A->key, B->key, (const int*)d->d_big, (const DsmcStatus*)d->d_status);
    int shift = 6;
    while (shift > 0 && (ncells >> shift) < DSMC_WAVES) shift--;
    hipLaunchKernelGGL(dsmc_collide, dim3((ncells + (1 << shift) - 1) >> shift), dim3(64), 0, ctx->stream, ctx->mp, sa, oa,
                       sb, ob, pp, shift, (const int32_t*)A->key, (const int32_t*)B->key, (const DsmcCell*)d->d_cells,
                       d->d_scm, d->d_count, d->d_real, d->d_status);
    SF_HIP(ctx, hipGetLastError());
    SF_HIP(ctx, hipMemcpyAsync(d->h_status, d->d_status, sizeof(DsmcStatus), hipMemcpyDeviceToHost, ctx->stream));
    SF_HIP(ctx, hipStreamSynchronize(ctx->stream));
    const int over = d->h_status->overflow;
    if (collisions) *collisions = (int64_t)d->h_status->ncol;
    if (over > 0)
        return sf_fail(ctx, SF_ERR_UNSUPPORTED, "sf_dsmc_perform: a cell holds %d particles of one species (limit %d);"
                       " its collisions were skipped", over, DSMC_MAXP);
    return SF_OK;
}

int sf_dsmc_field(sf_dsmc* d, int which, double* out) {
    if (!d) return SF_ERR_ARG;
    sf_ctx* ctx = d->ctx;
    if (!out || which < 0 || which > 4) return sf_fail(ctx, SF_ERR_ARG, "sf_dsmc_field: bad argument");
    SF_HIP(ctx, hipSetDevice(ctx->device));
    SF_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (which == 4) {   // sig_cr_max per cell, index j*(ni-1)+i
        const size_t nc = (size_t)ctx->mp.nci * ctx->mp.ncj;
        SF_HIP(ctx, hipMemcpy(out, d->d_scm, nc * 8, hipMemcpyDeviceToHost));
        return SF_OK;
    }
    const int64_t nn = (int64_t)ctx->mp.ni * ctx->mp.nj;
    double* d_out = nullptr;
    const int rc = field_workspace(ctx, &d_out);
    if (rc) return rc;
    const double inv_samples = d->num_samples > 0 ? 1.0 / d->num_samples : 0.0;
    // fc_nu = real_sum / (num_samples * frequency * dt) (DSMC.java:186-188)
    const double inv_time = 1.0 / (d->num_samples * d->desc.frequency * ctx->dt);
    hipLaunchKernelGGL(dsmc_fields_kernel, dim3((unsigned)((nn + 255) / 256 < 8192 ? (nn + 255) / 256 : 8192)),
                       dim3(256), 0, ctx->stream, nn, which, (const double*)d->d_count, (const double*)d->d_real,
                       inv_samples, inv_time, d_out);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(out, d_out, nn * 8, hipMemcpyDeviceToHost, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) return sf_fail(ctx, SF_ERR_HIP, "sf_dsmc_field: %s", hipGetErrorString(e));
    return SF_OK;
}

int sf_dsmc_clear_samples(sf_dsmc* d) {
    if (!d) return SF_ERR_ARG;
    sf_ctx* ctx = d->ctx;
    SF_HIP(ctx, hipSetDevice(ctx->device));
    const size_t nn = (size_t)ctx->mp.ni * ctx->mp.nj;
    SF_HIP(ctx, hipMemsetAsync(d->d_count, 0, nn * 8, ctx->stream));
    SF_HIP(ctx, hipMemsetAsync(d->d_real, 0, nn * 8, ctx->stream));
    SF_HIP(ctx, hipStreamSynchronize(ctx->stream));
    d->num_samples = 0;
    return SF_OK;
}

}  // extern "C"
