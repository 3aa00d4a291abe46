// spimc_kernels.h -- HIP kernels of the engine (included once, by spimc_engine.hip).
//
// Move stages run in rounds: every replica with attempts left performs one
// attempt per round.  Its parts:
//   propose      draws, bisection sampling of the coarse levels with their kinetic
//                Metropolis decisions, and the level-0 NEW beads
//   pair links   short-range pair action of the moved particle against all
//                others on every window link, OLD and NEW
//   rho_k items  a moved slice's chunk of k-vectors: incremental rho_k update into
//                the spare buffer fused with the long-range action sums, OLD and NEW
//   decide       level-0 Metropolis decision and commit
// In three launches, k_decide_propose_* decides the last round and proposes the next,
// k_pair_lds (tables in LDS) or k_pair takes the links, k_rho_loop the items.  Batches
// that fit the GPU at once run them in one, k_round, which for a bisection also makes
// the next proposal beside the pending one.  A single chain (the plain method) is the
// same launches with one replica.
#pragma once

#include "spimc_device.h"

namespace spimc {

constexpr int kPairBlock = 256;       // 4 wavefronts, one link each
constexpr int kRhoBlock = 256;
constexpr int kMaxIdx = 63;           // largest |n_d| of a k-vector
constexpr int kGrBins = 4096;

enum { WORK_PAIR_LINKS = 0, WORK_RHO_SLICEK = 1, WORK_COUNT = 2 };

// Per-replica estimator scratch: slots [slot][M] for slots 0..3, then the
// long-range k-chunk partials, then two results.
constexpr int kSlotKin = 0, kSlotPair = 1, kSlotCentroid = 2, kSlotVirial = 3;
__host__ __device__ inline size_t scratch_long(int M) { return (size_t)4 * M; }
__host__ __device__ inline size_t scratch_res(int M, int nk) { return (size_t)4 * M + (nk + kWave - 1) / kWave + 1; }
__host__ __device__ inline size_t scratch_size(int M, int nk) { return scratch_res(M, nk) + 4; }

// Blocks are dispatched round-robin over the 8 XCDs; this remap hands each XCD
// a contiguous range of logical blocks, so the items of one replica (sorted
// together) share an L2.
__device__ __forceinline__ int xcd_remap(int hw, int G) {
    const int X = 8;
    int q = G / X, rem = G % X;
    int xcd = hw % X, local = hw / X;
    return (xcd < rem) ? xcd * (q + 1) + local : rem * (q + 1) + (xcd - rem) * q + local;
}

// Loads through the global address space (replica arrays live in device
// memory; a generic pointer would compile to flat loads, which also count
// against the LDS wait counter).
template <class T>
__device__ __forceinline__ T gld(const T* p) {
    return *(const __attribute__((address_space(1))) T*)p;
}

// Loads of data that no kernel writes while this one runs, at an address all
// lanes share: scalar loads.  (Through a generic pointer the compiler would
// take the value for a per-lane one.)
template <class T>
__device__ __forceinline__ T uld(const T* p) {
    return *(const __attribute__((address_space(4))) T*)p;
}

// Partial sums passed between the workgroups of one launch (k_round): 64-bit
// atomic stores and loads at agent scope, which the memory model performs at
// the device's coherence point, so a workgroup on another XCD reads them
// without any L2 write-back or invalidation of the caches.
__device__ __forceinline__ void coh_store2(double2* p, double2 v) {
    __hip_atomic_store(&p->x, v.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&p->y, v.y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double2 coh_load2(const double2* p) {
    double2* q = const_cast<double2*>(p);
    return make_double2(__hip_atomic_load(&q->x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                        __hip_atomic_load(&q->y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// 16-byte global loads and stores of one rho_k value; NT marks them
// non-temporal (streamed through, not kept in the caches)
typedef double d2v __attribute__((ext_vector_type(2)));
template <bool NT>
__device__ __forceinline__ double2 ld2(const double2* p) {
    const __attribute__((address_space(1))) d2v* q = (const __attribute__((address_space(1))) d2v*)p;
    const d2v v = NT ? __builtin_nontemporal_load(q) : *q;
    return make_double2(v.x, v.y);
}
template <bool NT>
__device__ __forceinline__ void st2(double2* p, double2 v) {
    __attribute__((address_space(1))) d2v* q = (__attribute__((address_space(1))) d2v*)p;
    const d2v w = {v.x, v.y};
    if (NT)
        __builtin_nontemporal_store(w, q);
    else
        *q = w;
}

__device__ __forceinline__ double pos_at(const Rep& R, int d, int s, int p) {
    return gld(R.pos + ((size_t)d * R.M + s) * R.N + p);
}

// The NEW positions of a bisection or displacement; only k_round meets those
// made ahead.
__device__ __forceinline__ double* prop_beads(const Rep& R, const Prop& pr) {
    return pr.buf == 0 ? R.prop_new : pr.buf == 1 ? R.next_new[0] : R.next_new[1];
}

// NEW-mode position of the proposal's particle at slice s
__device__ __forceinline__ double pos_new(const Rep& R, const Prop& pr, int d, int s) {
    int m = s - pr.first;
    if (m < 0) m += R.M;
    return (m < pr.count) ? R.prop_new[3 * m + d] : pos_at(R, d, s, pr.p);
}

__device__ __forceinline__ double tape_get(const Rep& R, long long i, int* bad) {
    if (i < 0 || i >= R.tape_len) {
        *bad = 1;
        return 0.5;
    }
    return R.tape[i];
}

// Phase tables of moved bead m (OLD position xo, NEW position xn) for k_rho:
// chain c = o * 3 + d of length max_idx + 1, by the KSpace::CalcC recurrence.
__device__ __forceinline__ void moved_phase_chain(const Rep& R, int m, int c, const double* xo, const double* xn) {
    const int stride = R.max_idx + 1, o = c / 3, d = c % 3;
    phase_chain((o ? xn[d] : xo[d]) * R.box, R.max_idx, R.phase + ((size_t)m * 6 + c) * stride);
}

// Row descriptor of moved bead m at slice s: k_rho streams rho[sel][s] -> rho[1-sel][s].
__device__ __forceinline__ void moved_row(const Rep& R, int m, int s) { R.rho_rows[m] = make_int2(s, R.sel[s]); }

// The rho_k work items of a replica's round, written by its proposal kernel
// (one wavefront): item t = (moved bead t / n_chunks, k chunk t % n_chunks),
// valid when the proposal goes to level 0 and moves that bead (bead m sits at
// slice first + m).  Idle items (no attempt left, rejected at a coarse level,
// fewer moved beads) are marked invalid.
__device__ __forceinline__ void rho_items_write(const Rep& R, int move, int status, int count, int first, int lane,
                                                int nthr = kWave, const double2* phase = nullptr) {
    RhoItem* items = move == 0 ? R.ritems_bis : R.ritems_dis;
    const int n = move == 0 ? R.n_ritems_bis : R.n_ritems_dis;
    if (!items) return;
    const int stride = R.max_idx + 1, nch = R.n_chunks, ck = kRhoBlock * R.rho_kpt;
    for (int t = lane; t < n; t += nthr) {
        const int m = t / nch, ch = t % nch;
        RhoItem d{};
        if (status == 1 && m < count) {
            const int s = (first + m) % R.M, cur = R.sel[s];
            d.rc = R.rho + ((size_t)cur * R.M + s) * R.nk;
            d.rn = R.rho + ((size_t)(1 - cur) * R.M + s) * R.nk;
            d.ph = (phase ? phase : R.phase) + (size_t)m * 6 * stride;
            d.kidx = R.kidx;
            d.coef = R.coef_s;
            d.part = R.rho_part + m * nch + ch;
            d.k0 = ch * ck;
            d.k1 = min(R.nk, d.k0 + ck);
            d.stride = stride;
            d.valid = 1;
        }
        items[t] = d;
    }
}

// ---------------------------------------------------------------------------
// K3: rho_k of every slice (Species::InitRhoK, species_class.h:380-403);
// particle sums in particle order per k.
// ---------------------------------------------------------------------------
constexpr int kBuildTile = 16;
template <int KPT>
__global__ __launch_bounds__(256) void k_rho_build(const Rep* __restrict__ reps, int r) {
    const Rep& R = reps[r];
    const int b = blockIdx.x, chunk = blockIdx.y;
    const int mx = R.max_idx, stride = mx + 1;
    __shared__ double2 tab[kBuildTile * 3 * (kMaxIdx + 1)];
    double2 acc[KPT];
    int kk[KPT];
    for (int i = 0; i < KPT; ++i) {
        acc[i] = make_double2(0., 0.);
        int k = chunk * 256 * KPT + i * 256 + threadIdx.x;
        kk[i] = (k < R.nk) ? R.kidx[k] : -1;
    }
    for (int p0 = 0; p0 < R.N; p0 += kBuildTile) {
        __syncthreads();
        if (threadIdx.x < kBuildTile * 3) {
            int pp = threadIdx.x / 3, d = threadIdx.x % 3;
            if (p0 + pp < R.N) phase_chain(pos_at(R, d, b, p0 + pp) * R.box, mx, &tab[(pp * 3 + d) * stride]);
        }
        __syncthreads();
        const int np = min(kBuildTile, R.N - p0);
        for (int pp = 0; pp < np; ++pp)
            for (int i = 0; i < KPT; ++i)
                if (kk[i] >= 0) {
                    double2 e = phase_k(&tab[pp * 3 * stride], stride, kk[i]);
                    acc[i].x += e.x;
                    acc[i].y += e.y;
                }
    }
    double2* out = R.rho + ((size_t)R.sel[b] * R.M + b) * R.nk;
    for (int i = 0; i < KPT; ++i) {
        int k = chunk * 256 * KPT + i * 256 + threadIdx.x;
        if (k < R.nk) out[k] = acc[i];
    }
}

// K3 by columns: the k-vectors (n0, n1, +-n2) of one column share e^{i (n0 phi_0 +
// n1 phi_1)} = x + iy, and with e^{i n phi_2} = c + is both signs of n take the four
// sums of xc, ys, xs and yc: rho(+-n) = (xc -+ ys, yc +- xs).  A lane holds four
// consecutive n of a column (16 sums, 16 multiply-adds a particle for up to eight
// k-vectors, where k_rho_build spends two complex products and three LDS reads on
// each), a workgroup 64 such groups of one slice, its wavefronts every fourth
// particle; the wavefronts' sums are added in order.  Bound by its LDS reads (six
// of 16 bytes a particle and lane).  One slice array of N = 1024, M = 128 with 4012
// k-vectors: 306 us by k_rho_build, 88 us so.
__global__ __launch_bounds__(256) void k_rho_cols(const Rep* __restrict__ reps, int r, int tile) {
    extern __shared__ double lds[];
    const Rep& R = reps[r];
    const int b = blockIdx.x, lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const int mx = R.max_idx, stride = mx + 1, N = R.N, ng = R.n_col_k / 4, g = blockIdx.y * kWave + lane;
    double2* tab = reinterpret_cast<double2*>(lds);  // [tile][3][stride], and three values that a padded group reads
    const int2 cg = g < ng ? R.col_g[g] : make_int2(128 | 128 << 8, 0);
    const int n0 = (cg.x & 255) - 128, n1 = (cg.x >> 8) - 128;
    const int a0 = abs(n0), a1 = stride + abs(n1), a2 = 2 * stride + cg.y;
    const double g0 = n0 < 0 ? -1. : 1., g1 = n1 < 0 ? -1. : 1.;
    double s[4][4];
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i / 4][i % 4] = 0.;
    for (int p0 = 0; p0 < N; p0 += tile) {
        __syncthreads();
        const int np = min(tile, N - p0);
        for (int t = threadIdx.x; t < 3 * np; t += 256)
            phase_chain(pos_at(R, t % 3, b, p0 + t / 3) * R.box, mx, tab + t * stride);
        __syncthreads();
        for (int pp = w; pp < np; pp += 256 / kWave) {
            const double2* f = tab + pp * 3 * stride;
            double2 e0 = f[a0], e1 = f[a1];
            e0.y *= g0;
            e1.y *= g1;
            const double2 e = cmul(e0, e1);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const double2 z = f[a2 + i];
                s[i][0] = fma(e.x, z.x, s[i][0]);
                s[i][1] = fma(e.y, z.y, s[i][1]);
                s[i][2] = fma(e.x, z.y, s[i][2]);
                s[i][3] = fma(e.y, z.x, s[i][3]);
            }
        }
    }
    __syncthreads();
    if (w > 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) lds[((w - 1) * 16 + i) * kWave + lane] = s[i / 4][i % 4];
    }
    __syncthreads();
    if (w > 0 || g >= ng) return;
    double2* out = R.rho + ((size_t)R.sel[b] * R.M + b) * R.nk;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        for (int v = 0; v < 256 / kWave - 1; ++v)
            for (int q = 0; q < 4; ++q) s[i][q] += lds[(v * 16 + 4 * i + q) * kWave + lane];
        const int2 k = R.col_k[4 * g + i];
        if (k.x >= 0) out[k.x] = make_double2(s[i][0] - s[i][1], s[i][3] + s[i][2]);
        if (k.y >= 0) out[k.y] = make_double2(s[i][0] + s[i][1], s[i][3] - s[i][2]);
    }
}

// ---------------------------------------------------------------------------
// K4: Bisect::Attempt down to level 0 (bisect_class.h:39-124), one wavefront
// per replica.  Coarse levels carry only the kinetic action (the pair action
// returns 0 above max_level = 0, pair_action_class.h:269).
// ---------------------------------------------------------------------------
// Synchronisation of the one-wavefront bodies below (the whole 64-thread
// workgroup of the round kernels).
struct BlockSync {
    __device__ void operator()() const { __syncthreads(); }
};
// Ordering point of the one-wavefront bodies when they run in one wavefront of
// a larger workgroup: the wavefront's memory operations complete, and no code
// moves across it.
struct WaveSync {
    __device__ void operator()() const {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        __builtin_amdgcn_wave_barrier();
    }
};

// LDS of one bisection proposal (one wavefront): the window's beads, OLD and
// NEW; the attempt's normals, 3 per midpoint in level order, and level
// uniforms (device RNG), drawn before the level loop across the lanes; the
// attempt's counter step and first draws.
struct BisectLds {
    double x_old[(1 << kMaxLevel) + 1][3];
    double x_new[(1 << kMaxLevel) + 1][3];
    double z[3 * ((1 << kMaxLevel) - 1) + 1];
    double u[kMaxLevel];
    double sums[4][kMaxLevel];  // bisect_levels: sampling and kinetic sums, OLD then NEW
    int info[6];  // an attempt is left, p, b0, bad draw; of bisect_levels: status, moved beads
    long long cur;
    unsigned long long seq;
};

// The counter step of an attempt (one lane): whether one is left, and its
// sequence number (the device RNG's counter).
__device__ __forceinline__ void bisect_take(const Rep& R, BisectLds& S) {
    Counters* c = R.cnt;
    const unsigned int rem = c->remaining;
    S.info[0] = rem > 0;
    if (rem > 0) {
        c->remaining = rem - 1;
        S.seq = c->seq;
        c->seq = S.seq + 1;
    }
}

// The normals and level uniforms of attempt seq on the device RNG into S.
__device__ __forceinline__ void bisect_draws(const Rep& R, int lane, BisectLds& S, unsigned long long seq) {
    const int n = R.n_level, nb = 1 << n;
    Rng rng{make_uint2((uint32_t)R.key, (uint32_t)(R.key >> 32)), 1u, seq};
    // normal g is normal(1 + n + g / 2, g & 1): one call per pair of normals
    const int n_norm = 3 * (nb - 1);
    for (int q = lane; 2 * q < n_norm; q += kWave) {
        double z0, z1;
        rng.normal2(1 + n + q, &z0, &z1);
        S.z[2 * q] = z0;
        S.z[2 * q + 1] = z1;
    }
    for (int l = lane; l < n; l += kWave) S.u[l] = rng.unif(1 + l, 0);
}

// The window's beads of (p, b0) into S, and on the device RNG (draws) the
// attempt's normals and level uniforms, made while the loads are in flight
// (the window holds nb + 1 <= 65 beads: two per lane at most).
__device__ __forceinline__ void bisect_window(const Rep& R, int lane, BisectLds& S, int p, int p2, int b0,
                                              bool draws) {
    const int n = R.n_level, nb = 1 << n, M = R.M;
    double xw[2][3];
    for (int k = 0; k < 2; ++k) {
        const int j = lane + k * kWave;
        if (j > nb) break;
        const int s = (b0 + j) % M;
        const int lbl = (b0 + j >= M) ? p2 : p;
        for (int d = 0; d < 3; ++d) xw[k][d] = pos_at(R, d, s, lbl);
    }
    if (draws) bisect_draws(R, lane, S, S.seq);
    for (int k = 0; k < 2; ++k) {
        const int j = lane + k * kWave;
        if (j > nb) break;
        for (int d = 0; d < 3; ++d) {
            S.x_old[j][d] = xw[k][d];
            S.x_new[j][d] = xw[k][d];
        }
    }
}

// Particle and first bead of attempt seq on the device RNG: rng.index(0, 0, N) and
// rng.index(0, 1, M) from one call.
__device__ __forceinline__ void bisect_where(const Rep& R, unsigned long long seq, int* p, int* b0) {
    Rng rng{make_uint2((uint32_t)R.key, (uint32_t)(R.key >> 32)), 1u, seq};
    const uint4 w = rng.call(0);
    *p = (int)(((uint64_t)w.x * (uint32_t)R.N) >> 32);
    *b0 = (int)(((uint64_t)w.y * (uint32_t)R.M) >> 32);
}

// Bisect::Attempt of the attempt in S (info, window, draws) up to the level-0
// decision, on the W wavefronts of a workgroup: the same numbers as
// propose_bisect_impl, whose single wavefront walks levels of sums one after the
// other.  Only the new midpoints depend on the level above them, so the first
// wavefront lays all of them down while the others sum the OLD actions (levels in
// turn); then every wavefront takes levels of the NEW sums; the levels' decisions
// follow in order.  The proposal goes to pr, its beads and phase chains to the
// buffers given; after the last barrier S.info holds its status and moved beads.
template <int W>
__device__ __forceinline__ void bisect_levels(const Rep& R, BisectLds& S, int w, int lane, Prop* pr, double* beads,
                                              double2* phase, int buf) {
    const int n = R.n_level, nb = 1 << n, M = R.M, p = S.info[1], b0 = S.info[2];
    const int p2 = label_after_wrap(R, p);
    // (see propose_bisect_impl)
    const bool wraps = (nb % M) == 0 && p2 == p;
    if (w == 0) {
        int g = 3 * lane;
        for (int level = n - 1; level >= 0; --level) {
            const int skip = 1 << level, nmid = wraps ? 0 : nb >> (level + 1);
            const double sigma = sqrt(R.lambda * (R.tau * skip));
            if (lane < nmid) {
#pragma clang fp contract(off)
                const int a = 2 * lane * skip, b = a + skip, c = a + 2 * skip;
                for (int d = 0; d < 3; ++d) {
                    const double dn = minimg(sigma * S.z[g + d], R.L, R.iL);
                    const double t = minimg(S.x_new[c][d] - S.x_new[a][d], R.L, R.iL);
                    const double rbar = S.x_new[a][d] + 0.5 * t;
                    S.x_new[b][d] = rbar + dn;
                }
            }
            WaveSync{}();
            g += 3 * nmid;
        }
    }
    for (int half = 0; half < 2; ++half) {
        // half 0: OLD, beside the midpoints; half 1: NEW
        const double(*x)[3] = half ? S.x_new : S.x_old;
        const int first = half ? w : w - 1, step = half ? W : W - 1;
        for (int level = first < 0 ? n : first; level < n; level += step) {
            const int skip = 1 << level, nmid = wraps ? 0 : nb >> (level + 1), nlinks = wraps ? 0 : nb >> level;
            const double level_tau = R.tau * skip;
            const double i4lt_b = 1. / (4. * R.lambda * (0.5 * R.tau * (double)skip));
            double lsp = 0., k = 0.;
            if (lane < nmid) {
#pragma clang fp contract(off)
                const int a = 2 * lane * skip, b = a + skip, c = a + 2 * skip;
                double dd[3];
                if (half) {
                    const double sigma = sqrt(R.lambda * level_tau);
                    // the levels above drew for 1 + 2 + ... + nmid / 2 midpoints
                    const int g = 3 * (nmid - 1 + lane);
                    for (int d = 0; d < 3; ++d) dd[d] = minimg(sigma * S.z[g + d], R.L, R.iL);
                } else {
                    for (int d = 0; d < 3; ++d) {
                        const double t = minimg(x[c][d] - x[a][d], R.L, R.iL);
                        const double rbar = x[a][d] + 0.5 * t;
                        dd[d] = minimg(x[b][d] - rbar, R.L, R.iL);
                    }
                }
                lsp = -free_neg_log(&R.bis[level], R.bis_images, i4lt_b, dd);
            }
            const double i4lt_k = 1. / (4. * R.lambda * level_tau);
            for (int i = lane; i < nlinks; i += kWave) {
                const int a = i * skip, b = a + skip;
                double dd[3];
                for (int d = 0; d < 3; ++d) dd[d] = minimg(x[a][d] - x[b][d], R.L, R.iL);
                k += free_neg_log(&R.kin[level], R.kin_images, i4lt_k, dd);
            }
            lsp = wave_sum(lsp);
            k = wave_sum(k);
            if (lane == 0) {
                S.sums[2 * half][level] = lsp;
                S.sums[2 * half + 1][level] = k;
            }
        }
        __syncthreads();
    }
    const int nm = wraps ? 0 : nb - 1;
    if (w == 0) {
        // the levels' decisions, a log of each level's uniform per lane
        const double lu = lane < n ? log(S.u[lane]) : 0.;
        double prev = 0., lsr = 0., ko = 0., kn = 0.;
        int status = 1;
        for (int level = n - 1; level >= 0; --level) {
            lsr = -S.sums[2][level] + S.sums[0][level];
            ko = S.sums[1][level];
            kn = S.sums[3][level];
            if (level == 0) break;
            const double old_action = 0. + ko, new_action = 0. + kn;
            const double change = new_action - old_action;
            const double la = lsr - change + prev;
            if (la < __shfl(lu, level)) {
                status = 2;
                break;
            }
            prev = change;
        }
        if (lane == 0) {
            S.info[4] = status;
            S.info[5] = status == 1 ? nm : 0;
            pr->status = status;
            pr->move = 0;
            pr->p = p;
            pr->p2 = p2;
            // (see propose_bisect_impl)
            pr->generic = status == 1 && (p2 != p) && (b0 + nb > M);
            pr->buf = buf;
            pr->b0 = b0;
            pr->n_links = R.pair_type ? nb : 0;
            pr->first = (b0 + 1) % M;
            pr->count = status == 1 ? nm : 0;
            pr->lsr = lsr;
            pr->k_old = ko;
            pr->k_new = kn;
            pr->prev = prev;
            pr->u0 = S.u[0];
            pr->tape_next = 0;
        }
    }
    const int tid = w * kWave + lane;
    for (int t = tid; t < 3 * nm; t += W * kWave) beads[t] = S.x_new[1 + t / 3][t % 3];
    if (R.use_long_range) {
        const int stride = R.max_idx + 1;
        for (int t = tid; t < 6 * nm; t += W * kWave) {
            const int m = t / 6, c = t % 6, d = c % 3;
            phase_chain((c / 3 ? S.x_new[m + 1][d] : S.x_old[m + 1][d]) * R.box, R.max_idx,
                        phase + ((size_t)m * 6 + c) * stride);
        }
    }
    __syncthreads();
}

// Bisect::Attempt up to the level-0 decision, one wavefront (lane 0..63) on
// replica R; items: also write the round's rho_k work items.
template <class Sync>
__device__ __forceinline__ void propose_bisect_impl(const Rep& R, int lane, Sync sync, bool items, BisectLds& S) {
    Prop* pr = R.prop;
    if (lane == 0) bisect_take(R, S);
    sync();
    if (!S.info[0]) {
        if (lane == 0) pr->status = 0;
        if (items) rho_items_write(R, 0, 0, 0, 0, lane);
        return;
    }
    const int n = R.n_level, nb = 1 << n, N = R.N, M = R.M;
    const bool tape = R.tape != nullptr;
    int bad = 0;
    if (lane == 0) {
        int p, b0;
        long long cur = 0;
        if (tape) {
            cur = *R.tape_cursor;
            p = (int)tape_get(R, cur, &bad);
            b0 = (int)tape_get(R, cur + 1, &bad);
            cur += 2;
            if (p < 0 || p >= N || b0 < 0 || b0 >= M) {
                bad = 1;
                p = 0;
                b0 = 0;
            }
        } else {
            bisect_where(R, S.seq, &p, &b0);
        }
        S.info[1] = p;
        S.info[2] = b0;
        S.info[3] = bad;
        S.cur = cur;
    }
    sync();
    const int p = S.info[1], b0 = S.info[2];
    // the chain walked from (p, b0) carries label p2 after the wrap
    const int p2 = label_after_wrap(R, p);
    // 2^n_level == M and the chain closes on itself: the window's last bead is
    // its first one, so the reference's bead walks visit no midpoint and no
    // kinetic link (bisect_class.h:51-58,78)
    const bool wraps = (nb % M) == 0 && p2 == p;
    bisect_window(R, lane, S, p, p2, b0, !tape);
    sync();
    long long cur = S.cur;
    double prev = 0.;
    int g_base = 0;  // normals drawn so far (device RNG indexing)
    for (int level = n - 1; level >= 0; --level) {
        const int skip = 1 << level;
        const int nmid = wraps ? 0 : nb >> (level + 1);
        const double level_tau = R.tau * skip;
        const double sigma = sqrt(R.lambda * level_tau);
        const double i4lt_b = 1. / (4. * R.lambda * (0.5 * R.tau * (double)skip));
        double lspo = 0., lspn = 0.;
        if (lane < nmid) {
#pragma clang fp contract(off)
            const int a = 2 * lane * skip, b = a + skip, c = a + 2 * skip;
            double t[3], rbar[3], dold[3], dnew[3];
            for (int d = 0; d < 3; ++d) {
                t[d] = minimg(S.x_old[c][d] - S.x_old[a][d], R.L, R.iL);
                rbar[d] = S.x_old[a][d] + 0.5 * t[d];
                dold[d] = minimg(S.x_old[b][d] - rbar[d], R.L, R.iL);
            }
            for (int d = 0; d < 3; ++d) {
                double z;
                if (tape)
                    z = tape_get(R, cur + 3 * lane + d, &bad);
                else
                    z = S.z[g_base + 3 * lane + d];
                dnew[d] = sigma * z;
                dnew[d] = minimg(dnew[d], R.L, R.iL);
                t[d] = minimg(S.x_new[c][d] - S.x_new[a][d], R.L, R.iL);
                rbar[d] = S.x_new[a][d] + 0.5 * t[d];
                S.x_new[b][d] = rbar[d] + dnew[d];
            }
            lspo = -free_neg_log(&R.bis[level], R.bis_images, i4lt_b, dold);
            lspn = -free_neg_log(&R.bis[level], R.bis_images, i4lt_b, dnew);
        }
        sync();
        const int nlinks = wraps ? 0 : nb >> level;
        const double i4lt_k = 1. / (4. * R.lambda * level_tau);
        double ko = 0., kn = 0.;
        for (int i = lane; i < nlinks; i += kWave) {
            const int a = i * skip, b = a + skip;
            double dd[3];
            for (int d = 0; d < 3; ++d) dd[d] = minimg(S.x_old[a][d] - S.x_old[b][d], R.L, R.iL);
            ko += free_neg_log(&R.kin[level], R.kin_images, i4lt_k, dd);
            for (int d = 0; d < 3; ++d) dd[d] = minimg(S.x_new[a][d] - S.x_new[b][d], R.L, R.iL);
            kn += free_neg_log(&R.kin[level], R.kin_images, i4lt_k, dd);
        }
        lspo = wave_sum(lspo);
        lspn = wave_sum(lspn);
        ko = wave_sum(ko);
        kn = wave_sum(kn);
        const double lsr = -lspn + lspo;
        cur += 3 * nmid;
        g_base += 3 * nmid;
        double u;
        if (tape)
            u = tape_get(R, cur, &bad);
        else
            u = S.u[level];
        cur += 1;
        if (level > 0) {
            const double old_action = 0. + ko, new_action = 0. + kn;
            const double change = new_action - old_action;
            const double la = lsr - change + prev;
            if (la < log(u)) {
                if (lane == 0) {
                    pr->status = 2;
                    pr->move = 0;
                    pr->p = p;
                    pr->p2 = p2;
                    pr->generic = 0;
                    pr->buf = 0;
                    pr->b0 = b0;
                    pr->count = 0;
                    pr->tape_next = cur;
                }
                if (items) rho_items_write(R, 0, 2, 0, 0, lane);
                return;
            }
            prev = change;
        } else {
            const int any_bad = __any(bad);
            const int status = (any_bad || S.info[3]) ? 3 : 1;
            if (lane == 0) {
                pr->status = status;
                pr->move = 0;
                pr->p = p;
                pr->p2 = p2;
                // moved beads on both sides of the wrap under two labels: the
                // label-general pair kernel takes the proposal
                pr->generic = (p2 != p) && (b0 + nb > M);
                pr->buf = 0;
                pr->b0 = b0;
                pr->n_links = R.pair_type ? nb : 0;  // no pair action: no links to evaluate
                pr->first = (b0 + 1) % M;
                pr->count = wraps ? 0 : nb - 1;
                pr->lsr = lsr;
                pr->k_old = ko;
                pr->k_new = kn;
                pr->prev = prev;
                pr->u0 = u;
                pr->tape_next = cur;
            }
            for (int j = lane; j < (wraps ? 0 : nb - 1); j += kWave)
                for (int d = 0; d < 3; ++d) R.prop_new[3 * j + d] = S.x_new[j + 1][d];
            if (R.use_long_range) {
                for (int t = lane; t < (wraps ? 0 : 6 * (nb - 1)); t += kWave)
                    moved_phase_chain(R, t / 6, t % 6, S.x_old[t / 6 + 1], S.x_new[t / 6 + 1]);
                if (items) rho_items_write(R, 0, status, wraps ? 0 : nb - 1, (b0 + 1) % M, lane);
            }
        }
    }
}

__device__ __forceinline__ void propose_bisect_body(const Rep* __restrict__ reps, int n_reps) {
    const int r = blockIdx.x;
    if (r >= n_reps) return;
    __shared__ BisectLds S;
    propose_bisect_impl(reps[r], (int)threadIdx.x, BlockSync{}, true, S);
}

// DisplaceParticle::Attempt (displace_particle_class.h:28-72): NEW beads only.
// Kinetic::GetAction(0, M, {p}) walks from (p, 0) to the bead M links later:
// the walk is empty when the particle's path closes on itself, else it holds
// the wrap link (p, M-1) -> (perm[p], 0), the one link of the walk a rigid shift
// changes.  The link into (p, 0) from (iperm[p], M-1), which the shift also
// changes, is outside the walk and not counted, as in the reference.
// lane: the thread's index among the nthr that run the proposal (its draws and
// record on thread 0; the moved slices' positions, phase chains and rho_k
// items over all nthr).
template <class Sync>
__device__ __forceinline__ void propose_displace_impl(const Rep& R, int lane, Sync sync, bool items,
                                                      int nthr = kWave) {
    __shared__ int s_act, s_p, s_status;
    __shared__ double s_dr[3];
    Prop* pr = R.prop;
    if (lane == 0) {
        Counters* c = R.cnt;
        unsigned int rem = c->remaining;
        s_act = rem > 0;
        if (rem > 0) {
            c->remaining = rem - 1;
            unsigned long long seq = c->seq;
            c->seq = seq + 1;
            int bad = 0, p;
            double u0;
            long long cur = 0;
            if (R.tape) {
                cur = *R.tape_cursor;
                p = (int)tape_get(R, cur, &bad);
                for (int d = 0; d < 3; ++d) s_dr[d] = tape_get(R, cur + 1 + d, &bad);
                u0 = tape_get(R, cur + 4, &bad);
                cur += 5;
                if (p < 0 || p >= R.N) {
                    bad = 1;
                    p = 0;
                }
            } else {
                Rng rng{make_uint2((uint32_t)R.key, (uint32_t)(R.key >> 32)), 2u, seq};
                p = (int)rng.index(0, 0, R.N);
                s_dr[0] = R.step * (rng.unif(1, 0) - 0.5);
                s_dr[1] = R.step * (rng.unif(1, 1) - 0.5);
                s_dr[2] = R.step * (rng.unif(2, 0) - 0.5);
                u0 = rng.unif(2, 1);
            }
            s_p = p;
            double k_old = 0., k_new = 0.;
            const int pn = label_after_wrap(R, p);
            if (pn != p) {
                const double i4lt = 1. / (4. * R.lambda * R.tau);
                double dd[3];
                for (int d = 0; d < 3; ++d) dd[d] = minimg(pos_at(R, d, R.M - 1, p) - pos_at(R, d, 0, pn), R.L, R.iL);
                k_old = free_neg_log(&R.kin[0], R.kin_images, i4lt, dd);
                for (int d = 0; d < 3; ++d)
                    dd[d] = minimg((pos_at(R, d, R.M - 1, p) + s_dr[d]) - pos_at(R, d, 0, pn), R.L, R.iL);
                k_new = free_neg_log(&R.kin[0], R.kin_images, i4lt, dd);
            }
            pr->status = bad ? 3 : 1;
            pr->move = 1;
            pr->p = p;
            pr->p2 = p;
            pr->generic = 0;
            pr->buf = 0;
            pr->b0 = 0;
            pr->n_links = R.pair_type ? R.M : 0;
            pr->first = 0;
            pr->count = R.M;
            pr->lsr = 0.;
            pr->k_old = k_old;
            pr->k_new = k_new;
            pr->prev = 0.;
            pr->u0 = u0;
            pr->tape_next = cur;
            s_status = bad ? 3 : 1;
        } else {
            pr->status = 0;
        }
    }
    sync();
    if (!s_act) {
        if (items) rho_items_write(R, 1, 0, 0, 0, lane, nthr);
        return;
    }
    const int p = s_p;
    for (int s = lane; s < R.M; s += nthr)
        for (int d = 0; d < 3; ++d) R.prop_new[3 * s + d] = pos_at(R, d, s, p) + s_dr[d];
    if (R.use_long_range)
        for (int t = lane; t < 6 * R.M; t += nthr) {
            const int s = t / 6;
            double xo[3], xn[3];
            for (int d = 0; d < 3; ++d) {
                xo[d] = pos_at(R, d, s, p);
                xn[d] = xo[d] + s_dr[d];
            }
            moved_phase_chain(R, s, t % 6, xo, xn);
        }
    if (R.use_long_range) if (items) rho_items_write(R, 1, s_status, R.M, 0, lane, nthr);
}

__device__ __forceinline__ void propose_displace_body(const Rep* __restrict__ reps, int n_reps) {
    const int r = blockIdx.x;
    if (r >= n_reps) return;
    propose_displace_impl(reps[r], (int)threadIdx.x, BlockSync{}, true);
}

// ---------------------------------------------------------------------------
// K1: short-range pair action of the moved particle on the window links,
// OLD and NEW (pair_action_class.h:279-290), one wavefront per (replica, link).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void pair_block(const Rep* __restrict__ reps, const uint2* __restrict__ items, int n_items,
                                           int blk) {
    const int item = blk * (kPairBlock / kWave) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & (kWave - 1);
    if (item >= n_items) return;
    const uint2 it = items[item];
    const Rep& R = reps[it.x];
    const Prop pr = *R.prop;
    if (pr.status != 1 || pr.generic) return;
    const int j = (int)it.y;
    if (j >= pr.n_links) return;
    const int M = R.M, N = R.N, p = pr.p;
    const int s0 = (pr.b0 + j) % M, s1 = (s0 + 1) % M;
    double po0[3], po1[3], pn0[3], pn1[3];
    for (int d = 0; d < 3; ++d) {
        po0[d] = pos_at(R, d, s0, p);
        po1[d] = pos_at(R, d, s1, p);
        pn0[d] = pos_new(R, pr, d, s0);
        pn1[d] = pos_new(R, pr, d, s1);
    }
    double uo = 0., un = 0.;
    for (int q = lane; q < N; q += kWave) {
        if (q == p) continue;
        double q0[3], q1[3];
        for (int d = 0; d < 3; ++d) {
            q0[d] = pos_at(R, d, s0, q);
            q1[d] = pos_at(R, d, s1, q);
        }
        LinkGeom g;
        link_geom(po0, q0, po1, q1, R.L, R.iL, g);
        uo += pair_u(R, g.r, g.rp, g.s);
        link_geom(pn0, q0, pn1, q1, R.L, R.iL, g);
        un += pair_u(R, g.r, g.rp, g.s);
    }
    uo = wave_sum(uo);
    un = wave_sum(un);
    if (lane == 0) {
        R.pair_part[j] = make_double2(uo, un);
    }
}

// Device-side kernel clocks.  Block 0 of a timed launch (the first dispatched)
// stores its start on the constant-rate wall clock; every block stores its end
// in a slot of its own (plain stores; grids above KT_SLOTS blocks fold several
// blocks into a slot with atomicMax).  The round's decide kernel (its first
// wavefront) takes the latest end of each class, adds end - start to a running
// sum and clears the slots: a launch is timed from its first block's start to
// its last block's end, whatever runs beside it on other streams.
// kt[c]: open start of class c (0 = none); kt[2 + 2c], kt[3 + 2c]: summed
// ticks and launches; kt[KT_END + c * KT_SLOTS + slot]: block ends.
enum { KT_RHO = 0, KT_PAIR = 1, KT_CLASSES = 2, KT_SLOTS = 1024, KT_END = 8, KT_WORDS = KT_END + KT_CLASSES * KT_SLOTS };
__device__ __forceinline__ void kt_begin(unsigned long long* kt, int cls) {
    if (kt && blockIdx.x == 0 && threadIdx.x == 0) kt[cls] = (unsigned long long)wall_clock64();
}
__device__ __forceinline__ void kt_end(unsigned long long* kt, int cls) {
    if (!kt) return;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long* slot = kt + KT_END + cls * KT_SLOTS + blockIdx.x % KT_SLOTS;
        const unsigned long long now = (unsigned long long)wall_clock64();
        if (gridDim.x <= KT_SLOTS)
            *slot = now;
        else
            atomicMax(slot, now);
    }
}
// called by one full wavefront
__device__ __forceinline__ void kt_close(unsigned long long* kt) {
    const int lane = threadIdx.x & (kWave - 1);
    for (int c = 0; c < KT_CLASSES; ++c) {
        unsigned long long e = 0;
        for (int t = lane; t < KT_SLOTS; t += kWave) {
            unsigned long long* slot = kt + KT_END + c * KT_SLOTS + t;
            e = max(e, *slot);
            *slot = 0ull;
        }
        for (int o = kWave / 2; o > 0; o >>= 1) e = max(e, (unsigned long long)__shfl_xor(e, o));
        if (lane == 0) {
            const unsigned long long b = kt[c];
            if (b && e >= b) {
                kt[2 + 2 * c] += e - b;
                kt[3 + 2 * c] += 1ull;
            }
            kt[c] = 0ull;
        }
    }
}

// K1 with the link-action tables staged in LDS: one 1024-thread workgroup per
// replica loads its B-spline tables once, then each wavefront takes window links
// j = w, w + 16, ...; lanes run over the partners q.
constexpr int kPairLdsBlock = 1024;
// The window links j = j0, j0 + step, ... of a proposal, one wavefront: lanes
// run over the partners q; the OLD and NEW sums of link j go to pair_part[j]
// (COH: as agent-scope atomic stores).
// One lane's OLD and NEW sums of window link j over the partners q_lo + lane,
// q_lo + lane + 64, ... below q_hi (at least one: the lanes without one load q_lo).
// ONE: ranges of at most 64 partners take one each (k_pair_lds has none; the
// second copy of the evaluation would cost it registers).
template <int PT, int NORD, bool ONE = false>
__device__ __forceinline__ void pair_link_range(const Rep& R, const double* lds, const Prop& pr, int j, int q_lo,
                                                int q_hi, int lane, double& uo, double& un) {
    const int M = R.M, p = pr.p;
    const int s0 = (pr.b0 + j) % M, s1 = (s0 + 1) % M;
    double po0[3], po1[3], pn0[3], pn1[3];
    for (int d = 0; d < 3; ++d) {
        po0[d] = pos_at(R, d, s0, p);
        po1[d] = pos_at(R, d, s1, p);
        pn0[d] = pos_new(R, pr, d, s0);
        pn1[d] = pos_new(R, pr, d, s1);
    }
    uo = 0.;
    un = 0.;
    if (ONE && q_hi - q_lo <= kWave) {
        // one partner per lane
        const int q = q_lo + lane;
        const bool ok = q < q_hi && q != p;
        const int qa = q < q_hi ? q : q_lo;
        double a0[3], a1[3];
        for (int d = 0; d < 3; ++d) {
            a0[d] = pos_at(R, d, s0, qa);
            a1[d] = pos_at(R, d, s1, qa);
        }
        double r, rp, s2;
        link_rr_s2(po0, a0, po1, a1, R.L, R.iL, r, rp, s2);
        const double uo1 = pair_u_lds_s2<PT, NORD>(R, lds, r, rp, s2);
        link_rr_s2(pn0, a0, pn1, a1, R.L, R.iL, r, rp, s2);
        const double un1 = pair_u_lds_s2<PT, NORD>(R, lds, r, rp, s2);
        uo = ok ? uo1 : 0.;
        un = ok ? un1 : 0.;
    } else {
        const int N = q_hi;
        // two partners per lane per step: independent evaluation chains for the scheduler
        for (int q = q_lo + lane; q < N; q += 2 * kWave) {
            const int q2 = q + kWave;
            const bool ok1 = q != p, ok2 = (q2 < N) && (q2 != p);
            const int qq = (q2 < N) ? q2 : q;
            double a0[3], a1[3], b0[3], b1[3];
            for (int d = 0; d < 3; ++d) {
                a0[d] = pos_at(R, d, s0, q);
                a1[d] = pos_at(R, d, s1, q);
                b0[d] = pos_at(R, d, s0, qq);
                b1[d] = pos_at(R, d, s1, qq);
            }
            double r, rp, s2;
            link_rr_s2(po0, a0, po1, a1, R.L, R.iL, r, rp, s2);
            const double uo1 = pair_u_lds_s2<PT, NORD>(R, lds, r, rp, s2);
            link_rr_s2(pn0, a0, pn1, a1, R.L, R.iL, r, rp, s2);
            const double un1 = pair_u_lds_s2<PT, NORD>(R, lds, r, rp, s2);
            link_rr_s2(po0, b0, po1, b1, R.L, R.iL, r, rp, s2);
            const double uo2 = pair_u_lds_s2<PT, NORD>(R, lds, r, rp, s2);
            link_rr_s2(pn0, b0, pn1, b1, R.L, R.iL, r, rp, s2);
            const double un2 = pair_u_lds_s2<PT, NORD>(R, lds, r, rp, s2);
            uo += (ok1 ? uo1 : 0.) + (ok2 ? uo2 : 0.);
            un += (ok1 ? un1 : 0.) + (ok2 ? un2 : 0.);
        }
    }
}

template <int PT, int NORD, bool COH = false>
__device__ __forceinline__ void pair_links_lds(const Rep& R, const double* lds, const Prop& pr, int j0, int step,
                                               int lane) {
    for (int j = j0; j < pr.n_links; j += step) {
        double uo, un;
        pair_link_range<PT, NORD>(R, lds, pr, j, 0, R.N, lane, uo, un);
        uo = wave_sum(uo);
        un = wave_sum(un);
        if (lane == 0) {
            if (COH)
                coh_store2(R.pair_part + j, make_double2(uo, un));
            else
                R.pair_part[j] = make_double2(uo, un);
        }
    }
}

// The window links of a proposal on a W-wavefront workgroup (part of bpr for
// the replica), ns = pair_split<W>(N, qpw) wavefronts per link: wavefront w takes
// link jb + w / ns and partner range w % ns (pair_range; an empty one adds nothing).
// A link's sum adds its ranges' wavefront sums in range
// order; with ns = 1 it is pair_links_lds's.  Every wavefront of the
// workgroup calls it (it holds workgroup barriers); wpart: W entries of LDS.
template <int PT, int NORD, bool COH, int W>
__device__ __forceinline__ void pair_links_split(const Rep& R, const double* lds, const Prop& pr, int part, int bpr,
                                                 int qpw, int w, int lane, double2* wpart) {
    const int ns = pair_split<W>(R.N, qpw), lpb = W / ns;
    const int2 qr = pair_range(R.N, ns, w % ns);
    for (int jb = part * lpb; jb < pr.n_links; jb += bpr * lpb) {
        const int j = jb + w / ns;
        double uo = 0., un = 0.;
        if (w < lpb * ns && j < pr.n_links && qr.x < qr.y) {
            pair_link_range<PT, NORD, true>(R, lds, pr, j, qr.x, qr.y, lane, uo, un);
            uo = wave_sum(uo);
            un = wave_sum(un);
        }
        if (lane == 0) wpart[w] = make_double2(uo, un);
        __syncthreads();
        if ((int)threadIdx.x < lpb && jb + (int)threadIdx.x < pr.n_links) {
            double so = wpart[threadIdx.x * ns].x, sn = wpart[threadIdx.x * ns].y;
            for (int kk = 1; kk < ns; ++kk) {
                so += wpart[threadIdx.x * ns + kk].x;
                sn += wpart[threadIdx.x * ns + kk].y;
            }
            if (COH)
                coh_store2(R.pair_part + jb + threadIdx.x, make_double2(so, sn));
            else
                R.pair_part[jb + threadIdx.x] = make_double2(so, sn);
        }
        __syncthreads();
    }
}

// The window links of a proposal from the tables in global memory (tabulated
// Ilkka actions and grids that are not uniform), as pair_links_split: a link's
// OLD and NEW sums are wavefronts of their own (each is a serial chain of a
// grid search and loads that depend on it, which a small batch waits for in
// full), and so are its partner ranges.  An Ilkka table's axes are searched in
// LDS where the launch has room for them (ax_doubles values).  A range's sum is
// the one that k_pair forms over the same partners.  A bisection round of 24
// replicas of N = 33, M = 32: 31.6 us in three launches with k_pair, 20.6 so; of
// one replica of N = 200, M = 64: 62.7 and 24.0.
template <int W>
__host__ __device__ __forceinline__ int general_split(int N, int qpw) {
    return 2 * pair_split<W / 2>(N, qpw);
}
constexpr int kAxDoubles = 1024;
template <bool COH, int W>
__device__ __forceinline__ void pair_links_general(const Rep& R, double* lds, int ax_doubles, const Prop& pr, int part,
                                                   int bpr, int qpw, int w, int lane, double2* wpart) {
    const int ns = general_split<W>(R.N, qpw), lpb = W / ns, nq = ns / 2;
    const int q_len = ((R.N + nq - 1) / nq + kWave - 1) / kWave * kWave;
    const bool axes = R.pair_type == 3 && R.u2.nx + R.u2.ny <= ax_doubles;
    if (axes) {
        for (int t = threadIdx.x; t < R.u2.nx; t += W * kWave) lds[t] = R.u2.x[t];
        for (int t = threadIdx.x; t < R.u2.ny; t += W * kWave) lds[R.u2.nx + t] = R.u2.y[t];
        __syncthreads();
    }
    Spl2 T = R.u2;
    T.x = lds;
    T.y = lds + R.u2.nx;
    const int M = R.M, p = pr.p;
    for (int jb = part * lpb; jb < pr.n_links; jb += bpr * lpb) {
        const int j = jb + w / ns, k = w % ns;
        double u = 0.;
        if (w < lpb * ns && j < pr.n_links) {
            const int s0 = (pr.b0 + j) % M, s1 = (s0 + 1) % M, q_lo = (k >> 1) * q_len, q_hi = min(R.N, q_lo + q_len);
            double p0[3], p1[3];
            for (int d = 0; d < 3; ++d) {
                p0[d] = (k & 1) ? pos_new(R, pr, d, s0) : pos_at(R, d, s0, p);
                p1[d] = (k & 1) ? pos_new(R, pr, d, s1) : pos_at(R, d, s1, p);
            }
            for (int q = q_lo + lane; q < q_hi; q += kWave) {
                if (q == p) continue;
                double q0[3], q1[3];
                for (int d = 0; d < 3; ++d) {
                    q0[d] = pos_at(R, d, s0, q);
                    q1[d] = pos_at(R, d, s1, q);
                }
                LinkGeom g;
                link_geom(p0, q0, p1, q1, R.L, R.iL, g);
                u += axes ? ilkka_u(R, T, R.u_long_r, R.r_u_min, R.r_u_max, g.r, g.rp, g.s)
                          : pair_u(R, g.r, g.rp, g.s);
            }
            u = wave_sum(u);
        }
        double* part_u = reinterpret_cast<double*>(wpart);
        if (lane == 0) part_u[w] = u;
        __syncthreads();
        if ((int)threadIdx.x < lpb && jb + (int)threadIdx.x < pr.n_links) {
            const double* f = part_u + threadIdx.x * ns;
            double so = f[0], sn = f[1];
            for (int kk = 2; kk < ns; kk += 2) {
                so += f[kk];
                sn += f[kk + 1];
            }
            if (COH)
                coh_store2(R.pair_part + jb + threadIdx.x, make_double2(so, sn));
            else
                R.pair_part[jb + threadIdx.x] = make_double2(so, sn);
        }
        __syncthreads();
    }
}

// Copies values [t_lo, n) of the tables a | b (a holds the first na) into lds
// with nthr threads, 16 values per thread at a time, every load issued before
// the stores that wait on it (a large table then costs a few load latencies
// instead of one per value).
__device__ __forceinline__ void stage_batched(double* lds, const double* a, const double* b, int na, int n, int t_lo,
                                              int nthr) {
    for (int t0 = t_lo + (int)threadIdx.x; t0 < n; t0 += 16 * nthr) {
        double v[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const int t = t0 + k * nthr;
            v[k] = t < n ? (t < na ? a[t] : b[t - na]) : 0.;
        }
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const int t = t0 + k * nthr;
            if (t < n) lds[t] = v[k];
        }
    }
}

template <int PT, int NORD, int BS>
__device__ __forceinline__ void pair_lds_block(const Rep* __restrict__ reps, int n_reps, int bpr) {
    extern __shared__ double lds[];
    // bpr workgroups per replica (when replicas are few): part takes every bpr-th
    // group of BS/64 links
    const int idx = xcd_remap(blockIdx.x, gridDim.x), r = idx / bpr, part = idx % bpr;
    if (r >= n_reps) return;
    const Rep R = reps[r];  // by value: the fields used stay in registers across the loops
    const Prop pr = *R.prop;
    if (pr.status != 1 || pr.generic) return;
    stage_batched(lds, R.bt_a.c, R.bt_b.c, R.bt_a.ncoef * R.bt_a.ncomp, R.lds_doubles, 0, BS);
    __syncthreads();
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    if (part * (BS / kWave) >= pr.n_links) return;
    pair_links_lds<PT, NORD>(R, lds, pr, part * (BS / kWave) + w, bpr * (BS / kWave), lane);
}


// PT: 1 all replicas Bare, 2 all David, 0 mixed (type read per replica);
// NORD: the David expansion order when all replicas share it, else 0
// BS: workgroup size; with BS < 1024 a CU keeps room for other kernels' waves
// (at most 128 VGPRs per wave whatever BS is)
template <int PT, int NORD, int BS = kPairLdsBlock>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(4))) void k_pair_lds(
    const Rep* __restrict__ reps, int n_reps, int bpr, unsigned long long* __restrict__ kt) {
    kt_begin(kt, KT_PAIR);
    pair_lds_block<PT, NORD, BS>(reps, n_reps, bpr);
    kt_end(kt, KT_PAIR);
}

__global__ __launch_bounds__(kPairBlock) void k_pair(const Rep* __restrict__ reps, const uint2* __restrict__ items,
                                                     int n_items, unsigned long long* __restrict__ kt) {
    kt_begin(kt, KT_PAIR);
    pair_block(reps, items, n_items, xcd_remap(blockIdx.x, gridDim.x));
    kt_end(kt, KT_PAIR);
}

// ---------------------------------------------------------------------------
// K2: incremental rho_k of the moved slices (Species::UpdateRhoK,
// species_class.h:406-425) written to the spare buffer, fused with the
// long-range action sums of CalcULong (bare_pair_action_class.h:153-172,
// david_pair_action_class.h:105-123) for OLD and NEW.
// ---------------------------------------------------------------------------
// One rho_k work item on a whole kRhoBlock-thread workgroup: its rho_k, k-table
// and phase-chain loads are all issued before the first wait; the item's
// (OLD, NEW) sums go to *d.part.  The caller separates items that reuse tab and
// red with a workgroup barrier.  COH: the sums go out as agent-scope atomic
// stores.
template <int KPT, bool NT, bool COH = false>
__device__ __forceinline__ void rho_item(const RhoItem& d, double2* tab, double (*red)[kRhoBlock / kWave]) {
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const int k0 = d.k0 + threadIdx.x;
    double2 rv[KPT];
    int kp[KPT];
    double cf[KPT];
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
        const int k = k0 + i * kRhoBlock;
        const bool ok = k < d.k1;
        rv[i] = ok ? ld2<NT>(d.rc + k) : make_double2(0., 0.);
        kp[i] = ok ? gld(d.kidx + k) : (128 | (128 << 8) | (128 << 16));
        cf[i] = ok ? gld(d.coef + k) : 0.;
    }
    const int nt = 6 * d.stride, tx = (int)threadIdx.x;
    const double2 t0 = tx < nt ? ld2<false>(d.ph + tx) : make_double2(0., 0.);
    const double2 t1 = tx + kRhoBlock < nt ? ld2<false>(d.ph + tx + kRhoBlock) : make_double2(0., 0.);
    if (tx < nt) tab[tx] = t0;
    if (tx + kRhoBlock < nt) tab[tx + kRhoBlock] = t1;
    __syncthreads();
    double ao = 0., an = 0.;
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
        const int k = k0 + i * kRhoBlock;
        const double2 en = phase_k(&tab[3 * d.stride], d.stride, kp[i]);
        const double2 eo = phase_k(tab, d.stride, kp[i]);
        double2 nv;
        nv.x = rv[i].x + (en.x - eo.x);
        nv.y = rv[i].y + (en.y - eo.y);
        if (k < d.k1) st2<NT>(d.rn + k, nv);
        ao += cf[i] * (rv[i].x * rv[i].x + rv[i].y * rv[i].y);
        an += cf[i] * (nv.x * nv.x + nv.y * nv.y);
    }
    ao = wave_sum(ao);
    an = wave_sum(an);
    if (lane == 0) {
        red[0][w] = ao;
        red[1][w] = an;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double to = 0., tn = 0.;
        for (int i = 0; i < kRhoBlock / kWave; ++i) {
            to += red[0][i];
            tn += red[1][i];
        }
        if (COH)
            coh_store2(d.part, make_double2(to, tn));
        else
            *d.part = make_double2(to, tn);
    }
}

// K2 with a fixed number of workgroups that loop over the work items: the
// launch then holds at most that many workgroups per CU, so a concurrent pair
// kernel on another stream always finds room on every CU.
// Each item is one descriptor (scalar loads, prefetched while the previous
// item computes).
template <int KPT, bool NT>
__global__ __launch_bounds__(kRhoBlock) void k_rho_loop(const RhoItem* __restrict__ items, int n_items,
                                                        unsigned long long* __restrict__ kt) {
    kt_begin(kt, KT_RHO);
    __shared__ double2 tab[6 * (kMaxIdx + 1)];
    __shared__ double red[2][kRhoBlock / kWave];
    int it = blockIdx.x;
    RhoItem d;
    if (it < n_items) d = items[it];
    for (; it < n_items; it += gridDim.x) {
        RhoItem nd;
        const int nx = it + gridDim.x;
        if (nx < n_items) nd = items[nx];
        if (d.valid) {
            rho_item<KPT, NT>(d, tab, red);
            __syncthreads();  // tab and red are reused by the next item
        }
        d = nd;
    }
    kt_end(kt, KT_RHO);
}

// ---------------------------------------------------------------------------
// K5: level-0 Metropolis decision and commit (bisect_class.h:100-123,24-36,127-139;
// displace_particle_class.h:68-86), one wavefront per replica.
// ---------------------------------------------------------------------------
template <class Sync>
__device__ __forceinline__ void commit_impl(const Rep& R, const Prop& pr, int lane, int acc, const double* pre,
                                            unsigned char pre_sel, const double* beads, Sync sync);
// Raises the context's replay-error flag, a word of host memory that the host reads
// after the stage.
__device__ __forceinline__ void ctx_error_set(const Rep& R) {
    __hip_atomic_store(R.ctx_error, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// The counters, accept flag and action trace of one decided attempt (one lane):
// status as decided (3: replay error), po/pn/lo/ln the summed level-0 terms.
__device__ __forceinline__ void decide_book(const Rep& R, const Prop& pr, int acc, int status, double po, double pn,
                                            double lo, double ln) {
    Counters* c = R.cnt;
    if (pr.status == 1 && pr.move != 3) {  // the round's pair and rho_k work, for the roofline figures
        c->rho_slicek += (unsigned long long)pr.count * (unsigned long long)R.nk;
        if (R.pair_type) c->pair_links += 2ull * (unsigned long long)pr.n_links * (unsigned long long)(R.N - 1);
    }
    if (pr.move == 0) {
        c->bis_att += 1;
        c->bis_acc += acc;
        c->bead_updates += (1ull << R.n_level) - 1;
    } else if (pr.move == 3) {
        // Move::DoEvent counts every attempt; PermBisect counts per cycle length
        // the attempts that reached the bisection (perm_bisect_class.h:66-87)
        unsigned long long* pc = R.perm_cnt;
        pc[0] += 1;
        pc[1] += acc;
        if (pr.n_chain > 0) {
            pc[2 + pr.n_chain - 1] += 1;
            pc[2 + R.N + pr.n_chain - 1] += acc;
        }
        c->bead_updates += (unsigned long long)pr.n_chain * ((1ull << pr.n_level) - 1);
    } else {
        c->dis_att += 1;
        c->dis_acc += acc;
        c->bead_updates += R.M;
    }
    unsigned int si = c->stage_i;
    if (si < R.accepted_cap) R.accepted[si] = (unsigned char)acc;
    if (R.act_trace && si < R.accepted_cap) {
        // the terms of the level-0 decision as summed (NaN: no level-0 decision)
        double* t = R.act_trace + (size_t)si * kTraceWords;
        const bool l0 = pr.status == 1;
        const double nan = __builtin_nan("");
        t[0] = l0 ? pr.k_old : nan;
        t[1] = l0 ? pr.k_new : nan;
        t[2] = l0 ? po : nan;
        t[3] = l0 ? pn : nan;
        t[4] = l0 ? R.long_scale * lo : nan;
        t[5] = l0 ? R.long_scale * ln : nan;
        t[6] = l0 ? pr.lsr : nan;
        t[7] = l0 ? pr.prev : nan;
    }
    c->stage_i = si + 1;
    if (status == 3) {  // replay tape overrun / bad draw
        c->error = 1;
        ctx_error_set(R);
    }
}

// What decide_impl hands to a later decide_book when the caller defers it.
struct DecideOut {
    Prop pr;
    double po, pn, lo, ln;
    int acc, status;  // status 0: nothing was decided
};

// COH: the pair and rho_k sums are read with agent-scope atomic loads (they were
// written in the same launch, by workgroups on any XCD).  hint_links /
// hint_rho >= 0: the pair and rho_k sums the proposal is expected to hold,
// loaded before the proposal itself (summed again if it holds others).  out:
// the bookkeeping is left to the caller (decide_book), which receives what it
// needs there.  Returns the particle whose beads an accepted one-particle move
// committed, else -1.
template <bool COH = false, class Sync>
__device__ __forceinline__ int decide_impl(const Rep& R, int lane, Sync sync, int hint_links = -1, int hint_rho = -1,
                                           DecideOut* out = nullptr) {
    Prop* prp = R.prop;
    double po = 0., pn = 0., lo = 0., ln = 0.;
    if (hint_links >= 0) {
        for (int j = lane; j < hint_links; j += kWave) {
            const double2 v = COH ? coh_load2(R.pair_part + j) : R.pair_part[j];
            po += v.x;
            pn += v.y;
        }
        for (int j = lane; j < hint_rho; j += kWave) {
            const double2 v = COH ? coh_load2(R.rho_part + j) : R.rho_part[j];
            lo += v.x;
            ln += v.y;
        }
    }
    const Prop pr = *prp;
    if (pr.status == 0) return -1;
    const double* beads = COH ? prop_beads(R, pr) : R.prop_new;
    // the commit's loads of a one-particle move, issued before the sums: the
    // lane's first new bead and the selector of its slice
    double pre[3] = {0., 0., 0.};
    unsigned char pre_sel = 0;
    if (pr.status == 1 && pr.move != 3 && lane < pr.count) {
        for (int d = 0; d < 3; ++d) pre[d] = beads[3 * lane + d];
        if (R.use_long_range) pre_sel = R.sel[(pr.first + lane) % R.M];
    }
    if (pr.status == 1) {
        const int np = R.use_long_range ? pr.count * R.n_chunks : 0;
        if (pr.n_links != hint_links || np != hint_rho) {
            po = pn = lo = ln = 0.;
            for (int j = lane; j < pr.n_links; j += kWave) {
                const double2 v = COH ? coh_load2(R.pair_part + j) : R.pair_part[j];
                po += v.x;
                pn += v.y;
            }
            for (int j = lane; j < np; j += kWave) {
                const double2 v = COH ? coh_load2(R.rho_part + j) : R.rho_part[j];
                lo += v.x;
                ln += v.y;
            }
        }
        po = wave_sum(po);
        pn = wave_sum(pn);
        lo = wave_sum(lo);
        ln = wave_sum(ln);
    }
    __shared__ int s_acc;
    int acc = 0, status = pr.status;
    long long tape_next = pr.tape_next;
    if (lane == 0) {
        if (pr.status == 1) {
            const double pair_old = po + R.long_scale * lo, pair_new = pn + R.long_scale * ln;
            const double old_action = (0. + pr.k_old) + pair_old;
            const double new_action = (0. + pr.k_new) + pair_new;
            const double change = new_action - old_action;
            const double la = pr.lsr - change + pr.prev;
            acc = !(la < log(pr.u0));
        }
        if (acc && pr.move == 3 && pr.tab_on) {
            // PermBisectTable: the table of the new path (perm_bisect_table_class.h:216-225)
            int bad = 0;
            const double u = R.tape ? tape_get(R, tape_next++, &bad) : pr.u_tab;
            if (bad) status = 3;
            acc = !(pr.tab_ratio < u);
        }
        s_acc = acc;
    }
    sync();
    commit_impl(R, pr, lane, s_acc, pre, pre_sel, beads, sync);
    // bookkeeping after the commit's stores are issued
    if (lane == 0) {
        if (R.tape) *R.tape_cursor = tape_next;
        if (out) {
            out->pr = pr;
            out->acc = acc;
            out->status = status;
            out->po = po;
            out->pn = pn;
            out->lo = lo;
            out->ln = ln;
        } else {
            decide_book(R, pr, acc, status, po, pn, lo, ln);
        }
        prp->status = 0;
    }
    return (pr.status == 1 && s_acc && pr.move != 3) ? pr.p : -1;
}

// The commit of a decided proposal (part of decide_impl): Bisect::Accept /
// DisplaceParticle::Accept of its beads, or of every chain of a permuting
// proposal and its relabelling.  pre / pre_sel: the lane's first new bead and
// selector, loaded before the decision.
template <class Sync>
__device__ __forceinline__ void commit_impl(const Rep& R, const Prop& pr, int lane, int acc, const double* pre,
                                            unsigned char pre_sel, const double* beads, Sync sync) {
    const int M = R.M, N = R.N;
    const int s_acc = acc;
    if (s_acc && pr.move == 3) {
        // Bisect::Accept of every chain, then PermBisect::AssignParticleLabels
        // (perm_bisect_class.h:47-56): the slices after the relinked slice e take
        // the labels of the path they now continue, so chain label a_i there
        // holds what a_{ch_nxt[i]} held (each cycle of ch_nxt followed from its
        // first chain), and the wrap permutation follows.
        const int n = pr.n_chain, nm = pr.count, nb = nm + 1;
        for (int idx = lane; idx < n * nm; idx += kWave) {
            const int i = idx / nm, t = idx % nm + 1;
            const int s = (pr.b0 + t) % M, l = (pr.b0 + t >= M) ? R.ch_lbl2[i] : R.ch_lbl[i];
            for (int d = 0; d < 3; ++d) R.pos[((size_t)d * M + s) * N + l] = R.ch_new[(size_t)idx * 3 + d];
        }
        if (R.use_long_range)
            for (int m = lane; m < nm; m += kWave) R.sel[(pr.first + m) % M] ^= 1;
        sync();
        if (n > 1) {
            const bool wrapped = pr.b0 + nb - 1 >= M;
            const int e = pr.e_slice;
            const int* lbl = wrapped ? R.ch_lbl2 : R.ch_lbl;
            for (int idx = lane; idx < (M - 1 - e) * 3; idx += kWave) {
                const int s = e + 1 + idx / 3, d = idx % 3;
                double* col = R.pos + ((size_t)d * M + s) * N;
                for (int i0 = 0; i0 < n; ++i0) {
                    if (!R.ch_lead[i0]) continue;
                    const double keep = col[lbl[i0]];
                    int ai = lbl[i0];
                    for (int i = R.ch_nxt[i0]; i != i0; i = R.ch_nxt[i]) {
                        col[ai] = col[lbl[i]];
                        ai = lbl[i];
                    }
                    col[ai] = keep;
                }
            }
            if (lane == 0) {
                for (int i0 = 0; i0 < n; ++i0) {
                    if (!R.ch_lead[i0]) continue;
                    const int keep = R.perm[lbl[i0]];
                    int ai = lbl[i0];
                    for (int i = R.ch_nxt[i0]; i != i0; i = R.ch_nxt[i]) {
                        R.perm[ai] = R.perm[lbl[i]];
                        ai = lbl[i];
                    }
                    R.perm[ai] = keep;
                }
                for (int i = 0; i < n; ++i) {
                    const int a = wrapped ? R.ch_lbl2[i] : R.ch_lbl[i];
                    R.iperm[R.perm[a]] = a;
                }
            }
        }
    } else if (s_acc) {
        for (int m = lane; m < pr.count; m += kWave) {
            const int s = (pr.first + m) % M;
            // a bisection chain carries label p2 past the wrap
            const int l = (pr.move == 0 && pr.b0 + m + 1 >= M) ? pr.p2 : pr.p;
            const bool first = m == lane;
            for (int d = 0; d < 3; ++d) R.pos[((size_t)d * M + s) * N + l] = first ? pre[d] : beads[3 * m + d];
            if (R.use_long_range) R.sel[s] = (unsigned char)((first ? pre_sel : R.sel[s]) ^ 1);
        }
    }
    if (pr.move == 3 && pr.status == 1) {
        sync();
        for (int i = lane; i < pr.n_chain; i += kWave) {
            R.mv_pre[R.ch_lbl[i]] = -1;
            R.mv_post[R.ch_lbl2[i]] = -1;
        }
    }
}

__device__ __forceinline__ void decide_body(const Rep* __restrict__ reps, int n_reps,
                                            unsigned long long* __restrict__ kt) {
    if (kt && blockIdx.x == 0) kt_close(kt);
    const int r = blockIdx.x;
    if (r >= n_reps) return;
    decide_impl(reps[r], (int)threadIdx.x, BlockSync{});
}

__global__ __launch_bounds__(64) void k_propose_bisect(const Rep* __restrict__ reps, int n_reps) {
    propose_bisect_body(reps, n_reps);
}
__global__ __launch_bounds__(64) void k_propose_displace(const Rep* __restrict__ reps, int n_reps) {
    propose_displace_body(reps, n_reps);
}
__global__ __launch_bounds__(64) void k_decide(const Rep* __restrict__ reps, int n_reps,
                                               unsigned long long* __restrict__ kt) {
    decide_body(reps, n_reps, kt);
}
// K5 of one round and K4 of the next in one launch: a replica's pending
// proposal is decided and committed (nothing is pending at the first round of
// a stage), then its next proposal is made.  Saves one dependent launch per
// round; the stage's last decision is a k_decide of its own.  Four wavefronts
// per replica: the first decides while, on the device RNG of an unpermuted
// path, the second and third fetch the next attempt's window and draws; then
// all four make its levels (bisect_levels): 15 us for 512 replicas of N = 256,
// M = 128 beside 18 with the levels on one wavefront.  At most 128 registers: four
// workgroups a CU, 1024 replicas at once (with 135, three: a round of 780 replicas of
// N = 32, M = 32 77.7 us, 72.6 so; of 1024 of N = 12, M = 16 68.4 and 63.0).  Beyond
// them two wavefronts, the second with the window and the draws (1300 replicas 112
// and 107 us).
template <int W>
__global__ __launch_bounds__(W * kWave) __attribute__((amdgpu_waves_per_eu(4))) void k_decide_propose_bisect(
    const Rep* __restrict__ reps, int n_reps, unsigned long long* __restrict__ kt) {
    constexpr int BS = W * kWave;
    __shared__ BisectLds S;
    __shared__ DecideOut s_out;
    __shared__ int s_moved;
    const int r = blockIdx.x, w = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    if (kt && blockIdx.x == 0 && w == 0) kt_close(kt);
    if (r >= n_reps) return;
    const Rep& R = reps[r];
    // a window that crosses the wrap of a permuted path holds a second label,
    // which the window check after the decision does not follow
    const bool ahead = R.tape == nullptr && R.perm == nullptr;
    Counters* c = R.cnt;
    const unsigned int rem = c->remaining;
    const unsigned long long seq = c->seq;
    int p = -1, b0 = 0;
    if (ahead && rem > 0 && w > 0) bisect_where(R, seq, &p, &b0);
    if (w == 0) {
        if (lane == 0) s_out.status = 0;
        const int nb = 1 << R.n_level;
        const int moved = decide_impl(R, lane, WaveSync{}, R.pair_type ? nb : 0,
                                      R.use_long_range ? (nb - 1) * R.n_chunks : 0, &s_out);
        if (lane == 0) s_moved = moved;
    } else if (w == 1 && p >= 0) {
        if (lane == 0) {
            S.info[1] = p;
            S.info[2] = b0;
        }
        bisect_window(R, lane, S, p, p, b0, false);
        if (W == 2) bisect_draws(R, lane, S, seq);
    } else if (W > 2 && w == 2 && p >= 0) {
        bisect_draws(R, lane, S, seq);
    }
    __syncthreads();
    if (w == W - 1 && lane == 0 && s_out.status != 0)
        decide_book(R, s_out.pr, s_out.acc, s_out.status, s_out.po, s_out.pn, s_out.lo, s_out.ln);
    if (!ahead) {
        if (w == 0) propose_bisect_impl(R, lane, WaveSync{}, true, S);
        return;
    }
    if (rem == 0) {
        if (threadIdx.x == 0) R.prop->status = 0;
        rho_items_write(R, 0, 0, 0, 0, threadIdx.x, BS);
        return;
    }
    if (threadIdx.x == 0) {
        c->remaining = rem - 1;
        c->seq = seq + 1;
    }
    if (S.info[1] == s_moved) {
        // the decision just committed beads of the attempt's particle: its window again
        if (w == 0) bisect_window(R, lane, S, s_moved, s_moved, S.info[2], false);
        __syncthreads();
    }
    bisect_levels<W>(R, S, w, lane, R.prop, R.prop_new, R.phase, 0);
    rho_items_write(R, 0, S.info[4], S.info[5], (S.info[2] + 1) % R.M, threadIdx.x, BS);
}
// Displacement: the decision on the first wavefront, then the proposal, whose
// M moved slices (positions, phase chains, rho_k items) take all kDisBlock
// threads.
constexpr int kDisBlock = 256;
__global__ __launch_bounds__(kDisBlock) void k_decide_propose_displace(const Rep* __restrict__ reps, int n_reps,
                                                                       unsigned long long* __restrict__ kt) {
    const int r = blockIdx.x;
    if (threadIdx.x < kWave) {
        if (kt && blockIdx.x == 0) kt_close(kt);
        if (r < n_reps) decide_impl(reps[r], (int)threadIdx.x, WaveSync{});
    }
    __syncthreads();
    if (r >= n_reps) return;
    propose_displace_impl(reps[r], (int)threadIdx.x, BlockSync{}, true, kDisBlock);
}


// A whole round (MOVE 0 bisection, 1 displacement) in one launch, for batches
// too small to fill the GPU (a round is then bound by latency, not by
// throughput).  After the XCD remap the first n_reps workgroups (bisection) make
// the replicas' next proposals, the following n_reps * bpr run the window links
// of the LDS pair kernel, the others a group of up to ipb rho_k items of one
// replica each (rgrp: first item, items, replica; ipb > 1 only where one item per
// workgroup would exceed what the GPU holds at once).  Every workgroup then
// counts itself in on its replica's arrival counter; the replica's last one
// decides and commits its proposal (K5) and publishes the next, with its rho_k
// items.  A replica's round thus ends with its own last workgroup: no launch
// boundary separates the sums from the decision, and nothing waits (the counter
// is only read by the atomic that increments it).  The sums and the proposal pass
// between workgroups as agent-scope atomic stores and loads, each waited for
// before its workgroup arrives; agent-scope fences would instead write back a
// whole L2 per workgroup, which measured slower than three launches per round.
// The last workgroup resets the counter for the next round.
//
// A bisection draws from its sequence number alone and reads only its own
// particle's beads, so the proposal made beside the pending one is the one that
// would follow the decision, bit for bit, unless the decision commits beads of
// the same particle (an acceptance, 1 in N): then the last workgroup makes it
// again.  What remains after the last arrival is the decision.  A displacement
// (its M slices' phases) and a replayed tape (its cursor follows the decision)
// are proposed after the decision.  A bisection round with the proposal in the
// last workgroup, with it beside the pending one on one wavefront, and on four
// (bisect_levels): one replica of N = 256, M = 128 23, 18 and 14.5 us; of N = 32,
// M = 32 16, 15.5 and 12 us.
constexpr int kRoundBlock = kRhoBlock;
constexpr int kNextWords = sizeof(NextProp) / 8, kPropWords = sizeof(Prop) / 8;
static_assert(sizeof(NextProp) % 8 == 0 && sizeof(Prop) % 8 == 0 && kNextWords <= kWave, "one word a lane");

// Workgroup of k_round that makes replica R's next bisection while the others
// evaluate the pending one: the whole proposal, from the positions before the
// decision, into the set of buffers the pending one does not use.  It stands
// unless the decision commits beads of the same particle.
__device__ __forceinline__ void next_bisect(const Rep& R, BisectLds& S, NextProp& next) {
    if (R.tape != nullptr) return;
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    Counters* c = R.cnt;
    const unsigned int rem = c->remaining;
    const unsigned long long seq = c->seq;
    const int set = R.prop->buf == 1 ? 1 : 0;
    if (threadIdx.x < kNextWords) ((unsigned long long*)&next)[threadIdx.x] = 0;
    if (rem > 0) {
        int p, b0;
        bisect_where(R, seq, &p, &b0);
        if (threadIdx.x == 0) {
            S.info[1] = p;
            S.info[2] = b0;
            S.seq = seq;
        }
        if (w == 0) bisect_window(R, lane, S, p, label_after_wrap(R, p), b0, false);
        if (w == 1) bisect_draws(R, lane, S, seq);
    }
    __syncthreads();  // every wavefront has read the counters
    if (rem > 0) {
        if (threadIdx.x == 0) {
            c->remaining = rem - 1;
            c->seq = seq + 1;
            next.seq = seq;
            next.has = 1;
        }
        bisect_levels<kRoundBlock / kWave>(R, S, w, lane, &next.pr, R.next_new[set], R.next_phase[set], set + 1);
    }
    if (threadIdx.x < kNextWords)
        __hip_atomic_store((unsigned long long*)R.next + threadIdx.x, ((unsigned long long*)&next)[threadIdx.x],
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// PT 3: the tables stay in global memory, NORD the doubles of LDS for their axes.
template <int PT, int NORD, int KPT, bool NT, int MOVE>
__global__ __launch_bounds__(kRoundBlock) void k_round(const Rep* __restrict__ reps, int n_reps, int bpr, int qpw,
                                                       const RhoItem* __restrict__ items,
                                                       const int4* __restrict__ rgrp, int ipb,
                                                       unsigned int* __restrict__ arrive) {
    extern __shared__ double lds[];
    __shared__ double2 tab[6 * (kMaxIdx + 1)];
    __shared__ double red[2][kRhoBlock / kWave];
    __shared__ double2 wpart[kRoundBlock / kWave];
    __shared__ int s_last;
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    __shared__ BisectLds S;
    __shared__ NextProp s_next;
    const int n_next = MOVE == 0 ? n_reps : 0;
    const int n_pair = n_reps * bpr, idx = (int)xcd_remap(blockIdx.x, gridDim.x) - n_next;
    int r;
    if (MOVE == 0 && idx < 0) {
        r = idx + n_next;
        next_bisect(reps[r], S, s_next);
    } else if (idx < n_pair) {
        r = idx / bpr;
        const int part = idx % bpr;
        Rep R = reps[r];
        if constexpr (PT == 3) {
            constexpr int W = kRoundBlock / kWave;
            const Prop pr = *R.prop;
            R.prop_new = prop_beads(reps[r], pr);
            if (pr.status == 1 && !pr.generic && part * (W / general_split<W>(R.N, qpw)) < pr.n_links)
                pair_links_general<true, W>(R, lds, NORD, pr, part, bpr, qpw, w, lane, wpart);
        } else {
            // the tables' first kRoundBlock * 4 values are loaded while the proposal is
            const int na = R.bt_a.ncoef * R.bt_a.ncomp, nd = R.lds_doubles;
            double tv[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int t = threadIdx.x + k * kRoundBlock;
                tv[k] = t < nd ? (t < na ? R.bt_a.c[t] : R.bt_b.c[t - na]) : 0.;
            }
            const Prop pr = *R.prop;
            R.prop_new = prop_beads(reps[r], pr);
            constexpr int W = kRoundBlock / kWave;
            if (pr.status == 1 && !pr.generic && part * (W / pair_split<W>(R.N, qpw)) < pr.n_links) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int t = threadIdx.x + k * kRoundBlock;
                    if (t < nd) lds[t] = tv[k];
                }
                // the rest (large tables: 96 KB for David's)
                stage_batched(lds, R.bt_a.c, R.bt_b.c, na, nd, 4 * kRoundBlock, kRoundBlock);
                __syncthreads();
                pair_links_split<PT, NORD, true, W>(R, lds, pr, part, bpr, qpw, w, lane, wpart);
            }
        }
    } else {
        // a group of up to ipb rho_k items of one replica, one after the other
        const int4 g = rgrp[idx - n_pair];  // first item, items, replica
        r = g.z;
        RhoItem d = items[g.x];
        for (int i = 0; i < g.y; ++i) {
            RhoItem nd;
            if (i + 1 < g.y) nd = items[g.x + i + 1];
            if (d.valid) {
                rho_item<KPT, NT, true>(d, tab, red);
                __syncthreads();  // tab and red are reused by the next item
            }
            d = nd;
        }
    }
    // every wavefront's sums are performed before the workgroup arrives
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) {
        const Rep& R = reps[r];
        const int n_items = MOVE == 0 ? R.n_ritems_bis : R.n_ritems_dis;
        const unsigned int expect = (MOVE == 0 ? 1u : 0u) + (unsigned int)bpr + (unsigned int)((n_items + ipb - 1) / ipb);
        s_last = atomicAdd(arrive + r, 1u) + 1u == expect;
    }
    __syncthreads();
    if (!s_last) return;
    // the replica's last workgroup: its first wavefront decides while its second
    // fetches the proposal made ahead
    __shared__ DecideOut s_out;
    __shared__ int s_moved;
    const Rep& R = reps[r];
    const bool ahead = MOVE == 0 && R.tape == nullptr;
    if (w == 0) {
        if (lane == 0) {
            __hip_atomic_store(arrive + r, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            s_out.status = 0;
        }
        // the pair and rho_k sums of a proposal that reached level 0 (bisection:
        // 2^l links and 2^l - 1 moved slices; displacement: M of each), loaded
        // before the proposal itself
        const int nl = MOVE == 0 ? 1 << R.n_level : R.M, nm = MOVE == 0 ? nl - 1 : R.M;
        const int moved = decide_impl<true>(R, lane, WaveSync{}, R.pair_type ? nl : 0,
                                            R.use_long_range ? nm * R.n_chunks : 0, &s_out);
        if (lane == 0) s_moved = moved;
    } else if (w == 1 && ahead) {
        unsigned long long *to = (unsigned long long*)&s_next, *from = (unsigned long long*)R.next;
        if (lane < kNextWords) to[lane] = __hip_atomic_load(from + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (w == 2 && lane == 0 && s_out.status != 0)
        // the decision's counters and flags, off the proposal's path
        decide_book(R, s_out.pr, s_out.acc, s_out.status, s_out.po, s_out.pn, s_out.lo, s_out.ln);
    if (MOVE == 1) {
        propose_displace_impl(R, (int)threadIdx.x, BlockSync{}, true, kRoundBlock);
        return;
    }
    if (!ahead) {
        if (w == 0) propose_bisect_impl(R, lane, WaveSync{}, true, S);
        return;
    }
    const int p = s_next.pr.p;
    if (!(s_next.has && p == s_moved)) {
        // the decision left the attempt's particle where it was: the proposal made
        // ahead stands, its rho_k rows are known now
        if (w == 2) return;
        const int t = w == 3 ? lane + 2 * kWave : (int)threadIdx.x;
        if (t < kPropWords) ((unsigned long long*)R.prop)[t] = ((const unsigned long long*)&s_next.pr)[t];
        rho_items_write(R, 0, s_next.pr.status, s_next.pr.count, s_next.pr.first, t, 3 * kWave,
                        s_next.pr.buf ? R.next_phase[s_next.pr.buf - 1] : nullptr);
        return;
    }
    // the decision just committed beads of the attempt's particle: the proposal
    // again, from the same draws
    if (threadIdx.x == 0) {
        S.info[1] = p;
        S.info[2] = s_next.pr.b0;
    }
    if (w == 0) bisect_window(R, lane, S, p, label_after_wrap(R, p), s_next.pr.b0, false);
    if (w == 1) bisect_draws(R, lane, S, s_next.seq);
    __syncthreads();
    bisect_levels<kRoundBlock / kWave>(R, S, w, lane, R.prop, R.prop_new, R.phase, 0);
    rho_items_write(R, 0, S.info[4], S.info[5], (S.info[2] + 1) % R.M, threadIdx.x, kRoundBlock);
}

// Sums the per-replica work counters into work[WORK_PAIR_LINKS], work[WORK_RHO_SLICEK].
__global__ __launch_bounds__(64) void k_work_sum(const Rep* __restrict__ reps, int n_reps,
                                                 unsigned long long* __restrict__ work) {
    unsigned long long a = 0, b = 0;
    for (int r = threadIdx.x; r < n_reps; r += kWave) {
        a += reps[r].cnt->pair_links;
        b += reps[r].cnt->rho_slicek;
    }
    for (int o = kWave / 2; o > 0; o >>= 1) {
        a += __shfl_xor(a, o);
        b += __shfl_xor(b, o);
    }
    if (threadIdx.x == 0) {
        work[WORK_PAIR_LINKS] = a;
        work[WORK_RHO_SLICEK] = b;
    }
}

// ---------------------------------------------------------------------------
// What a block's write reads and resets.  A small copy between device memory and
// the caller's costs 8-10 us each (a blocking copy or fill of a few bytes), and a
// write of R replicas made 6 R fills and 6 R copies: 1.85 ms for 12 replicas, more
// than the estimators.  One kernel clears every replica's accumulators, and one
// gathers the pieces of a read into pinned host memory, ready after the stream's
// synchronisation: 0.55 ms.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_obs_reset(const Rep* __restrict__ reps, unsigned int which, unsigned int n_r) {
    const Rep& R = reps[blockIdx.x];
    if (which & 1u) {
        if (threadIdx.x < 2) R.e_acc[threadIdx.x] = 0.;
        if (threadIdx.x == 0) R.n_measure[0] = 0;
    }
    if (which & 2u) {
        for (int k = threadIdx.x; k < max(R.nk, 1); k += 256) R.sk_acc[k] = 0.;
        if (threadIdx.x == 0) R.n_measure[1] = 0;
    }
    if (which & 4u) {
        for (unsigned int i = threadIdx.x; i < n_r; i += 256) R.gr_cnt[i] = 0;
        if (threadIdx.x == 0) R.n_measure[2] = 0;
    }
}
// n_a and n_b 8-byte words from a and b, one after the other
__global__ __launch_bounds__(256) void k_pack(unsigned long long* __restrict__ out, const unsigned long long* __restrict__ a,
                                              int n_a, const unsigned long long* __restrict__ b, int n_b) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t < n_a)
        out[t] = a[t];
    else if (t < n_a + n_b)
        out[t] = b[t - n_a];
}
// accept flags of every replica's last stage, rows of mx bytes
__global__ __launch_bounds__(256) void k_pack_accepted(const Rep* __restrict__ reps, const unsigned int* __restrict__ counts,
                                                       unsigned int mx, unsigned char* __restrict__ out) {
    const unsigned int n = counts[blockIdx.x];
    const unsigned char* a = reps[blockIdx.x].accepted;
    for (unsigned int i = threadIdx.x; i < n; i += 256) out[(size_t)blockIdx.x * mx + i] = a[i];
}
// the committed rho_k rows of the slices from first in order
__global__ __launch_bounds__(256) void k_gather_rho(const Rep* __restrict__ reps, int r, int first, double2* __restrict__ out) {
    const Rep& R = reps[r];
    const int b = first + blockIdx.x;
    const double2* row = R.rho + ((size_t)R.sel[b] * R.M + b) * R.nk;
    for (int k = threadIdx.x; k < R.nk; k += 256) out[(size_t)blockIdx.x * R.nk + k] = row[k];
}

// Stage set-up on the device (kept out of hipMemset so captured graphs stay plain kernels)
__global__ void k_stage_begin(const Rep* __restrict__ reps, int n_reps, const unsigned int* __restrict__ counts) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n_reps) return;
    reps[r].cnt->remaining = counts[r];
    reps[r].cnt->stage_i = 0;
}

// ---------------------------------------------------------------------------
// Interface kernels (Action::GetAction in a chosen mode).  A query is a few
// microseconds of work, so launches, copies and synchronisations are its cost:
// the proposal's record comes as a kernel argument (NEW beads of up to 64 slices
// too), a pair query is one launch whose last workgroup adds the terms, and the
// result goes to pinned host memory.  An attempt of N = 32, M = 32 (proposal, four
// queries, accept) took 238 us with 10 blocking copies and 14 launches,
// 81 us so.
// ---------------------------------------------------------------------------
constexpr int kPropArg = 64;
struct PropBeads {
    double x[3 * kPropArg];
};
__global__ __launch_bounds__(3 * kPropArg) void k_set_proposal(const Rep* __restrict__ reps, int r, int n, PropBeads v) {
    if ((int)threadIdx.x < 3 * n) reps[r].prop_new[threadIdx.x] = v.x[threadIdx.x];
}
__device__ __forceinline__ void host_result(double* out, double v) {
    __hip_atomic_store(out, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Kinetic::GetAction (kinetic_class.h:105-122) for the proposal's particle p.
__global__ __launch_bounds__(64) void k_kinetic_window(const Rep* __restrict__ reps, int r, Prop pr, int mode, int p,
                                                        int b0, int n_links, int level, double* __restrict__ out) {
    const Rep& R = reps[r];
    const int skip = 1 << level, M = R.M;
    const double i4lt = 1. / (4. * R.lambda * (R.tau * (double)skip));
    double tot = 0.;
    // the walk from (p, b0) carries label perm[p] past the wrap; NEW mode reads
    // the proposal's beads where the label is the proposal's particle
    const int p2 = label_after_wrap(R, p);
    for (int i = threadIdx.x; i < n_links; i += kWave) {
        const int ta = i * skip, tb = ta + skip;
        const int a = (b0 + ta) % M, b = (b0 + tb) % M;
        const int la = (b0 + ta >= M) ? p2 : p, lb = (b0 + tb >= M) ? p2 : p;
        double dd[3];
        for (int d = 0; d < 3; ++d) {
            double xa = (mode && pr.p == la) ? pos_new(R, pr, d, a) : pos_at(R, d, a, la);
            double xb = (mode && pr.p == lb) ? pos_new(R, pr, d, b) : pos_at(R, d, b, lb);
            dd[d] = minimg(xa - xb, R.L, R.iL);
        }
        tot += free_neg_log(&R.kin[level], R.kin_images, i4lt, dd);
    }
    tot = wave_sum(tot);
    if (threadIdx.x == 0) host_result(out, tot);
}

// PairAction::GetAction (pair_action_class.h:267-302) of particle p at level 0 in
// one mode.  Workgroups: one per window link (its partners over the threads), then
// one per slice the proposal moves whose NEW rho_k is not there yet (n_update:
// Species::UpdateRhoK, species_class.h:406-425, with the slice's CalcULong sum when
// it lies in the window), then one per other window slice (CalcULong on the
// committed rho_k, or on the spare row where NEW mode updated it before).  The
// terms pass between workgroups as agent-scope atomic stores and loads (see
// k_round); the last one to arrive adds them in link and slice order.
constexpr int kIfaceBlock = 256;
__global__ __launch_bounds__(kIfaceBlock) void k_iface_pair(const Rep* __restrict__ reps, int r, Prop pr, int mode, int b0,
                                                            int n_links, int n_update, int n_long, int rho_updated,
                                                            double* __restrict__ part, unsigned int* __restrict__ arrive,
                                                            double* __restrict__ out) {
    const Rep& R = reps[r];
    const int M = R.M, N = R.N, p = pr.p, tid = threadIdx.x;
    __shared__ double sh[kIfaceBlock / kWave];
    __shared__ double2 tab[6 * (kMaxIdx + 1)];
    __shared__ int s_last;
    const int blk = blockIdx.x;
    double t = 0.;
    double* to = nullptr;
    if (blk < n_links) {
        const int s0 = (b0 + blk) % M, s1 = s0 + 1 == M ? 0 : s0 + 1;
        double a0[3], a1[3];
        for (int d = 0; d < 3; ++d) {
            a0[d] = mode ? pos_new(R, pr, d, s0) : pos_at(R, d, s0, p);
            a1[d] = mode ? pos_new(R, pr, d, s1) : pos_at(R, d, s1, p);
        }
        for (int q = tid; q < N; q += kIfaceBlock) {
            if (q == p) continue;
            double c0[3], c1[3];
            for (int d = 0; d < 3; ++d) {
                c0[d] = pos_at(R, d, s0, q);
                c1[d] = pos_at(R, d, s1, q);
            }
            LinkGeom g;
            link_geom(a0, c0, a1, c1, R.L, R.iL, g);
            t += pair_u(R, g.r, g.rp, g.s);
        }
        to = &R.pair_part[blk].x;
    } else if (blk < n_links + n_update) {
        const int m = blk - n_links, s = (pr.first + m) % M, stride = R.max_idx + 1;
        int w = s - b0 % M;
        if (w < 0) w += M;
        const int cur = R.sel[s];
        const double2* rc = R.rho + ((size_t)cur * M + s) * R.nk;
        double2* rn = R.rho + ((size_t)(1 - cur) * M + s) * R.nk;
        if (tid < 6) {
            const int d = tid % 3;
            phase_chain((tid >= 3 ? R.prop_new[3 * m + d] : pos_at(R, d, s, p)) * R.box, R.max_idx, tab + tid * stride);
        }
        __syncthreads();
        for (int k = tid; k < R.nk; k += kIfaceBlock) {
            const double2 v = ld2<false>(rc + k);
            const int kp = gld(R.kidx + k);
            const double2 en = phase_k(&tab[3 * stride], stride, kp), eo = phase_k(tab, stride, kp);
            double2 nv;
            nv.x = v.x + (en.x - eo.x);
            nv.y = v.y + (en.y - eo.y);
            rn[k] = nv;
            t += gld(R.coef_s + k) * (nv.x * nv.x + nv.y * nv.y);
        }
        if (w < n_long) to = part + w;
    } else {
        const int w = blk - n_links - n_update, s = (b0 + w) % M;
        int m = s - pr.first;
        if (m < 0) m += M;
        const bool moved = mode && m < pr.count;
        if (!(moved && n_update)) {  // (else its update's workgroup has the sum)
            const int buf = moved && rho_updated ? 1 - R.sel[s] : R.sel[s];
            const double2* rb = R.rho + ((size_t)buf * M + s) * R.nk;
            for (int k = tid; k < R.nk; k += kIfaceBlock) {
                const double2 v = ld2<false>(rb + k);
                t += gld(R.coef_s + k) * (v.x * v.x + v.y * v.y);
            }
            to = part + w;
        }
    }
    t = block_sum<kIfaceBlock>(t, sh);
    if (tid == 0) {
        if (to) __hip_atomic_store(to, t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_s_waitcnt(0);  // the term is performed before the workgroup arrives
        s_last = atomicAdd(arrive, 1u) + 1u == gridDim.x;
    }
    __syncthreads();
    if (!s_last || tid >= kWave) return;
    double a = 0., l = 0.;
    for (int j = tid; j < n_links; j += kWave)
        a += __hip_atomic_load(&R.pair_part[j].x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int j = tid; j < n_long; j += kWave) l += __hip_atomic_load(part + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    a = wave_sum(a);
    l = wave_sum(l);
    if (tid == 0) {
        __hip_atomic_store(arrive, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        host_result(out, a + R.long_scale * l);
    }
}

// PairAction::GetActionLaplacian (pair_action_class.h:336-363) of particle p at
// level 0: for the window beads b0 <= b < b1, the links (b, b + 1) and
// (b, b - 1 + M) with every other particle, each through CalcLaplacianU
// (:167-199), the central second difference (eps 1e-4) of the link action in
// each coordinate of bead (p, b).  The long-range part is left out, as in the
// reference.  NEW mode reads the pending interface proposal's beads.  One
// workgroup; the thread sums are added in thread order.
constexpr int kLapBlock = 256;
__global__ __launch_bounds__(kLapBlock) void k_pair_laplacian(const Rep* __restrict__ reps, int r, Prop pr, int mode,
                                                              int b0, int b1, int p, double* __restrict__ out) {
    const Rep& R = reps[r];
    const int M = R.M, N = R.N, nb = b1 - b0;
    const double eps = 1.e-4;
    __shared__ double red[kLapBlock / kWave];
    auto at = [&](int d, int s, int lbl) { return (mode && pr.p == lbl) ? pos_new(R, pr, d, s) : pos_at(R, d, s, lbl); };
    double tot = 0.;
    for (int it = threadIdx.x; it < nb * (N - 1); it += kLapBlock) {
        const int bi = b0 + it / (N - 1), qi = it % (N - 1), q = qi < p ? qi : qi + 1;
        const int si = bi % M;
        double lap = 0.;
        for (int side = 0; side < 2; ++side) {
            const int sj = side == 0 ? (bi + 1) % M : (bi - 1 + M) % M;
            double a0[3], c0[3], a1[3], c1[3];
            for (int d = 0; d < 3; ++d) {
                a0[d] = at(d, si, p);
                c0[d] = at(d, si, q);
                a1[d] = at(d, sj, p);
                c1[d] = at(d, sj, q);
            }
            LinkGeom g;
            link_geom(a0, c0, a1, c1, R.L, R.iL, g);
            const double f0 = pair_u(R, g.r, g.rp, g.s);
            double part = 0.;
            for (int d = 0; d < 3; ++d) {
                const double x0 = a0[d];
                a0[d] = x0 + eps;
                link_geom(a0, c0, a1, c1, R.L, R.iL, g);
                const double fp1 = pair_u(R, g.r, g.rp, g.s);
                a0[d] = x0 - eps;
                link_geom(a0, c0, a1, c1, R.L, R.iL, g);
                const double fm1 = pair_u(R, g.r, g.rp, g.s);
                part += (fp1 + fm1 - 2 * f0) / (eps * eps);
                a0[d] = x0;
            }
            lap += part;
        }
        tot += lap;
    }
    tot = wave_sum(tot);
    if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x / kWave] = tot;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.;
        for (int w = 0; w < kLapBlock / kWave; ++w) t += red[w];
        host_result(out, t);
    }
}

// Move::Accept / Reject of an interface proposal.
__global__ void k_commit(const Rep* __restrict__ reps, int r, Prop pr, int accept, int rho_updated) {
    const Rep& R = reps[r];
    if (accept)
        for (int m = threadIdx.x; m < pr.count; m += blockDim.x) {
            const int s = (pr.first + m) % R.M;
            for (int d = 0; d < 3; ++d) R.pos[((size_t)d * R.M + s) * R.N + pr.p] = R.prop_new[3 * m + d];
            if (rho_updated && R.use_long_range) R.sel[s] ^= 1;
        }
}

// ---------------------------------------------------------------------------
// K6: whole-path estimators (thermal energy, potential)
// ---------------------------------------------------------------------------
// Kinetic::DActionDBeta summand per slice (kinetic_class.h:35-45)
__global__ __launch_bounds__(256) void k_kin_dbeta(const Rep* __restrict__ reps, int slot) {
    const Rep& R = reps[blockIdx.y];
    const int b = blockIdx.x;
    if (b >= R.M) return;
    const int b1 = (b + 1) % R.M;
    double t = 0.;
    for (int p = threadIdx.x; p < R.N; p += 256) {
        const int pn = next_label(R, b, p);
        double dd[3];
        for (int d = 0; d < 3; ++d) dd[d] = minimg(pos_at(R, d, b, p) - pos_at(R, d, b1, pn), R.L, R.iL);
        double img = 0.;
        if (R.kin_images > 0)
            for (int d = 0; d < 3; ++d) img -= spl_eval1(R.kin_dtau, dd[d]);
        t += img - (dd[0] * dd[0] + dd[1] * dd[1] + dd[2] * dd[2]) * R.kin_i4ltt;
    }
    __shared__ double sh[4];
    t = block_sum<256>(t, sh);
    if (threadIdx.x == 0) R.scratch[slot * R.M + b] = t;
}

// Pair sums over all pairs on link (b, b+1): which 0 = CalcdUdBeta
// (pair_action_class.h:241-264), 1 = CalcV on plain minimum images
// (pair_action_class.h:369-395).  Pairs (i, i+d mod N), d = 1..N/2.
__global__ __launch_bounds__(256) void k_pair_whole(const Rep* __restrict__ reps, int which, int slot) {
    const Rep& R = reps[blockIdx.y];
    const int b = blockIdx.x;
    if (b >= R.M || R.pair_type == 0) {
        if (b < R.M && threadIdx.x == 0) R.scratch[slot * R.M + b] = 0.;
        return;
    }
    const int N = R.N, M = R.M, b1 = (b + 1) % M;
    double t = 0.;
    const int half = N / 2;
    for (int i = threadIdx.x; i < N; i += 256) {
        double a0[3], a1[3];
        for (int d = 0; d < 3; ++d) {
            a0[d] = pos_at(R, d, b, i);
            a1[d] = pos_at(R, d, b1, i);
        }
        for (int dd = 1; dd <= half; ++dd) {
            if ((N % 2 == 0) && dd == half && i >= half) continue;
            const int j = (i + dd) % N;
            double c0[3], c1[3];
            for (int d = 0; d < 3; ++d) {
                c0[d] = pos_at(R, d, b, j);
                c1[d] = pos_at(R, d, b1, j);
            }
            // pair (lo, hi): r = r_hi - r_lo; magnitudes do not depend on the orientation
            LinkGeom g;
            if (i < j)
                link_geom(a0, c0, a1, c1, R.L, R.iL, g);
            else
                link_geom(c0, a0, c1, a1, R.L, R.iL, g);
            if (which == 0) {
                t += pair_du_dbeta(R, g.r, g.rp, g.s);
            } else {
                double v0[3], v1[3];
                for (int d = 0; d < 3; ++d) {
                    v0[d] = minimg(a0[d] - c0[d], R.L, R.iL);
                    v1[d] = minimg(a1[d] - c1[d], R.L, R.iL);
                }
                t += pair_v(R, sqrt(v0[0] * v0[0] + v0[1] * v0[1] + v0[2] * v0[2]),
                            sqrt(v1[0] * v1[0] + v1[1] * v1[1] + v1[2] * v1[2]));
            }
        }
    }
    __shared__ double sh[4];
    t = block_sum<256>(t, sh);
    if (threadIdx.x == 0) R.scratch[slot * R.M + b] = t;
}

// sum_b |rho(b,k)|^2 for the 64 k-vectors of a workgroup (k the lane's; valid on the
// first wavefront): its wavefronts (16 at most, and no more than have four slices each)
// share the slices, four loads in flight each, and are added in order.  (A thread per k-vector that walked the
// slices, each load behind its buffer selector, left 8 workgroups for 1979
// k-vectors: 73 us for M = 128, 5 us so.)
constexpr int kSumBlock = 1024;
__device__ __forceinline__ double sum_rho2(const Rep& R, int k, double* sh) {
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave, M = R.M;
    const int W = blockDim.x / kWave;
    double t = 0.;
    if (k < R.nk)
        for (int b = w; b < M; b += 4 * W) {
            double2 v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int s = b + i * W;
                v[i] = s < M ? ld2<false>(R.rho + ((size_t)R.sel[s] * M + s) * R.nk + k) : make_double2(0., 0.);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) t += v[i].x * v[i].x + v[i].y * v[i].y;
        }
    sh[threadIdx.x] = t;
    __syncthreads();
    t = 0.;
    if (w == 0)
        for (int i = 0; i < W; ++i) t += sh[i * kWave + lane];
    return t;
}

// sum_k coef(k) sum_b |rho(b,k)|^2 per 64 k-vectors, plus (the first) the k=0 and
// r=0 constants: which 0 CalcdUdBetaLong (coef_b, const_du), 1 CalcVLong (coef_v,
// const_v)
__global__ __launch_bounds__(kSumBlock) void k_long_whole(const Rep* __restrict__ reps, int which) {
    const Rep& R = reps[blockIdx.y];
    __shared__ double sh[kSumBlock];
    const int k = (int)(blockIdx.x * kWave + (threadIdx.x & (kWave - 1)));
    if ((int)blockIdx.x * kWave >= R.nk || !R.use_long_range) return;
    double t = sum_rho2(R, k, sh);
    if (threadIdx.x >= kWave) return;
    t = k < R.nk ? t * (which ? R.coef_v[k] : R.coef_b[k]) : 0.;
    t = wave_sum(t);
    if (threadIdx.x == 0)
        R.scratch[scratch_long(R.M) + blockIdx.x] = t + (blockIdx.x == 0 ? (which ? R.const_v : R.const_du) : 0.);
}

// Kinetic::VirialEnergy (kinetic_class.h:48-102): -1 / (4 lambda tau W tau) times
// the sum over the beads of D . d, d the link leaving the bead and D the W links
// from it, for 64 particles per workgroup; the walks follow the path: past slice
// M - 1 a bead is followed by slice 0 of the particle perm[label], however often a
// window goes round.  A window of whole turns of a path that closes on itself has
// the same D (its windings) at every bead, and a particle's sum is D . D of one
// turn: its links are shared by the workgroup's 16 wavefronts.  Otherwise each
// wavefront takes a share of the beads, adds the first one's W links and then moves
// the window.  (A thread per particle took two dependent walks of M slices on one
// workgroup: 493 us for N = 1024, M = 128, 10 us so.)
constexpr int kVirBlock = 1024;
// A walk along the path from slice b of label l.
struct PathWalk {
    int b, l;
    double x[3];
    __device__ __forceinline__ PathWalk(const Rep& R, int b_, int l_) : b(b_), l(l_) {
        for (int d = 0; d < 3; ++d) x[d] = pos_at(R, d, b, l);
    }
    // the link to the next bead into t
    __device__ __forceinline__ void step(const Rep& R, double* t) {
        if (++b == R.M) {
            b = 0;
            l = label_after_wrap(R, l);
        }
        for (int d = 0; d < 3; ++d) {
            const double y = pos_at(R, d, b, l);
            t[d] = minimg(y - x[d], R.L, R.iL);
            x[d] = y;
        }
    }
};
__global__ __launch_bounds__(kVirBlock) void k_kin_virial(const Rep* __restrict__ reps, unsigned int W_in,
                                                          double* __restrict__ part) {
    const Rep& R = reps[blockIdx.y];
    const int M = R.M, N = R.N;
    const unsigned int W = W_in > 0 ? W_in : (unsigned int)M;
    constexpr int G = kVirBlock / kWave;
    __shared__ double sh[kVirBlock * 3];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave, p = blockIdx.x * kWave + lane;
    if ((int)blockIdx.x * kWave >= N) return;
    const bool valid = p < N;
    const int lo = (int)((long long)M * w / G), hi = (int)((long long)M * (w + 1) / G);
    const bool ring = W % (unsigned int)M == 0 && R.perm == nullptr;
    double D[3] = {0., 0., 0.}, t[3], tot = 0.;
    if (valid && lo < hi) {
        PathWalk end(R, lo, p);
        if (ring) {
            for (int c = lo; c < hi; ++c) {
                end.step(R, t);
                for (int d = 0; d < 3; ++d) D[d] += t[d];
            }
        } else {
            unsigned long long left = W;
            if (W > (unsigned int)M) {
                // whole turns of the closed path (M slices of every label of its
                // cycle) are walked once
                unsigned long long turn = M;
                for (int l = label_after_wrap(R, p); l != p; l = label_after_wrap(R, l)) turn += M;
                if (W >= turn) {
                    for (unsigned long long i = 0; i < turn; ++i) {
                        end.step(R, t);
                        for (int d = 0; d < 3; ++d) D[d] += t[d];
                    }
                    for (int d = 0; d < 3; ++d) D[d] *= (double)(W / turn);
                    left = W % turn;
                }
            }
            for (; left > 0; --left) {
                end.step(R, t);
                for (int d = 0; d < 3; ++d) D[d] += t[d];
            }
            PathWalk start(R, lo, p);
            for (int c = lo; c < hi; ++c) {
                double a[3];
                start.step(R, a);
                tot += D[0] * a[0] + D[1] * a[1] + D[2] * a[2];
                if (c + 1 == hi) break;
                end.step(R, t);
                for (int d = 0; d < 3; ++d) D[d] += t[d] - a[d];
            }
        }
    }
    for (int d = 0; d < 3; ++d) sh[threadIdx.x * 3 + d] = ring ? D[d] : d == 0 ? tot : 0.;
    __syncthreads();
    if (w) return;
    double v[3] = {0., 0., 0.};
    for (int i = 0; i < G; ++i)
        for (int d = 0; d < 3; ++d) v[d] += sh[(i * kWave + lane) * 3 + d];
    tot = wave_sum(ring ? v[0] * v[0] + v[1] * v[1] + v[2] * v[2] : v[0]);
    if (ring) tot *= (double)(W / (unsigned int)M);
    if (lane == 0) part[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = -tot * R.kin_i4lt / (W * R.tau);
}
// its workgroups' sums and the constant into the replica's scratch
__global__ __launch_bounds__(64) void k_kin_virial_sum(const Rep* __restrict__ reps, unsigned int W_in, int n_part, int slot,
                                                       const double* __restrict__ part) {
    const Rep& R = reps[blockIdx.x];
    double t = 0.;
    for (int i = threadIdx.x; i < (R.N + kWave - 1) / kWave; i += kWave) t += part[(size_t)blockIdx.x * n_part + i];
    t = wave_sum(t);
    if (threadIdx.x == 0) R.scratch[slot * R.M] = R.kin_dbeta_const / (W_in > 0 ? W_in : (unsigned int)R.M) + t;
}

// ---------------------------------------------------------------------------
// K7: gradients.  Thread per bead (b, p); output grad[b][p][3].
// ---------------------------------------------------------------------------
// Reference-compatible PairAction::GetActionGradient(b, b+1, {p}, 0):
// CalcGradientU by central difference, eps = 1e-4 (pair_action_class.h:135-155,305-337)
__global__ __launch_bounds__(64) void k_grad_compat(const Rep* __restrict__ reps, int out_est, int short_on) {
    const Rep& R = reps[blockIdx.z];
    const int p = blockIdx.x * 64 + threadIdx.x, b = blockIdx.y;
    if (p >= R.N || b >= R.M) return;
    const int M = R.M, N = R.N;
    const int bj = (b + 1) % M, bk = (b + M - 1) % M;
    double r0[3], pj[3], pk[3], g[3] = {0., 0., 0.};
    for (int d = 0; d < 3; ++d) {
        r0[d] = pos_at(R, d, b, p);
        pj[d] = pos_at(R, d, bj, p);
        pk[d] = pos_at(R, d, bk, p);
    }
    const double eps = 1.e-4;
    if (!short_on) {
    } else if (R.pair_type == 3 && N > 1) {
        // IlkkaPairAction::CalcGradientU (ilkka_pair_action_class.h:172-222) per link,
        // as the reference forms it from DrDrpDrrp's r = r_q - r_p (path_class.h:153-166):
        // -(1/2)[U_x (r/|r| + (r - r')/|r - r'|) + U_y (r/|r| - (r - r')/|r - r'|)]
        // - (1/2) u_long'(|r|) r/|r|, |r| and |r'| clamped to the u/diag grid.  The
        // first term is dU/dr_p; the second has the opposite sign of d/dr_p of the
        // -(1/2) u_long(|r|) term of CalcU.
        for (int q = 0; q < N; ++q) {
            if (q == p) continue;
            double q0[3];
            for (int d = 0; d < 3; ++d) q0[d] = pos_at(R, d, b, q);
            for (int lk = 0; lk < 2; ++lk) {
                const double* a1 = lk ? pk : pj;
                double c1[3];
                for (int d = 0; d < 3; ++d) c1[d] = pos_at(R, d, lk ? bk : bj, q);
                LinkGeom gg;
                link_geom(r0, q0, a1, c1, R.L, R.iL, gg);
                const double qq = 0.5 * (gg.r + gg.rp);
                double ux, uy;
                spl2_eval(R.u2, qq + 0.5 * gg.s, qq - 0.5 * gg.s, &ux, &uy);
                double dl = 0.;
                if (R.use_long_range) {
                    double a = gg.r, bb = gg.rp;
                    clamp2(R.r_u_min, R.r_u_max, a, bb);
                    const int ia = spl_locate(R.u_long_r, a);
                    dl = spl_der(R.u_long_r, ia, 0, a - R.u_long_r.x[ia]);
                }
                for (int d = 0; d < 3; ++d) {
                    const double rh = gg.r == 0. ? 0. : gg.rv[d] / gg.r, sh = gg.s == 0. ? 0. : gg.sv[d] / gg.s;
                    g[d] += -0.5 * (ux * (rh + sh) + uy * (rh - sh)) - 0.5 * dl * rh;
                }
            }
        }
    } else if (R.pair_type != 0 && N > 1)
        for (int q = 0; q < N; ++q) {
            if (q == p) continue;
            double q0[3], qj[3], qk[3];
            for (int d = 0; d < 3; ++d) {
                q0[d] = pos_at(R, d, b, q);
                qj[d] = pos_at(R, d, bj, q);
                qk[d] = pos_at(R, d, bk, q);
            }
            for (int lk = 0; lk < 2; ++lk) {
                const double* a1 = lk ? pk : pj;
                const double* c1 = lk ? qk : qj;
                for (int d = 0; d < 3; ++d) {
                    double a0[3] = {r0[0], r0[1], r0[2]};
                    LinkGeom gg;
                    a0[d] = r0[d] + eps;
                    link_geom(a0, q0, a1, c1, R.L, R.iL, gg);
                    const double f1 = pair_u(R, gg.r, gg.rp, gg.s);
                    a0[d] = r0[d] - eps;
                    link_geom(a0, q0, a1, c1, R.L, R.iL, gg);
                    const double f2 = pair_u(R, gg.r, gg.rp, gg.s);
                    g[d] += (f1 - f2) / (2. * eps);
                }
            }
        }
    double* o = (out_est ? R.grad_est : R.grad) + 3 * ((size_t)b * N + p);
    o[0] = g[0];
    o[1] = g[1];
    o[2] = g[2];
}

// Loads a replica's link-action tables into LDS.
__device__ __forceinline__ void stage_tables(const Rep& R, double* lds) {
    stage_batched(lds, R.bt_a.c, R.bt_b.c, R.bt_a.ncoef * R.bt_a.ncomp, R.lds_doubles, 0, (int)blockDim.x);
    __syncthreads();
}

// The same differences for the Bare and David actions, a bead's partners shared by
// a workgroup.  blockIdx.x: slice; np particles per workgroup (a tile blockIdx.y of
// the slice's), whose blockDim.x / np groups of threads (at most one a partner) each
// take a range of the partners; the groups' sums are added in order.  The bead's own distance is the same in the
// links (b, b + 1) and (b, b - 1), and r' moves with the bead only where its image
// does: 6 radial terms at r and 2 at r' per pair instead of 48.  Every link action
// is added up from its terms in k_grad_compat's order, from the same cubics: a
// difference over 2 eps magnifies the rounding of a link action 5000 times, and
// terms left out or in another form (B-splines in LDS: 102 us) come out several
// times further from 64-bit arithmetic.  Bound by FP64 arithmetic and table
// gathers: N = 77, M = 50, 12 replicas 1243 us with a thread per bead, 189 us so.
constexpr int kCompatBlock = 512;  // (1024 spills)
struct RadialTerms {
    double a, l;  // the action's own table (or 0.5 / r) and the long-range one
};
__device__ __forceinline__ RadialTerms radial_terms(const Rep& R, bool bare, double r) {
    RadialTerms t{0., 0.};
    if (bare) {
        // (clamps as in bare_v: one range after the other)
        r = clampd(r, R.r_v_min, R.r_v_max);
        t.a = R.is_coulomb ? 0.5 / r : spl_eval1(R.v_r, r);
        if (R.use_long_range) {
            r = clampd(r, R.r_l_min, R.r_l_max);
            t.l = spl_eval1(R.v_long_r, r);
        }
    } else {
        r = clampd(r, R.g_min, R.g_max);
        const int i = spl_locate(R.u, r);
        t.a = spl_val(R.u, i, 1, r - R.u.x[i]);
    }
    return t;
}
// pair_u from the radial terms at r and r'
__device__ __forceinline__ double pair_u_terms(const Rep& R, bool bare, const RadialTerms& t0, const RadialTerms& t1,
                                               double r0, double r1, double s) {
    if (bare) {
        double v = 0.;
        if (R.is_coulomb) {
            v += t0.a + t1.a;
        } else {
            v += 0.5 * t0.a;
            v += 0.5 * t1.a;
        }
        if (R.use_long_range) {
            v -= 0.5 * t0.l;
            v -= 0.5 * t1.l;
        }
        return R.tau * v;
    }
    const double q = 0.5 * (r0 + r1), z = r0 - r1;
    double u = 0.5 * (t0.a + t1.a);
    if (s > 0.0 && q < R.g_max) {
        const int iq = spl_locate(R.u, q);
        u += david_offdiag(R.u, R.n_order, iq, q - R.u.x[iq], z, s);
    }
    return u;
}
template <int PT>
__global__ __launch_bounds__(kCompatBlock) void k_grad_compat_split(const Rep* __restrict__ reps, int out_est, int short_on,
                                                                    int np) {
    extern __shared__ double lds[];  // [group][np][3]
    const Rep& R = reps[blockIdx.z];
    const int b = blockIdx.x, p0 = blockIdx.y * np, N = R.N, M = R.M;
    if (b >= M || p0 >= N) return;
    const bool on = short_on && R.pair_type != 0 && N > 1;
    const int n = min(np, N - p0), n_grp = min((int)blockDim.x / n, N);
    const int grp = threadIdx.x / n, lp = threadIdx.x % n, p = p0 + lp;
    const bool bare = PT == 1 || (PT == 0 && R.pair_type == 1);
    const double eps = 1.e-4;
    if (on && grp < n_grp) {
        double g[3] = {0., 0., 0.};
        const int b1[2] = {b + 1 == M ? 0 : b + 1, b == 0 ? M - 1 : b - 1};
        const int q_lo = (int)((long long)N * grp / n_grp), q_hi = (int)((long long)N * (grp + 1) / n_grp);
        double r0[3], p1[2][3];
        for (int d = 0; d < 3; ++d) {
            r0[d] = pos_at(R, d, b, p);
            for (int lk = 0; lk < 2; ++lk) p1[lk][d] = pos_at(R, d, b1[lk], p);
        }
        for (int q = q_lo; q < q_hi; ++q) {
            if (q == p) continue;
            double q0[3], q1[2][3], rp[2];
            RadialTerms tp[2];
            LinkGeom gg;
            for (int d = 0; d < 3; ++d) {
                q0[d] = pos_at(R, d, b, q);
                for (int lk = 0; lk < 2; ++lk) q1[lk][d] = pos_at(R, d, b1[lk], q);
            }
#pragma unroll
            for (int lk = 0; lk < 2; ++lk) {
                link_geom(r0, q0, p1[lk], q1[lk], R.L, R.iL, gg);
                rp[lk] = gg.rp;
                tp[lk] = radial_terms(R, bare, gg.rp);
            }
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                double f[2][2];
#pragma unroll
                for (int sg = 0; sg < 2; ++sg) {
                    double a0[3] = {r0[0], r0[1], r0[2]};
                    a0[d] = sg ? r0[d] - eps : r0[d] + eps;
                    RadialTerms t;
#pragma unroll
                    for (int lk = 0; lk < 2; ++lk) {
                        link_geom(a0, q0, p1[lk], q1[lk], R.L, R.iL, gg);
                        if (lk == 0) t = radial_terms(R, bare, gg.r);
                        RadialTerms t1 = tp[lk];
                        if (gg.rp != rp[lk]) t1 = radial_terms(R, bare, gg.rp);  // another image of r'
                        f[lk][sg] = pair_u_terms(R, bare, t, t1, gg.r, gg.rp, gg.s);
                    }
                }
                g[d] += (f[0][0] - f[0][1]) + (f[1][0] - f[1][1]);
            }
        }
        for (int d = 0; d < 3; ++d) lds[((size_t)grp * n + lp) * 3 + d] = g[d] / (2. * eps);
    }
    __syncthreads();
    double* o = (out_est ? R.grad_est : R.grad) + 3 * ((size_t)b * N + p0);
    for (int t = threadIdx.x; t < 3 * n; t += blockDim.x) {
        double v = 0.;
        if (on)
            for (int i = 0; i < n_grp; ++i) v += lds[(size_t)i * 3 * n + t];
        o[t] = v;
    }
}

// radial part of the Bare link action / tau at one distance
__device__ __forceinline__ double bare_radial_lds(const Rep& R, const double* lds, double r) {
    r = clampd(r, R.r_v_min, R.r_v_max);
    double v = R.is_coulomb ? 0.5 / r : 0.5 * bt_apply(lds, bt_basis(R.bt_a, r));
    if (R.use_long_range) {
        const double* vl = lds + (R.is_coulomb ? 0 : R.bt_a.ncoef);
        v -= 0.5 * bt_apply(vl, bt_basis(R.bt_b, clampd(r, R.r_l_min, R.r_l_max)));
    }
    return v;
}
// Analytic adjoint, local terms: kinetic links (b-1,b), (b,b+1) and short-range
// pair links of every other particle.  Writes (overwrites) grad.
__global__ __launch_bounds__(64) void k_adjoint_local(const Rep* __restrict__ reps, unsigned int terms, int out_est) {
    const Rep& R = reps[blockIdx.z];
    const int i = blockIdx.x * 64 + threadIdx.x, b = blockIdx.y;
    if (i >= R.N || b >= R.M) return;
    const int M = R.M, N = R.N;
    const int bn = (b + 1) % M, bp = (b + M - 1) % M;
    double ri[3], rn[3], rp[3], g[3] = {0., 0., 0.};
    for (int d = 0; d < 3; ++d) {
        ri[d] = pos_at(R, d, b, i);
        rn[d] = pos_at(R, d, bn, i);
        rp[d] = pos_at(R, d, bp, i);
    }
    if (terms & 1u) {
        // K(d) = sum_x img(d_x) + |d|^2 i4lt, d = r_b - r_{b+1}: dK/dr_b = K'(d_fwd) - K'(d_bwd);
        // the kinetic links follow the path across the wrap
        const int kn = next_label(R, b, i), kp = prev_label(R, b, i);
        double df[3], db[3];
        for (int d = 0; d < 3; ++d) {
            df[d] = minimg(ri[d] - (kn == i ? rn[d] : pos_at(R, d, bn, kn)), R.L, R.iL);
            db[d] = minimg((kp == i ? rp[d] : pos_at(R, d, bp, kp)) - ri[d], R.L, R.iL);
        }
        for (int d = 0; d < 3; ++d) {
            double kf = 2. * df[d] * R.kin_i4lt, kb = 2. * db[d] * R.kin_i4lt;
            if (R.kin_images > 0) {
                int ia = spl_locate(R.kin[0], df[d]), ib = spl_locate(R.kin[0], db[d]);
                kf += spl_der(R.kin[0], ia, 0, df[d] - R.kin[0].x[ia]);
                kb += spl_der(R.kin[0], ib, 0, db[d] - R.kin[0].x[ib]);
            }
            g[d] += kf - kb;
        }
    }
    if ((terms & 2u) && R.pair_type != 0)
        for (int j = 0; j < N; ++j) {
            if (j == i) continue;
            double j0[3], jn[3], jp[3];
            for (int d = 0; d < 3; ++d) {
                j0[d] = pos_at(R, d, b, j);
                jn[d] = pos_at(R, d, bn, j);
                jp[d] = pos_at(R, d, bp, j);
            }
            LinkGeom gg;
            double ur, urp, us;
            // link (b, b+1), i first: r = r_j(b) - r_i(b); dU/dr_i(b) = -(U_r rhat + U_s shat)
            link_geom(ri, j0, rn, jn, R.L, R.iL, gg);
            pair_u_grad(R, gg.r, gg.rp, gg.s, ur, urp, us);
            for (int d = 0; d < 3; ++d)
                g[d] -= ur * gg.rv[d] / gg.r + ((gg.s > 0.) ? us * gg.sv[d] / gg.s : 0.);
            // link (b-1, b), i first: r' = r_j(b) - r_i(b); dU/dr_i(b) = -(U_r' rphat - U_s shat)
            link_geom(rp, jp, ri, j0, R.L, R.iL, gg);
            pair_u_grad(R, gg.r, gg.rp, gg.s, ur, urp, us);
            for (int d = 0; d < 3; ++d)
                g[d] -= urp * gg.rpv[d] / gg.rp - ((gg.s > 0.) ? us * gg.sv[d] / gg.s : 0.);
        }
    double* o = (out_est ? R.grad_est : R.grad) + 3 * ((size_t)b * N + i);
    o[0] = g[0];
    o[1] = g[1];
    o[2] = g[2];
}

// Analytic adjoint, local terms with LDS tables: one 1024-thread workgroup per
// replica; thread t owns particle i = t % N over a contiguous slice range and
// walks it in order, so each link (b, b+1) of (i, j) is evaluated once for i:
// its r_i(b) part goes to bead b, its r_i(b+1) part is carried to bead b+1.
constexpr int kAdjLdsBlock = 1024;
// PT, NORD: the pair type and David order shared by all replicas (0: per replica)
template <int PT, int NORD>
__global__ __launch_bounds__(kAdjLdsBlock) void k_adjoint_local_lds(const Rep* __restrict__ reps, unsigned int terms,
                                                                    int out_est) {
    extern __shared__ double lds[];
    // gridDim.y workgroups per replica (when replicas are few), each taking a
    // contiguous block of the slice ranges
    const Rep R = reps[blockIdx.x];  // by value: the fields used stay in registers
    stage_tables(R, lds);
    const int M = R.M, N = R.N, bpr = gridDim.y;
    const int per_blk = kAdjLdsBlock / N > 0 ? kAdjLdsBlock / N : 1;  // slice ranges per particle in one workgroup
    const int per = min(M, per_blk * bpr);                               // ... over the replica's workgroups
    const int p_lo = (int)((long long)per * blockIdx.y / bpr), p_hi = (int)((long long)per * (blockIdx.y + 1) / bpr);
    const int n_units = N * (p_hi - p_lo);
    for (int unit = threadIdx.x; unit < n_units; unit += kAdjLdsBlock) {
        const int i = unit % N, part = p_lo + unit / N;
        const int b_lo = (int)((long long)M * part / per), b_hi = (int)((long long)M * (part + 1) / per);
        if (b_lo >= b_hi) continue;
        double carry[3] = {0., 0., 0.};  // d/dr_i(b) from link (b-1, b)
        // the link entering the range
        {
            const int bp = (b_lo + M - 1) % M;
            double rp_[3], ri_[3];
            for (int d = 0; d < 3; ++d) {
                rp_[d] = pos_at(R, d, bp, i);
                ri_[d] = pos_at(R, d, b_lo, i);
            }
            if ((terms & 2u) && R.pair_type != 0)
                for (int j = 0; j < N; ++j) {
                    if (j == i) continue;
                    double jp[3], j0[3];
                    for (int d = 0; d < 3; ++d) {
                        jp[d] = pos_at(R, d, bp, j);
                        j0[d] = pos_at(R, d, b_lo, j);
                    }
                    LinkGeom gg;
                    double ur, urp, us;
                    link_geom_fast(rp_, jp, ri_, j0, R.L, R.iL, gg);
                    pair_u_grad_lds<PT, NORD>(R, lds, gg.r, gg.rp, gg.s, ur, urp, us);
                    const double frp = urp / gg.rp, so = (gg.s > 0.) ? us / gg.s : 0.;
                    for (int d = 0; d < 3; ++d) carry[d] -= frp * gg.rpv[d] - so * gg.sv[d];
                }
        }
        for (int b = b_lo; b < b_hi; ++b) {
            const int bn = (b + 1) % M, bp = (b + M - 1) % M;
            double ri[3], rn[3], rpv[3], g[3], nxt[3] = {0., 0., 0.};
            for (int d = 0; d < 3; ++d) {
                ri[d] = pos_at(R, d, b, i);
                rn[d] = pos_at(R, d, bn, i);
                rpv[d] = pos_at(R, d, bp, i);
                g[d] = carry[d];
            }
            if (terms & 1u) {
                // the kinetic links follow the path across the wrap
                const int kn = next_label(R, b, i), kp = prev_label(R, b, i);
                for (int d = 0; d < 3; ++d) {
                    const double xn = kn == i ? rn[d] : pos_at(R, d, bn, kn), xp = kp == i ? rpv[d] : pos_at(R, d, bp, kp);
                    const double df = minimg(ri[d] - xn, R.L, R.iL), db = minimg(xp - ri[d], R.L, R.iL);
                    double kf = 2. * df * R.kin_i4lt, kb = 2. * db * R.kin_i4lt;
                    if (R.kin_images > 0) {
                        int ia = spl_locate(R.kin[0], df), ib = spl_locate(R.kin[0], db);
                        kf += spl_der(R.kin[0], ia, 0, df - R.kin[0].x[ia]);
                        kb += spl_der(R.kin[0], ib, 0, db - R.kin[0].x[ib]);
                    }
                    g[d] += kf - kb;
                }
            }
            if ((terms & 2u) && R.pair_type != 0)
                for (int j = 0; j < N; ++j) {
                    if (j == i) continue;
                    double j0[3], jn[3];
                    for (int d = 0; d < 3; ++d) {
                        j0[d] = pos_at(R, d, b, j);
                        jn[d] = pos_at(R, d, bn, j);
                    }
                    LinkGeom gg;
                    double ur, urp, us;
                    link_geom_fast(ri, j0, rn, jn, R.L, R.iL, gg);
                    pair_u_grad_lds<PT, NORD>(R, lds, gg.r, gg.rp, gg.s, ur, urp, us);
                    const double fr = ur / gg.r, frp = urp / gg.rp, so = (gg.s > 0.) ? us / gg.s : 0.;
                    for (int d = 0; d < 3; ++d) {
                        g[d] -= fr * gg.rv[d] + so * gg.sv[d];
                        nxt[d] -= frp * gg.rpv[d] - so * gg.sv[d];
                    }
                }
            double* o = (out_est ? R.grad_est : R.grad) + 3 * ((size_t)b * N + i);
            o[0] = g[0];
            o[1] = g[1];
            o[2] = g[2];
            carry[0] = nxt[0];
            carry[1] = nxt[1];
            carry[2] = nxt[2];
        }
    }
}

// dK/dr_i(b) of the two kinetic links at bead (b, i); the links follow the path
// across the wrap.
__device__ __forceinline__ void adj_kinetic(const Rep& R, int b, int i, double* g) {
    const int M = R.M, bn = (b + 1) % M, bp = (b + M - 1) % M;
    const int kn = next_label(R, b, i), kp = prev_label(R, b, i);
    for (int d = 0; d < 3; ++d) {
        const double ri = pos_at(R, d, b, i);
        const double df = minimg(ri - pos_at(R, d, bn, kn), R.L, R.iL), db = minimg(pos_at(R, d, bp, kp) - ri, R.L, R.iL);
        double kf = 2. * df * R.kin_i4lt, kb = 2. * db * R.kin_i4lt;
        if (R.kin_images > 0) {
            int ia = spl_locate(R.kin[0], df), ib = spl_locate(R.kin[0], db);
            kf += spl_der(R.kin[0], ia, 0, df - R.kin[0].x[ia]);
            kb += spl_der(R.kin[0], ib, 0, db - R.kin[0].x[ib]);
        }
        g[d] = kf - kb;
    }
}

// One pair-link's shares of dS/dr: with r = r_q(b) - r_p(b),
// dU/dr_p(b) = -(U_r rhat + U_s shat) = -e0, dU/dr_p(b+1) = -(U_r' rphat - U_s shat) = -e1,
// and q's are e0, e1.  The geometry is link_geom_fast's.
template <int PT, int NORD>
__device__ __forceinline__ void adj_pair_eval(const Rep& R, const double* lds, const double* a0, const double* c0,
                                              const double* a1, const double* c1, double* rv, double* rpv, double* e0,
                                              double* e1) {
    double rr = 0., pp = 0., ss = 0.;
    for (int d = 0; d < 3; ++d) {
        rv[d] = c0[d] - a0[d];
        rpv[d] = c1[d] - a1[d];
        rv[d] -= rint(rv[d] * R.iL) * R.L;
        rpv[d] += rint((rv[d] - rpv[d]) * R.iL) * R.L;
        const double sv = rv[d] - rpv[d];
        rr += rv[d] * rv[d];
        pp += rpv[d] * rpv[d];
        ss += sv * sv;
    }
    const double r = sqrt_pos(rr), rp = sqrt_pos(pp), sl = sqrt_pos(ss);
    double ur, urp, us;
    pair_u_grad_lds<PT, NORD>(R, lds, r, rp, sl, ur, urp, us);
    const double fr = ur / r, frp = urp / rp, so = (sl > 0.) ? us / sl : 0.;
    for (int d = 0; d < 3; ++d) {
        const double sv = rv[d] - rpv[d];
        e0[d] = fr * rv[d] + so * sv;
        e1[d] = frp * rpv[d] - so * sv;
    }
}

// Adds the short-range pair terms of link (b, b+1) to dS/dr at beads b and b+1,
// one wave, each pair-link evaluated once for both of its particles.  The
// particles are taken in tiles of 64.  For a tile pair (I, J >= I), lane l holds
// particle p = 64I + l and at step s evaluates its link with q = 64J + (l + s)
// mod 64 (I = J: (l + s) mod n for s = 1 .. n/2, the last step on half the lanes
// when n is even).  p's share stays in registers; q's, the same vector with the
// opposite sign, is added to q's slot in the wave's LDS slots (6 x 64 doubles,
// component-major): at one step the lanes touch distinct slots, and one wave's
// LDS operations complete in order, so every sum is formed in a fixed order.
template <int PT, int NORD>
__device__ void adj_link_pairs(const Rep& R, const double* lds, double* slot, double* __restrict__ o, int b, int lane) {
    const int M = R.M, N = R.N, b1 = (b + 1) % M, T = (N + kWave - 1) / kWave;
    for (int I = 0; I < T; ++I) {
        const int nI = min(kWave, N - I * kWave), p = I * kWave + lane;
        const bool pv = lane < nI;
        double a0[3], a1[3], acc[6] = {0., 0., 0., 0., 0., 0.};
        for (int d = 0; d < 3; ++d) {
            a0[d] = pv ? pos_at(R, d, b, p) : 0.;
            a1[d] = pv ? pos_at(R, d, b1, p) : 0.;
        }
        for (int J = I; J < T; ++J) {
            const bool diag = J == I;
            const int nJ = min(kWave, N - J * kWave);
            const int s0 = diag ? 1 : 0, s1 = diag ? nI / 2 : kWave - 1;
            for (int k = 0; k < 6; ++k) slot[k * kWave + lane] = 0.;
            for (int s = s0; s <= s1; ++s) {
                const int ql = diag ? (pv ? (lane + s) % nI : lane) : ((lane + s) & (kWave - 1));
                const bool act = pv && (diag ? !((nI % 2 == 0) && s == nI / 2 && lane >= nI / 2) : ql < nJ);
                if (!act) continue;
                const int q = J * kWave + ql;
                double c0[3], c1[3];
                for (int d = 0; d < 3; ++d) {
                    c0[d] = pos_at(R, d, b, q);
                    c1[d] = pos_at(R, d, b1, q);
                }
                double rv[3], rpv[3], e0[3], e1[3];
                adj_pair_eval<PT, NORD>(R, lds, a0, c0, a1, c1, rv, rpv, e0, e1);
                for (int d = 0; d < 3; ++d) {
                    acc[d] -= e0[d];
                    acc[3 + d] -= e1[d];
                    slot[d * kWave + ql] += e0[d];
                    slot[(3 + d) * kWave + ql] += e1[d];
                }
            }
            if (diag) {
                for (int k = 0; k < 6; ++k) acc[k] += slot[k * kWave + lane];
            } else if (lane < nJ) {
                double* o0 = o + 3 * ((size_t)b * N + J * kWave + lane);
                double* o1 = o + 3 * ((size_t)b1 * N + J * kWave + lane);
                for (int d = 0; d < 3; ++d) {
                    o0[d] += slot[d * kWave + lane];
                    o1[d] += slot[(3 + d) * kWave + lane];
                }
            }
        }
        if (pv) {
            double* o0 = o + 3 * ((size_t)b * N + p);
            double* o1 = o + 3 * ((size_t)b1 * N + p);
            for (int d = 0; d < 3; ++d) {
                o0[d] += acc[d];
                o1[d] += acc[3 + d];
            }
        }
    }
}

// Analytic adjoint, local terms, each pair-link evaluated once: one 1024-thread
// workgroup per replica (gridDim.y per replica when replicas are few); wave w
// owns links [b_lo, b_hi) of n_rng contiguous ranges of at least two links.
// Phase 0 writes the kinetic term of beads b_lo+1 .. b_hi and adds the pair
// terms of links b_lo+1 .. b_hi-1, all of whose beads it owns; phase 1, the
// next launch, adds those of link b_lo, whose bead b_lo the previous range
// wrote.  Every bead's sum is formed in a fixed order.  Dynamic LDS: the
// replica's tables, then kAdjSlotDoubles per wave.
constexpr int kAdjPairWaves = kAdjLdsBlock / kWave;
constexpr int kAdjSlotDoubles = 6 * kWave;  // one wave's partner slots
template <int PT, int NORD>
__global__ __launch_bounds__(kAdjLdsBlock) void k_adjoint_pairs_lds(const Rep* __restrict__ reps, unsigned int terms,
                                                                    int out_est, int phase) {
    extern __shared__ double lds[];
    const Rep R = reps[blockIdx.x];
    const bool pairs = (terms & 2u) && R.pair_type != 0 && R.N > 1;
    if (phase == 1 && !pairs) return;
    if (pairs) stage_tables(R, lds);
    const int M = R.M, N = R.N;
    const int n_rng = max(1, min(kAdjPairWaves * (int)gridDim.y, M / 2));
    const int w = blockIdx.y * kAdjPairWaves + threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    if (w >= n_rng) return;
    const int b_lo = (int)((long long)M * w / n_rng), b_hi = (int)((long long)M * (w + 1) / n_rng);
    double* o = out_est ? R.grad_est : R.grad;
    // the wave's partner slots follow the replica's tables
    double* slot = lds + R.lds_doubles + (threadIdx.x / kWave) * kAdjSlotDoubles;
    if (phase == 1) {
        adj_link_pairs<PT, NORD>(R, lds, slot, o, b_lo, lane);
        return;
    }
    for (int b = b_lo + 1; b <= b_hi; ++b) {
        const int bb = b % M;
        for (int p = lane; p < N; p += kWave) {
            double g[3] = {0., 0., 0.};
            if (terms & 1u) adj_kinetic(R, bb, p, g);
            double* op = o + 3 * ((size_t)bb * N + p);
            op[0] = g[0];
            op[1] = g[1];
            op[2] = g[2];
        }
    }
    if (pairs)
        for (int b = b_lo + 1; b < b_hi; ++b) adj_link_pairs<PT, NORD>(R, lds, slot, o, b, lane);
}

// Analytic adjoint, local terms, for few replicas: each pair-link evaluated once,
// with a whole workgroup per link (h workgroups when M links alone leave CUs
// idle).  A range of links per wavefront, as above, needs thousands of links in
// flight; here the 64 partner rotations of a tile pair (64 x 64 particles) are
// dealt to the workgroup's 16 wavefronts, so one chain fills the chip.  What
// bounds it then is the evaluation itself, at LDS-gather latency: N = 256,
// M = 128, one replica, 75 us, against 563 us for a thread per bead
// on the LDS tables (twice the evaluations, a quarter of the threads busy) and
// 1177 us for a thread per bead on the global ones.
// Each tile pair's sums are added over the wavefronts in order and go to the
// link's own share of part, [h][M][link's first and second slice][3][particle]
// (strides: max_M, max_N), which k_adjoint_gather adds up: every sum is formed
// in a fixed order, with no atomics.
template <int PT, int NORD>
__global__ __launch_bounds__(kAdjLdsBlock) void k_adjoint_links(const Rep* __restrict__ reps, int h, int max_M, int max_N,
                                                                double* __restrict__ part) {
    extern __shared__ double lds[];
    const Rep R = reps[blockIdx.y];
    const int b = blockIdx.x / h, hh = blockIdx.x % h;
    if (b >= R.M || R.N < 2 || R.pair_type == 0) return;
    stage_tables(R, lds);
    const int M = R.M, N = R.N, b1 = b + 1 == M ? 0 : b + 1, T = (N + kWave - 1) / kWave;
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    double* slots = lds + R.lds_doubles;  // [wavefront][6][64]
    double* slot = slots + w * kAdjSlotDoubles;
    double* P = part + (((size_t)blockIdx.y * h + hh) * max_M + b) * 6 * max_N;
    // thread t < 384 owns component t / 64 of the particles t % 64 + 64 J
    const bool own = threadIdx.x < kAdjSlotDoubles;
    double* Pt = P + (size_t)(threadIdx.x >> 6) * max_N + lane;
    if (own)
        for (int J = 0; J * kWave + lane < N; ++J) Pt[J * kWave] = 0.;
    const int n_pairs = T * (T + 1) / 2;
    const int u_lo = (int)((long long)n_pairs * hh / h), u_hi = (int)((long long)n_pairs * (hh + 1) / h);
    int I = 0, J = u_lo;  // tile pair u is (I, J >= I), row by row
    while (J >= T - I) {
        J -= T - I;
        ++I;
    }
    J += I;
    for (int u = u_lo; u < u_hi; ++u) {
        const bool diag = J == I;
        const int nI = min(kWave, N - I * kWave), nJ = min(kWave, N - J * kWave), p = I * kWave + lane;
        const bool pv = lane < nI;
        double a0[3], a1[3], acc[6] = {0., 0., 0., 0., 0., 0.};
        for (int d = 0; d < 3; ++d) {
            a0[d] = pv ? pos_at(R, d, b, p) : 0.;
            a1[d] = pv ? pos_at(R, d, b1, p) : 0.;
        }
        for (int k = 0; k < 6; ++k) slot[k * kWave + lane] = 0.;
        const int s1 = diag ? nI / 2 : kWave - 1;
        for (int s = (diag ? 1 : 0) + w; s <= s1; s += kAdjPairWaves) {
            const int ql = diag ? (pv ? (lane + s) % nI : lane) : ((lane + s) & (kWave - 1));
            const bool act = pv && (diag ? !((nI % 2 == 0) && s == nI / 2 && lane >= nI / 2) : ql < nJ);
            if (!act) continue;
            const int q = J * kWave + ql;
            double c0[3], c1[3];
            for (int d = 0; d < 3; ++d) {
                c0[d] = pos_at(R, d, b, q);
                c1[d] = pos_at(R, d, b1, q);
            }
            double rv[3], rpv[3], e0[3], e1[3];
            adj_pair_eval<PT, NORD>(R, lds, a0, c0, a1, c1, rv, rpv, e0, e1);
            for (int d = 0; d < 3; ++d) {
                acc[d] -= e0[d];
                acc[3 + d] -= e1[d];
                slot[d * kWave + ql] += e0[d];
                slot[(3 + d) * kWave + ql] += e1[d];
            }
        }
        __syncthreads();
        double v = 0.;
        if (own) {
            for (int i = 0; i < kAdjPairWaves; ++i) v += slots[i * kAdjSlotDoubles + threadIdx.x];
            if (lane < nJ) Pt[J * kWave] += v;
        }
        __syncthreads();
        for (int k = 0; k < 6; ++k) slot[k * kWave + lane] = acc[k];
        __syncthreads();
        if (own) {
            v = 0.;
            for (int i = 0; i < kAdjPairWaves; ++i) v += slots[i * kAdjSlotDoubles + threadIdx.x];
            if (pv) Pt[I * kWave] += v;
        }
        __syncthreads();
        if (++J == T) J = ++I;
    }
}

// dS/dr of every bead from k_adjoint_links's shares: the kinetic term, then the
// link the bead begins and the one it ends, share by share.
__global__ __launch_bounds__(256) void k_adjoint_gather(const Rep* __restrict__ reps, unsigned int terms, int out_est,
                                                        int h, int max_M, int max_N, const double* __restrict__ part) {
    const Rep& R = reps[blockIdx.y];
    const int b = blockIdx.x;
    if (b >= R.M) return;
    const int bp = b == 0 ? R.M - 1 : b - 1;
    const bool pairs = (terms & 2u) && R.pair_type != 0 && R.N > 1;
    for (int p = threadIdx.x; p < R.N; p += 256) {
        double g[3] = {0., 0., 0.};
        if (terms & 1u) adj_kinetic(R, b, p, g);
        if (pairs)
            for (int hh = 0; hh < h; ++hh) {
                const double* P = part + ((size_t)blockIdx.y * h + hh) * max_M * 6 * max_N + p;
                for (int d = 0; d < 3; ++d)
                    g[d] += P[((size_t)b * 6 + d) * max_N] + P[((size_t)bp * 6 + 3 + d) * max_N];
            }
        double* o = (out_est ? R.grad_est : R.grad) + 3 * ((size_t)b * R.N + p);
        o[0] = g[0];
        o[1] = g[1];
        o[2] = g[2];
    }
}

// Whole-path pair sums with LDS tables (which 0: CalcdUdBeta over every link, 1:
// CalcV on plain minimum images), one partial sum per workgroup, S x Q workgroups
// per replica (blockIdx.y): S contiguous slice ranges, Q parts of the pairs
// (i, i + d mod N), d = 1..N/2.  A thread walks each of its pairs along its range
// of slices.  What bounds it is the gathers from the LDS tables (36 doubles a link
// with every term read), so a link reads fewer: dU/dbeta takes the sum of the
// potential and the first component as one table (stage_whole), and the radial
// term at a link's second slice is the next link's first where both see the same
// image, which leaves 24; on plain minimum images the two are always the same, and
// a potential is one term per slice.  dU/dbeta and the potential of N = 1024,
// M = 128, one replica, 862 us together, 2495 us with a workgroup per slice (half
// the CUs) and every term read; dU/dbeta of 512 replicas of N = 256, M = 128
// 18.8 ms, 26.5 ms before; of one 51 us, 114 us before.
constexpr int kWholeBlock = 1024;
// The tables of the whole-path sums.  Bare: [v_r][v_long_r].  David: which 0 the
// sum of components 0 and 1 of du_kj_dbeta, then components 2..n_val; which 1
// component 0.
__device__ __forceinline__ void stage_whole(const Rep& R, double* lds, int which) {
    if (R.pair_type != 2) {
        stage_batched(lds, R.bt_a.c, R.bt_b.c, R.bt_a.ncoef * R.bt_a.ncomp, R.lds_doubles, 0, (int)blockDim.x);
    } else {
        const int nc = R.bt_du.ncoef, n = which ? nc : nc * (R.bt_du.ncomp - 1);
        for (int t = threadIdx.x; t < n; t += (int)blockDim.x)
            lds[t] = which ? R.bt_du.c[t] : t < nc ? R.bt_du.c[t] + R.bt_du.c[nc + t] : R.bt_du.c[nc + t];
    }
    __syncthreads();
}
template <int PT, int NORD>
__global__ __launch_bounds__(kWholeBlock) void k_pair_whole_lds(const Rep* __restrict__ reps, int which, int S, int Q,
                                                                double* __restrict__ part) {
    extern __shared__ double lds[];
    const Rep R = reps[blockIdx.x];
    __shared__ double red[kWholeBlock / kWave];
    const int s = blockIdx.y / Q, q = blockIdx.y % Q, N = R.N, M = R.M, half = N / 2;
    const int b_lo = (int)((long long)M * s / S), b_hi = (int)((long long)M * (s + 1) / S);
    const bool on = R.pair_type != 0 && half > 0 && b_lo < b_hi;
    double t = 0.;
    if (on) {
        stage_whole(R, lds, which);
        const bool bare = PT == 1 || (PT == 0 && R.pair_type == 1);
        const BTab& T = R.bt_du;
        auto radial = [&](double r) {
            return bare ? bare_radial_lds(R, lds, r) : 0.5 * bt_apply(lds, bt_basis(T, clampd(r, R.g_min, R.g_max)));
        };
        const long long n_pairs = (long long)N * half;
        const long long u_lo = n_pairs * q / Q, u_hi = n_pairs * (q + 1) / Q;
        for (long long u = u_lo + threadIdx.x; u < u_hi; u += kWholeBlock) {
            const int dd = 1 + (int)(u / N), i = (int)(u % N);
            if ((N % 2 == 0) && dd == half && i >= half) continue;
            const int j = i + dd < N ? i + dd : i + dd - N;
            double rv[3];
            for (int d = 0; d < 3; ++d) rv[d] = minimg(pos_at(R, d, b_lo, j) - pos_at(R, d, b_lo, i), R.L, R.iL);
            double r = sqrt_pos(rv[0] * rv[0] + rv[1] * rv[1] + rv[2] * rv[2]);
            double f = radial(r);
            if (which) {
                // sum over the links of (v(r_b) + v(r_b+1)) / 2 = sum over the slices of v(r_b)
                t += 2. * f;
                for (int b = b_lo + 1; b < b_hi; ++b) {
                    double rr = 0.;
                    for (int d = 0; d < 3; ++d) {
                        const double x = minimg(pos_at(R, d, b, j) - pos_at(R, d, b, i), R.L, R.iL);
                        rr += x * x;
                    }
                    t += 2. * radial(sqrt_pos(rr));
                }
                continue;
            }
            // the link's second slice is loaded one link ahead
            double xi[3], xj[3];
            int bn = b_lo + 1 == M ? 0 : b_lo + 1;
            for (int d = 0; d < 3; ++d) {
                xi[d] = pos_at(R, d, bn, i);
                xj[d] = pos_at(R, d, bn, j);
            }
            for (int b = b_lo; b < b_hi; ++b) {
                double rp[3], nx[3], dx[3], pp = 0., s2 = 0.;
                for (int d = 0; d < 3; ++d) dx[d] = xj[d] - xi[d];
                bn = bn + 1 == M ? 0 : bn + 1;
                for (int d = 0; d < 3; ++d) {
                    xi[d] = pos_at(R, d, bn, i);
                    xj[d] = pos_at(R, d, bn, j);
                }
                bool same = true;  // r' is the next link's r
                for (int d = 0; d < 3; ++d) {
                    const double x = dx[d];
                    const double shift = rint((rv[d] - x) * R.iL), home = rint(x * R.iL);
                    rp[d] = x + shift * R.L;
                    nx[d] = x - home * R.L;
                    same = same && shift == -home;
                    const double sv = rv[d] - rp[d];
                    pp += rp[d] * rp[d];
                    s2 += sv * sv;
                }
                const double r1 = sqrt_pos(pp), f1 = radial(r1);
                t += f + f1;
                if (!bare) {
                    const double qm = 0.5 * (r + r1), z = r - r1;
                    if (s2 > 0.0 && qm < R.g_max) {
                        const BBasis bq = bt_basis(T, qm);
                        const double z2 = z * z;
                        double sp[4], zp[4];
                        sp[0] = 1.;
                        zp[0] = 1.;
#pragma unroll
                        for (int e = 1; e <= (NORD ? NORD : 3); ++e) {
                            sp[e] = sp[e - 1] * s2;
                            zp[e] = zp[e - 1] * z2;
                        }
                        const int n_order = NORD ? NORD : R.n_order;
#pragma unroll
                        for (int k = 1; k <= (NORD ? NORD : 3); ++k) {
                            if (k > n_order) break;
#pragma unroll
                            for (int e = 0; e <= k; ++e)
                                t += bt_apply(lds + (size_t)(k * (k + 1) / 2 + e) * T.ncoef, bq) * zp[e] * sp[k - e];
                        }
                    }
                }
                r = r1;
                f = f1;
                if (!same) {
                    r = sqrt_pos(nx[0] * nx[0] + nx[1] * nx[1] + nx[2] * nx[2]);
                    f = radial(r);
                }
                for (int d = 0; d < 3; ++d) rv[d] = nx[d];
            }
        }
    }
    t = wave_sum(t);
    if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x / kWave] = t;
    __syncthreads();
    if (threadIdx.x == 0) {
        double tt = 0.;
        for (int w = 0; w < kWholeBlock / kWave; ++w) tt += red[w];
        part[(size_t)blockIdx.x * S * Q + blockIdx.y] = tt;
    }
}

// Factor on the long-range gradient: 1 for the adjoint; with compat, the
// reference's GetActionGradient (pair_action_class.h:331-334) adds
// IlkkaPairAction::CalcGradientULong (ilkka_pair_action_class.h:231-249), half
// the adjoint term, once per particle pair, i.e. (N - 1) / 2; the Bare and David
// actions add nothing (pair_action_class.h:158-165).
__device__ __forceinline__ double long_grad_scale(const Rep& R, int compat) {
    if (!compat) return 1.;
    return R.pair_type == 3 ? 0.5 * (R.N - 1.) : 0.;
}

// Analytic adjoint, Ewald term: d/dr_i of long_scale sum_k coef_s |rho(b,k)|^2
// = -2 long_scale sum_k coef_s k Im(conj(rho) e^{i k.r_i}).  Block = 64 beads of
// one slice; rho(b,:) staged through LDS in k tiles; per-bead phase tables in LDS.
constexpr int kAdjTile = 128;
__global__ __launch_bounds__(64) void k_adjoint_long(const Rep* __restrict__ reps, int out_est, int compat) {
    const Rep& R = reps[blockIdx.z];
    const int b = blockIdx.y;
    if (b >= R.M || (int)blockIdx.x * 64 >= R.N || !R.use_long_range || R.pair_type == 0) return;
    const int i = blockIdx.x * 64 + threadIdx.x;
    const int mx = R.max_idx, stride = mx + 1;
    extern __shared__ double2 dyn[];
    double2* tab = dyn;                            // [64][3][stride]
    double2* rho_t = dyn + 64 * 3 * stride;        // [kAdjTile]
    int* kp_t = (int*)(rho_t + kAdjTile);          // [kAdjTile]
    double* cf_t = (double*)(kp_t + kAdjTile);     // [kAdjTile]
    const bool valid = i < R.N;
    double2* my = tab + threadIdx.x * 3 * stride;
    if (valid)
        for (int d = 0; d < 3; ++d) phase_chain(pos_at(R, d, b, i) * R.box, mx, my + d * stride);
    double g[3] = {0., 0., 0.};
    const double2* rb = R.rho + ((size_t)R.sel[b] * R.M + b) * R.nk;
    for (int k0 = 0; k0 < R.nk; k0 += kAdjTile) {
        __syncthreads();
        for (int t = threadIdx.x; t < kAdjTile; t += 64) {
            const int k = k0 + t;
            if (k < R.nk) {
                rho_t[t] = rb[k];
                kp_t[t] = R.kidx[k];
                cf_t[t] = R.coef_s[k];
            }
        }
        __syncthreads();
        if (valid) {
            const int nt = min(kAdjTile, R.nk - k0);
            for (int t = 0; t < nt; ++t) {
                const int kp = kp_t[t];
                const double2 e = phase_k(my, stride, kp);
                const double2 rv = rho_t[t];
                // Im(conj(rho) e) = rho.x e.y - rho.y e.x
                const double im = cf_t[t] * (rv.x * e.y - rv.y * e.x);
                g[0] += im * ((kp & 255) - 128);
                g[1] += im * (((kp >> 8) & 255) - 128);
                g[2] += im * (((kp >> 16) & 255) - 128);
            }
        }
    }
    if (valid) {
        double* o = (out_est ? R.grad_est : R.grad) + 3 * ((size_t)b * R.N + i);
        const double f = -2. * long_grad_scale(R, compat) * R.long_scale * R.box;
        o[0] += f * g[0];
        o[1] += f * g[1];
        o[2] += f * g[2];
    }
}

// Long-range adjoint: dS_long/dr_p(b) = -2 s box sum_k c_k n_k Im(conj(rho_k) e^{ik.r}).
// The k-vectors are grouped in columns (n0, n1) of n2 = -m..m.  With w = c conj(rho)
// and c_n = e^{i n phi_2}, a column's sums over n >= 0,
//   A = sum w(n) c_n + w(-n) conj(c_n),   B = sum n (w(n) c_n - w(-n) conj(c_n)),
// take four real weights per n (k_adjoint_weights writes them, once per slice):
//   s1 = Re(w+ + w-), s2 = Im(w- - w+), s3 = Re(w+ - w-), s4 = Im(w+ + w-):
//   A = (s1 cx + s2 cy, s3 cy + s4 cx),   B = n (s3 cx - s4 cy, s1 cy - s2 cx),
// and the gradient takes Im(E A) n0, Im(E A) n1, Im(E B), E = e^{i (n0 phi_0 + n1 phi_1)}.
// So both signs of n2 cost eight multiply-adds, all independent, with a
// particle's c_n and n c_n in registers (NM of them); walking the runs of
// consecutive n2 (k_adjoint_long_runs, kept for |n2| above 15) is one serial
// chain of complex products, nine operations a k-vector.  The weights are the
// same for every lane: they come through the scalar cache, which leaves LDS
// and the vector memory path free (a broadcast LDS read costs as much as a
// gather).  A wavefront takes 64 particles of a slice and one of the block's
// segments of the columns; the segments' sums are added in order.
// N = 256, M = 128, 1979 k-vectors: one replica 170 us by runs with a thread per
// particle, 57 us by runs in 16 segments, 47 us so (36 us and the weights' 11);
// 512 replicas 14.6 ms by runs, 14.1 ms (17 ms with a tile per workgroup: the
// weights then miss the scalar cache); N = 1024, 4012 k-vectors, 8 replicas
// 2.9 ms by runs, 1.6 ms.
constexpr int kAdjColMax = 16;  // |n2| + 1 at most
constexpr int kAdjColPad = 4;   // a column's entries are padded (k = -1) to whole groups of this
__global__ __launch_bounds__(256) void k_adjoint_weights(const Rep* __restrict__ reps, int max_M, int stride,
                                                         double4* __restrict__ wts) {
    const Rep& R = reps[blockIdx.y];
    const int b = blockIdx.x;
    if (b >= R.M || !R.use_long_range || R.pair_type == 0) return;
    const double2* rb = R.rho + ((size_t)R.sel[b] * R.M + b) * R.nk;
    double4* o = wts + ((size_t)blockIdx.y * max_M + b) * stride;
    for (int t = threadIdx.x; t < R.n_col_k; t += 256) {
        const int2 k = R.col_k[t];  // the k-vectors at n2 and -n2, or -1
        double2 p = make_double2(0., 0.), m = p;
        if (k.x >= 0) {
            const double2 v = rb[k.x];
            const double c = R.coef_s[k.x];
            p = make_double2(c * v.x, -c * v.y);
        }
        if (k.y >= 0) {
            const double2 v = rb[k.y];
            const double c = R.coef_s[k.y];
            m = make_double2(c * v.x, -c * v.y);
        }
        o[t] = make_double4(p.x + m.x, m.y - p.y, p.x - m.x, p.y + m.y);
    }
}
// blockDim.x = 64 n_seg tiles-per-block: n_seg > 1 splits one tile's columns; with
// one segment up to four tiles of a slice share a workgroup, and so its weights
// in the scalar cache.
template <int NM>
__global__ __launch_bounds__(512) void k_adjoint_cols(const Rep* __restrict__ reps, int n_seg, int max_M, int stride,
                                                      const double4* __restrict__ wts, int out_est, int compat) {
    const Rep& R = reps[blockIdx.z];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
    const int seg = n_seg > 1 ? wave : 0, b = blockIdx.y;
    const int p0 = (n_seg > 1 ? (int)blockIdx.x : (int)blockIdx.x * (int)(blockDim.x / kWave) + wave) * kWave;
    if (b >= R.M || p0 >= R.N || !R.use_long_range || R.pair_type == 0) return;
    __shared__ double sums[512 * 3];
    const int p = min(p0 + lane, R.N - 1);
    // the segment's columns, about as many weights each
    const int4* __restrict__ cols = R.cols;
    const int n_cols = R.n_cols;
    auto first = [&](int t) {
        int lo = 0, hi = n_cols;
        while (lo < hi) {
            const int m = (lo + hi) >> 1;
            if (uld(&cols[m].z) < t)
                lo = m + 1;
            else
                hi = m;
        }
        return lo;
    };
    const int u_lo = n_seg > 1 ? first(R.n_col_k * seg / n_seg) : 0;
    const int u_hi = n_seg > 1 ? first(R.n_col_k * (seg + 1) / n_seg) : n_cols;
    const double4* __restrict__ W = wts + ((size_t)blockIdx.z * max_M + b) * stride;
    double2 st[3], c[NM], nc[NM];
    for (int d = 0; d < 3; ++d) {
        double sn, cs;
        sincos(pos_at(R, d, b, p) * R.box, &sn, &cs);
        st[d] = make_double2(cs, sn);
    }
    c[0] = make_double2(1., 0.);
    nc[0] = make_double2(0., 0.);
#pragma unroll
    for (int n = 1; n < NM; ++n) {
        c[n] = cmul(st[2], c[n - 1]);
        nc[n] = make_double2(n * c[n].x, n * c[n].y);
    }
    const double2 cst0 = make_double2(st[0].x, -st[0].y), cst1 = make_double2(st[1].x, -st[1].y);
    double2 e0 = make_double2(1., 0.), e1 = make_double2(1., 0.);
    int c0 = 0, c1 = 0;
    double g0 = 0., g1 = 0., g2 = 0.;
    for (int u = u_lo; u < u_hi; ++u) {
        // n0 + 128 | (n1 + 128) << 8, entries (n = 0 .. entries - 1), first entry
        const int n01 = uld(&cols[u].x), len = uld(&cols[u].y);
        const int n0 = (n01 & 255) - 128, n1 = (n01 >> 8) - 128;
        for (; c0 < n0; ++c0) e0 = cmul(e0, st[0]);
        for (; c0 > n0; --c0) e0 = cmul(e0, cst0);
        for (; c1 < n1; ++c1) e1 = cmul(e1, st[1]);
        for (; c1 > n1; --c1) e1 = cmul(e1, cst1);
        const double* w = reinterpret_cast<const double*>(W + uld(&cols[u].z));
        double ax = 0., ay = 0., bx = 0., by = 0.;
#pragma unroll
        for (int q = 0; q < NM; q += kAdjColPad) {
            if (q < len) {  // (a break would keep the loop from unrolling: c and nc would go to scratch)
                double s[kAdjColPad][4];
#pragma unroll
                for (int i = 0; i < 4 * kAdjColPad; ++i) s[i / 4][i % 4] = uld(w + 4 * q + i);
#pragma unroll
                for (int i = 0; i < kAdjColPad; ++i) {
                    const int n = q + i;
                    ax = fma(s[i][1], c[n].y, fma(s[i][0], c[n].x, ax));
                    ay = fma(s[i][3], c[n].x, fma(s[i][2], c[n].y, ay));
                    if (n > 0) {
                        bx = fma(-s[i][3], nc[n].y, fma(s[i][2], nc[n].x, bx));
                        by = fma(-s[i][1], nc[n].x, fma(s[i][0], nc[n].y, by));
                    }
                }
            }
        }
        const double2 e = cmul(e0, e1);
        const double ia = fma(e.x, ay, e.y * ax);
        g0 = fma((double)n0, ia, g0);
        g1 = fma((double)n1, ia, g1);
        g2 = fma(e.x, by, fma(e.y, bx, g2));
    }
    const double f = -2. * long_grad_scale(R, compat) * R.long_scale * R.box;
    double* o = (out_est ? R.grad_est : R.grad) + 3 * ((size_t)b * R.N + p0);
    if (n_seg > 1) {
        double* mine = sums + threadIdx.x * 3;
        mine[0] = g0;
        mine[1] = g1;
        mine[2] = g2;
        __syncthreads();
        for (int t = threadIdx.x; t < 3 * kWave && p0 + t / 3 < R.N; t += blockDim.x) {
            double g = 0.;
            for (int i = 0; i < n_seg; ++i) g += sums[i * 3 * kWave + t];
            o[t] += f * g;
        }
    } else if (p0 + lane < R.N) {
        o[3 * lane] += f * g0;
        o[3 * lane + 1] += f * g1;
        o[3 * lane + 2] += f * g2;
    }
}

// Long-range adjoint by runs: dS_long/dr_p(b) = -2 s box sum_k c_k n_k Im(conj(rho_k) e^{ik.r}).
// One workgroup per (slice, replica), a thread per particle.  The k-vectors are
// walked in runs of consecutive n2 at fixed (n0, n1), so each phase is the
// previous one times e^{+-i phi_2} (one complex product), and the weights
// w_k = c_k conj(rho_k) sit in LDS in run order: every lane reads the same
// address (a broadcast).  Run starts step running phases e^{i n0 phi_0},
// e^{i n1 phi_1}; the runs are ordered by (n0, n1) so those steps are short.
constexpr int kAdjRunBlock = 256;
__global__ __launch_bounds__(kAdjRunBlock) void k_adjoint_long_runs(const Rep* __restrict__ reps, int out_est, int compat) {
    const Rep& R = reps[blockIdx.y];
    const int b = blockIdx.x;
    if (b >= R.M || !R.use_long_range || R.pair_type == 0) return;
    extern __shared__ double2 wsh[];
    int4* runs = (int4*)(wsh + R.nk);
    const int nk = R.nk, n_runs = R.n_runs;
    const double2* rb = R.rho + ((size_t)R.sel[b] * R.M + b) * nk;
    for (int t = threadIdx.x; t < nk; t += kAdjRunBlock) {
        const int k = R.k_order[t];
        const double2 rv = rb[k];
        const double cf = R.coef_s[k];
        wsh[t] = make_double2(cf * rv.x, -cf * rv.y);
    }
    for (int t = threadIdx.x; t < n_runs; t += kAdjRunBlock) runs[t] = R.k_runs[t];
    __syncthreads();
    const double f = -2. * long_grad_scale(R, compat) * R.long_scale * R.box;
    for (int p = threadIdx.x; p < R.N; p += kAdjRunBlock) {
        double2 st[3];
        for (int d = 0; d < 3; ++d) {
            double sn, cs;
            sincos(pos_at(R, d, b, p) * R.box, &sn, &cs);
            st[d] = make_double2(cs, sn);
        }
        const double2 cst0 = make_double2(st[0].x, -st[0].y), cst1 = make_double2(st[1].x, -st[1].y);
        const double2 cst2 = make_double2(st[2].x, -st[2].y);
        double2 e0 = make_double2(1., 0.), e1 = make_double2(1., 0.);
        int c0 = 0, c1 = 0, off = 0;
        double g0 = 0., g1 = 0., g2 = 0.;
        for (int u = 0; u < n_runs; ++u) {
            const int4 h = runs[u];
            for (; c0 < h.x; ++c0) e0 = cmul(e0, st[0]);
            for (; c0 > h.x; --c0) e0 = cmul(e0, cst0);
            for (; c1 < h.y; ++c1) e1 = cmul(e1, st[1]);
            for (; c1 > h.y; --c1) e1 = cmul(e1, cst1);
            double2 e = cmul(e0, e1);
            const int n2 = h.z, len = h.w > 0 ? h.w : -h.w;
            for (int m = 0; m < n2; ++m) e = cmul(e, st[2]);
            for (int m = 0; m > n2; --m) e = cmul(e, cst2);
            const double2 step = h.w > 0 ? st[2] : cst2;
            const double dn = h.w > 0 ? 1. : -1.;
            double sr = 0., tr = 0., n2d = (double)n2;
            for (int i = 0; i < len; ++i) {
                const double2 w = wsh[off + i];
                const double im = w.x * e.y + w.y * e.x;  // Im(w e)
                sr += im;
                tr = fma(im, n2d, tr);
                n2d += dn;
                e = cmul(e, step);
            }
            off += len;
            g0 = fma((double)h.x, sr, g0);
            g1 = fma((double)h.y, sr, g1);
            g2 += tr;
        }
        double* o = (out_est ? R.grad_est : R.grad) + 3 * ((size_t)b * R.N + p);
        o[0] += f * g0;
        o[1] += f * g1;
        o[2] += f * g2;
    }
}

// Centroid term of Energy::VirialEstimator (energy_class.h:79-94):
// sum_p grad_nonkinetic(b,p) . Dr(r_p(b), r_p(0)), per slice.  from_sweep: the
// gradient is the sweep's full dS/dr, whose kinetic term is removed here.
__global__ __launch_bounds__(256) void k_centroid(const Rep* __restrict__ reps, int slot, int from_sweep) {
    const Rep& R = reps[blockIdx.y];
    const int b = blockIdx.x;
    if (b >= R.M) return;
    const int bn = (b + 1) % R.M, bp = (b + R.M - 1) % R.M;
    double t = 0.;
    for (int p = threadIdx.x; p < R.N; p += 256) {
        const double* g = (from_sweep ? R.grad : R.grad_est) + 3 * ((size_t)b * R.N + p);
        for (int d = 0; d < 3; ++d) {
            double gd = g[d];
            if (from_sweep) {
                const double x = pos_at(R, d, b, p);
                const double df = minimg(x - pos_at(R, d, bn, next_label(R, b, p)), R.L, R.iL);
                const double db = minimg(pos_at(R, d, bp, prev_label(R, b, p)) - x, R.L, R.iL);
                double kf = 2. * df * R.kin_i4lt, kb = 2. * db * R.kin_i4lt;
                if (R.kin_images > 0) {
                    int ia = spl_locate(R.kin[0], df), ib = spl_locate(R.kin[0], db);
                    kf += spl_der(R.kin[0], ia, 0, df - R.kin[0].x[ia]);
                    kb += spl_der(R.kin[0], ib, 0, db - R.kin[0].x[ib]);
                }
                gd -= kf - kb;
            }
            t += gd * minimg(pos_at(R, d, b, p) - pos_at(R, d, 0, p), R.L, R.iL);
        }
    }
    __shared__ double sh[4];
    t = block_sum<256>(t, sh);
    if (threadIdx.x == 0) R.scratch[slot * R.M + b] = t;
}

// Combines estimator partials (fixed order) into results res[0..1] of a replica.
//   what 0: kinetic dbeta -> res[0]; 1: pair dbeta or potential -> res[1];
//   what 2: virial kinetic (virial slot + centroid / 2 tau) -> res[0]
//   acc: add res[0..1] into the energy accumulators
// Scratch layout per replica: [slot][M] for slots 0..3, then long-range chunk
// partials, then the two results.

// One workgroup per replica; the partials are added lane by lane, then the lanes.
// pair_part: the pair sums' n_pair partials per replica (nullptr: per slice in the
// scratch, from the global-table kernel).
__global__ __launch_bounds__(256) void k_finalize(const Rep* __restrict__ reps, int what, int acc,
                                                  const double* __restrict__ pair_part, int n_pair) {
    const Rep& R = reps[blockIdx.x];
    const int M = R.M;
    const double* S = R.scratch;
    double* res = R.scratch + scratch_res(M, R.nk);
    __shared__ double sh[4];
    const int slot = what == 0 ? kSlotKin : what == 1 ? kSlotPair : kSlotCentroid;
    const bool parts = what == 1 && pair_part;
    const double* v = parts ? pair_part + (size_t)blockIdx.x * n_pair : S + slot * M;
    const int n = parts ? n_pair : M;
    double t = 0., l = 0.;
    for (int b = threadIdx.x; b < n; b += 256) t += v[b];
    if (what == 1 && R.use_long_range && R.pair_type != 0) {
        const double* lw = R.scratch + scratch_long(M);
        for (int c = threadIdx.x; c < (R.nk + kWave - 1) / kWave; c += 256) l += lw[c];
    }
    t = block_sum<256>(t, sh);
    l = block_sum<256>(l, sh);
    if (threadIdx.x) return;
    if (what == 0)
        res[0] = R.kin_dbeta_const + t;
    else if (what == 1)
        res[1] = t + l;
    else
        res[0] = S[kSlotVirial * M] + t / (2. * R.tau);
    if (acc) {
        R.e_acc[0] += res[0];
        R.e_acc[1] += res[1];
        R.n_measure[0] += 1;
    }
}

// ---------------------------------------------------------------------------
// K8: StructureFactor::Accumulate (structure_factor_class.h:15-32)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kSumBlock) void k_sk(const Rep* __restrict__ reps, double k_cut) {
    const Rep& R = reps[blockIdx.y];
    __shared__ double sh[kSumBlock];
    if ((int)blockIdx.x * kWave >= R.nk) return;
    const int k = blockIdx.x * kWave + (threadIdx.x & (kWave - 1));
    if (threadIdx.x == 0 && blockIdx.x == 0) R.n_measure[1] += 1;
    const double t = sum_rho2(R, k, sh);
    if (threadIdx.x < kWave && k < R.nk && R.kmag[k] < k_cut) R.sk_acc[k] += t;
}

// ---------------------------------------------------------------------------
// K9: PairCorrelation::Accumulate (pair_correlation_class.h:15-28) with
// LinearGrid::ReverseMap (observable_class.h:56-62); LDS histogram per slice.
// The workgroup's threads share the pairs (i, i + d mod N), i fastest; 1024 of
// them while the slices alone do not fill the chip (N = 256, M = 128, one replica
// 54 us with 256 threads, a particle each, 27 us so).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(1024) void k_gr(const Rep* __restrict__ reps, double r_min, double d_ir, int n_r,
                                            const double* __restrict__ r_max_per_rep) {
    const Rep& R = reps[blockIdx.y];
    const int b = blockIdx.x;
    if (b >= R.M) return;
    __shared__ unsigned int hist[kGrBins];
    const int nthr = blockDim.x;
    for (int i = threadIdx.x; i < n_r; i += nthr) hist[i] = 0;
    __syncthreads();
    const int N = R.N, half = N / 2;
    double dir = d_ir;
    if (r_max_per_rep) dir = 1. / ((r_max_per_rep[blockIdx.y] - r_min) / (n_r - 1.));
    const int groups = max(1, nthr / N);  // threads per particle
    for (int u = threadIdx.x; u < N * groups; u += nthr) {
        const int i = u % N, grp = u / N;
        double a[3];
        for (int d = 0; d < 3; ++d) a[d] = pos_at(R, d, b, i);
        for (int dd = 1 + grp; dd <= half; dd += groups) {
            if ((N % 2 == 0) && dd == half && i >= half) continue;
            const int j = i + dd < N ? i + dd : i + dd - N;
            const int lo = min(i, j), hi = max(i, j);
            double v[3];
            {
#pragma clang fp contract(off)
                for (int d = 0; d < 3; ++d) {
                    const double x = (lo == i) ? a[d] : pos_at(R, d, b, lo);
                    const double y = (hi == i) ? a[d] : pos_at(R, d, b, hi);
                    v[d] = minimg(x - y, R.L, R.iL);
                }
                const double rr = sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
                const double f = rint((rr - r_min) * dir - 0.5);
                const unsigned int bin = (unsigned int)(long long)f;
                if (f >= 0. && bin < (unsigned int)n_r) atomicAdd(&hist[bin], 1u);
            }
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n_r; i += nthr)
        if (hist[i]) atomicAdd(&R.gr_cnt[i], (unsigned long long)hist[i]);
    if (threadIdx.x == 0 && b == 0) R.n_measure[2] += 1;
}

}  // namespace spimc
