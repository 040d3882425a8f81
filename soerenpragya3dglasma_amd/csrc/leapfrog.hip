// The fused FP64 leapfrog kernel: one launch per Dynamics::SUNc::Update (SC/DYNAMICS/SUNcDynamics.cpp:353-378).
//
// A block of 256 threads advances one tile of 64 sites (step_tile4): wavefronts 0, 1, 2 own link
// direction 0, 1, 2 of every site (link_update in site.h), wavefront 3 forms J+-stat'(x) and
// J+-stat'(x+z) and hands them to wavefront 2 through LDS, which applies the J advection with its own
// half-step link.  Splitting a site over wavefronts keeps each wavefront's live state to a few matrices.
// The link operands on the tile's own rows (own links and their x neighbours, 18 of the 41 matrix loads per site) come
// from an LDS copy made once per block, with the few x neighbours outside the tile in halo slots; the kernel runs three
// wavefronts per SIMD.
//
// HBM traffic per site-update: read U (432 B) + E (192 B) + J (256 B), write the same: 1760 B, the
// compulsory minimum.  The neighbour link matrices are re-read through L2 / MALL, so the order in
// which the 8 XCDs (each with its own 4 MB L2) visit the lattice matters: workgroups are dealt to the
// XCDs round-robin, and with the column-band orders (TileMap mode 2 in site.h) each XCD walks its bands
// through z, so the y and z neighbours of a tile are read by the same XCD shortly before or after it (L2
// hits).  Measured at 256 x 256 x 1024 with the tuned 1 x 16 bands and three waves per SIMD, reads come to
// 1.40x the compulsory bytes (the y-halo rows of a band belong to another XCD, and the tiles in flight
// outgrow an XCD's 4 MB L2); writes are exactly compulsory.
//
// GLASMA_STEP_WAVES (2 or 3: register budget of 256 or 168 per lane, for lattices below 2^32 sites) and
// GLASMA_STEP_MAP / _BW / _BH select variants for measurement sweeps; the defaults are the fastest measured on MI355X.
#include <cstdlib>

#include "internal.h"

namespace glasma {

constexpr int kCus = 256;  // compute units of the chip

static int env_int(const char* name, int dflt) {
    const char* v = std::getenv(name);
    return v ? std::atoi(v) : dflt;
}


// The links of a tile's sites in LDS, slot 1 + lane.  A tile is any 64 consecutive sites: the end of one row, whole rows
// and the start of another (x periodic within each row); at most four x neighbours lie outside it (row_slots).
constexpr int kRow = kTile + 2;     // whole rows or one row segment (row_form 1): halo slots 0 and 65 at most
constexpr int kRowSeg = kTile + 4;  // any rows (row_form 2): halo slots 0, 65, 66, 67

// LDS of one block of the four-wavefront step (RL slots per row: kRow or kRowSeg).  The row length is a template
// parameter so that the whole-row form keeps the 66-slot layout, whose LDS offsets let it fit 168 registers
// without spills (68 slots cost two spilled doubles).
template <int RL>
struct StepShared {
    double row[3][18][RL];  // U_mu on the tile's row(s) and halo sites, plane pairs as in ldm (re, im of element k)
    double j[6][8][kTile];  // J+stat'(x), J-stat'(x), J+stat'(x+z), J-stat'(x+z), J+(x), J-(x)
    int ready;
};

template <int RL>
__device__ __forceinline__ void ld_row(const double (*r)[RL], int slot, M3& M) {
#pragma unroll
    for (int k = 0; k < 9; k++) {
        M.re[k] = r[2 * k][slot];
        M.im[k] = r[2 * k + 1][slot];
    }
}

// The two staples of link MU in transverse direction NU (link_update's loop body) with the operands on
// the tile's own rows -- U_nu(x), U_nu(x+x) for MU = x, U_mu(x+-x) and U_x(x-x) for NU = x -- read from
// the LDS copy instead of global memory (slots: own 1 + lane, x+1 at sp, x-1 at sm).  Same products in the
// same order as link_update.
// PRE: the forward staple's operands from global memory, U_nu(x+mu) (MU != 0) and U_mu(x+nu) (NU != 0), come in
// pre[0] and pre[1] (read before the row copy's barrier, first_staple_operands).
template <class I, int MU, int NU, int RL, bool PRE = false>
__device__ __forceinline__ void staples_row(const StepArgs& A, I s, int x, int y, int z, int lane, int sp, int sm,
                                            const double (*row)[18][RL], M3& Sig, const M3* pre = nullptr) {
    const Geom& g = A.g;
    const double cn = A.cE[NU];
    M3 P1, P2, T;
    // forward staple U_nu(x+mu) U_mu^dag(x+nu) U_nu^dag(x)
    if (MU == 0) ld_row(row[NU], sp, P1);
    else if (PRE) P1 = pre[0];
    else ldm<I>(A.U, kUPlanes, 18 * NU, nbr<I>(g, x, y, z, MU, 1, NU, 0), P1);
    if (NU == 0) ld_row(row[MU], sp, P2);
    else if (PRE) P2 = pre[1];
    else ldm<I>(A.U, kUPlanes, 18 * MU, nbr<I>(g, x, y, z, NU, 1, MU, 0), P2);
    mul_nd(P1, P2, T);
    ld_row(row[NU], lane + 1, P1);
    acc_mul_nd(cn, T, P1, Sig);
    // backward staple U_nu^dag(x+mu-nu) U_mu^dag(x-nu) U_nu(x-nu)
    ldm<I>(A.U, kUPlanes, 18 * NU, nbr<I>(g, x, y, z, MU, 1, NU, -1), P1);
    if (NU == 0) {
        ld_row(row[MU], sm, P2);
    } else {
        ldm<I>(A.U, kUPlanes, 18 * MU, nbr<I>(g, x, y, z, NU, -1, MU, 0), P2);
    }
    mul_dd(P1, P2, T);
    if (NU == 0) ld_row(row[0], sm, P1);
    else ldm<I>(A.U, kUPlanes, 18 * NU, nbr<I>(g, x, y, z, NU, -1, MU, 0), P1);
    acc_mul_nn(cn, T, P1, Sig);
}

// wait for the J wavefront's hand-over (set unconditionally once its LDS stores are complete).  The wait is
// capped so that no wave can spin forever; false if the cap was reached, and the caller then writes NaN
// currents (glasma_bulk reports non-finite sums as GLASMA_ERR_NUMERIC) instead of silently using stale values.
template <class SH>
__device__ __forceinline__ bool wait_ready(SH& sh) {
    bool ok = false;
    for (int spin = 0; spin < (1 << 24); spin++) {
        if (__hip_atomic_load(&sh.ready, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) {
            ok = true;
            break;
        }
        __builtin_amdgcn_s_sleep(2);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    return ok;
}

// the global operands of link MU's first forward staple (NU = MU + 1), read before the row copy's barrier so that
// their latency overlaps the barrier's wait: pre[0] = U_nu(x+mu) when MU != 0, pre[1] = U_mu(x+nu) when NU != 0
template <class I, int MU>
__device__ __forceinline__ void first_staple_operands(const StepArgs& A, int x, int y, int z, M3* pre) {
    constexpr int NU = (MU + 1) % 3;
    if (MU != 0) ldm<I>(A.U, kUPlanes, 18 * NU, nbr<I>(A.g, x, y, z, MU, 1, NU, 0), pre[0]);
    if (NU != 0) ldm<I>(A.U, kUPlanes, 18 * MU, nbr<I>(A.g, x, y, z, NU, 1, MU, 0), pre[1]);
}

// link_update with the row operands from LDS (PRE: the first staple's global operands in pre, first_staple_operands)
template <class I, int MU, int RL, bool PRE = false>
__device__ __forceinline__ void link_update_row(const StepArgs& A, I s, int x, int y, int z, int lane, int sp,
                                                int sm, const double (*row)[18][RL], M3& Uh,
                                                const M3* pre = nullptr) {
    M3 Sig;
#pragma unroll
    for (int k = 0; k < 9; k++) { Sig.re[k] = 0.0; Sig.im[k] = 0.0; }
    // scheduling barriers keep the compiler from hoisting the next staple pair's loads into this one:
    // that fits the form into 168 registers without spills (three waves per SIMD, 31.3 -> 30.1 ms at
    // 256 x 256 x 1024), the waves hiding the latency instead
    staples_row<I, MU, (MU + 1) % 3, RL, PRE>(A, s, x, y, z, lane, sp, sm, row, Sig, pre);
    __builtin_amdgcn_sched_barrier(0);
    staples_row<I, MU, (MU + 2) % 3, RL>(A, s, x, y, z, lane, sp, sm, row, Sig);
    __builtin_amdgcn_sched_barrier(0);
    M3 Uo;
    ld_row(row[MU], lane + 1, Uo);
    link_finish<I, MU>(A, s, Uo, Sig, Uh);
}

// Four-wavefront step of the tile starting at site `first`.  Waves 0-2 update the link directions; wave 3
// forms J+-stat'(x) and J+-stat'(x+z) (the cheaper work) and hands them, with the J+-(x) it read, to
// wave 2 through LDS.  Wave 2 applies the J advection with its own U_h,z as soon as its link is done, so
// the block ends with its slowest link wavefront instead of a serial advection after a block barrier.
// The hand-over is a workgroup-scope flag: wave 3 sets it unconditionally once its stores to LDS are
// complete, so wave 2's wait always ends; the wait is capped all the same.
//
// Waves 0-2 first copy U_w of the tile and of its halo sites into LDS, and the 18 of 41 link operands per site that lie
// on those rows are read from there.  This takes about a third of the vector-memory accesses off the L1, whose pipeline is
// what the kernel waits on.  Reading all 41 from global memory, at two waves per SIMD, took 583 us at 81 x 75 x 125 (357
// now).
template <class I>
__device__ __forceinline__ void step_tile4(const StepArgs& A, long first, StepShared<kRow>& sh) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const long sl = first + lane;
    const bool valid = sl < A.g.S;
    const I s = (I)(valid ? sl : 0);
    int x, y, z;
    site_coords<I>(A.g, s, x, y, z);
    // LDS slots of x+1 and x-1: the next / previous lane, or halo slots; in a tile of several short rows, the
    // lane of the periodic neighbour in the same row
    const bool one_row = A.g.nx % kTile == 0;
    const int sp = one_row ? lane + 2 : lane + 1 + (x + 1 == A.g.nx ? 1 - A.g.nx : 1);
    const int sm = one_row ? lane : lane + 1 + (x == 0 ? A.g.nx - 1 : -1);
    const int nhalo = one_row ? 2 : 0;
    if (wave < 3) {
        // lanes past the end of the lattice (last tile only) copy site 0; no valid lane reads their slots
        M3 M;
        ldm<I>(A.U, kUPlanes, 18 * wave, s, M);
#pragma unroll
        for (int k = 0; k < 9; k++) {
            sh.row[wave][2 * k][lane + 1] = M.re[k];
            sh.row[wave][2 * k + 1][lane + 1] = M.im[k];
        }
        if (lane < nhalo) {
            const int xt = x - lane;  // the tile's first x
            const long hs = (long)s - x + (lane == 0 ? xwrap(xt - 1, A.g.nx) : xwrap(xt + kTile, A.g.nx));
            ldm<I>(A.U, kUPlanes, 18 * wave, (I)hs, M);
            const int slot = lane == 0 ? 0 : kTile + lane;
#pragma unroll
            for (int k = 0; k < 9; k++) {
                sh.row[wave][2 * k][slot] = M.re[k];
                sh.row[wave][2 * k + 1][slot] = M.im[k];
            }
        }
    }
    if (threadIdx.x == 0) sh.ready = 0;
    __syncthreads();
    if (wave == 0) {
        M3 Uh;
        if (valid) link_update_row<I, 0, kRow>(A, s, x, y, z, lane, sp, sm, sh.row, Uh);
    } else if (wave == 1) {
        M3 Uh;
        if (valid) link_update_row<I, 1, kRow>(A, s, x, y, z, lane, sp, sm, sh.row, Uh);
    } else if (wave == 3) {
        if (valid) {
            double jps[8], jms[8], jp[8], jm[8];
            const int zm = zdn(A.g, z);
            jstat_new_keep<I>(A, s, (I)(sl + A.g.P * (long)(zm - z)), jps, jms, jp, jm);
            stv<I>(A.Jn, kJPlanes, JPS * 8, s, jps);
            stv<I>(A.Jn, kJPlanes, JMS * 8, s, jms);
#pragma unroll
            for (int a = 0; a < 8; a++) {
                sh.j[0][a][lane] = jps[a];
                sh.j[1][a][lane] = jms[a];
                sh.j[4][a][lane] = jp[a];
                sh.j[5][a][lane] = jm[a];
            }
            // U_z(x) of J+-stat'(x+z) from the row copy; on the open top layer J+-stat'(x+z) is
            // J+-stat'(x) itself (jstat_new_up), already in jps, jms
            const int zp = zup(A.g, z);
            if (zp != z) {
                M3 Uz;
                ld_row(sh.row[2], lane + 1, Uz);
                jstat_core<I>(A, (I)(sl + A.g.P * (long)(zp - z)), s, Uz, jps, jms);
            }
#pragma unroll
            for (int a = 0; a < 8; a++) {
                sh.j[2][a][lane] = jps[a];
                sh.j[3][a][lane] = jms[a];
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        if (lane == 0) __hip_atomic_store(&sh.ready, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    } else {
        M3 Uh;
        if (valid) link_update_row<I, 2, kRow>(A, s, x, y, z, lane, sp, sm, sh.row, Uh);
        const bool handed_over = wait_ready(sh);
        if (valid) {
            double jps[8], jms[8], jpsU[8], jmsU[8], jp[8], jm[8];
#pragma unroll
            for (int a = 0; a < 8; a++) {
                jps[a] = sh.j[0][a][lane];
                jms[a] = sh.j[1][a][lane];
                jpsU[a] = sh.j[2][a][lane];
                jmsU[a] = sh.j[3][a][lane];
                jp[a] = sh.j[4][a][lane];
                jm[a] = sh.j[5][a][lane];
            }
            if (!handed_over) jp[0] = jm[0] = __builtin_nan("");
            j_advect_with<I>(A, s, Uh, jps, jms, jpsU, jmsU, jp, jm);
        }
    }
}

// One link wavefront of step_tile4_seg (link direction MU): the row copy of U_MU with the first staple's global
// operands read in the same burst, the block barrier, the link update and, for MU = 2, the J advection after the J
// wavefront's hand-over.  Each wavefront's branch holds its own barrier (the branches are uniform: every wavefront
// runs exactly one), so that the operands read before it stay live in that branch only.
template <class I, int MU>
__device__ __forceinline__ void link_wave(const StepArgs& A, long first, I s, bool valid, int x, int y, int z, int lane,
                                          int x0, StepShared<kRowSeg>& sh) {
    const RowSlots rs = row_slots(A.g, lane, x);
    M3 pre[2];
    // lanes past the end of the lattice (last tile only) copy site 0; no valid lane reads their slots
    M3 M;
    ldm<I>(A.U, kUPlanes, 18 * MU, s, M);
    first_staple_operands<I, MU>(A, x, y, z, pre);
#pragma unroll
    for (int k = 0; k < 9; k++) {
        sh.row[MU][2 * k][lane + 1] = M.re[k];
        sh.row[MU][2 * k + 1][lane + 1] = M.im[k];
    }
    if (lane < 4) {
        ldm<I>(A.U, kUPlanes, 18 * MU, (I)halo_site(A.g, first, x0, lane), M);
        const int slot = lane == 0 ? 0 : kTile + lane;
#pragma unroll
        for (int k = 0; k < 9; k++) {
            sh.row[MU][2 * k][slot] = M.re[k];
            sh.row[MU][2 * k + 1][slot] = M.im[k];
        }
    }
    if (MU == 0 && lane == 0) sh.ready = 0;
    __syncthreads();
    M3 Uh;
    if (valid) link_update_row<I, MU, kRowSeg, true>(A, s, x, y, z, lane, rs.sp, rs.sm, sh.row, Uh, pre);
    if (MU == 2) {
        const bool handed_over = wait_ready(sh);
        if (valid) {
            double jps[8], jms[8], jpsU[8], jmsU[8], jp[8], jm[8];
#pragma unroll
            for (int a = 0; a < 8; a++) {
                jps[a] = sh.j[0][a][lane];
                jms[a] = sh.j[1][a][lane];
                jpsU[a] = sh.j[2][a][lane];
                jmsU[a] = sh.j[3][a][lane];
                jp[a] = sh.j[4][a][lane];
                jm[a] = sh.j[5][a][lane];
            }
            if (!handed_over) jp[0] = jm[0] = __builtin_nan("");
            j_advect_with<I>(A, s, Uh, jps, jms, jpsU, jmsU, jp, jm);
        }
    }
}

// step_tile4 for tiles that start and end anywhere in a row (row_form 2), with each link wavefront's branch holding its
// own barrier and the first staple's global operands read before it (link_wave): no spilled registers where the shared
// form above spills 4 with the longer rows, 1.69-1.72 against 1.71-1.75 ms at 96 x 96 x 384.  For whole rows it was slower
// (29.96 against 29.62 ms at 256 x 256 x 1024: 4 spilled registers).
template <class I>
__device__ __forceinline__ void step_tile4_seg(const StepArgs& A, long first, StepShared<kRowSeg>& sh) {
    // the wave index through readfirstlane: uniform to the compiler, so the per-wave branches are scalar branches
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const long sl = first + lane;
    const bool valid = sl < A.g.S;
    const I s = (I)(valid ? sl : 0);
    int x, y, z;
    site_coords<I>(A.g, s, x, y, z);
    if (wave == 3) {
        __syncthreads();
        if (valid) {
            double jps[8], jms[8], jp[8], jm[8];
            const int zm = zdn(A.g, z);
            jstat_new_keep<I>(A, s, (I)(sl + A.g.P * (long)(zm - z)), jps, jms, jp, jm);
            stv<I>(A.Jn, kJPlanes, JPS * 8, s, jps);
            stv<I>(A.Jn, kJPlanes, JMS * 8, s, jms);
#pragma unroll
            for (int a = 0; a < 8; a++) {
                sh.j[0][a][lane] = jps[a];
                sh.j[1][a][lane] = jms[a];
                sh.j[4][a][lane] = jp[a];
                sh.j[5][a][lane] = jm[a];
            }
            // U_z(x) of J+-stat'(x+z) from the row copy; on the open top layer J+-stat'(x+z) is
            // J+-stat'(x) itself (jstat_new_up), already in jps, jms
            const int zp = zup(A.g, z);
            if (zp != z) {
                M3 Uz;
                ld_row(sh.row[2], lane + 1, Uz);
                jstat_core<I>(A, (I)(sl + A.g.P * (long)(zp - z)), s, Uz, jps, jms);
            }
#pragma unroll
            for (int a = 0; a < 8; a++) {
                sh.j[2][a][lane] = jps[a];
                sh.j[3][a][lane] = jms[a];
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        if (lane == 0) __hip_atomic_store(&sh.ready, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        return;
    }
    const int x0 = __builtin_amdgcn_readfirstlane(x);  // lane 0's x: every lane of the wave is active here
    if (wave == 0) link_wave<I, 0>(A, first, s, valid, x, y, z, lane, x0, sh);
    else if (wave == 1) link_wave<I, 1>(A, first, s, valid, x, y, z, lane, x0, sh);
    else link_wave<I, 2>(A, first, s, valid, x, y, z, lane, x0, sh);
}

template <class I, int W, bool SEG>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(W, W))) k_step4(StepArgs A, TileMap tm) {
    __shared__ StepShared<SEG ? kRowSeg : kRow> sh;
    if constexpr (SEG) step_tile4_seg<I>(A, tile_site(A.g, tm, blockIdx.x), sh);
    else step_tile4<I>(A, tile_site(A.g, tm, blockIdx.x), sh);
}

// Ensemble step: one launch per form advances every event of a batch.  Block b works on the tile starting
// at site block_site[b] of event e = block_event[b] (each event's blocks in the order tile_site gives it
// alone); the event's arguments come from a device table (uniform per block, so they are read with scalar
// loads).  The per-site arithmetic is that of k_step4.  The blocks come in two groups by row_form.
template <bool SEG>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3)))
k_step_batch(const StepArgs* __restrict__ table, const int* __restrict__ block_event,
             const unsigned* __restrict__ block_site) {
    __shared__ StepShared<SEG ? kRowSeg : kRow> sh;
    const StepArgs A = table[block_event[blockIdx.x]];
    if constexpr (SEG) step_tile4_seg<unsigned int>(A, (long)block_site[blockIdx.x], sh);
    else step_tile4<unsigned int>(A, (long)block_site[blockIdx.x], sh);
}

int launch_step_batch(hipStream_t st, const StepArgs* table, const int* block_event, const unsigned* block_site,
                      long nrow, long nseg) {
    if (nrow < 0 || nseg < 0 || nrow + nseg <= 0 || nrow > 0x7fffffffL || nseg > 0x7fffffffL) return GLASMA_ERR_ARG;
    if (nrow > 0)
        hipLaunchKernelGGL(k_step_batch<false>, dim3((unsigned)nrow), dim3(256), 0, st, table, block_event, block_site);
    if (nseg > 0)
        hipLaunchKernelGGL(k_step_batch<true>, dim3((unsigned)nseg), dim3(256), 0, st, table, block_event + nrow,
                           block_site + nrow);
    return hipGetLastError() == hipSuccess ? 0 : GLASMA_ERR_HIP;
}

// the arguments of one step of a context (current buffers, optional UOld)
StepArgs step_args(const glasma_ctx* ctx, int cur, bool write_old) {
    StepArgs A;
    A.U = ctx->U[cur];
    A.Un = ctx->U[cur ^ 1];
    A.E = ctx->E;
    A.J = ctx->J[cur];
    A.Jn = ctx->J[cur ^ 1];
    A.UOld = write_old ? ctx->UOld : nullptr;
    A.g = ctx->g;
    fill_step_coefficients(A, ctx->p.a, ctx->p.dt);
    return A;
}

template <class I, int W>
static void launch(const TileMap& tm, const StepArgs& A, hipStream_t st) {
    dim3 grid((unsigned)(pad_sites(A.g.S) / kTile));
    if (row_form(A.g) == 2) hipLaunchKernelGGL((k_step4<I, W, true>), grid, dim3(256), 0, st, A, tm);
    else hipLaunchKernelGGL((k_step4<I, W, false>), grid, dim3(256), 0, st, A, tm);
}

// Waves per SIMD of the step, that is workgroups (one tile each) per CU: three with 168 registers or two with 183.
// Three keep more loads in flight (64 x 64 x 64 0.120 ms against 0.124, 256 x 256 x 1024 30.1 against 31.8).  Two are
// the better where three have nothing to add: up to two tiles per CU, all resident either way, gain by the registers
// (256 tiles 11.3 us against 12.5, 512 tiles 18.8 against 19.0), and four per CU run as 2 + 2
// instead of 3 + 1 (960 tiles 32.6 us against 34.5, 1024 tiles 33.5 against 36.3).  Three per CU are a single round
// (768 tiles 26.7 us against 29.5), and from five on the tail matters less (1152 tiles 39.4 against 39.6, 1536 tiles
// 48.5 against 50.0).
static int step_waves(const Geom& g) {
    static const int env = env_int("GLASMA_STEP_WAVES", 0);
    if (env == 2 || env == 3) return env;
    const long per_cu = (pad_sites(g.S) / kTile + kCus - 1) / kCus;
    return per_cu <= 2 || per_cu == 4 ? 2 : 3;
}

// tile order for a geometry: the requested mode when the lattice fits it, else the next simpler one
TileMap tile_map(const Geom& g, int mode, int bw, int bh) {
    TileMap m = {0, 0, 0, 0, 0, 0};
    if (mode == 2 && g.nx % kTile == 0 && bw > 0 && bh > 0) {
        const int tpr = g.nx / kTile;
        if (tpr % bw == 0 && g.ny % bh == 0) {
            const long bands = (long)(tpr / bw) * (g.ny / bh);
            if (bands % kXcds == 0) {
                m.mode = 2;
                m.bw = bw;
                m.bh = bh;
                m.nbx = tpr / bw;
                m.tpbp = bw * bh;
                return m;
            }
        }
    }
    if (mode == 3) {
        const long nt = pad_sites(g.S) / kTile;
        if (nt / kXcds <= 0x7fffffffL) {
            m.mode = 3;
            m.bpb = (int)(nt / kXcds);
            m.nbx = (int)(nt % kXcds);
            return m;
        }
    }
    if (mode >= 1) {
        const long bpb = (g.P + kXcds * kTile / 2) / (kXcds * kTile);
        if (bpb > 0) {
            m.mode = 1;
            m.bpb = (int)bpb;
        }
    }
    return m;
}

TileMap default_tile_map(const Geom& g) {
    // GLASMA_STEP_MAP = mode (0, 1, 2) and, for mode 2, the band width in tiles and height in rows
    // (mode 2 with 4 x 4 bands measured fastest at 256 x 256 x 1024: 33.9 ms against 36.6 ms for mode 1)
    static const int map_mode = env_int("GLASMA_STEP_MAP", 2);
    static const int map_bw = env_int("GLASMA_STEP_BW", 4);
    static const int map_bh = env_int("GLASMA_STEP_BH", 4);
    const TileMap m = tile_map(g, map_mode, map_bw, map_bh);
    // Planes that do not split into column bands: an eighth of every plane per XCD where the plane is about a multiple of
    // 8 tiles or has many (81 x 75 x 125: 0.357 ms, z slabs 0.387, linear 0.459; 225 x 250 x 300: 8.4, 9.4 and 11.3;
    // 40 x 72 x 100: 0.137, 0.142, 0.180), z slabs for the small ones, whose bands would be a few tiles that drift against
    // the planes (48 x 48 x 128: 0.146 ms, bands 0.148, linear 0.176; 36 x 20 x 64: 0.027, 0.037, 0.036).
    if (map_mode == 2 && m.mode < 2 && g.P % (kXcds * kTile) != 0 && m.bpb < 6) return tile_map(g, 3, 0, 0);
    return m;
}

TileMap ctx_tile_map(const glasma_ctx* ctx) { return ctx->tm_tuned ? ctx->tm : default_tile_map(ctx->g); }

// one step with explicit buffers and tile order (the context supplies the stream)
int launch_step_map(glasma_ctx* ctx, const StepArgs& A, const TileMap& tm, hipStream_t st) {
    if (!st) st = ctx->stream;
    if (A.g.S >= (1L << 32)) launch<unsigned long, 3>(tm, A, st);
    else if (step_waves(A.g) == 2) launch<unsigned int, 2>(tm, A, st);
    else launch<unsigned int, 3>(tm, A, st);
    return 0;
}

// one step with explicit buffers (the context supplies geometry, stream and tile order)
int launch_step_args(glasma_ctx* ctx, const StepArgs& A, hipStream_t st) {
    return launch_step_map(ctx, A, ctx_tile_map(ctx), st);
}

int launch_step(glasma_ctx* ctx, bool write_old) {
    const int rc = launch_step_args(ctx, step_args(ctx, ctx->cur, write_old));
    ctx->cur ^= 1;
    return rc;
}

}  // namespace glasma
