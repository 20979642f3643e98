// The two kernels of an integrator step inside a segment of steps.
//
// k_advance closes one step and opens the next: the forces summed per particle, the closing
// half-kick, the next step's position update and its largest displacement.  One pass over the
// state instead of two (k_finish and k_baoab_a / k_gjf_a), with no force array written in between:
// 184 instead of 320 bytes a particle for a Lennard-Jones fluid.
//
// k_forces evaluates every interaction of a small system in one launch, its blocks split into one
// run per interaction, and keeps the neighbour lists: every block takes the step's skin decision
// for itself from the same two words, and on a rebuild each row group first finds its own row
// among all participants.  A step of a small system is a chain of dependent launches, each about
// 1 us of dispatch plus two or three levels of loads that miss to memory (0.5 to 1 us each), so
// what counts is their number: two here, where separate kernels for the skin check, the cell sort,
// the list build, the local terms, the pairs, each 3SPN2 interaction, the force sum and the
// position update make 6 (a fluid) to 17 (a DNA duplex).  A rebuild by brute force is np^2 distance
// tests without any ordering between blocks: a launch with one takes 71 us at 4096 participants (6.9 without),
// where the cell sort and the build from it took 180.  Measured per FP64 step, before and after: a fluid of 512
// particles 17.0 -> 9.4 us, of 4096 18.9 -> 11.1, a chain of 1000 beads 27.5 -> 11.4, a 200-bp duplex
// 64 -> 18; mixed chain of 3001 beads 29 -> 11.6.
#pragma once
#include "force_kernels.hpp"
#include "nlist_kernels.hpp"

namespace mjg
{
// the lists that k_forces keeps: their margins are settled by the next k_advance.  Four are what the largest
// of the framework's own force fields has (3SPN2: excluded volume, Debye-Hueckel, base pairing, cross
// stacking; four local interactions beside them); the table of them travels in the kernel's arguments.  A
// system with more takes the separate launches (a chain of 1000 beads with five lists 29.7 us a step, with
// its two 11.4).
constexpr int kMaxSelfLists = 4;
struct SelfLists
{
    ListCtl* ctl[kMaxSelfLists];
    double abs_margin[kMaxSelfLists];
    int never[kMaxSelfLists];          // Naive: built once
    int n;
};

// The skin decision of step k of the segment (ForceField::reduce_margin, ForceField.hpp:75-92): the
// margin left after the step's largest displacement, below zero when the list must be rebuilt.
__device__ __forceinline__ double margin_after(const ListCtl* ctl, const StepCtl* sctl, uint32_t k)
{
    // both slots are read with the step count, not after it
    const unsigned long long d0 = sctl->maxdisp2[0], d1 = sctl->maxdisp2[1];
    return ctl->margin - 2 * sqrt(__longlong_as_double((long long)(((sctl->step + k) & 1) ? d1 : d0)));
}

struct AdvanceArgs
{
    GatherArgs g;
    SelfLists lists;
    double4* pos;
    double4* vel;
    double4* force;
    const double* rmass;
    const double* c1;
    const double* c2;
    const double* c3;
    const double4* noise;      // the step's draws where k_forces made them (null: drawn here)
    StepCtl* ctl;
    const ListCtl* lctl;       // every list's control words
    ListCtl* h_lctl;           // their pinned copy, and that of the step control, for the host
    StepCtl* h_ctl;
    double dt, halfdt;
    uint64_t seed;
    Box box;
    uint32_t n;
    uint32_t k;                // steps since the segment began (ctl->step does not move inside it)
    int nlists;
};

// STAGED: the system has local terms.  A block of 256 threads then serves 64 particles and brings their
// term-force slots, one contiguous run, to LDS in a single round of loads (a thread that walked its
// own dozen slots waited for three or four rounds: k_advance of a 1000-bead chain 6.5 us, of a
// fluid of that size 3.9).
// FIRST: opens step 0 from the stored force.  LAST: closes step k - 1 only, stores the force,
// advances the step count by k and reports to the host.
constexpr uint32_t kStagedParticles = 64;
constexpr uint32_t kStagedRounds = 12;       // words a thread brings; longer runs are read where they lie
template<bool GJF, bool FIRST, bool LAST, bool STAGED>
__global__ void __launch_bounds__(256)
k_advance(AdvanceArgs a)
{
    const uint32_t per = STAGED ? kStagedParticles : blockDim.x;
    const uint32_t i = (threadIdx.x < per) ? blockIdx.x * per + threadIdx.x : a.n;
    const uint64_t step0 = a.ctl->step;
    const double* slots = nullptr;
    uint32_t slot0 = 0;
    if constexpr(STAGED && !FIRST)
    {
        __shared__ double staged[kStagedRounds * 256];
        const uint32_t i0 = blockIdx.x * per, i1 = (i0 + per < a.n) ? i0 + per : a.n;
        const uint32_t b = a.g.gstart[i0], words = 3 * (a.g.gstart[i1] - b);
        if(words <= kStagedRounds * 256)
        {
            double v[kStagedRounds];
#pragma unroll
            for(uint32_t m = 0; m < kStagedRounds; ++m)
            {
                const uint32_t q = m * 256 + threadIdx.x;
                v[m] = (q < words) ? a.g.tf[3 * (size_t)b + q] : 0.0;
            }
#pragma unroll
            for(uint32_t m = 0; m < kStagedRounds; ++m) {staged[m * 256 + threadIdx.x] = v[m];}
            slots = staged;
            slot0 = b;
        }
        __syncthreads();
    }
    if constexpr(!FIRST)
    {
        // the previous step's skin decision, taken by every block of its k_forces, is made final
        if(blockIdx.x == 0 && threadIdx.x < (uint32_t)kWave)
        {
            bool spent = false;
            if(threadIdx.x < (uint32_t)a.lists.n && !a.lists.never[threadIdx.x])
            {
                ListCtl* c = a.lists.ctl[threadIdx.x];
                const double m = margin_after(c, a.ctl, a.k - 1);
                spent = m < 0;
                c->margin = spent ? a.lists.abs_margin[threadIdx.x] : m;
            }
            const uint32_t built = (uint32_t)__popcll(__ballot(spent));
            if(threadIdx.x == 0 && built > 0) {a.ctl->rebuilds += built;}
        }
    }
    double d2 = 0.0;
    if(i < a.n)
    {
        double fx, fy, fz;
        const double rm = a.rmass[i];
        double4 v = a.vel[i];
        double4 p;
        if constexpr(!LAST) {p = a.pos[i];}
        double Rx = 0, Ry = 0, Rz = 0;
        double b = 0, c = 0, cc = 0;
        if constexpr(!LAST)
        {
            b = a.c1[i]; c = a.c2[i];
            if constexpr(GJF) {cc = a.c3[i];}
            if(!FIRST && a.noise) {const double4 r = a.noise[i]; Rx = r.x; Ry = r.y; Rz = r.z;}
            else {noise3(a.seed, step0 + a.k, i, Rx, Ry, Rz);}
        }
        if constexpr(FIRST) {const double4 f = a.force[i]; fx = f.x; fy = f.y; fz = f.z;}
        else
        {
            gather_force<true>(a.g, a.n, i, fx, fy, fz, slots, slot0);
            // closing half-kick (BAOABLangevinIntegrator.hpp:222-229, GJFNVTLangevinIntegrator.hpp:222-229)
            const double hrm = a.halfdt * rm;
            v.x += hrm * fx; v.y += hrm * fy; v.z += hrm * fz;
        }
        if constexpr(LAST) {a.force[i] = make_double4(fx, fy, fz, 0.0);}
        else
        {
            double dpx, dpy, dpz;
            if constexpr(!GJF)
            {
                // BAOABLangevinIntegrator.hpp:176-200
                const double hrm = a.halfdt * rm;
                v.x += hrm * fx; v.y += hrm * fy; v.z += hrm * fz;
                dpx = a.halfdt * v.x; dpy = a.halfdt * v.y; dpz = a.halfdt * v.z;
                v.x *= b; v.y *= b; v.z *= b;
                v.x += c * Rx; v.y += c * Ry; v.z += c * Rz;
                dpx += a.halfdt * v.x; dpy += a.halfdt * v.y; dpz += a.halfdt * v.z;
            }
            else
            {
                // GJFNVTLangevinIntegrator.hpp:172-197
                const double r2m = 0.5 * rm;
                const double bx = Rx * c, by = Ry * c, bz = Rz * c;
                const double bdt = b * a.dt;
                dpx = bdt * (v.x + r2m * (a.dt * fx + bx));
                dpy = bdt * (v.y + r2m * (a.dt * fy + by));
                dpz = bdt * (v.z + r2m * (a.dt * fz + bz));
                const double dtr2m = a.dt * r2m, brm = b * rm;
                v.x = cc * (v.x + dtr2m * fx) + brm * bx;
                v.y = cc * (v.y + dtr2m * fy) + brm * by;
                v.z = cc * (v.z + dtr2m * fz) + brm * bz;
            }
            double x = p.x + dpx, y = p.y + dpy, z = p.z + dpz;
            adjust_position(a.box, x, y, z);
            p.x = x; p.y = y; p.z = z;
            a.pos[i] = p;
            d2 = length_sq(dpx, dpy, dpz);
            if(!isfinite(x) || !isfinite(y) || !isfinite(z)) {a.ctl->nonfinite = 1;}
        }
        a.vel[i] = v;
    }
    if constexpr(!LAST) {block_max_to(d2, a.ctl, step0 + a.k);}
    else if(blockIdx.x == 0)
    {
        // every other kernel of the segment has ended: the control words are final after this
        __syncthreads();
        if(threadIdx.x == 0)
        {
            StepCtl c = *a.ctl;
            c.step += a.k;
            a.ctl->step = c.step;
            *a.h_ctl = c;
        }
        if(threadIdx.x < (uint32_t)a.nlists) {a.h_lctl[threadIdx.x] = a.lctl[threadIdx.x];}
    }
}

// The segment's start, from which a segment whose list overflowed runs again.
struct BackupArgs
{
    const double4* src[3];
    double4* dst[3];
    const StepCtl* ctl;
    StepCtl* bak_ctl;
    const ListCtl* lctl;
    ListCtl* bak_lctl;
    uint32_t n;
    int nlists;
};
__global__ void __launch_bounds__(256)
k_backup(BackupArgs a)
{
    for(uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < a.n; i += gridDim.x * blockDim.x)
    {
#pragma unroll
        for(int k = 0; k < 3; ++k) {a.dst[k][i] = a.src[k][i];}
    }
    if(blockIdx.x == 0)
    {
        if(threadIdx.x == 0) {*a.bak_ctl = *a.ctl;}
        if(threadIdx.x < (uint32_t)a.nlists) {a.bak_lctl[threadIdx.x] = a.lctl[threadIdx.x];}
    }
}

// ------------------------------------------------------------------------------------
// all forces of a small system
// ------------------------------------------------------------------------------------
constexpr int kMaxSmallLocals = 8;

// one global interaction: its rows and what keeps its list
struct RowSeg
{
    uint32_t block_begin;
    int never;
    PairSeg p;                 // LJ / EV / DH / 3SPN2 excluded volume
    unsigned long long* acc;   // 3SPN2 multibody: fixed-point sums
    ListCtl* ctl;
    uint32_t* nl;
    uint32_t* nn;
    const uint32_t* part;
    const uint32_t* pslot;
    const uint32_t* mol;
    const uint32_t* ex_start;
    const uint32_t* ex;
    ListRule rule;
};
struct SmallForces
{
    RowSeg row[kMaxSelfLists];
    LocalSeg local[kMaxSmallLocals];
    int nrow, nlocal;
    uint32_t local_begin, noise_begin;   // first blocks of the local terms and of the noise
    const uint32_t* lidx;
    const double* lpar;
    const uint32_t* ldst;
    double* tf;
    double4* noise;
    uint64_t seed;
    StepCtl* sctl;
    uint32_t n, k;
};
constexpr uint32_t kScanTile = 256;   // candidates staged at a time by a rebuild
constexpr uint32_t kScanEx = 4096;    // exclusions staged by a block, shared out over its rows

// The rows of one block found among all participants, in participant order; the pairs are k_verlet's
// (the same distance test, pair_allowed's rules).  A candidate near enough used to read the participant,
// base and exclusion tables in a dependent chain of about 3 us, on nearly every round of a chain's or
// a duplex's rows (251 us for a force launch of the 200-bp duplex with a rebuild, 92 now, 9.5 without one);
// here a tile's tables are staged with its positions, loaded while the tile before is tested, and a row
// keeps its own exclusions in LDS (an exclusion holds both ways, so the owner's list decides).  Every thread
// of the block calls it; `valid`: the thread's row exists.
__device__ __forceinline__ void self_build(const RowSeg& s, const Box& box, const double4* __restrict__ pos, uint32_t t,
                                           uint32_t l, bool valid)
{
    __shared__ double cx[kScanTile], cy[kScanTile], cz[kScanTile];
    __shared__ uint32_t cj[kScanTile], cslot[kScanTile], cmol[kScanTile];
    __shared__ int cbase[kScanTile];
    __shared__ uint32_t ex[kScanEx];
    const uint32_t tid = threadIdx.x, lane = tid % kWave;
    const uint32_t np = s.p.np, tpp = s.p.tpp, cap = s.p.cap;
    const ListRule& rule = s.rule;
    const uint32_t i = valid ? s.p.spart[t] : 0u;
    const double4 ri = pos[i];
    const uint32_t islot = s.pslot[i], imol = rule.ignore_mol ? s.mol[i] : 0u;
    const int ibase = rule.base_rule ? (int)rule.base_par[(size_t)i * rule.base_stride] : 0;
    const uint64_t gmask = group_mask_of(tpp, lane), below = gmask & ((1ull << lane) - 1ull);
    // the row's exclusions: those within 32 indices of i as bits, the first `excap` of the others in
    // LDS, any more read where they lie
    const uint32_t exb = s.ex_start[i], exn = rule.simple ? 0u : s.ex_start[i + 1] - exb;
    const uint32_t excap = kScanEx / (blockDim.x / tpp), exo = (tid / tpp) * excap;
    unsigned long long near = 0;
    uint32_t nfar = 0, over = exn;
    for(uint32_t k0 = 0; k0 < exn; k0 += tpp)
    {
        const uint32_t k = k0 + l;
        const uint32_t e = (k < exn) ? s.ex[exb + k] : i;
        const uint32_t d = e - i + 32u;
        const bool far = d >= 64u;
        if(!far) {near |= 1ull << d;}
        const uint64_t f = __ballot(far) & gmask;
        const uint32_t at = nfar + (uint32_t)__popcll(f & below);
        if(far && at < excap) {ex[exo + at] = e;}
        nfar += (uint32_t)__popcll(f);
        if(nfar > excap && over == exn) {over = k0;}       // words from here on may not be staged
    }
    for(uint32_t o = tpp / 2; o > 0; o >>= 1) {near |= (unsigned long long)__shfl_xor((long long)near, o, kWave);}
    const uint32_t exl = (nfar < excap) ? nfar : excap;
    uint32_t* row = s.nl + (size_t)(valid ? t : 0u) * cap;
    uint32_t count = 0;

    double4 nr = ri;
    uint32_t nj = 0, nslot = 0, nmol = 0;
    int nbase = 0;
    auto fetch = [&](uint32_t base) {
        const uint32_t q = base + tid;
        if(q >= np) {return;}
        nj = s.part[q];
        nr = pos[nj];
        nslot = s.pslot[nj];
        if(rule.ignore_mol) {nmol = s.mol[nj];}
        if(rule.base_rule) {nbase = (int)rule.base_par[(size_t)nj * rule.base_stride];}
    };
    fetch(0);
    for(uint32_t base = 0; base < np; base += kScanTile)
    {
        __syncthreads();
        cx[tid] = nr.x; cy[tid] = nr.y; cz[tid] = nr.z;
        cj[tid] = nj; cslot[tid] = nslot; cmol[tid] = nmol; cbase[tid] = nbase;
        __syncthreads();
        fetch(base + kScanTile);
        const uint32_t m = (np - base < kScanTile) ? np - base : kScanTile;
        for(uint32_t b = 0; b < m; b += tpp)
        {
            const uint32_t c = b + l;
            bool accept = valid && c < m;
            const uint32_t q = accept ? c : 0u;
            const uint32_t j = cj[q];
            accept = accept && j != i;
            const bool up = i < j;
            if(accept && rule.use_distance)
            {
                // the reference measures the pair from its lower index (same operands, same order)
                const double4 rj = make_double4(cx[q], cy[q], cz[q], 0.0);
                const double4 from = up ? ri : rj, to = up ? rj : ri;
                double dx, dy, dz;
                adjust_direction(box, from.x, from.y, from.z, to.x, to.y, to.z, dx, dy, dz);
                accept = length_sq(dx, dy, dz) < rule.r_list2;
            }
            if(accept)
            {
                const uint32_t slo = up ? islot : cslot[q], shi = up ? cslot[q] : islot;
                accept = rule.pairwise ? slo <= shi : slo != rule.last_slot;
                if(rule.ignore_mol == 1) {accept = accept && imol != cmol[q];}
                if(rule.ignore_mol == 2) {accept = accept && imol == cmol[q];}
                const int jbase = cbase[q];
                if(rule.base_rule == 1)
                {
                    accept = accept && !(ibase >= 2 && jbase >= 2 && complementary_bases(ibase - 2, jbase - 2));
                }
                else if(rule.base_rule == 2) {accept = accept && complementary_bases(ibase, jbase);}
                const uint32_t d = j - i + 32u;
                if(d < 64u) {accept = accept && ((near >> d) & 1ull) == 0ull;}
                else
                {
                    for(uint32_t k = 0; accept && k < exl; ++k) {accept = ex[exo + k] != j;}
                    for(uint32_t k = over; accept && k < exn; ++k) {accept = s.ex[exb + k] != j;}
                }
            }
            const uint64_t took = __ballot(accept) & gmask;
            if(accept)
            {
                const uint32_t k = count + (uint32_t)__popcll(took & below);
                if(k < cap) {row[k] = j;}
            }
            count += (uint32_t)__popcll(took);
        }
    }
    if(valid && l == 0) {s.nn[t] = (count < cap) ? count : cap;}
    block_max2_to(valid ? count : 0u, 0u, &s.ctl->maxcount, nullptr);
    __threadfence_block();     // the rows are read back by the block that wrote them
}

// TSP: the system has 3SPN2 terms (their long arithmetic costs the other systems registers).
template<bool MIXED, bool TSP>
__global__ void __launch_bounds__(256)
k_forces(const double4* __restrict__ pos, Box box, SmallForces a)
{
    const uint32_t block = blockIdx.x;
    if(block >= a.noise_begin)
    {
        // the next step's draws, ready when k_advance opens it
        const uint32_t i = (block - a.noise_begin) * blockDim.x + threadIdx.x;
        if(i < a.n)
        {
            double x, y, z;
            noise3(a.seed, a.sctl->step + a.k + 1, i, x, y, z);
            a.noise[i] = make_double4(x, y, z, 0.0);
        }
        return;
    }
    if(block >= a.local_begin)
    {
        const uint32_t lb = block - a.local_begin;
        int si = 0;
        while(si + 1 < a.nlocal && lb >= a.local[si + 1].block_begin) {++si;}
        const LocalSeg& s = a.local[si];
        const uint32_t t = (lb - s.block_begin) * blockDim.x + threadIdx.x;
        if(t < s.n_terms) {local_term<false, TSP>(s, t, pos, box, a.lidx, a.lpar, a.ldst, a.tf, nullptr);}
        return;
    }
    int si = 0;
    while(si + 1 < a.nrow && block >= a.row[si + 1].block_begin) {++si;}
    const RowSeg& s = a.row[si];
    // a row's lanes: tpp, four times as many for cross stacking (one pair on four lanes); a rebuild
    // takes tpp of them, the lanes of one wave
    const uint32_t lanes = (TSP && s.p.kind == kCrossStack) ? 4 * s.p.tpp : s.p.tpp;
    const uint32_t rows = 256 / lanes, row0 = (block - s.block_begin) * rows;
    const uint32_t t = row0 + threadIdx.x / lanes, l = threadIdx.x % lanes;
    const bool valid = t < s.p.np;
    // the row's head is on its way while the skin decision's words are
    RowHead h = row_head(s.p, valid ? t : 0u, l);
    if(!s.never && margin_after(s.ctl, a.sctl, a.k) < 0)
    {
        const uint32_t r = threadIdx.x / s.p.tpp;
        self_build(s, box, pos, row0 + r, threadIdx.x % s.p.tpp, r < rows && row0 + r < s.p.np);
        h = row_head(s.p, valid ? t : 0u, l);
    }
    if(!valid) {return;}   // whole groups leave together
    if(TSP && (s.p.kind == kBasePair || s.p.kind == kCrossStack))
    {
        TspSeg ts;
        ts.kind = s.p.kind; ts.np = s.p.np; ts.cap = s.p.cap; ts.tpp = s.p.tpp;
        ts.spart = s.p.spart; ts.nl = s.p.nl; ts.nn = s.p.nn; ts.ppar = s.p.ppar;
        ts.acc = s.acc; ts.n = a.n; ts.eout = nullptr;
        if(s.p.kind == kBasePair) {tsp_row<false, 1>(ts, t, l, pos, box);}
        else {tsp_row<false, 4>(ts, t, l, pos, box);}
    }
    else if constexpr(MIXED) {pair_row_mixed_store<false>(s.p, h, t, l, pos, box);}
    else {pair_row_store<false>(s.p, h, t, l, pos, box);}
}

} // mjg
