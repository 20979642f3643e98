// Cell-tile pair kernel of the engine (periodic cell lists).
//
// One workgroup per cell of the interaction's grid.  It stages the 27 surrounding cells' slots
// (TileSlot, written in slot order by k_tile_slots each step) in LDS, in the order the list
// build walks them (z outer, then y, then x; each cell's sorted slots in order), and walks the
// rows of its own cell's participants.  A row entry's staging slot is written by k_verlet beside
// its particle index (nl16), so a partner is read from LDS instead of gathered from global memory:
// the rows of one cell share their 27-cell neighbourhood, which the full-list kernels fetch again
// for every row entry (about 130 scattered 32-byte loads per particle at r_l = 15 A in the
// Lennard-Jones fluid).
//
// The lanes of a row and their sum order are those of k_pairs / k_pairs_mixed when tpp is theirs
// (entries k = l, l + tpp, ... per lane, then the same butterfly): the FP64 result is theirs bit
// for bit; the mixed result is an exact fixed-point sum, the same for any lane split.  A build
// whose largest neighbourhood exceeded the staging capacity (ListCtl::maxnbr > cap_nbr) is served
// by those kernels' global gathers instead, inside this kernel, until the host grows the capacity.
#pragma once
#include "force_kernels.hpp"
#include "nlist_kernels.hpp"

#include <type_traits>

namespace mjg
{
// One sorted slot as the tile stages it.  FP64: the position and both parameter columns.  Mixed: the
// FP32 hi and lo parts of the offset from the centre of the slot's own cell (at the image nearest to
// it), the parameter columns in their w.
template<bool MIXED> struct TileSlot;
template<> struct TileSlot<false> {double x, y, z, p0, p1, pad;};
template<> struct TileSlot<true> {float4 hi, lo;};

struct TileSeg
{
    PairSeg ps;                   // rows, lists, parameters and outputs as k_pairs reads them
    const uint16_t* nl16;         // staging slot of each row entry (row-major like nl)
    const uint32_t* spart;        // sorted slot -> particle
    const void* slots;            // this call's positions and parameters in slot order (k_tile_slots)
    const uint32_t* cell_start;
    const uint32_t* cell_end;
    Grid grid;                    // a periodic box's grid is fixed
    float wh[3], wl[3];           // cell widths, hi and lo parts
    const ListCtl* ctl;
    uint32_t cap_nbr;             // staging capacity in particles
    uint32_t tpp;                 // lanes per row of this kernel
    uint16_t* in16;               // staging slots of the inner list's entries (null: no inner list in
                                  // this launch); rows served from global memory walk the whole list
};
constexpr uint32_t kTileThreads = 256;
constexpr int kTileBatch = 4;

// staged per-particle parameters (column 0 and 1)
struct StagePar
{
    const double* s0;
    const double* s1;
    __device__ __forceinline__ double get(uint32_t k, int c) const {return c ? s1[k] : s0[k];}
};

// LDS bytes per staged particle: x, y, z, two parameter columns, particle index
constexpr size_t kTileBytesPerParticle = 5 * sizeof(double) + sizeof(uint32_t);

// What a lane needs of its row before any position, read before the neighbourhood is staged (a
// word past the row's end is dropped by length afterwards).
struct TileHead
{
    uint32_t i, cnt;
    uint32_t w[kTileBatch];
};
template<int USE>
__device__ __forceinline__ TileHead tile_head(const TileSeg& s, uint32_t t, uint32_t l)
{
    TileHead h;
    h.i = s.spart[t];
    h.cnt = (USE == kListInner) ? s.ps.nin[t] : s.ps.nn[t];
    const uint16_t* row = ((USE == kListInner) ? (const uint16_t*)s.in16 : s.nl16) + (size_t)t * s.ps.cap;
#pragma unroll
    for(int m = 0; m < kTileBatch; ++m)
    {
        const uint32_t k = l + m * s.tpp;
        h.w[m] = row[(k < s.ps.cap) ? k : 0u];
    }
    return h;
}

// Block b's cell: consecutive blocks go to the eight XCDs in turn, so each XCD gets a contiguous
// eighth of the cells, whose neighbourhoods overlap in its own L2 (ncell when there is none).
constexpr uint32_t kXcds = 8;
__device__ __forceinline__ uint32_t tile_cell_index(uint32_t b, uint32_t ncell)
{
    const uint32_t per = (ncell + kXcds - 1) / kXcds;
    const uint32_t c = (b % kXcds) * per + b / kXcds;
    return (b / kXcds < per && c < ncell) ? c : ncell;
}

template<bool MIXED, bool ENERGY, int KIND, int USE>
__device__ __forceinline__ void tile_rows(const TileSeg& s, const TileHead& head, const Box& box, uint32_t cs, uint32_t nhome, uint32_t home0,
                                          const double* sx, const double* sy, const double* sz, const StagePar& par,
                                          const uint32_t* sid)
{
    const PairSeg& ps = s.ps;
    const uint32_t tpp = s.tpp;
    const uint32_t tid = threadIdx.x;
    const PairConstsF K = pair_consts_f(ps.pp);
    for(uint32_t u = tid; u < nhome * tpp; u += kTileThreads)
    {
        const uint32_t h = u / tpp, l = u % tpp;
        const uint32_t t = cs + h, ki = home0 + h;
        const TileHead hd = (u == tid) ? head : tile_head<USE>(s, t, l);
        const uint32_t i = hd.i;
        const double xi = sx[ki], yi = sy[ki], zi = sz[ki];
        const uint32_t cnt = hd.cnt;
        const uint16_t* row = ((USE == kListInner) ? (const uint16_t*)s.in16 : s.nl16) + (size_t)t * ps.cap;
        uint32_t at = 0;
        double fx = 0, fy = 0, fz = 0, e = 0;
        long long ax = 0, ay = 0, az = 0;
        // the entries k = l, l + tpp, ... in order, kTileBatch at a time: a batch's row words come
        // from global memory, so the next batch's are requested before the current one is computed
        constexpr int B = kTileBatch;
        uint32_t nxt[B];
#pragma unroll
        for(int m = 0; m < B; ++m) {const uint32_t k = l + m * tpp; nxt[m] = (k < cnt) ? hd.w[m] : ki;}
        for(uint32_t k0 = l; k0 < cnt; k0 += B * tpp)
        {
            uint32_t kj[B];
#pragma unroll
            for(int m = 0; m < B; ++m) {kj[m] = nxt[m];}
#pragma unroll
            for(int m = 0; m < B; ++m)
            {
                const uint32_t k = k0 + (B + m) * tpp;
                nxt[m] = (k < cnt) ? row[k] : ki;
            }
#pragma unroll
            for(int m = 0; m < B; ++m)
            {
                if(k0 + m * tpp >= cnt) {break;}
                const uint32_t j = sid[kj[m]];
                double dx, dy, dz;
                adjust_direction(box, xi, yi, zi, sx[kj[m]], sy[kj[m]], sz[kj[m]], dx, dy, dz);
                if constexpr(USE == kListPrune)
                {
                    const bool keep = length_sq(dx, dy, dz) < ps.r_in2;
                    const uint32_t k = group_append(keep, tpp, at);
                    if(keep) {s.in16[(size_t)t * ps.cap + k] = (uint16_t)kj[m];}
                }
                if constexpr(MIXED)
                {
                    float c;
                    if(!pair_term_f32<KIND, ENERGY>(K, ps.pp, par, i, j, ki, kj[m], dx, dy, dz, c, e)) {continue;}
                    long long gx, gy, gz;
                    fix3r<float>((float)dx * c, (float)dy * c, (float)dz * c, gx, gy, gz);
                    ax += gx; ay += gy; az += gz;
                }
                else
                {
                    pair_term_p<KIND, ENERGY>(ps.pp, i, j, par, ki, kj[m], dx, dy, dz, fx, fy, fz, e);
                }
            }
        }
        for(uint32_t o = tpp / 2; o > 0; o >>= 1)
        {
            if constexpr(MIXED)
            {
                ax += shfl_xor_ll(ax, (int)o);
                ay += shfl_xor_ll(ay, (int)o);
                az += shfl_xor_ll(az, (int)o);
            }
            else
            {
                fx += __shfl_xor(fx, o, kWave);
                fy += __shfl_xor(fy, o, kWave);
                fz += __shfl_xor(fz, o, kWave);
            }
            if(ENERGY) {e += __shfl_xor(e, o, kWave);}
        }
        if(l == 0)
        {
            if(USE == kListPrune) {ps.nin[t] = at;}
            if constexpr(MIXED)
            {
                const bool bad = fix_insane((unsigned long long)ax) || fix_insane((unsigned long long)ay) ||
                                 fix_insane((unsigned long long)az);
                const double nan = bad ? __builtin_nan("") : 0.0;
                ps.fout[i] = make_double4(from_fix<float>((unsigned long long)ax) + nan,
                                          from_fix<float>((unsigned long long)ay) + nan,
                                          from_fix<float>((unsigned long long)az) + nan, 0.0);
            }
            else
            {
                ps.fout[i] = make_double4(fx, fy, fz, 0.0);
            }
            if(ENERGY) {ps.eout[t] = e;}
        }
    }
}

// The rows of one cell with the full-list kernels' global gathers (a neighbourhood that does not
// fit the staging capacity).
template<bool MIXED, bool ENERGY, int KIND>
__device__ __forceinline__ void tile_rows_global(const TileSeg& s, const double4* __restrict__ pos, const Box& box,
                                                 uint32_t cs, uint32_t nhome)
{
    const PairSeg& ps = s.ps;
    const uint32_t tpp = ps.tpp;
    for(uint32_t u = threadIdx.x; u < nhome * tpp; u += kTileThreads)
    {
        const uint32_t t = cs + u / tpp, l = u % tpp;
        const RowHead hd = row_head(ps, t, l);
        const uint32_t i = hd.i;
        double e = 0;
        if constexpr(MIXED)
        {
            long long ax = 0, ay = 0, az = 0;
            pair_row_mixed<KIND, ENERGY>(ps, hd, t, l, pos, box, ax, ay, az, e);
            for(uint32_t o = tpp / 2; o > 0; o >>= 1)
            {
                ax += shfl_xor_ll(ax, (int)o);
                ay += shfl_xor_ll(ay, (int)o);
                az += shfl_xor_ll(az, (int)o);
                if(ENERGY) {e += __shfl_xor(e, o, kWave);}
            }
            if(l == 0)
            {
                const bool bad = fix_insane((unsigned long long)ax) || fix_insane((unsigned long long)ay) ||
                                 fix_insane((unsigned long long)az);
                const double nan = bad ? __builtin_nan("") : 0.0;
                ps.fout[i] = make_double4(from_fix<float>((unsigned long long)ax) + nan,
                                          from_fix<float>((unsigned long long)ay) + nan,
                                          from_fix<float>((unsigned long long)az) + nan, 0.0);
                if(ENERGY) {ps.eout[t] = e;}
            }
        }
        else
        {
            double fx = 0, fy = 0, fz = 0;
            pair_row<KIND, ENERGY>(ps, hd, t, l, pos, box, fx, fy, fz, e);
            for(uint32_t o = tpp / 2; o > 0; o >>= 1)
            {
                fx += __shfl_xor(fx, o, kWave);
                fy += __shfl_xor(fy, o, kWave);
                fz += __shfl_xor(fz, o, kWave);
                if(ENERGY) {e += __shfl_xor(e, o, kWave);}
            }
            if(l == 0)
            {
                ps.fout[i] = make_double4(fx, fy, fz, 0.0);
                if(ENERGY) {ps.eout[t] = e;}
            }
        }
    }
}

// The 27 neighbour cells of `cell` (m = 9 (dz + 1) + 3 (dy + 1) + (dx + 1), wrapped as k_verlet wraps
// them): first sorted slot and staging offsets (c_off[27] = neighbourhood size).
__device__ __forceinline__ void tile_neighbourhood(const uint32_t* __restrict__ cell_start,
                                                   const uint32_t* __restrict__ cell_end, const Grid& g, uint32_t cell,
                                                   uint32_t* c_beg, uint32_t* c_off)
{
    const uint32_t tid = threadIdx.x;
    uint32_t count = 0;
    if(tid < 27)
    {
        const int dz = (int)(tid / 9) - 1, dy = (int)((tid / 3) % 3) - 1, dx = (int)(tid % 3) - 1;
        const int cx = (int)(cell % (uint32_t)g.dim[0]);
        const int cy = (int)((cell / (uint32_t)g.dim[0]) % (uint32_t)g.dim[1]);
        const int cz = (int)(cell / ((uint32_t)g.dim[0] * (uint32_t)g.dim[1]));
        int x = cx + dx, y = cy + dy, z = cz + dz;
        x = (x < 0) ? g.dim[0] - 1 : (x >= g.dim[0] ? 0 : x);
        y = (y < 0) ? g.dim[1] - 1 : (y >= g.dim[1] ? 0 : y);
        z = (z < 0) ? g.dim[2] - 1 : (z >= g.dim[2] ? 0 : z);
        const uint32_t c2 = (uint32_t)x + (uint32_t)g.dim[0] * ((uint32_t)y + (uint32_t)g.dim[1] * (uint32_t)z);
        const uint32_t b = cell_start[c2], en = cell_end[c2];
        c_beg[tid] = b;
        count = (en > b) ? en - b : 0u;
    }
    // running sums over the first wave's lanes
    if(tid < (uint32_t)kWave)
    {
        uint32_t sum = count;
#pragma unroll
        for(int o = 1; o < 32; o <<= 1)
        {
            const uint32_t v = (uint32_t)__shfl_up((int)sum, o, kWave);
            if((int)tid >= o) {sum += v;}
        }
        if(tid < 27) {c_off[tid + 1] = sum;}
        if(tid == 0) {c_off[0] = 0;}
    }
    __syncthreads();
}

// f(staging slot, neighbour cell, sorted slot) for every particle of the neighbourhood.  A wave takes one
// of the nine runs of three cells at a time, a lane a particle (a run of a liquid at r_list = 15 A
// holds about 57): its cell is two comparisons away, and consecutive lanes read consecutive sorted
// slots.
template<typename F>
__device__ __forceinline__ void tile_stage(const uint32_t* c_beg, const uint32_t* c_off, F&& f)
{
    const uint32_t wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    for(uint32_t r = wave; r < 9; r += kTileThreads / kWave)
    {
        const uint32_t o0 = c_off[3 * r], o1 = c_off[3 * r + 1], o2 = c_off[3 * r + 2], o3 = c_off[3 * r + 3];
        for(uint32_t k = o0 + lane; k < o3; k += kWave)
        {
            const uint32_t c = (k >= o1 ? 1u : 0u) + (k >= o2 ? 1u : 0u);
            const uint32_t m = 3 * r + c;
            f(k, m, c_beg[m] + (k - (c == 0 ? o0 : c == 1 ? o1 : o2)));
        }
    }
}

// neighbour cell of staging slot k (binary search over the 27 offsets)
__device__ __forceinline__ uint32_t tile_cell_of(const uint32_t* c_off, uint32_t k)
{
    uint32_t m = 0;
#pragma unroll
    for(uint32_t w = 16; w > 0; w >>= 1) {if(m + w < 27 && c_off[m + w] <= k) {m += w;}}
    return m;
}

template<bool MIXED, bool ENERGY, int KIND, int USE>
__device__ __forceinline__ void tile_cell(const TileSeg& s, const double4* __restrict__ pos, const Box& box,
                                          unsigned char* smem)
{
    __shared__ uint32_t c_beg[27], c_off[28];
    const uint32_t cell = tile_cell_index(blockIdx.x, s.grid.ncell);
    if(cell >= s.grid.ncell) {return;}
    const uint32_t tid = threadIdx.x;
    const uint32_t cs = s.cell_start[cell], ce = s.cell_end[cell];
    if(ce <= cs) {return;}                                   // empty cell: no rows (uniform)
    const uint32_t nhome = ce - cs;
    if(s.ctl->maxnbr > s.cap_nbr)                            // uniform: one word for the launch
    {
        tile_rows_global<MIXED, ENERGY, KIND>(s, pos, box, cs, nhome);
        return;
    }
    // the first row of the thread (its own row again where the cell has fewer)
    const uint32_t h0 = (tid / s.tpp < nhome) ? tid / s.tpp : 0u;
    const TileHead head = tile_head<USE>(s, cs + h0, tid % s.tpp);
    tile_neighbourhood(s.cell_start, s.cell_end, s.grid, cell, c_beg, c_off);
    const uint32_t cap = s.cap_nbr;
    double* sx = reinterpret_cast<double*>(smem);
    double* sy = sx + cap;
    double* sz = sy + cap;
    double* s0 = sz + cap;
    double* s1 = s0 + cap;
    uint32_t* sid = reinterpret_cast<uint32_t*>(s1 + cap);
    tile_stage(c_beg, c_off, [&](uint32_t k, uint32_t, uint32_t q) {
        const TileSlot<false> v = static_cast<const TileSlot<false>*>(s.slots)[q];
        sx[k] = v.x; sy[k] = v.y; sz[k] = v.z;
        s0[k] = v.p0; s1[k] = v.p1;
        sid[k] = s.spart[q];
    });
    __syncthreads();
    tile_rows<MIXED, ENERGY, KIND, USE>(s, head, box, cs, nhome, c_off[13], sx, sy, sz, StagePar{s0, s1}, sid);
}

// ------------------------------------------------------------------------------------
// Mixed precision (MJG_FP32_FIXED) with FP32 staging.  Each staged particle holds its position
// relative to the home cell's centre, seen through the neighbour cell's periodic image, split into
// two FP32 parts (hi = the FP32 rounding of the FP64 offset, lo = the FP32 rounding of what
// remains), so that (hi_j - hi_i) + (lo_j - lo_i) is the displacement to about FP32 precision of
// the displacement itself; no minimum-image branches remain in the pair loop.  The cutoff test is
// taken on that r^2 in FP32 where it is clear by more than kTileBand (relative); a pair inside the
// band is decided by the FP64 path's own test (adjust_direction on the FP64 positions and the FP64
// parameters), so the pair set inside the cutoff stays the FP64 path's.  The staged parameters are
// FP32 (column 0 with the hi part, column 1 with the lo part).  No particle index is staged: a
// row's own index comes from the cell-sorted order, a neighbour's only for a pair inside the band
// (through its cell, as staging found it), and each row adds half of every pair energy, so a
// pair's energy is counted once over its two rows.
// ------------------------------------------------------------------------------------
constexpr float kTileBand = 1.0e-5f;          // the FP32 r^2 and threshold errors are below 2e-6 relative
constexpr size_t kTileBytesPerParticleF32 = 2 * sizeof(float4);

// (hi, lo) + (eh, el) as (h, l): h the rounded sum of the large parts, its rounding error kept in l
__device__ __forceinline__ void tile_shift(float hi, float lo, float eh, float el, float& h, float& l)
{
#pragma clang fp contract(off)
    h = hi + eh;
    const float b = h - hi;
    const float err = (hi - (h - b)) + (eh - b);
    l = (lo + el) + err;
}

// The positions and parameters of one tiled interaction in slot order, for the force call that follows:
// staging then reads each neighbour cell as one contiguous run.  Without it every staged particle
// (27 cells stage each one) went through its index to scattered position and parameter loads, and the
// mixed kernel formed the split FP64 offset 27 times; the tile kernel of the 262,144-particle fluid
// spent more time staging than on its pairs (mixed 98 us a step on the inner list).
template<bool MIXED>
__global__ void __launch_bounds__(256)
k_tile_slots(const double4* __restrict__ pos, Box box, const uint32_t* __restrict__ spart,
             const uint32_t* __restrict__ skeys, const Grid* __restrict__ grid, const double* __restrict__ ppar, int npar,
             uint32_t np, void* __restrict__ out)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if(t >= np) {return;}
    const uint32_t i = spart[t];
    const double4 r = pos[i];
    const double p0 = ppar[(size_t)i * npar], p1 = (npar > 1) ? ppar[(size_t)i * npar + 1] : 0.0;
    TileSlot<MIXED> v;
    if constexpr(MIXED)
    {
        // A particle has moved less than half the skin since the build that put it in this cell, and
        // positions are wrapped into the box every step: its image nearest to the cell's centre is the one
        // within half a cell plus that drift, fewer than half a box width, since a periodic grid has at
        // least three cells a dimension.  Seen from a neighbouring home cell this image is a partner's nearest
        // one, or out of reach, where (dim - 2) cell widths are at least r_list on every axis: the other
        // image lies (dim - 2) widths away at the build and r_list less the skin, the cutoff, later.  An
        // axis of three cells narrower than r_list has pairs inside the cutoff through its other side;
        // this kernel is not launched for such boxes.
        const Grid g = *grid;
        const uint32_t cell = skeys[t];
        const int cx = (int)(cell % (uint32_t)g.dim[0]);
        const int cy = (int)((cell / (uint32_t)g.dim[0]) % (uint32_t)g.dim[1]);
        const int cz = (int)(cell / ((uint32_t)g.dim[0] * (uint32_t)g.dim[1]));
        double X = r.x - (box.lower[0] + ((double)cx + 0.5) * (box.width[0] / g.dim[0]));
        double Y = r.y - (box.lower[1] + ((double)cy + 0.5) * (box.width[1] / g.dim[1]));
        double Z = r.z - (box.lower[2] + ((double)cz + 0.5) * (box.width[2] / g.dim[2]));
        X -= box.width[0] * rint(X * (1.0 / box.width[0]));
        Y -= box.width[1] * rint(Y * (1.0 / box.width[1]));
        Z -= box.width[2] * rint(Z * (1.0 / box.width[2]));
        const float hx = (float)X, hy = (float)Y, hz = (float)Z;
        v.hi = make_float4(hx, hy, hz, (float)p0);
        v.lo = make_float4((float)(X - (double)hx), (float)(Y - (double)hy), (float)(Z - (double)hz), (float)p1);
    }
    else
    {
        v.x = r.x; v.y = r.y; v.z = r.z; v.p0 = p0; v.p1 = p1; v.pad = 0.0;
    }
    static_cast<TileSlot<MIXED>*>(out)[t] = v;
}

// the FP64 path's inside-cutoff decision of the pair (i, j) (pair_term_f32's)
template<int KIND>
__device__ __forceinline__ bool tile_inside_fp64(const PairParams& pp, const double* __restrict__ ppar,
                                              const double4* __restrict__ pos, const Box& box, uint32_t i, uint32_t j)
{
    const double4 ri = pos[i], rj = pos[j];
    double dx, dy, dz;
    adjust_direction(box, ri.x, ri.y, ri.z, rj.x, rj.y, rj.z, dx, dy, dz);
    const double l_sq = length_sq(dx, dy, dz);
    if(KIND == kPairLJ)
    {
        const double sg = (ppar[2 * (size_t)i] + ppar[2 * (size_t)j]) / 2;
        return !(sg * sg * pp.cutoff_ratio2 < l_sq);
    }
    if(KIND == kPairEV)
    {
        const double rad = ppar[i] + ppar[j];
        return !(rad * rad * pp.cutoff_ratio2 < l_sq);
    }
    if(KIND == kPair3SPN2EV)
    {
        const double sg = (tsp::ev_sigma((int)ppar[i]) + tsp::ev_sigma((int)ppar[j])) * 0.5;
        return sg * sg > l_sq;
    }
    return pp.abs_cutoff * pp.abs_cutoff > l_sq;
}

// the particle index of staging slot k (its cell found among the 27 offsets)
__device__ __forceinline__ uint32_t tile_slot_particle(const TileSeg& s, const uint32_t* c_beg, const uint32_t* c_off,
                                                       uint32_t k)
{
    const uint32_t m = tile_cell_of(c_off, k);
    return s.spart[c_beg[m] + (k - c_off[m])];
}

template<bool ENERGY, int KIND, int USE>
__device__ __forceinline__ void tile_rows_f32(const TileSeg& s, const TileHead& head, const double4* __restrict__ pos, const Box& box,
                                              uint32_t cs, uint32_t nhome, uint32_t home0, const float4* hi,
                                              const float4* lo, const uint32_t* c_beg, const uint32_t* c_off)
{
#pragma clang fp contract(fast)
    const PairSeg& ps = s.ps;
    const uint32_t tpp = s.tpp;
    const uint32_t tid = threadIdx.x;
    const PairConstsF K = pair_consts_f(ps.pp);
    const float acut2 = (float)(ps.pp.abs_cutoff * ps.pp.abs_cutoff);
    const float rin2 = (float)ps.r_in2 * (1.0f + kTileBand);
    for(uint32_t u = tid; u < nhome * tpp; u += kTileThreads)
    {
        const uint32_t h = u / tpp, l = u % tpp;
        const uint32_t t = cs + h, ki = home0 + h;
        const TileHead hd = (u == tid) ? head : tile_head<USE>(s, t, l);
        const uint32_t i = hd.i;
        const float4 ah = hi[ki], al = lo[ki];
        const uint32_t cnt = hd.cnt;
        const uint16_t* row = ((USE == kListInner) ? (const uint16_t*)s.in16 : s.nl16) + (size_t)t * ps.cap;
        uint32_t at = 0;
        double e = 0;
        long long ax = 0, ay = 0, az = 0;
        constexpr int B = kTileBatch;
        uint32_t nxt[B];
#pragma unroll
        for(int m = 0; m < B; ++m) {const uint32_t k = l + m * tpp; nxt[m] = (k < cnt) ? hd.w[m] : ki;}
        for(uint32_t k0 = l; k0 < cnt; k0 += B * tpp)
        {
            uint32_t kj[B];
#pragma unroll
            for(int m = 0; m < B; ++m) {kj[m] = nxt[m];}
#pragma unroll
            for(int m = 0; m < B; ++m)
            {
                const uint32_t k = k0 + (B + m) * tpp;
                nxt[m] = (k < cnt) ? row[k] : ki;
            }
#pragma unroll
            for(int m = 0; m < B; ++m)
            {
                if(k0 + m * tpp >= cnt) {break;}
                const float4 bh = hi[kj[m]], bl = lo[kj[m]];
                const float dx = (bh.x - ah.x) + (bl.x - al.x);
                const float dy = (bh.y - ah.y) + (bl.y - al.y);
                const float dz = (bh.z - ah.z) + (bl.z - al.z);
                const float l_sq = dx * dx + dy * dy + dz * dz;
                if constexpr(USE == kListPrune)
                {
                    const bool keep = l_sq < rin2;
                    const uint32_t k = group_append(keep, tpp, at);
                    if(keep) {s.in16[(size_t)t * ps.cap + k] = (uint16_t)kj[m];}
                }
                float thr, sg = 0.0f;
                if(KIND == kPairLJ) {sg = (ah.w + bh.w) * 0.5f; thr = sg * sg * K.cut2;}
                else if(KIND == kPairEV) {sg = ah.w + bh.w; thr = sg * sg * K.cut2;}
                else if(KIND == kPair3SPN2EV)
                {
                    sg = (float)((tsp::ev_sigma((int)ah.w) + tsp::ev_sigma((int)bh.w)) * 0.5);
                    thr = sg * sg;
                }
                else {thr = acut2;}
                if(l_sq > thr * (1.0f + kTileBand)) {continue;}
                if(l_sq >= thr * (1.0f - kTileBand) &&
                   !tile_inside_fp64<KIND>(ps.pp, ps.ppar, pos, box, i, tile_slot_particle(s, c_beg, c_off, kj[m])))
                {
                    continue;
                }
                float c;
                if(KIND == kPairLJ)
                {
                    const float e1 = al.w, e2 = bl.w;
                    const float eps = (e1 == e2) ? e1 : RMath<float>::sqrt(e1 * e2);
                    const float rcp = RMath<float>::rcp(l_sq);
                    const float s2l2 = sg * sg * rcp;
                    const float s6 = s2l2 * s2l2 * s2l2;
                    c = 24.0f * eps * (s6 - 2.0f * s6 * s6) * rcp;
                    if(ENERGY) {e += 0.5 * (double)(4.0f * eps * (s6 * s6 - s6 - K.cac));}
                }
                else if(KIND == kPairEV)
                {
                    const float rcp = RMath<float>::rcp(l_sq);
                    const float s2l2 = sg * sg * rcp;
                    const float s6 = s2l2 * s2l2 * s2l2;
                    c = -(K.eps * 12.0f) * s6 * s6 * rcp;
                    if(ENERGY) {e += 0.5 * (double)(K.eps * (s6 * s6 - K.cac));}
                }
                else if(KIND == kPair3SPN2EV)
                {
                    const float rl = RMath<float>::rsqrt(l_sq);
                    const float r1s1 = sg * rl;
                    const float r3s3 = r1s1 * r1s1 * r1s1;
                    const float r6s6 = r3s3 * r3s3;
                    c = 12.0f * K.eps * rl * r6s6 * (1.0f - r6s6) * rl;
                    if(ENERGY) {e += 0.5 * (double)(K.eps * (r6s6 * (r6s6 - 2.0f) + 1.0f));}
                }
                else
                {
                    const float qq = K.qk * ah.w * bh.w;
                    const float rl = RMath<float>::rsqrt(l_sq);
                    const float ll = l_sq * rl;
                    const float ex = RMath<float>::exp(-ll * K.idebye);
                    const float f_mag = -qq * (K.debye + ll) * K.idebye * (rl * rl) * ex;
                    c = f_mag * rl;
                    if(ENERGY) {e += 0.5 * (double)(qq * (ex * rl - K.cac));}
                }
                long long gx, gy, gz;
                fix3r<float>(dx * c, dy * c, dz * c, gx, gy, gz);
                ax += gx; ay += gy; az += gz;
            }
        }
        for(uint32_t o = tpp / 2; o > 0; o >>= 1)
        {
            ax += shfl_xor_ll(ax, (int)o);
            ay += shfl_xor_ll(ay, (int)o);
            az += shfl_xor_ll(az, (int)o);
            if(ENERGY) {e += __shfl_xor(e, o, kWave);}
        }
        if(l == 0)
        {
            if(USE == kListPrune) {ps.nin[t] = at;}
            const bool bad = fix_insane((unsigned long long)ax) || fix_insane((unsigned long long)ay) ||
                             fix_insane((unsigned long long)az);
            const double nan = bad ? __builtin_nan("") : 0.0;
            ps.fout[i] = make_double4(from_fix<float>((unsigned long long)ax) + nan,
                                      from_fix<float>((unsigned long long)ay) + nan,
                                      from_fix<float>((unsigned long long)az) + nan, 0.0);
            if(ENERGY) {ps.eout[t] = e;}
        }
    }
}

template<bool ENERGY, int KIND, int USE>
__device__ __forceinline__ void tile_cell_f32(const TileSeg& s, const double4* __restrict__ pos, const Box& box,
                                              unsigned char* smem)
{
    __shared__ uint32_t c_beg[27], c_off[28];
    const uint32_t cell = tile_cell_index(blockIdx.x, s.grid.ncell);
    if(cell >= s.grid.ncell) {return;}
    const uint32_t tid = threadIdx.x;
    const uint32_t cs = s.cell_start[cell], ce = s.cell_end[cell];
    if(ce <= cs) {return;}
    const uint32_t nhome = ce - cs;
    if(s.ctl->maxnbr > s.cap_nbr)
    {
        tile_rows_global<true, ENERGY, KIND>(s, pos, box, cs, nhome);
        return;
    }
    // the first row of the thread (its own row again where the cell has fewer)
    const uint32_t h0 = (tid / s.tpp < nhome) ? tid / s.tpp : 0u;
    const TileHead head = tile_head<USE>(s, cs + h0, tid % s.tpp);
    tile_neighbourhood(s.cell_start, s.cell_end, s.grid, cell, c_beg, c_off);
    const uint32_t cap = s.cap_nbr;
    float4* hi = reinterpret_cast<float4*>(smem);
    float4* lo = hi + cap;
    const float hx = s.wh[0], hy = s.wh[1], hz = s.wh[2], lx = s.wl[0], ly = s.wl[1], lz = s.wl[2];
    tile_stage(c_beg, c_off, [&](uint32_t k, uint32_t m, uint32_t q) {
        // the slot's offset from its own cell's centre, seen from the home cell: that cell lies dx, dy, dz
        // cell widths away.  hi + the width's hi part is split again exactly (two-sum), so the staged
        // parts are as good as those of the slot.
        const TileSlot<true> v = static_cast<const TileSlot<true>*>(s.slots)[q];
        const float dx = (float)((int)(m % 3) - 1), dy = (float)((int)((m / 3) % 3) - 1), dz = (float)((int)(m / 9) - 1);
        float4 h, l;
        tile_shift(v.hi.x, v.lo.x, dx * hx, dx * lx, h.x, l.x);
        tile_shift(v.hi.y, v.lo.y, dy * hy, dy * ly, h.y, l.y);
        tile_shift(v.hi.z, v.lo.z, dz * hz, dz * lz, h.z, l.z);
        h.w = v.hi.w; l.w = v.lo.w;
        hi[k] = h;
        lo[k] = l;
    });
    __syncthreads();
    tile_rows_f32<ENERGY, KIND, USE>(s, head, pos, box, cs, nhome, c_off[13], hi, lo, c_beg, c_off);
}

// ------------------------------------------------------------------------------------
// Cell-tiled list build for the interactions the cell-tile kernel serves.  A workgroup takes a
// cell at a time (a grid-stride loop over the cells, at most kVerletMaxBlocks workgroups, so that
// the launch a step makes when no list is rebuilt stays small), stages the slot-ordered positions
// (k_sorted_slots) and particles of its 27-cell neighbourhood in LDS in k_verlet's order, and builds
// the cell's rows from there: each candidate is loaded once per cell instead of once per row.  The
// candidates are tested in k_verlet's order by its own test (verlet_consider), so every row is
// k_verlet's, entry for entry, whatever the lanes per row.  A neighbourhood larger than the staging
// capacity builds its rows as k_verlet does.
//
// FAST: candidates are staged as FP32 offsets from the home cell's centre (each at its own cell's
// image) and tested there; only one within a relative band of 1e-5 around r_list^2 is decided on the
// FP64 positions as verlet_near does, so the rows are the same (the offsets reach 1.5 cell widths,
// and the FP32 error of a squared distance near r_list^2 is below 1e-6 of it).  A test is a third of
// the FP64 minimum image's instructions, which bound the build: of the 262,144-particle fluid 795 ->
// 405 us, of 30,000 particles 153 -> 83.  Valid where no pair within r_list sees another image
// nearer than the staged one, (dim - 2) cell widths at least r_list in every dimension; a grid
// clamped to three cells narrower than that is built in FP64.
// ------------------------------------------------------------------------------------
constexpr size_t kBuildBytesPerParticle = 3 * sizeof(double) + sizeof(uint32_t);
constexpr size_t kBuildBytesPerParticleF32 = sizeof(float4);

template<bool FAST>
__global__ void __launch_bounds__(kTileThreads)
k_verlet_tiled(const double4* __restrict__ pos, Box box, ListSeg s, uint32_t cap_nbr)
{
    if(s.ctl->rebuild == 0) {return;}
    extern __shared__ __align__(16) unsigned char tile_smem[];
    __shared__ uint32_t c_beg[27], c_off[28];
    double* sx = reinterpret_cast<double*>(tile_smem);
    double* sy = sx + cap_nbr;
    double* sz = sy + cap_nbr;
    uint32_t* sj = reinterpret_cast<uint32_t*>(sz + cap_nbr);
    float4* sf = reinterpret_cast<float4*>(tile_smem);
    const Grid g = *s.grid;
    const uint32_t tid = threadIdx.x, lane = tid % kWave;
    const uint32_t tpp = s.tpp;
    const float r2 = (float)s.rule.r_list2, r2_in = r2 * (1.0f - kTileBand), r2_out = r2 * (1.0f + kTileBand);
    uint32_t mc = 0, mn = 0;                                 // longest row, largest neighbourhood
    const uint32_t rounds = kXcds * ((g.ncell + kXcds - 1) / kXcds);
    for(uint32_t b = blockIdx.x; b < rounds; b += gridDim.x)
    {
        const uint32_t cell = tile_cell_index(b, g.ncell);
        if(cell >= g.ncell) {continue;}                      // uniform over the workgroup
        const uint32_t cs = s.cell_start[cell], ce = s.cell_end[cell];
        if(ce <= cs) {continue;}                             // uniform over the workgroup
        const uint32_t nhome = ce - cs;
        tile_neighbourhood(s.cell_start, s.cell_end, g, cell, c_beg, c_off);
        const uint32_t total = c_off[27];
        if(total > cap_nbr)
        {
            for(uint32_t u = tid; u < nhome * tpp; u += kTileThreads)
            {
                verlet_row(s, cs + u / tpp, u % tpp, pos, box, mc, mn);
            }
        }
        else
        {
            if constexpr(FAST)
            {
                const int hx = (int)(cell % (uint32_t)g.dim[0]);
                const int hy = (int)((cell / (uint32_t)g.dim[0]) % (uint32_t)g.dim[1]);
                const int hz = (int)(cell / ((uint32_t)g.dim[0] * (uint32_t)g.dim[1]));
                const double wx = box.width[0] / g.dim[0], wy = box.width[1] / g.dim[1], wz = box.width[2] / g.dim[2];
                const double ox = box.lower[0] + ((double)hx + 0.5) * wx, oy = box.lower[1] + ((double)hy + 0.5) * wy;
                const double oz = box.lower[2] + ((double)hz + 0.5) * wz;
                tile_stage(c_beg, c_off, [&](uint32_t k, uint32_t m, uint32_t q) {
                    // the image that lies in the neighbour cell as the home cell sees it
                    const int dx = (int)(m % 3) - 1, dy = (int)((m / 3) % 3) - 1, dz = (int)(m / 9) - 1;
                    const double4 r = s.spos[q];
                    const double X = r.x - ox + ((hx + dx < 0) ? -box.width[0] : (hx + dx >= g.dim[0]) ? box.width[0] : 0.0);
                    const double Y = r.y - oy + ((hy + dy < 0) ? -box.width[1] : (hy + dy >= g.dim[1]) ? box.width[1] : 0.0);
                    const double Z = r.z - oz + ((hz + dz < 0) ? -box.width[2] : (hz + dz >= g.dim[2]) ? box.width[2] : 0.0);
                    sf[k] = make_float4((float)X, (float)Y, (float)Z, __uint_as_float(s.spart[q]));
                });
            }
            else
            {
                tile_stage(c_beg, c_off, [&](uint32_t k, uint32_t, uint32_t q) {
                    const double4 rj = s.spos[q];
                    sx[k] = rj.x; sy[k] = rj.y; sz[k] = rj.z;
                    sj[k] = s.spart[q];
                });
            }
            __syncthreads();
            for(uint32_t u = tid; u < nhome * tpp; u += kTileThreads)
            {
                const uint32_t h = u / tpp, l = u % tpp;
                const uint32_t t = cs + h, ki = c_off[13] + h;
                RowBuild rb;
                rb.gmask = group_mask_of(tpp, lane);
                rb.below = rb.gmask & ((1ull << lane) - 1ull);
                rb.count = 0;
                rb.row = s.nl + (size_t)t * s.cap;
                rb.row16 = s.nl16 + (size_t)t * s.cap;
                if constexpr(FAST)
                {
                    const float4 a = sf[ki];
                    rb.i = __float_as_uint(a.w);
                    for(uint32_t base = 0; base < total; base += tpp)
                    {
                        const uint32_t k = base + l;
                        const bool v = k < total && k != ki;
                        const float4 c = sf[v ? k : ki];
                        const float dx = c.x - a.x, dy = c.y - a.y, dz = c.z - a.z;
                        const float d2 = dx * dx + dy * dy + dz * dz;
                        const uint32_t j = __float_as_uint(c.w);
                        bool near = v && d2 < r2_in;
                        if(v && !near && d2 <= r2_out)
                        {
                            const uint32_t m = tile_cell_of(c_off, k);
                            near = verlet_near(box, s.rule.r_list2, rb.i, j, s.spos[t], s.spos[c_beg[m] + (k - c_off[m])]);
                        }
                        verlet_append(s, rb, j, near, k);
                    }
                }
                else
                {
                    rb.i = sj[ki];
                    rb.ri = make_double4(sx[ki], sy[ki], sz[ki], 0.0);
                    for(uint32_t base = 0; base < total; base += tpp)
                    {
                        const uint32_t k = base + l;
                        const bool v = k < total;
                        verlet_consider(s, box, rb, v ? sj[k] : 0u, v, k,
                                        v ? make_double4(sx[k], sy[k], sz[k], 0.0) : rb.ri);
                    }
                }
                if(l == 0) {s.nn[t] = (rb.count < s.cap) ? rb.count : s.cap;}
                mc = max(mc, rb.count);
                mn = max(mn, total);
            }
        }
        __syncthreads();                                     // the next cell's staging overwrites this one's
    }
    block_max2_to(mc, mn, &s.ctl->maxcount, &s.ctl->maxnbr);
}

// one kernel per kind: a kind's registers do not weigh on the others' waves per SIMD
template<bool MIXED, bool ENERGY, int KIND>
__global__ void __launch_bounds__(kTileThreads)
k_pairs_tiled(const double4* __restrict__ pos, Box box, TileSeg s)
{
    extern __shared__ __align__(16) unsigned char tile_smem[];
    auto cell = [&](auto use) {
        constexpr int USE = decltype(use)::value;
        if constexpr(MIXED) {tile_cell_f32<ENERGY, KIND, USE>(s, pos, box, tile_smem);}
        else {tile_cell<false, ENERGY, KIND, USE>(s, pos, box, tile_smem);}
    };
    // the launch's use of the lists (uniform: one word); an energy call walks the whole list
    if(ENERGY || s.in16 == nullptr) {cell(std::integral_constant<int, kListWhole>{});}
    else if(s.ctl->prune) {cell(std::integral_constant<int, kListPrune>{});}
    else {cell(std::integral_constant<int, kListInner>{});}
}

using TileKernel = void (*)(const double4*, Box, TileSeg);
template<bool MIXED, bool ENERGY>
inline TileKernel tile_kernel(int kind)
{
    if(kind == kPairLJ) {return k_pairs_tiled<MIXED, ENERGY, kPairLJ>;}
    if(kind == kPairEV) {return k_pairs_tiled<MIXED, ENERGY, kPairEV>;}
    if(kind == kPair3SPN2EV) {return k_pairs_tiled<MIXED, ENERGY, kPair3SPN2EV>;}
    return k_pairs_tiled<MIXED, ENERGY, kPairDH>;
}
inline TileKernel tile_kernel(bool mixed, bool energy, int kind)
{
    if(mixed) {return energy ? tile_kernel<true, true>(kind) : tile_kernel<true, false>(kind);}
    return energy ? tile_kernel<false, true>(kind) : tile_kernel<false, false>(kind);
}

} // mjg
