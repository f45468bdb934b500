// Neighbour lists and the list-driven field kernels of the MPIDForce PME path.
//
// The solver applies the real-space dipole field operator once per iteration,
// so the pairs within the cutoff are found once per evaluation and kept as a
// full (both directions) per-atom list.  Each atom then sums only its own
// field: no atomics per pair, no second pass over pair slots that fail the
// cutoff, and the same list serves the permanent-field pass.
//
// Construction, all in the Morton-sorted order of the atoms:
//   1. block rows: for every 64-atom block I, the blocks J whose bounding
//      boxes come within the cutoff (both J < I and J >= I), in ascending J;
//   2. neighbour masks: one wavefront per block pair (I, J >= I) tests each
//      pair once and writes the 64-bit masks of both directions (the second
//      by a bit-matrix transpose), skipping self pairs and scaled covalent
//      partners (those pairs go to the covalent-pair kernels);
//   3. atom lists: lane i of block I walks its row in ascending J and appends
//      the atoms of each mask.
// Both steps are deterministic, so the summation order of every field is.
// The solver needs fields at polarisable sites only: an atom without
// polarisability carries no induced dipole (mu = S y with S = 0) and its
// row of the solver's operator is multiplied by S = 0.  An evaluation
// therefore lists the polarisable atoms only, each with its full list (for
// the permanent field) and a list of its polarisable neighbours (for the
// solver's operator); the inspection entry points, which want fields at
// every atom, ask for full lists of all atoms.
//
// List layout: entry k of list row l sits at ((k / S) * rows + l) * S + k % S
// with S = kNlSplit, so the S threads that share an atom read S adjacent
// words and a wavefront reads 64 consecutive words per step.
#include "pair_math.h"

namespace mpid {

__device__ __forceinline__ size_t nl_index(int l, int k, int rows) {
    return ((size_t)(k / kNlSplit) * rows + l) * kNlSplit + (k % kNlSplit);
}

// Whether an axis-aligned box of half-widths h, centred at separation d
// from a point, comes within rc of that point under some periodic image:
// the point-to-box gap of every image is at most the distance between any
// point of the box and the given point, so a pair within rc passes.  A
// rectangular cell wraps each axis alone.  A triclinic cell (reduced form)
// tries every lattice shift k c + j b + i a that brings the z, then the y,
// then the x separation within rc + h (one shift more on each side for the
// float rounding of the bounds); such a shift exists for any pair within rc,
// whichever image the pair's own minimum image picks.
__device__ __forceinline__ bool gap_within(float dx, float dy, float dz, float hx, float hy, float hz,
                                           const Box<float>& box, float rc) {
    const float rc2 = rc * rc;
    if (box.bx == 0.f && box.cx == 0.f && box.cy == 0.f) {
        const float d[3] = {dx, dy, dz}, h[3] = {hx, hy, hz};
        float d2 = 0.f;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const float dk = d[k] - box.L[k] * floorf(d[k] * box.inv[k] + 0.5f);
            const float g = fmaxf(0.f, fabsf(dk) - h[k]);
            d2 += g * g;
        }
        return d2 <= rc2;
    }
    const V3<float> d = min_image(mk(dx, dy, dz), box);
    const int k0 = (int)floorf((-rc - hz - d.z) * box.inv[2]) - 1, k1 = (int)ceilf((rc + hz - d.z) * box.inv[2]) + 1;
    for (int k = k0; k <= k1; k++) {
        const float z = d.z + (float)k * box.L[2];
        const float gz = fmaxf(0.f, fabsf(z) - hz);
        if (gz * gz > rc2) continue;
        const float y0 = d.y + (float)k * box.cy, x0 = d.x + (float)k * box.cx;
        const int j0 = (int)floorf((-rc - hy - y0) * box.inv[1]) - 1, j1 = (int)ceilf((rc + hy - y0) * box.inv[1]) + 1;
        for (int j = j0; j <= j1; j++) {
            const float y = y0 + (float)j * box.L[1];
            const float gy = fmaxf(0.f, fabsf(y) - hy);
            if (gz * gz + gy * gy > rc2) continue;
            const float x1 = x0 + (float)j * box.bx;
            const int i0 = (int)floorf((-rc - hx - x1) * box.inv[0]) - 1,
                      i1 = (int)ceilf((rc + hx - x1) * box.inv[0]) + 1;
            for (int i = i0; i <= i1; i++) {
                const float gx = fmaxf(0.f, fabsf(x1 + (float)i * box.L[0]) - hx);
                if (gz * gz + gy * gy + gx * gx <= rc2) return true;
            }
        }
    }
    return false;
}

// Bounding boxes of blocks I and J within the cutoff (the gap test above on
// the separation of the box centres with the summed half-widths, with a
// little slack for the float rounding of the bounds).
__device__ __forceinline__ bool blocks_within(float4 a0, float4 a1, float4 b0, float4 b1, const Box<float>& box,
                                              float cutoff) {
    const float rc = cutoff * 1.0001f + 1e-5f;
    return gap_within(0.5f * (b0.x + b1.x) - 0.5f * (a0.x + a1.x), 0.5f * (b0.y + b1.y) - 0.5f * (a0.y + a1.y),
                      0.5f * (b0.z + b1.z) - 0.5f * (a0.z + a1.z), 0.5f * (a1.x - a0.x) + 0.5f * (b1.x - b0.x),
                      0.5f * (a1.y - a0.y) + 0.5f * (b1.y - b0.y), 0.5f * (a1.z - a0.z) + 0.5f * (b1.z - b0.z), box,
                      rc);
}

// One wavefront per block I.  Count mode (rows == nullptr) writes counts[I]
// and upper[I], the number of those blocks J with J >= I; fill mode writes
// the row at rows[start[I] ...] in ascending J, and I into owner[] at the
// same positions; *nact takes the number of entries with J >= I (ustart[nb]),
// or 0 when the rows overflow their capacity.
__global__ __launch_bounds__(64) void k_block_rows(int nb, const float4* __restrict__ bmin,
                                                   const float4* __restrict__ bmax, Box<float> box, float cutoff,
                                                   const int* __restrict__ start, int* __restrict__ counts,
                                                   int* __restrict__ upper, int* __restrict__ rows,
                                                   int* __restrict__ owner, int cap, const int* __restrict__ ustart,
                                                   int* __restrict__ nact) {
    const int I = blockIdx.x, lane = threadIdx.x;
    const float4 a0 = bmin[I], a1 = bmax[I];
    const int base = rows ? start[I] : 0;
    int c = 0, cu = 0;
    for (int J0 = 0; J0 < nb; J0 += kTile) {
        const int J = J0 + lane;
        const bool hit = J < nb && blocks_within(a0, a1, bmin[J], bmax[J], box, cutoff);
        const unsigned long long m = __ballot(hit);
        if (hit && rows) {
            const int at = base + c + __popcll(m & ((1ull << lane) - 1ull));
            if (at < cap) {  // entries beyond the capacity: the host grows it and builds again
                rows[at] = J;
                owner[at] = I;
            }
        }
        c += __popcll(m);
        cu += __popcll(__ballot(hit && J >= I));
    }
    if (lane == 0 && !rows) {
        counts[I] = c;
        upper[I] = cu;
    }
    if (rows && I == 0 && lane == 0) *nact = start[nb] <= cap ? ustart[nb] : 0;
}

// Exclusive scans, one workgroup each: start[k] = counts[0] + ... +
// counts[k-1] for k = 0..m.  The first one's total also goes to *total.
struct Scans {
    const int* counts[3];
    int* start[3];
};
__global__ __launch_bounds__(1024) void k_exclusive_scans(int m, Scans sc, int* total) {
    __shared__ int part[1024];
    const int* __restrict__ counts = sc.counts[blockIdx.x];
    int* __restrict__ start = sc.start[blockIdx.x];
    const int t = threadIdx.x;
    const int per = (m + 1023) / 1024;
    const int b = min(t * per, m), e = min(b + per, m);
    int s = 0;
    for (int k = b; k < e; k++) s += counts[k];
    part[t] = s;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const int v = t >= off ? part[t - off] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    int run = t ? part[t - 1] : 0;
    for (int k = b; k < e; k++) {
        start[k] = run;
        run += counts[k];
    }
    if (t == 1023) {
        start[m] = part[1023];
        if (blockIdx.x == 0) *total = part[1023];
    }
}

// At most kOneRows blocks: counting, the three scans and the rows in one
// workgroup (the boxes and the hit masks stay in LDS, so each block pair is
// tested once): 6 us at 11 blocks against 20-25 us for the two passes and the
// scans as three dependent dispatches.  At 192 blocks one CU needs 45 us for
// the 36,864 tests, so that larger systems take the three.
__global__ __launch_bounds__(1024) void k_block_rows_one(int nb, const float4* __restrict__ bmin,
                                                         const float4* __restrict__ bmax, Box<float> box, float cutoff,
                                                         const int* __restrict__ polcnt, int* __restrict__ start,
                                                         int* __restrict__ ustart, int* __restrict__ polstart,
                                                         int* __restrict__ rows, int* __restrict__ owner, int cap,
                                                         int* total, int* __restrict__ nact) {
    constexpr int kWords = kOneRows / kTile;
    __shared__ float4 s0[kOneRows], s1[kOneRows];
    __shared__ unsigned long long hit[kOneRows][kWords];
    __shared__ int cnt[3][kOneRows];  // entries, entries with J >= I, polarisable atoms: then inclusive sums
    const int lane = threadIdx.x & (kTile - 1), w = threadIdx.x / kTile;
    for (int k = threadIdx.x; k < nb; k += 1024) {
        s0[k] = bmin[k];
        s1[k] = bmax[k];
    }
    if (threadIdx.x < kOneRows) cnt[2][threadIdx.x] = (int)threadIdx.x < nb ? polcnt[threadIdx.x] : 0;
    __syncthreads();
    for (int I = w; I < kOneRows; I += 1024 / kTile) {
        int c = 0, cu = 0;
        if (I < nb) {
            const float4 a0 = s0[I], a1 = s1[I];
            for (int J0 = 0; J0 < nb; J0 += kTile) {
                const int J = J0 + lane;
                const bool h = J < nb && blocks_within(a0, a1, s0[min(J, nb - 1)], s1[min(J, nb - 1)], box, cutoff);
                const unsigned long long m = __ballot(h);
                c += __popcll(m);
                cu += __popcll(__ballot(h && J >= I));
                if (lane == 0) hit[I][J0 / kTile] = m;
            }
        }
        if (lane == 0) {
            cnt[0][I] = c;
            cnt[1][I] = cu;
        }
    }
    __syncthreads();
    for (int off = 1; off < kOneRows; off <<= 1) {
        int v[3] = {0, 0, 0};
        const int t = threadIdx.x;
        if (t < kOneRows && t >= off)
            for (int q = 0; q < 3; q++) v[q] = cnt[q][t - off];
        __syncthreads();
        if (t < kOneRows)
            for (int q = 0; q < 3; q++) cnt[q][t] += v[q];
        __syncthreads();
    }
    if ((int)threadIdx.x <= nb) {
        const int t = threadIdx.x;
        start[t] = t ? cnt[0][t - 1] : 0;
        ustart[t] = t ? cnt[1][t - 1] : 0;
        polstart[t] = t ? cnt[2][t - 1] : 0;
        if (t == nb) {
            *total = cnt[0][nb - 1];
            *nact = cnt[0][nb - 1] <= cap ? cnt[1][nb - 1] : 0;
        }
    }
    for (int I = w; I < nb; I += 1024 / kTile) {
        int at = I ? cnt[0][I - 1] : 0;
        for (int J0 = 0; J0 < nb; J0 += kTile) {
            const unsigned long long m = hit[I][J0 / kTile];
            const int k = at + __popcll(m & ((1ull << lane) - 1ull));
            if (((m >> lane) & 1ull) && k < cap) {  // entries beyond the capacity: the host grows it and builds again
                rows[k] = J0 + lane;
                owner[k] = I;
            }
            at += __popcll(m);
        }
    }
}

// Phase 1 of the atom lists, one wavefront per row entry r = (I, J), J >= I
// (entries with J < I return): lane i of block I tests the atoms of J (FP64
// distances, the test of the reference: r2 > cutoff^2 is out), skipping
// itself and its scaled covalent partners (those pairs go to the
// covalent-pair kernels), and writes the 64-bit neighbour mask of i within J
// to nmask[r * 64 + lane].  For J > I the masks of J's atoms within I (one
// ballot per tested atom) go to the mirrored entry (J, I) of J's row; the
// block-box test is symmetric, so that entry exists (if not, flag[0] is set
// and the host raises an error).
//
// One workgroup of W wavefronts per entry; each tests every W-th atom of J
// against the 64 of I.  A ballot per tested atom, kept in LDS, gives its
// pairs (j > i); a scan of their counts places them in the tile's pair list by
// class (TileList, kernels_pairs.hip).  (The electrostatics kernel used to rank
// the masks' bits itself, one lane per row i stepping through its set bits:
// 44% of that kernel's instructions.)  A tile is a chain over the tested atoms:
// four wavefronts shorten it where there are few tiles (81 atoms: 18 us with
// one, 9 with four), and repeat the setup and the scan where there are many
// (98,304 atoms: 160 us with one, 349 with four; 12,288 atoms are even).
// Evaluations with direct polarization, four and one: 1,111 tiles 215 and 221 us,
// 3,292 268 and 274, 9,892 335 both, 17,000 442 and 419.  (The line is taken on the
// row entries launched: the capacity while the count of the build is pending.)
constexpr int kOneWaveRows = 16384;  // row entries (twice the tiles)
template <int W>
__global__ __launch_bounds__(W * kTile) void k_nl_masks(int n, const int* __restrict__ rstart, const int* __restrict__ rows,
                                                 const int* __restrict__ owner, const float4* __restrict__ bmin,
                                                 const float4* __restrict__ bmax, const double4* __restrict__ pos,
                                                 const int* __restrict__ partners, const int* __restrict__ npart,
                                                 int pstride, Box<double> box, double rc2,
                                                 const unsigned long long* __restrict__ bmask,
                                                 unsigned long long* __restrict__ nmask,
                                                 int* __restrict__ flag, int cap, int4* __restrict__ act,
                                                 unsigned short* __restrict__ plist, int tcap,
                                                 int2* __restrict__ groups, int group,
                                                 const int* __restrict__ ustart) {
    __shared__ double4 sp[kTile];
    __shared__ unsigned long long shits[kTile];             // [atom of J]: the atoms of I within the cutoff
    __shared__ unsigned long long sm[W][kTile];             // [][atom of I]: a wavefront's part of its mask
    const int r = blockIdx.x, lane = threadIdx.x & (kTile - 1), wave = threadIdx.x / kTile;
    const int nbk = (n + kTile - 1) / kTile;
    if (r >= min(rstart[nbk], cap)) return;  // uniform: the grid may cover the capacity, not the count
    const int I = owner[r], J = rows[r];
    if (J < I) return;  // uniform: written by the mirrored entry
    const int i = I * kTile + lane, j = J * kTile + lane;
    const bool iv = i < n, jv = j < n;
    const int ic = iv ? i : n - 1, jc = jv ? j : n - 1;
    const double4 pi = pos[ic], pj = pos[jc];
    const unsigned long long ibare = bmask[I], jbare = bmask[J];
    if (wave == 0) {
        sp[lane] = pj;
        shits[lane] = 0ull;
    }
    // candidates: atoms of J whose distance to block I's box is within the
    // cutoff (minimum image; never rejects a pair within the cutoff)
    bool cand;
    // A rectangular cell's pairs within the cutoff all take the image that
    // brings the blocks' centres nearest, if |centre distance| + half widths
    // stays below L - cutoff on every axis (another image of the pair is then
    // farther than the cutoff): the image is subtracted once, which leaves a
    // third of the instructions of a tested atom (98,304 atoms:
    // 200 to 160 us beside the spreading).
    bool one_image = box.bx == 0.0 && box.cx == 0.0 && box.cy == 0.0;
    double si[3] = {pi.x, pi.y, pi.z};  // this lane's atom in the image nearest to J
    {
        const float4 b0 = bmin[I], b1 = bmax[I], j0 = bmin[J], j1 = bmax[J];
        const float jlo[3] = {j0.x, j0.y, j0.z}, jhi[3] = {j1.x, j1.y, j1.z};
        const float cI[3] = {0.5f * (b0.x + b1.x), 0.5f * (b0.y + b1.y), 0.5f * (b0.z + b1.z)};
        const float hI[3] = {0.5f * (b1.x - b0.x), 0.5f * (b1.y - b0.y), 0.5f * (b1.z - b0.z)};
        const float rcf = sqrtf((float)rc2) * 1.0001f + 1e-5f;
        Box<float> fb;
        for (int k = 0; k < 3; k++) {
            fb.L[k] = (float)box.L[k];
            fb.inv[k] = (float)box.inv[k];
        }
        fb.bx = (float)box.bx;
        fb.cx = (float)box.cx;
        fb.cy = (float)box.cy;
        for (int k = 0; k < 3; k++) {
            const double d = 0.5 * ((double)jlo[k] + (double)jhi[k]) - (double)cI[k];
            const double s = floor(d * box.inv[k] + 0.5) * box.L[k];
            one_image = one_image && fabs(d - s) + (double)hI[k] + 0.5 * ((double)jhi[k] - (double)jlo[k]) <
                                         box.L[k] - (double)rcf - 1e-4;
            si[k] += s;
        }
        cand = jv && gap_within((float)pj.x - cI[0], (float)pj.y - cI[1], (float)pj.z - cI[2], hI[0], hI[1], hI[2],
                                fb, rcf);
    }
    const unsigned long long cmask = __ballot(cand);
    unsigned long long skip = J == I ? 1ull << lane : 0ull;
    const int np = iv ? npart[ic] : 0;
    const int* parts = partners + (size_t)ic * pstride;
    for (int k = 0; k < np; k++) {
        const int p = parts[k] >> 2;
        if ((p >> 6) == J) skip |= 1ull << (p & 63);
    }
    __syncthreads();
    // the tile's entry in the electrostatics kernels' work list: the row
    // entries J >= I of row I are its last upper[I] entries, placed at
    // ustart[I] (the exclusive scan of upper) in the same order.  When the rows
    // exceed their capacity, the stored ones can hold more such entries than
    // the tile list: those have no tile, but their masks and the mirrored ones
    // are written all the same, since k_nl_fill reads the mask of every stored
    // row entry (the host then builds again).
    const int u = ustart[I + 1] - (rstart[I + 1] - r);
    const bool tile = u < tcap;  // uniform
    unsigned short* list = plist + (size_t)(tile ? u : 0) * kTilePairs;
    const unsigned long long below = (1ull << lane) - 1ull;
    const bool mine = ((ibare >> lane) & 1ull) != 0;  // this lane's atom of I is a bare charge
    const unsigned long long part = W == 4 ? cmask & (0x1111111111111111ull << wave) : cmask;
    unsigned long long m = 0;
    for (unsigned long long cm = part; cm;) {
        constexpr int kAhead = 4;  // distances formed at once
        unsigned long long bit[kAhead];
        int jj[kAhead];
        bool hit[kAhead];
#pragma unroll
        for (int k = 0; k < kAhead; k++) {
            bit[k] = cm & (0ull - cm);  // the lowest one left, or none
            jj[k] = __ffsll((long long)cm) - 1;
            cm &= cm - 1ull;
            const double4 q = sp[max(jj[k], 0)];
            V3<double> dr = mk(q.x - si[0], q.y - si[1], q.z - si[2]);
            if (!one_image) dr = min_image(mk(q.x - pi.x, q.y - pi.y, q.z - pi.z), box);  // uniform
            hit[k] = iv && dot(dr, dr) <= rc2 && (bit[k] & ~skip) != 0ull;
        }
#pragma unroll
        for (int k = 0; k < kAhead; k++) {
            const unsigned long long hits = __ballot(hit[k]);
            if (hit[k]) m |= bit[k];
            if (lane == 0 && bit[k]) shits[jj[k]] = hits;
        }
    }
    sm[wave][lane] = m;
    __syncthreads();
    // lane jj: the pairs of J's atom jj.  Those whose two sites are alike (both
    // bare, or neither) go to the front, two bare charges first; those with
    // one bare site to the back.
    const unsigned long long hits = shits[lane];
    const bool jb = ((jbare >> lane) & 1ull) != 0;
    const unsigned long long pairs = J > I ? hits : hits & below;  // j > i
    const unsigned long long alike = jb ? pairs & ibare : pairs & ~ibare, mixed = pairs & ~alike;
    const int na = __popcll(alike), nm = __popcll(mixed);
    int front = jb ? na : na << 16, back = nm;  // scans: two bare | general << 16, one bare
#pragma unroll
    for (int off = 1; off < kTile; off <<= 1) {
        const int f = __shfl_up(front, off), k = __shfl_up(back, off);
        if (lane >= off) {
            front += f;
            back += k;
        }
    }
    const int totals = __builtin_amdgcn_readlane(front, kTile - 1);
    const int ncc = totals & 0xffff, nup = ncc + (int)((unsigned)totals >> 16);
    const int none = __builtin_amdgcn_readlane(back, kTile - 1);
    front = jb ? (front & 0xffff) - na : ncc + (int)((unsigned)front >> 16) - na;
    back = kTilePairs - 1 - (back - nm);
    const unsigned long long own = (mine ? ibare : ~ibare) & below;  // this lane's class, the atoms before it
    // the entry without its atom of J, for a bare one and for another one there
    const int ent = lane << 8, ent_bare = ent, ent_other = mine ? ent | 0x8000 : ent;
    for (unsigned long long cm = tile ? part : 0ull; cm; cm &= cm - 1ull) {
        const int jj = __ffsll((long long)cm) - 1;  // uniform
        const unsigned lo = __builtin_amdgcn_readlane((unsigned)pairs, jj);
        const unsigned hi = __builtin_amdgcn_readlane((unsigned)(pairs >> 32), jj);
        const unsigned long long all = ((unsigned long long)hi << 32) | lo;
        const bool jbb = ((jbare >> jj) & 1ull) != 0, same = mine == jbb;
        const int f = __builtin_amdgcn_readlane(front, jj), k = __builtin_amdgcn_readlane(back, jj);
        const int rank = __popcll(all & own);
        if ((all >> lane) & 1ull)
            list[same ? f + rank : k - rank] = (unsigned short)((jbb ? ent_bare : ent_other) | jj);
    }
    if (wave != 0) return;
    m = 0;
#pragma unroll
    for (int w = 0; w < W; w++) m |= sm[w][lane];
    nmask[(size_t)r * kTile + lane] = m;
    if (tile && lane == 0) {
        act[u] = make_int4(ncc | ((nup - ncc) << 16), I, J, none);
        if (group > 1) {
            const int u0 = ustart[I], u1 = ustart[I + 1], slot = u0 / group + I, k = u - u0;
            if (k % group == 0) groups[slot + k / group] = make_int2(u, min(group, u1 - u));
            if (u + 1 == u1)  // the row's slot that it does not need, if there is one
                for (int s = slot + (u1 - u0 + group - 1) / group; s <= u1 / group + I; s++) groups[s] = make_int2(0, 0);
        }
    }
    if (J > I) {
        // the mirrored entry: I in the ascending row of J
        int lo = min(rstart[J], cap), hi = min(rstart[J + 1], cap) - 1;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (rows[mid] < I) lo = mid + 1;
            else hi = mid;
        }
        if (lo <= hi && rows[lo] == I) nmask[(size_t)lo * kTile + lane] = hits;
        else if (lane == 0) atomicOr(flag, 1);
    }
}

// Phase 2, one workgroup of kFillWaves wavefronts per block I: the row of I
// is cut into kFillWaves contiguous chunks in ascending J.  Each wavefront
// counts its chunk's entries per atom, and a prefix over the chunks gives
// each its offsets.  The entries are then written atom by atom: for each
// row entry, the wavefront takes in turn each stored atom whose mask is not
// empty, and lane jj writes neighbour jj at the atom's offset plus the
// number of mask bits below jj (all lanes work; a lane-per-atom walk over
// the mask bits would idle the lanes of non-stored atoms and of short
// masks).  all != 0: the full list of every atom, stored by atom index.
// all == 0: for the polarisable atoms only, the full list and the list of
// polarisable neighbours (polmask of the neighbour's block), stored by the
// atom's position p in the sorted index of polarisable atoms
// (p = polstart[I] + rank in the block, npol = polstart[nb] rows).
// count[i] (and pcount[i] when all == 0) are stored for every atom.  Entries
// beyond cap are counted but not stored; maxcount takes the largest stored
// list's length, and the host grows the lists and rebuilds.
constexpr int kFillWaves = 16;
__global__ __launch_bounds__(kFillWaves * kTile) void k_nl_fill(
    int n, int all, const int* __restrict__ rstart, const int* __restrict__ rows,
    const unsigned long long* __restrict__ polmask, const int* __restrict__ polstart,
    const unsigned long long* __restrict__ nmask, int cap, int* __restrict__ nbr, int* __restrict__ count,
    int* __restrict__ maxcount, int* __restrict__ pnbr, int* __restrict__ pcount, int rcap, int* __restrict__ pol_idx,
    int ntiles, const int* __restrict__ tstart, int* __restrict__ tpstart) {
    __shared__ int scnt[kFillWaves][kTile], spcnt[kFillWaves][kTile];
    const int I = blockIdx.x, lane = threadIdx.x & (kTile - 1), w = threadIdx.x / kTile;
    const int nb = (n + kTile - 1) / kTile;
    const int i = I * kTile + lane;
    const bool iv = i < n;
    const unsigned long long pmI = polmask[I];
    const bool ipol = ((pmI >> lane) & 1ull) != 0;
    const bool store = iv && (all || ipol);
    const int li = all ? i : polstart[I] + __popcll(pmI & ((1ull << lane) - 1ull));
    const int nrows = all ? n : polstart[nb];
    // the sorted index of the polarisable atoms, and its spreading tiles: a
    // tile's first polarisable atom is the first one at or after its first atom
    if (w == 0 && ipol) pol_idx[polstart[I] + __popcll(pmI & ((1ull << lane) - 1ull))] = i;
    if (tpstart)
        for (int t = I * kFillWaves * kTile + threadIdx.x; t <= ntiles; t += nb * kFillWaves * kTile) {
            const int f = tstart[t], B = f / kTile;
            tpstart[t] = B >= nb ? polstart[nb]
                                 : polstart[B] + __popcll(polmask[B] & ((1ull << (f & (kTile - 1))) - 1ull));
        }
    // (rows beyond the capacity rcap were not stored; the host grows it and builds again)
    const int r0 = min(rstart[I], rcap), r1 = min(rstart[I + 1], rcap);
    const int per = (r1 - r0 + kFillWaves - 1) / kFillWaves;
    const int a = min(r0 + w * per, r1), b = min(a + per, r1);
    int c = 0, pc = 0;
    for (int r = a; r < b; r++) {
        const unsigned long long m = iv ? nmask[(size_t)r * kTile + lane] : 0ull;
        c += __popcll(m);
        pc += __popcll(m & polmask[rows[r]]);
    }
    scnt[w][lane] = c;
    spcnt[w][lane] = pc;
    __syncthreads();
    int cnt = 0, pcnt = 0, tot = 0, ptot = 0;
    for (int v = 0; v < kFillWaves; v++) {
        if (v == w) {
            cnt = tot;
            pcnt = ptot;
        }
        tot += scnt[v][lane];
        ptot += spcnt[v][lane];
    }
    const unsigned long long below = (1ull << lane) - 1ull;  // mask bits of the lanes below this one
    for (int r = a; r < b; r++) {
        const unsigned long long mrow = iv ? nmask[(size_t)r * kTile + lane] : 0ull;
        const int J = rows[r];
        const unsigned long long polJ = all ? 0ull : polmask[J];
        unsigned long long act = __ballot(store && mrow != 0ull);
        while (act) {
            const int t = __ffsll((long long)act) - 1;  // uniform: the atom of lane t
            act &= act - 1ull;
            const unsigned lo = __builtin_amdgcn_readlane((unsigned)mrow, t);
            const unsigned hi = __builtin_amdgcn_readlane((unsigned)(mrow >> 32), t);
            const unsigned long long m = ((unsigned long long)hi << 32) | lo;
            const int base = __builtin_amdgcn_readlane(cnt, t);
            const int lt = __builtin_amdgcn_readlane(li, t);
            if ((m >> lane) & 1ull) {
                const int k = base + __popcll(m & below);
                if (k < cap) nbr[nl_index(lt, k, nrows)] = J * kTile + lane;
            }
            const unsigned long long mp = m & polJ;
            if (!all) {
                const int pbase = __builtin_amdgcn_readlane(pcnt, t);
                if ((mp >> lane) & 1ull) {
                    const int k = pbase + __popcll(mp & below);
                    if (k < cap) pnbr[nl_index(lt, k, nrows)] = J * kTile + lane;
                }
            }
            if (lane == t) {
                cnt += __popcll(m);
                pcnt += __popcll(mp);
            }
        }
    }
    if (w == 0) {
        if (iv) {
            count[i] = min(tot, cap);
            if (!all) pcount[i] = min(ptot, cap);
        }
        // the block's longest list, then one atomic per block (atomics from
        // every lane on one word serialise across the chip)
        int lmax = store ? tot : 0;
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) lmax = max(lmax, __shfl_xor(lmax, off));
        if (lane == 0 && lmax > 0) atomicMax(maxcount, lmax);
    }
}

// ---------------------------------------------------------------------------
// list-driven field kernels: kNlSplit threads per atom, each taking every
// kNlSplit-th entry; the partial fields meet in a lane reduction and are
// added once per atom.
// ---------------------------------------------------------------------------
template <class R>
__global__ __launch_bounds__(256) void k_nl_fixed_field(NbrList L, const int* __restrict__ atoms, int natoms,
                                                        PairAtoms<R> A, PairParams<R> P, acc_t* __restrict__ field) {
    const unsigned g = blockIdx.x * blockDim.x + threadIdx.x;
    const int t = (int)(g / kNlSplit), sub = (int)(g % kNlSplit);
    const int n = P.n;
    const bool iv = t < natoms;
    const int i = atoms ? atoms[iv ? t : natoms - 1] : (iv ? t : n - 1);
    const int ic = i;
    const R4<R> pi = A.pos[ic];
    const R2<R> tdi = A.td[ic];
    R mi[kMP];
#pragma unroll
    for (int k = 0; k < kMP; k++) mi[k] = A.lab[(size_t)ic * kMP + k];
    const int cnt = iv ? L.count[ic] : 0;
    // entry k of atom i: lp advances by n * kNlSplit per step of kNlSplit
    // lists of an atoms index are stored by position in the index
    const int li = atoms ? (iv ? t : natoms - 1) : ic;
    const int* lp = L.nbr + (size_t)li * kNlSplit + sub;
    const size_t stride = (size_t)(atoms ? natoms : n) * kNlSplit;
    int jn = sub < cnt ? lp[0] : 0;
    R ex = 0, ey = 0, ez = 0;
    for (int k = sub; k < cnt; k += kNlSplit) {
        const int j = jn;
        lp += stride;
        if (k + kNlSplit < cnt) jn = *lp;  // next index in flight during this pair
        const R4<R> pj = A.pos[j];
        const V3<R> dr = min_image(mk(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z), P.box);
        R mj[kMP];
#pragma unroll
        for (int c = 0; c < kMP; c++) mj[c] = A.lab[(size_t)j * kMP + c];
        // listed pairs are not covalent partners: scale 1, default Thole width
        const FixedRadial<R> gr = fixed_field_radial<R>(dot(dr, dr), tdi, R2<R>{R(0), pj.w}, R(1), P);
        const V3<R> fi = fixed_field_from<R>(mj, dr, gr);
        ex += fi.x;
        ey += fi.y;
        ez += fi.z;
    }
#pragma unroll
    for (int off = 1; off < kNlSplit; off <<= 1) {
        ex += __shfl_xor(ex, off);
        ey += __shfl_xor(ey, off);
        ez += __shfl_xor(ez, off);
    }
    if (iv && sub == 0) {
        acc_add(&field[3 * (size_t)i + 0], ex);
        acc_add(&field[3 * (size_t)i + 1], ey);
        acc_add(&field[3 * (size_t)i + 2], ez);
    }
}

template <class R>
__global__ __launch_bounds__(256) void k_nl_induced_field(NbrList L, const int* __restrict__ atoms, int natoms,
                                                          PairAtoms<R> A, const R* __restrict__ mu, PairParams<R> P,
                                                          acc_t* __restrict__ field) {
    const unsigned g = (unsigned)xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    const int t = (int)(g / kNlSplit), sub = (int)(g % kNlSplit);
    const int n = P.n;
    const bool iv = t < natoms;
    const int i = atoms ? atoms[iv ? t : natoms - 1] : (iv ? t : n - 1);
    const int ic = i;
    const R4<R> pi = A.pos[ic];
    const int cnt = iv ? L.count[ic] : 0;
    // lists of an atoms index are stored by position in the index
    const int li = atoms ? (iv ? t : natoms - 1) : ic;
    const int* lp = L.nbr + (size_t)li * kNlSplit + sub;
    const size_t stride = (size_t)(atoms ? natoms : n) * kNlSplit;
    int jn = sub < cnt ? lp[0] : 0;
    R ex = 0, ey = 0, ez = 0;
    for (int k = sub; k < cnt; k += kNlSplit) {
        const int j = jn;
        lp += stride;
        if (k + kNlSplit < cnt) jn = *lp;
        const R4<R> pj = A.pos[j];
        const V3<R> dr = min_image(mk(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z), P.box);
        const V3<R> uj = mk(mu[3 * (size_t)j], mu[3 * (size_t)j + 1], mu[3 * (size_t)j + 2]);
        // listed pairs are not covalent partners: polarization scale 1, default Thole width
        const V3<R> fi =
            induced_field_from<R>(uj, dr, induced_field_radial<R>(dot(dr, dr), pi.w, pj.w, P.default_thole, P));
        ex += fi.x;
        ey += fi.y;
        ez += fi.z;
    }
#pragma unroll
    for (int off = 1; off < kNlSplit; off <<= 1) {
        ex += __shfl_xor(ex, off);
        ey += __shfl_xor(ey, off);
        ez += __shfl_xor(ez, off);
    }
    if (iv && sub == 0) {
        acc_add(&field[3 * (size_t)i + 0], ex);
        acc_add(&field[3 * (size_t)i + 1], ey);
        acc_add(&field[3 * (size_t)i + 2], ez);
    }
}

// Thole damping derivatives of the energy gradients: h = u dE/du of each
// listed pair of polarisable sites (thole_u_derivative; listed pairs are not
// covalent partners: polarization scale 1, default Thole width), summed over
// the atom's polarisable neighbours into hd[i] and hdef[i].  Each pair is
// visited from both of its atoms.
template <class R>
__global__ __launch_bounds__(256) void k_nl_thole(NbrList L, const int* __restrict__ atoms, int natoms, PairAtoms<R> A,
                                                  const R* __restrict__ mu, PairParams<R> P, acc_t* __restrict__ hd,
                                                  acc_t* __restrict__ hdef) {
    const unsigned g = blockIdx.x * blockDim.x + threadIdx.x;
    const int t = (int)(g / kNlSplit), sub = (int)(g % kNlSplit);
    const bool iv = t < natoms;
    const int i = atoms[iv ? t : natoms - 1];
    const R4<R> pi = A.pos[i];
    R mi[kMP];
#pragma unroll
    for (int k = 0; k < kMP; k++) mi[k] = A.lab[(size_t)i * kMP + k];
    const V3<R> ui = mk(mu[3 * (size_t)i], mu[3 * (size_t)i + 1], mu[3 * (size_t)i + 2]);
    const int cnt = iv ? L.count[i] : 0;
    const int* lp = L.nbr + (size_t)(iv ? t : natoms - 1) * kNlSplit + sub;
    const size_t stride = (size_t)natoms * kNlSplit;
    int jn = sub < cnt ? lp[0] : 0;
    R h = 0;
    for (int k = sub; k < cnt; k += kNlSplit) {
        const int j = jn;
        lp += stride;
        if (k + kNlSplit < cnt) jn = *lp;
        const R4<R> pj = A.pos[j];
        const V3<R> dr = min_image(mk(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z), P.box);
        R mj[kMP];
#pragma unroll
        for (int c = 0; c < kMP; c++) mj[c] = A.lab[(size_t)j * kMP + c];
        const V3<R> uj = mk(mu[3 * (size_t)j], mu[3 * (size_t)j + 1], mu[3 * (size_t)j + 2]);
        h += thole_u_derivative<R>(dr, dot(dr, dr), mi, mj, ui, uj, pi.w, pj.w, P.default_thole, R(1), P.mutual != 0);
    }
#pragma unroll
    for (int off = 1; off < kNlSplit; off <<= 1) h += __shfl_xor(h, off);
    if (iv && sub == 0 && h != R(0)) {
        acc_add(&hd[i], h);
        acc_add(&hdef[i], h);
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
void launch_block_rows(hipStream_t s, int nb, const float4* bmin, const float4* bmax, Box<float> box, float cutoff,
                       const int* polcnt, int* work, int* start, int* ustart, int* polstart, int* rows, int* owner,
                       int cap, int* total, int* nact) {
    if (nb <= kOneRows) {
        hipLaunchKernelGGL(k_block_rows_one, dim3(1), dim3(1024), 0, s, nb, bmin, bmax, box, cutoff, polcnt, start,
                           ustart, polstart, rows, owner, cap, total, nact);
        return;
    }
    hipLaunchKernelGGL(k_block_rows, dim3(nb), dim3(kTile), 0, s, nb, bmin, bmax, box, cutoff, nullptr, work, work + nb,
                       nullptr, nullptr, 0, nullptr, nullptr);
    const Scans sc{{work, work + nb, polcnt}, {start, ustart, polstart}};
    hipLaunchKernelGGL(k_exclusive_scans, dim3(3), dim3(1024), 0, s, nb, sc, total);
    if (cap > 0)
        hipLaunchKernelGGL(k_block_rows, dim3(nb), dim3(kTile), 0, s, nb, bmin, bmax, box, cutoff, start, nullptr,
                           nullptr, rows, owner, cap, ustart, nact);
}
void launch_nl_build(hipStream_t s, int n, int nrows, int rcap, bool all, const int* rstart, const int* rows,
                     const int* owner, const float4* bmin, const float4* bmax, const double4* pos,
                     const int* partners, const int* npart, int pstride, Box<double> box, double rc2, int cap,
                     unsigned long long* nmask, const unsigned long long* polmask, const int* polstart, int* nbr,
                     int* count, int* scalars, int* pnbr, int* pcount, const unsigned long long* bmask, int4* act,
                     unsigned short* plist, int tcap, int2* groups, int group, const int* ustart, int* pol_idx, int ntiles,
                     const int* tstart, int* tpstart) {
    const int nb = (n + kTile - 1) / kTile;
    if (nrows > 0) {
        const bool one = nrows > kOneWaveRows;
        hipLaunchKernelGGL((one ? &k_nl_masks<1> : &k_nl_masks<4>), dim3(nrows), dim3(one ? kTile : 4 * kTile), 0, s, n,
                           rstart, rows, owner, bmin, bmax, pos, partners, npart, pstride, box, rc2, bmask, nmask,
                           scalars + 1, rcap, act, plist, tcap, groups, group, ustart);
    }
    hipLaunchKernelGGL(k_nl_fill, dim3(nb), dim3(kFillWaves * kTile), 0, s, n, all ? 1 : 0, rstart, rows, polmask,
                       polstart, nmask, cap, nbr, count, scalars, pnbr, pcount, rcap, pol_idx, ntiles, tstart, tpstart);
}
template <class R>
void launch_nl_fixed_field(hipStream_t s, int natoms, const int* atoms, NbrList l, PairAtoms<R> a, PairParams<R> p,
                           acc_t* field) {
    if (natoms <= 0) return;
    const size_t threads = (size_t)natoms * kNlSplit;
    hipLaunchKernelGGL(k_nl_fixed_field<R>, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, l, atoms, natoms,
                       a, p, field);
}
template <class R>
void launch_nl_induced_field(hipStream_t s, int natoms, const int* atoms, NbrList l, PairAtoms<R> a, const R* mu,
                             PairParams<R> p, acc_t* field) {
    if (natoms <= 0) return;
    const size_t threads = (size_t)natoms * kNlSplit;
    hipLaunchKernelGGL(k_nl_induced_field<R>, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, l, atoms,
                       natoms, a, mu, p, field);
}

template <class R>
void launch_nl_thole(hipStream_t s, int natoms, const int* atoms, NbrList l, PairAtoms<R> a, const R* mu,
                     PairParams<R> p, acc_t* hd, acc_t* hdef) {
    if (natoms <= 0) return;
    const size_t threads = (size_t)natoms * kNlSplit;
    hipLaunchKernelGGL(k_nl_thole<R>, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, l, atoms, natoms, a,
                       mu, p, hd, hdef);
}

#define MPID_INSTANTIATE(R)                                                                                         \
    template void launch_nl_thole<R>(hipStream_t, int, const int*, NbrList, PairAtoms<R>, const R*, PairParams<R>,  \
                                     acc_t*, acc_t*);                                                              \
    template void launch_nl_fixed_field<R>(hipStream_t, int, const int*, NbrList, PairAtoms<R>, PairParams<R>,       \
                                           acc_t*);                                                                \
    template void launch_nl_induced_field<R>(hipStream_t, int, const int*, NbrList, PairAtoms<R>, const R*,          \
                                             PairParams<R>, acc_t*);
MPID_INSTANTIATE(float)
MPID_INSTANTIATE(double)
#undef MPID_INSTANTIATE

}  // namespace mpid
