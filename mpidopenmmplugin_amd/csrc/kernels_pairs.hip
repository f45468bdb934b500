// Real-space electrostatics (energy, forces, torques) of the MPIDForce PME
// path on gfx950, and the covalent-pair kernels.
//
// Atoms are sorted along a Morton curve and cut into blocks of 64 (one
// wavefront).  A tile is a pair of blocks (I, J >= I) whose bounding boxes
// come within the cutoff; the neighbour-list build leaves, for every tile, the
// list of its pairs within the cutoff that are not covalent partners, sorted
// into three classes (two bare charges, general, one bare charge; TileList).
// One workgroup (four wavefronts) owns a tile, or two of one block row, and its
// wavefronts take chunks of 64 entries of a class.  Every thread works on a pair
// inside the cutoff, whatever the tile's fill, and each class runs its own
// formula without divergence.  Both sides accumulate in LDS (atomic adds) and
// are flushed to the fixed-point global accumulators once per tile.
//
// The pair formulas are in pair_math.h (MPIDReferenceForce.cpp:4335-4920).
#include "pair_math.h"

#include <algorithm>

namespace mpid {

constexpr int kElecThreads = 256;  // four wavefronts share one workgroup's tiles

// kPot (the energy gradients): also the potential vectors dE/dm of every
// pair (20 stored lab components per atom, induced dipoles fixed) into pot;
// all_general: every pair takes the general formula, so that sites that are
// bare charges get all 20 components (else they get the charge one only).
// kGen: the general pairs too (else they are k_general_pairs').
//
// A workgroup takes `tiles` (at most kM) consecutive tiles of one block row.
// They share block I's side, which is staged and flushed once, and their lists
// are walked as one, so that a class leaves one partly filled chunk per group
// and not one per tile.  The chunks are claimed in turn, the longest formula
// first, and a chunk's entries are loaded while the one before is worked on.
//
// What bounds it: vector instructions (64% of the issue slots at 98,304 atoms
// in FP32; per pair about 210 for two bare charges, 400 with one, 1,600 for a
// general one) and the LDS adds beside them (43%); 128 registers and the LDS of
// four workgroups per CU keep four wavefronts per SIMD.  Times at 98,304 atoms,
// 20 million pairs: FP32 625 us with one tile and fixed roles per workgroup,
// 520 with two and claimed chunks (four tiles and 512 threads 677: two large
// workgroups per CU wait for their slowest wavefront); FP64, without the
// general pairs, 579 and 440 (one tile: two need the LDS of three blocks, three
// workgroups per CU, 497).
typedef int per_tile __attribute__((ext_vector_type(4)));  // (in registers, where the compiler kept arrays in memory)
template <class R, bool kPot> struct TileShape {
    static constexpr int kM = kPot ? 1 : sizeof(R) == 4 ? 2 : 1;  // tiles per workgroup
};
template <class R, bool kPot, bool kGen>
__device__ __forceinline__ void electrostatics_tiles(int tiles, const TileList& T,
                                                     const unsigned long long* __restrict__ bmask,
                                                     const PairAtoms<R>& A, const R* __restrict__ mu,
                                                     const PairParams<R>& P, const double4* __restrict__ pos64,
                                                     const double* __restrict__ lab64, const PairParams<double>& P64,
                                                     acc_t* __restrict__ force, acc_t* __restrict__ torque,
                                                     acc_t* __restrict__ energy, acc_t* __restrict__ pot,
                                                     int all_general) {
    constexpr int kM = TileShape<R, kPot>::kM, kT = kElecThreads;
    constexpr int kWaves = kT / kTile, kSides = 1 + kM;
    // Multipole rows of 20 reals, read as 16-byte vectors: with a 20-word
    // stride, 16 lanes reading 16 different rows cover each bank once.
    constexpr int kV = 16 / (int)sizeof(R);  // reals per 16-byte vector
    constexpr int kVA = kMP / kV;            // vectors per row
    typedef R vec __attribute__((ext_vector_type(kV)));
    // [side][component][atom], side 0: atoms of block I, 1 + t: atoms of tile
    // t's block J; components: force x, y, z, torque x, y, z.  FP64 in both
    // precisions (LDS atomic adds of doubles keep up on gfx950, those of
    // floats stall).
    __shared__ double acc[kSides][6][kTile];
    // potential vectors (kPot): [side][component][atom]
    __shared__ double pacc[kPot ? kSides : 1][kPot ? kMP : 1][kTile];
    __shared__ __align__(16) R smp[kSides][kTile * kMP];
    __shared__ R smu[kSides][kTile * 3];
    __shared__ R4<R> spos[kSides][kTile];  // x, y, z in the working precision, damping factor
    __shared__ int san[kSides][kTile];
    __shared__ double4 spos64[kSides][kTile];  // x, y, z, charge
    __shared__ double sen[kWaves];
    __shared__ int snext;
    const int tid = threadIdx.x, lane = tid & (kTile - 1), wave = tid / kTile;
    const int n = P.n;
    double en = 0.0;
    // this workgroup's tiles u .. u + nt - 1, of one block row (the launch
    // covers an upper bound of the list's length)
    const int nact = *T.nact;
    int u = blockIdx.x, nt = 1;
    if (tiles == 1) {
        if (u >= nact) return;
    } else {
        if (nact == 0 || u >= tile_groups(nact, P.n, tiles)) return;
        const int2 g = T.groups[u];
        u = g.x;
        nt = g.y;
        if (nt == 0) return;
    }
    // where each class of each tile starts in their common list: entry q of
    // tile t is at q + the tile's offset
    static_assert(kM <= 4, "one vector element per tile");
    per_tile J = -1, of = 0, pf = 0, og = 0, pg = 0, ob = 0, pb = 0;
    int nf = 0, ng = 0, nb = 0, front = 0;
    const int I = T.act[u].y;
#pragma unroll
    for (int t = 0; t < kM; t++) {
        const int4 e = t < nt ? T.act[u + t] : make_int4(0, 0, 0, 0);
        const int cc = e.x & 0xffff, gen = e.x >> 16;
        J[t] = cc + gen + e.w > 0 ? e.z : -1;
        pf[t] = t < nt ? nf : 0x7fffffff;
        of[t] = t * kTilePairs - nf;
        nf += cc + gen;
        pg[t] = t < nt ? ng : 0x7fffffff;
        og[t] = t * kTilePairs + cc - ng;
        ng += gen;
        pb[t] = t < nt ? nb : 0x7fffffff;
        ob[t] = t * kTilePairs + kTilePairs - 1 + nb;
        nb += e.w;
        front = cc + gen;
    }
    const unsigned short* list = T.list + (size_t)u * kTilePairs;
    if (kPot && all_general) {  // every pair is general (kM = 1: one tile)
        ng = front + nb;
        og[0] = 0;
        nf = ng;
        of[0] = 0;
        nb = 0;
    }
    if (nf + nb == 0) return;  // uniform
    const int cg = kGen ? (ng + kTile - 1) / kTile : 0;  // chunks: general,
    const int cb = cg + (nb + kTile - 1) / kTile;        // one bare charge,
    const int cf = cb + (nf + kTile - 1) / kTile;        // and the charge-charge channel
    // Within a chunk of 64 entries, lane l takes entry 8 (l mod 8) + l / 8:
    // entries of one atom are adjacent in the list, and spreading them
    // over the lanes keeps the atomic adds of one instruction off a common
    // address.
    const int perm = ((lane & 7) << 3) | (lane >> 3);
    // this lane's entry of chunk c: tile << 16 | the list's entry, or -1
    auto fetch = [&](int c) {
        if (c >= cf) return -1;  // uniform
        const int mg = c < cg ? -1 : 0, mb = c < cb ? ~mg : 0, mf = ~(mg | mb);
        const int q = (c - ((cg & mb) | (cb & mf))) * kTile + perm, last = ((ng & mg) | (nb & mb) | (nf & mf)) - 1;
        const int k = min(q, last);
        const per_tile start = (pg & mg) | (pb & mb) | (pf & mf), off = (og & mg) | (ob & mb) | (of & mf);
        int t = 0, o = off[0];
#pragma unroll
        for (int v = 1; v < kM; v++) {
            t = k >= start[v] ? v : t;
            o = k >= start[v] ? off[v] : o;
        }
        // One load at a selected place, not a load on each side of a branch:
        // with lanes on both sides, the compiler (ROCm 7.2) put the loops'
        // register spills ahead of the join's exec restore, and half the
        // lanes kept the loop counter of an earlier trip.
        int at = o + (mb ? -k : k);
        if (kPot && all_general) at = k < front ? k : kTilePairs - 1 - (k - front);
        const int e = list[at] & (kPot && all_general ? 0x7fff : 0xffff);
        return q <= last ? (t << 16) | e : -1;
    };
    int c = wave, cur = fetch(c);

    // Stage the run's atoms: tile t's block J by kWaves / kM wavefronts,
    // block I by all.  Every load is issued before any of it is used.  A
    // bare charge's row is its charge and zeros, so only its first vector
    // is read; atoms past the last take no part.
    constexpr int kParts = kWaves / kM;
    constexpr int kHJ = (kVA + kParts - 1) / kParts, kHI = (kVA + kWaves - 1) / kWaves;
    const int jt = wave / kParts, part = wave % kParts;
    int Jw = -1;
#pragma unroll
    for (int t = 0; t < kM; t++) Jw = jt == t ? J[t] : Jw;
    const int ja = min(max(Jw, 0) * kTile + lane, n - 1), ia = min(I * kTile + lane, n - 1);
    const bool jbare = ((bmask[max(Jw, 0)] >> lane) & 1ull) != 0, ibare = ((bmask[I] >> lane) & 1ull) != 0;
    vec vj[kHJ], vi[kHI];
    const vec* rj = reinterpret_cast<const vec*>(A.lab + (size_t)ja * kMP);
    const vec* ri = reinterpret_cast<const vec*>(A.lab + (size_t)ia * kMP);
#pragma unroll
    for (int h = 0; h < kHJ; h++) {
        const int v = part + h * kParts;
        vj[h] = (Jw >= 0 && v < kVA && (v == 0 || !jbare)) ? rj[v] : vec(R(0));
    }
#pragma unroll
    for (int h = 0; h < kHI; h++) {
        const int v = wave + h * kWaves;
        vi[h] = (v < kVA && (v == 0 || !ibare)) ? ri[v] : vec(R(0));
    }
    // the other fields: block J by its first wavefront, block I by the last
    const bool si = wave == kWaves - 1, sj = part == 0 && Jw >= 0;
    R fd[2][4] = {}, fm[2][3] = {};
    int fa[2] = {};
    double4 fp[2] = {};
    double fq[2] = {};
#pragma unroll
    for (int h = 0; h < 2; h++)
        if (h == 0 ? sj : si) {
            const size_t a = h == 0 ? ja : ia;
            const R4<R> d = A.pos[a];
            fd[h][0] = d.x;
            fd[h][1] = d.y;
            fd[h][2] = d.z;
            fd[h][3] = d.w;
#pragma unroll
            for (int k = 0; k < 3; k++) fm[h][k] = mu[3 * a + k];
            fa[h] = A.aniso[a];
            fp[h] = pos64[a];
            fq[h] = lab64[a * kMP];
        }
    for (int k = tid; k < (1 + nt) * 6 * kTile; k += kT) (&acc[0][0][0])[k] = 0.0;
    if constexpr (kPot)
        for (int k = tid; k < kSides * kMP * kTile; k += kT) (&pacc[0][0][0])[k] = 0.0;
#pragma unroll
    for (int h = 0; h < kHJ; h++) {
        const int v = part + h * kParts;
        if (v < kVA) reinterpret_cast<vec*>(&smp[1 + jt][0])[lane * kVA + v] = vj[h];
    }
#pragma unroll
    for (int h = 0; h < kHI; h++) {
        const int v = wave + h * kWaves;
        if (v < kVA) reinterpret_cast<vec*>(&smp[0][0])[lane * kVA + v] = vi[h];
    }
#pragma unroll
    for (int h = 0; h < 2; h++)
        if (h == 0 ? sj : si) {
            const int side = h == 0 ? 1 + jt : 0;
            spos[side][lane] = R4<R>{fd[h][0], fd[h][1], fd[h][2], fd[h][3]};
#pragma unroll
            for (int k = 0; k < 3; k++) smu[side][3 * lane + k] = fm[h][k];
            san[side][lane] = fa[h];
            spos64[side][lane] = make_double4(fp[h].x, fp[h].y, fp[h].z, fq[h]);
        }
    if (tid == 0) snext = kWaves;
    __syncthreads();

    // the next chunk of this wavefront
    auto claim = [&] {
        int v = 0;
        if (lane == 0) v = atomicAdd(&snext, 1);
        return __builtin_amdgcn_readfirstlane(v);
    };
    // General pairs: the quasi-internal-frame interaction without its
    // charge-charge channel, in the working precision.
    if constexpr (kGen)
        while (c < cg) {
            c = claim();
            const int e = cur;
            cur = fetch(c);
            if (e < 0) continue;
            const int il = (e >> 8) & 63, jj = e & 63, sd = 1 + (e >> 16);
            const R4<R> pi = spos[0][il], pj = spos[sd][jj];
            const V3<R> dr = min_image(mk(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z), P.box);
            R mi[kMP], mj[kMP];
            const vec* ri = reinterpret_cast<const vec*>(&smp[0][il * kMP]);
            const vec* rj = reinterpret_cast<const vec*>(&smp[sd][jj * kMP]);
#pragma unroll
            for (int v = 0; v < kVA; v++) {
                const vec a = ri[v], b = rj[v];
#pragma unroll
                for (int k = 0; k < kV; k++) {
                    mi[v * kV + k] = a[k];
                    mj[v * kV + k] = b[k];
                }
            }
            const V3<R> ui = mk(smu[0][3 * il], smu[0][3 * il + 1], smu[0][3 * il + 2]);
            const V3<R> uj = mk(smu[sd][3 * jj], smu[sd][3 * jj + 1], smu[sd][3 * jj + 2]);
            R pot_i[kPot ? kMP : 1] = {}, pot_j[kPot ? kMP : 1] = {};
            const ElecOut<R> o = elec_pair<R, kPot>(dr, dot(dr, dr), mi, mj, ui, uj, R2<R>{R(0), pi.w},
                                                    R2<R>{R(0), pj.w}, san[0][il] != 0,
                                                    san[sd][jj] != 0, R(1), R(1), P, false, pot_i, pot_j);
            if constexpr (kPot) {
#pragma unroll
                for (int k = 0; k < kMP; k++) {
                    atomicAdd(&pacc[0][k][il], (double)pot_i[k]);
                    atomicAdd(&pacc[1][k][jj], (double)pot_j[k]);
                }
            }
            en += (double)o.energy;
            atomicAdd(&acc[0][0][il], -(double)o.f.x);
            atomicAdd(&acc[0][1][il], -(double)o.f.y);
            atomicAdd(&acc[0][2][il], -(double)o.f.z);
            atomicAdd(&acc[0][3][il], (double)o.ti.x);
            atomicAdd(&acc[0][4][il], (double)o.ti.y);
            atomicAdd(&acc[0][5][il], (double)o.ti.z);
            atomicAdd(&acc[sd][0][jj], (double)o.f.x);
            atomicAdd(&acc[sd][1][jj], (double)o.f.y);
            atomicAdd(&acc[sd][2][jj], (double)o.f.z);
            atomicAdd(&acc[sd][3][jj], (double)o.tj.x);
            atomicAdd(&acc[sd][4][jj], (double)o.tj.y);
            atomicAdd(&acc[sd][5][jj], (double)o.tj.z);
        }
    // Pairs with one bare charge b: the FP64 charge-charge channel, and
    // b's charge against a's moments and induced dipole in the working
    // precision (the Cartesian form, elec_pair_bare_cart).
    while (c < cb) {
        c = claim();
        const int e = cur;
        cur = fetch(c);
        if (e < 0) continue;
        const int il = (e >> 8) & 63, jj = e & 63, sd = 1 + (e >> 16);
        const bool ib_ = (e & 0x8000) != 0;  // I's site is the bare one
        const int sa = ib_ ? sd : 0, xa = ib_ ? jj : il;
        const int sb = ib_ ? 0 : sd, xb = ib_ ? il : jj;
        const double4 qa = spos64[sa][xa], qb = spos64[sb][xb];
        const V3<double> d = min_image(mk(qb.x - qa.x, qb.y - qa.y, qb.z - qa.z), P64.box);
        const R4<R> pa = spos[sa][xa], pb = spos[sb][xb];
        const V3<R> dr = min_image(mk(pb.x - pa.x, pb.y - pa.y, pb.z - pa.z), P.box);
        R ma[kMP];
        const vec* ra = reinterpret_cast<const vec*>(&smp[sa][xa * kMP]);
#pragma unroll
        for (int v = 0; v < kVA; v++) {
            const vec x = ra[v];
#pragma unroll
            for (int k = 0; k < kV; k++) ma[v * kV + k] = x[k];
        }
        const V3<R> ua = mk(smu[sa][3 * xa], smu[sa][3 * xa + 1], smu[sa][3 * xa + 2]);
        R pot_a[kPot ? kMP : 1] = {};
        R pot_b0 = R(0);
        const ElecBareOut<R> o = elec_pair_bare_cart<R, kPot>(dr, dot(dr, dr), ma, smp[sb][xb * kMP], ua,
                                                              san[sa][xa] != 0, P, pot_a, &pot_b0);
        V3<double> f;
        double ec;
        if constexpr (kPot) {
            double phi_a = 0.0, phi_b = 0.0;
            charge_pair<double, true>(d, dot(d, d), qa.w, qb.w, P64, f, ec, &phi_a, &phi_b);
            atomicAdd(&pacc[sa][0][xa], phi_a);
            atomicAdd(&pacc[sb][0][xb], phi_b + (double)pot_b0);
#pragma unroll
            for (int k = 1; k < kMP; k++) atomicAdd(&pacc[sa][k][xa], (double)pot_a[k]);
        } else {
            charge_pair<double>(d, dot(d, d), qa.w, qb.w, P64, f, ec);
        }
        en += ec + (double)o.energy;
        f.x += (double)o.f.x;
        f.y += (double)o.f.y;
        f.z += (double)o.f.z;
        atomicAdd(&acc[sa][0][xa], -f.x);
        atomicAdd(&acc[sa][1][xa], -f.y);
        atomicAdd(&acc[sa][2][xa], -f.z);
        atomicAdd(&acc[sa][3][xa], (double)o.ta.x);
        atomicAdd(&acc[sa][4][xa], (double)o.ta.y);
        atomicAdd(&acc[sa][5][xa], (double)o.ta.z);
        atomicAdd(&acc[sb][0][xb], f.x);
        atomicAdd(&acc[sb][1][xb], f.y);
        atomicAdd(&acc[sb][2][xb], f.z);
    }
    // The charge-charge channel runs in FP64 in both precision modes for
    // every pair: it carries most of the magnitude of the real-space
    // energy, and FP32 rounding of the charges, alpha and the Coulomb
    // constant would bias all its terms alike.  This loop takes it for the
    // pairs of two bare charges (where it is the whole interaction) and
    // for the general pairs (apart from their formula, whose registers it
    // would otherwise hold); the one-bare loop takes it with the rest.
    while (c < cf) {
        c = claim();
        const int e = cur;
        cur = fetch(c);
        if (e < 0) continue;
        const int il = (e >> 8) & 63, jj = e & 63, sd = 1 + (e >> 16);
        const double4 pi = spos64[0][il], pj = spos64[sd][jj];
        const V3<double> dr = min_image(mk(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z), P64.box);
        V3<double> f;
        double ec;
        if constexpr (kPot) {
            double phi_i = 0.0, phi_j = 0.0;
            charge_pair<double, true>(dr, dot(dr, dr), pi.w, pj.w, P64, f, ec, &phi_i, &phi_j);
            atomicAdd(&pacc[0][0][il], phi_i);
            atomicAdd(&pacc[1][0][jj], phi_j);
        } else {
            charge_pair<double>(dr, dot(dr, dr), pi.w, pj.w, P64, f, ec);
        }
        en += ec;
        atomicAdd(&acc[0][0][il], -f.x);
        atomicAdd(&acc[0][1][il], -f.y);
        atomicAdd(&acc[0][2][il], -f.z);
        atomicAdd(&acc[sd][0][jj], f.x);
        atomicAdd(&acc[sd][1][jj], f.y);
        atomicAdd(&acc[sd][2][jj], f.z);
    }
    __syncthreads();
    // flush: the threads run over each block's 64 x 3 consecutive words
    // (the memory side takes adds in pieces of 64 bytes: one component of
    // 64 atoms per instruction would be spread over 24 such pieces).  A
    // bare charge takes no torque, and an atom without pairs in the tile
    // nothing at all (atoms past the last have no pairs).
    for (int k = tid; k < (1 + nt) * 3 * kTile; k += kT) {
        const int side = k / (3 * kTile), e = k - side * 3 * kTile, al = e / 3, x = e - 3 * al;
        int B = I;
#pragma unroll
        for (int t = 0; t < kM; t++) B = side == 1 + t ? J[t] : B;
        const double f = acc[side][x][al], t = acc[side][3 + x][al];
        const size_t at = (size_t)3 * kTile * B + e;
        if (f != 0.0) acc_add(&force[at], f);
        if (t != 0.0) acc_add(&torque[at], t);
    }
    if constexpr (kPot)
        for (int k = tid; k < kSides * kMP * kTile; k += kT) {
            const int side = k / (kMP * kTile), e = k - side * kMP * kTile, al = e / kMP, x = e - al * kMP;
            const double v = pacc[side][x][al];
            if (v != 0.0) acc_add(&pot[(size_t)kMP * kTile * (side ? J[0] : I) + e], v);
        }
    // wavefront sums of the pair energies
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) en += __shfl_xor(en, off);
    if (lane == 0) sen[wave] = en;
    __syncthreads();
    if (tid == 0) {
        double e = 0.0;
        for (int k = 0; k < kWaves; k++) e += sen[k];
        if (e != 0.0) acc_add(energy + (blockIdx.x & (kEnergySlots - 1)), e);
    }
}

// The general pairs (neither site a bare charge) of an evaluation, without
// their charge-charge channel (the tile kernel's).  One workgroup per block I
// and split: it collects the general pairs of its tiles (I, J >= I) from their
// lists into an LDS queue and works through that 64 pairs at a time.  A tile of
// a water box holds about 26 general pairs among its 250, so that tile by tile
// the lanes of this class, the one with by far the longest formula, were 40%
// full, and in FP64 its registers (308) held the tile kernel to one wavefront
// per SIMD; here the chunks are full to the last one of a row, and the tile
// kernel needs 132.
//
// Both sides accumulate in LDS in FP64: block I's over the row, and those of the
// tiles' blocks J over a pass, in one slot per site that is not a bare charge
// (kGenSlots hold the 21 of 64 of 72 water tiles, or 24 tiles of general
// sites).  One workgroup per CU is what the registers leave, so its LDS is
// free.  A slot goes to the fixed-point accumulators once per tile.  (Adding
// every pair's J side there truncated each of them to 2^-32, and six adds a
// pair bound the kernel wherever tiles are dense.)  Three lanes hold a site's
// three consecutive words: the memory side takes adds in 64-byte pieces, and
// one component per instruction was 2-3 times slower.
// splits: workgroups per block row, so that small systems fill the chip.
// FP64, with every pair's J side added to the fixed-point accumulators in
// brackets: 98,304 atoms of water 258 us (303) beside 500 in the tile kernel,
// where one kernel for all pairs took 1,870; 64,000 general sites 565 us of
// electrostatics (747), 3,000 without a cutoff 715 (1,615).
constexpr int kGenTiles = 64;             // tiles ranked per pass
constexpr int kGenQueue = kTilePairs;     // queue entries: at least one tile's most
constexpr int kGenSlots = 1536;           // sites of the pass's blocks J, a multiple of 32
constexpr int kGenPitch = kGenSlots + 21;  // a flush reads components of 21 slots: 63 different places
template <class R>
__global__ __launch_bounds__(kElecThreads) void k_general_pairs(int splits, TileList T, const int* __restrict__ ustart,
                                                                const unsigned long long* __restrict__ bmask,
                                                                PairAtoms<R> A, const R* __restrict__ mu,
                                                                PairParams<R> P, acc_t* __restrict__ force,
                                                                acc_t* __restrict__ torque,
                                                                acc_t* __restrict__ energy) {
    constexpr int kV = 16 / (int)sizeof(R);  // reals per 16-byte vector
    constexpr int kWaves = kElecThreads / kTile;
    typedef R vec __attribute__((ext_vector_type(kV)));
    __shared__ unsigned queue[kGenQueue];  // slot of J's site << 6 | atom of I
    __shared__ int sfirst[kGenTiles], soff[kGenTiles + 1], sslot[kGenTiles + 1], sfit, sJ[kGenTiles];
    __shared__ unsigned long long sgen[kGenTiles];  // the sites of J that are not bare charges
    static_assert(kGenTiles == kTile, "a pass's tiles are ranked by one wavefront");
    static_assert(kGenSlots >= kTile && kGenQueue >= kTilePairs, "a pass takes at least one tile");
    __shared__ double accj[6][kGenPitch];
    __shared__ int satom[kGenSlots];
    __shared__ double acc[6][kTile];
    __shared__ R4<R> spos[kTile];
    __shared__ __align__(16) R smp[kTile * kMP];
    __shared__ R smu[kTile * 3];
    __shared__ int san[kTile];
    __shared__ double sen[kWaves];
    if (*T.nact == 0) return;
    const int n = P.n;
    const int tid = threadIdx.x, lane = tid & (kTile - 1), wave = tid / kTile;
    const int I = blockIdx.x / splits, y = blockIdx.x - I * splits;
    const int u0 = ustart[I] + y;
    const int ntiles = (ustart[I + 1] - u0 + splits - 1) / splits;
    const int i0 = I * kTile + lane;
    const bool bare = i0 >= n || ((bmask[I] >> lane) & 1ull) != 0;
    if (ntiles <= 0 || __ballot(!bare) == 0ull) return;  // uniform over the workgroup
    // block I's side
    for (int k = tid; k < kTile * (kMP / kV); k += kElecThreads) {
        const int a = min(I * kTile + k / (kMP / kV), n - 1);
        reinterpret_cast<vec*>(smp)[k] = reinterpret_cast<const vec*>(A.lab + (size_t)a * kMP)[k % (kMP / kV)];
    }
    if (wave == 0) {
        const int a = min(i0, n - 1);
        spos[lane] = A.pos[a];
        san[lane] = A.aniso[a];
#pragma unroll
        for (int k = 0; k < 3; k++) smu[3 * lane + k] = mu[3 * (size_t)a + k];
#pragma unroll
        for (int k = 0; k < 6; k++) acc[k][lane] = 0.0;
    }
    for (int k = tid; k < 6 * kGenPitch; k += kElecThreads) (&accj[0][0])[k] = 0.0;
    double en = 0.0;
    // as in the tile kernel: neighbours in the queue share a site, and spreading
    // them over the lanes keeps one instruction's atomic adds off a common address
    const int perm = ((lane & 7) << 3) | (lane >> 3);
    for (int b0 = 0; b0 < ntiles;) {
        const int nt = min(kGenTiles, ntiles - b0);
        if (wave == 0) {
            const int4 t = T.act[u0 + (b0 + min(lane, nt - 1)) * splits];
            int c = lane < nt ? t.x >> 16 : 0;
            const unsigned long long gen = c > 0 ? ~bmask[t.z] : 0ull;  // (atoms past the last have slots, no pairs)
            int sl = __popcll(gen);
            sfirst[lane] = t.x & 0xffff;
            sJ[lane] = t.z;
            sgen[lane] = gen;
#pragma unroll
            for (int off = 1; off < kTile; off <<= 1) {
                const int v = __shfl_up(c, off), w = __shfl_up(sl, off);
                if (lane >= off) {
                    c += v;
                    sl += w;
                }
            }
            soff[lane + 1] = c;
            sslot[lane + 1] = sl;
            // tiles of this pass (at least one)
            const int fit = __popcll(__ballot(lane < nt && c <= kGenQueue && sl <= kGenSlots));
            if (lane == 0) {
                soff[0] = sslot[0] = 0;
                sfit = fit;
            }
        }
        __syncthreads();
        const int fit = sfit, total = soff[fit], nslots = sslot[fit];
        // the tiles' general entries and sites, 16 lanes per tile
        for (int k = tid >> 4; k < fit; k += kElecThreads >> 4) {
            const unsigned short* list = T.list + (size_t)(u0 + (b0 + k) * splits) * kTilePairs + sfirst[k];
            const int o = soff[k], c = soff[k + 1] - o, so = sslot[k], a0 = sJ[k] * kTile;
            const unsigned long long gen = sgen[k];
            for (int a = tid & 15; a < kTile; a += 16)
                if ((gen >> a) & 1ull) satom[so + __popcll(gen & ((1ull << a) - 1ull))] = a0 + a;
            for (int e = tid & 15; e < c; e += 16) {
                const unsigned ent = list[e];
                const int slot = so + __popcll(gen & ((1ull << (ent & 63u)) - 1ull));
                queue[o + e] = ((unsigned)slot << 6) | (ent >> 8);
            }
        }
        __syncthreads();
        for (int q0 = wave * kTile; q0 < total; q0 += kElecThreads) {
            const int q = q0 + perm;
            const bool qv = q < total;
            const unsigned ent = queue[qv ? q : total - 1];
            const int il = (int)(ent & 63u), slot = (int)(ent >> 6);
            const size_t j = satom[slot];
            const R4<R> pi = spos[il], pj = A.pos[j];
            const V3<R> dr = min_image(mk(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z), P.box);
            R mi[kMP], mj[kMP];
            const vec* ri = reinterpret_cast<const vec*>(smp + il * kMP);
            const vec* rj = reinterpret_cast<const vec*>(A.lab + j * kMP);
#pragma unroll
            for (int v = 0; v < kMP / kV; v++) {
                const vec a = ri[v], b = rj[v];
#pragma unroll
                for (int c = 0; c < kV; c++) {
                    mi[v * kV + c] = a[c];
                    mj[v * kV + c] = b[c];
                }
            }
            const V3<R> ui = mk(smu[3 * il], smu[3 * il + 1], smu[3 * il + 2]);
            const V3<R> uj = mk(mu[3 * j], mu[3 * j + 1], mu[3 * j + 2]);
            const ElecOut<R> o =
                elec_pair<R>(dr, dot(dr, dr), mi, mj, ui, uj, R2<R>{R(0), pi.w}, R2<R>{R(0), pj.w}, san[il] != 0,
                             A.aniso[j] != 0, R(1), R(1), P, false);
            if (qv) {
                en += (double)o.energy;
                atomicAdd(&acc[0][il], -(double)o.f.x);
                atomicAdd(&acc[1][il], -(double)o.f.y);
                atomicAdd(&acc[2][il], -(double)o.f.z);
                atomicAdd(&acc[3][il], (double)o.ti.x);
                atomicAdd(&acc[4][il], (double)o.ti.y);
                atomicAdd(&acc[5][il], (double)o.ti.z);
                atomicAdd(&accj[0][slot], (double)o.f.x);
                atomicAdd(&accj[1][slot], (double)o.f.y);
                atomicAdd(&accj[2][slot], (double)o.f.z);
                atomicAdd(&accj[3][slot], (double)o.tj.x);
                atomicAdd(&accj[4][slot], (double)o.tj.y);
                atomicAdd(&accj[5][slot], (double)o.tj.z);
            }
        }
        b0 += fit;
        __syncthreads();
        // the slots, left zero for the next pass
        for (int e = tid; e < 3 * nslots; e += kElecThreads) {
            const int slot = e / 3, k = e - 3 * slot;
            const double f = accj[k][slot], t = accj[3 + k][slot];
            accj[k][slot] = 0.0;
            accj[3 + k][slot] = 0.0;
            const size_t at = 3 * (size_t)satom[slot] + k;
            if (f != 0.0) acc_add(&force[at], f);
            if (t != 0.0) acc_add(&torque[at], t);
        }
        __syncthreads();  // the queue and the slots are read before the next pass rewrites them
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) en += __shfl_xor(en, off);
    if (lane == 0) sen[wave] = en;
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int u = 0; u < 3; u++) {
            const int e = u * kTile + lane, al = e / 3, k = e - 3 * al;  // a bare charge has no general pairs
            const double f = acc[k][al], t = acc[3 + k][al];
            if (f != 0.0) acc_add(&force[3 * (size_t)I * kTile + e], f);
            if (t != 0.0) acc_add(&torque[3 * (size_t)I * kTile + e], t);
        }
    }
    if (tid == 0) {
        double e = 0.0;
        for (int k = 0; k < kWaves; k++) e += sen[k];
        if (e != 0.0) acc_add(energy + (blockIdx.x & (kEnergySlots - 1)), e);
    }
}

// Where the general pairs run.  FP32: in the tile kernel, whose registers they
// do not raise above 128 (98,304 atoms: the evaluation took 2,280 us with the
// kernel of their own, 2,195 without).  FP64: in their own kernel, except for
// systems of at most kSmallTiles tiles, which leave CUs idle whatever the
// registers: they are spared the dependent dispatch.  Evaluations with direct
// polarization, in the tile kernel and apart: 66 tiles 188 and 198 us, 190 193
// and 195, 560 to 1,111 even, 3,292 317 and 286.
constexpr int kSmallTiles = 256;

// FP32: at most 128 VGPRs, so that four wavefronts fit per SIMD
__global__ __launch_bounds__(kElecThreads) __attribute__((amdgpu_waves_per_eu(4)))
void k_electrostatics_f32(int tiles, TileList T, const unsigned long long* __restrict__ bmask, PairAtoms<float> A,
                          const float* __restrict__ mu, PairParams<float> P, const double4* __restrict__ pos64,
                          const double* __restrict__ lab64, PairParams<double> P64, acc_t* __restrict__ force,
                          acc_t* __restrict__ torque, acc_t* __restrict__ energy) {
    electrostatics_tiles<float, false, true>(tiles, T, bmask, A, mu, P, pos64, lab64, P64, force, torque,
                                                                energy, nullptr, 0);
}
__global__ __launch_bounds__(kElecThreads) __attribute__((amdgpu_waves_per_eu(4)))
void k_electrostatics_f64(int tiles, TileList T, const unsigned long long* __restrict__ bmask, PairAtoms<double> A,
                          const double* __restrict__ mu, PairParams<double> P, const double4* __restrict__ pos64,
                          const double* __restrict__ lab64, PairParams<double> P64, acc_t* __restrict__ force,
                          acc_t* __restrict__ torque, acc_t* __restrict__ energy) {
    electrostatics_tiles<double, false, false>(tiles, T, bmask, A, mu, P, pos64, lab64, P64, force, torque,
                                                                  energy, nullptr, 0);
}
__global__ __launch_bounds__(kElecThreads)
void k_electrostatics_f64_small(int tiles, TileList T, const unsigned long long* __restrict__ bmask,
                                PairAtoms<double> A, const double* __restrict__ mu, PairParams<double> P,
                                const double4* __restrict__ pos64, const double* __restrict__ lab64,
                                PairParams<double> P64, acc_t* __restrict__ force, acc_t* __restrict__ torque,
                                acc_t* __restrict__ energy) {
    electrostatics_tiles<double, false, true>(tiles, T, bmask, A, mu, P, pos64, lab64, P64, force, torque, energy,
                                              nullptr, 0);
}
// The final pass of the energy gradients: the same, with the potential vectors.
template <class R>
__global__ __launch_bounds__(kElecThreads)
void k_electrostatics_pot(TileList T, const unsigned long long* __restrict__ bmask, PairAtoms<R> A,
                          const R* __restrict__ mu, PairParams<R> P, const double4* __restrict__ pos64,
                          const double* __restrict__ lab64, PairParams<double> P64, acc_t* __restrict__ force,
                          acc_t* __restrict__ torque, acc_t* __restrict__ energy, acc_t* __restrict__ pot,
                          int all_general) {
    electrostatics_tiles<R, true, true>(1, T, bmask, A, mu, P, pos64, lab64, P64, force, torque, energy, pot, all_general);
}
// the kernel, and whether one of them leaves the general pairs to k_general_pairs
template <class R> struct ElecKernel;
template <> struct ElecKernel<float> {
    static constexpr bool kSplit = false;
    static constexpr auto fn(int) { return k_electrostatics_f32; }
};
template <> struct ElecKernel<double> {
    static constexpr bool kSplit = true;  // above kSmallTiles
    static constexpr auto fn(int tiles) { return tiles > kSmallTiles ? k_electrostatics_f64 : k_electrostatics_f64_small; }
};

// ---------------------------------------------------------------------------
// Covalent pairs.  The pairs on the scaled covalent lists (1-2, 1-3 and 1-4
// partners) are few, O(N), and carry the largest terms of the real-space sum:
// at 0.1 nm the screened and unscreened Coulomb parts cancel to a few percent,
// and the same geometry repeats in every molecule, so single-precision
// rounding would add up coherently.  The tile kernels skip them; these
// kernels evaluate each once (thread = atom i, partners j > i), in the
// precision they are instantiated with (FP64 for the permanent field and the
// final electrostatics in both precision modes).
// ---------------------------------------------------------------------------
template <class R>
__global__ __launch_bounds__(256) void k_cov_fixed_field(PairAtoms<R> A, PairParams<R> P, acc_t* __restrict__ field) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P.n) return;
    const int np = A.npart[i];
    if (np == 0) return;
    const R4<R> pi = A.pos[i];
    const R* mi = A.lab + (size_t)i * kMP;
    const R2<R> tdi = A.td[i];
    R ex = 0, ey = 0, ez = 0;
    for (int k = 0; k < np; k++) {
        const int e = A.partners[(size_t)i * A.pstride + k];
        const int j = e >> 2;
        if (j <= i) continue;
        const R4<R> pj = A.pos[j];
        const V3<R> dr = min_image(mk(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z), P.box);
        const R r2 = dot(dr, dr);
        if (r2 > P.rc2) continue;
        V3<R> fi, fj;
        fixed_field_pair<R>(dr, r2, mi, A.lab + (size_t)j * kMP, tdi, A.td[j], partner_scale<R>(e, P.scale14), P, fi,
                            fj);
        ex += fi.x;
        ey += fi.y;
        ez += fi.z;
        acc_add(&field[3 * (size_t)j + 0], fj.x);
        acc_add(&field[3 * (size_t)j + 1], fj.y);
        acc_add(&field[3 * (size_t)j + 2], fj.z);
    }
    acc_add(&field[3 * (size_t)i + 0], ex);
    acc_add(&field[3 * (size_t)i + 1], ey);
    acc_add(&field[3 * (size_t)i + 2], ez);
}

// pol_only: only pairs of two polarisable sites (the solver's operator).
template <class R>
__global__ __launch_bounds__(256) void k_cov_induced_field(PairAtoms<R> A, const R* __restrict__ mu, PairParams<R> P,
                                                           int pol_only, acc_t* __restrict__ field) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P.n) return;
    const int np = A.npart[i];
    if (np == 0) return;
    const R4<R> pi = A.pos[i];
    const V3<R> ui = mk(mu[3 * (size_t)i], mu[3 * (size_t)i + 1], mu[3 * (size_t)i + 2]);
    const R2<R> tdi = A.td[i];
    if (pol_only && tdi.y == R(0)) return;
    R ex = 0, ey = 0, ez = 0;
    for (int k = 0; k < np; k++) {
        const int e = A.partners[(size_t)i * A.pstride + k];
        const int j = e >> 2;
        if (j <= i) continue;
        if (pol_only && A.td[j].y == R(0)) continue;
        const R4<R> pj = A.pos[j];
        const V3<R> dr = min_image(mk(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z), P.box);
        const R r2 = dot(dr, dr);
        if (r2 > P.rc2) continue;
        V3<R> fi, fj;
        const R2<R> tdj = A.td[j];
        const R a = partner_scale<R>(e, P.scale14) == R(0) ? tdi.x + tdj.x : P.default_thole;
        const V3<R> uj = mk(mu[3 * (size_t)j], mu[3 * (size_t)j + 1], mu[3 * (size_t)j + 2]);
        induced_field_pair<R>(dr, r2, ui, uj, tdi.y, tdj.y, a, P, fi, fj);
        ex += fi.x;
        ey += fi.y;
        ez += fi.z;
        acc_add(&field[3 * (size_t)j + 0], fj.x);
        acc_add(&field[3 * (size_t)j + 1], fj.y);
        acc_add(&field[3 * (size_t)j + 2], fj.z);
    }
    acc_add(&field[3 * (size_t)i + 0], ex);
    acc_add(&field[3 * (size_t)i + 1], ey);
    acc_add(&field[3 * (size_t)i + 2], ez);
}

// Covalent electrostatics with the potential vectors (the energy gradients;
// an evaluation's are in the per-atom kernel of its final pass).
template <class R>
__global__ __launch_bounds__(128) void k_cov_electrostatics_pot(PairAtoms<R> A, const R* __restrict__ mu,
                                                                PairParams<R> P, acc_t* __restrict__ force,
                                                                acc_t* __restrict__ torque,
                                                                acc_t* __restrict__ energy, acc_t* __restrict__ pot) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    double en = i < P.n ? cov_electrostatics<R, true>(i, A, mu, P, force, torque, pot) : 0.0;
    // every lane reaches the reduction
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) en += __shfl_xor(en, off);
    if ((threadIdx.x & 63) == 0 && en != 0.0) acc_add(energy + (blockIdx.x & (kEnergySlots - 1)), en);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
template <class R>
void launch_electrostatics_pairs(hipStream_t s, int n, int maxtiles, int group, const TileList& t, const int* ustart,
                                 const unsigned long long* bmask, PairAtoms<R> a, const R* mu, PairParams<R> p,
                                 const double4* pos64, const double* lab64, PairParams<double> p64, acc_t* force,
                                 acc_t* torque, acc_t* energy) {
    if (maxtiles <= 0) return;
    hipLaunchKernelGGL(ElecKernel<R>::fn(maxtiles), dim3(group == 1 ? maxtiles : tile_groups(maxtiles, n, group)),
                       dim3(kElecThreads), 0, s, group, t, bmask, a, mu, p, pos64, lab64, p64, force,
                       torque, energy);
    if constexpr (ElecKernel<R>::kSplit) {
        if (maxtiles <= kSmallTiles) return;
        // About 512 workgroups, two for each that the chip holds (the first rows
        // have most tiles J >= I), at most 32 per block row.  Where tiles are
        // sparse longer queues would do: evaluations of 192 blocks of water with
        // direct polarization take 350 us with one workgroup per row, 359 with two,
        // 372 with four and 409 with eight.  Where they are dense a row has to be
        // cut: 3,000 general sites without a cutoff (47 blocks) take 1,230 us of
        // electrostatics with five per row and 713 with ten.
        const int nb = (n + kTile - 1) / kTile;
        const int splits = std::max(1, std::min(32, 512 / nb));
        hipLaunchKernelGGL(k_general_pairs<R>, dim3(nb * splits), dim3(kElecThreads), 0, s, splits, t, ustart, bmask, a,
                           mu, p, force, torque, energy);
    }
}

template <class R> void launch_cov_fixed_field(hipStream_t s, int n, PairAtoms<R> a, PairParams<R> p, acc_t* field) {
    hipLaunchKernelGGL(k_cov_fixed_field<R>, dim3((n + 255) / 256), dim3(256), 0, s, a, p, field);
}
template <class R>
void launch_cov_induced_field(hipStream_t s, int n, PairAtoms<R> a, const R* mu, PairParams<R> p, int pol_only,
                              acc_t* field) {
    hipLaunchKernelGGL(k_cov_induced_field<R>, dim3((n + 255) / 256), dim3(256), 0, s, a, mu, p, pol_only, field);
}
template <class R>
void launch_cov_electrostatics_pot(hipStream_t s, int n, PairAtoms<R> a, const R* mu, PairParams<R> p, acc_t* force,
                                   acc_t* torque, acc_t* energy, acc_t* pot) {
    hipLaunchKernelGGL(k_cov_electrostatics_pot<R>, dim3((n + 127) / 128), dim3(128), 0, s, a, mu, p, force, torque,
                       energy, pot);
}

// ---------------------------------------------------------------------------
// Thole damping of the covalent pairs (energy gradients): h = u dE/du of
// each pair of polarisable partners, once per pair (thread = atom i,
// partners j > i).  hd takes h at both atoms (the damping factors); a pair
// at polarization scale 0 has the width thole_i + thole_j, so ht takes h/a
// at both atoms; any other pair has the default width, and hdef takes 2h
// (hdef sums h over both atoms of every pair, like the neighbour-list kernel).
// ---------------------------------------------------------------------------
template <class R>
__global__ __launch_bounds__(256) void k_cov_thole(PairAtoms<R> A, const R* __restrict__ mu, PairParams<R> P,
                                                   acc_t* __restrict__ hd, acc_t* __restrict__ hdef,
                                                   acc_t* __restrict__ ht) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P.n) return;
    const int np = A.npart[i];
    const R2<R> tdi = A.td[i];
    if (np == 0 || tdi.y == R(0)) return;
    const R4<R> pi = A.pos[i];
    const R* mi = A.lab + (size_t)i * kMP;
    const V3<R> ui = mk(mu[3 * (size_t)i], mu[3 * (size_t)i + 1], mu[3 * (size_t)i + 2]);
    R hi = 0, hdi = 0, hti = 0;
    for (int k = 0; k < np; k++) {
        const int e = A.partners[(size_t)i * A.pstride + k];
        const int j = e >> 2;
        if (j <= i) continue;
        const R2<R> tdj = A.td[j];
        if (tdj.y == R(0)) continue;
        const R4<R> pj = A.pos[j];
        const V3<R> dr = min_image(mk(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z), P.box);
        const R r2 = dot(dr, dr);
        if (r2 > P.rc2) continue;
        const R ps = partner_scale<R>(e, P.scale14);
        const R a = ps == R(0) ? tdi.x + tdj.x : P.default_thole;
        const V3<R> uj = mk(mu[3 * (size_t)j], mu[3 * (size_t)j + 1], mu[3 * (size_t)j + 2]);
        const R h = thole_u_derivative<R>(dr, r2, mi, A.lab + (size_t)j * kMP, ui, uj, tdi.y, tdj.y, a, ps,
                                          P.mutual != 0);
        if (h == R(0)) continue;
        hi += h;
        acc_add(&hd[j], h);
        if (ps == R(0)) {
            const R t = h / a;
            hti += t;
            acc_add(&ht[j], t);
        } else {
            hdi += R(2) * h;
        }
    }
    if (hi != R(0)) acc_add(&hd[i], hi);
    if (hti != R(0)) acc_add(&ht[i], hti);
    if (hdi != R(0)) acc_add(&hdef[i], hdi);
}
template <class R>
void launch_cov_thole(hipStream_t s, int n, PairAtoms<R> a, const R* mu, PairParams<R> p, acc_t* hd, acc_t* hdef,
                      acc_t* ht) {
    hipLaunchKernelGGL(k_cov_thole<R>, dim3((n + 255) / 256), dim3(256), 0, s, a, mu, p, hd, hdef, ht);
}
template <class R>
void launch_electrostatics_pot(hipStream_t s, int maxtiles, const TileList& t, const unsigned long long* bmask,
                               PairAtoms<R> a, const R* mu, PairParams<R> p, const double4* pos64,
                               const double* lab64, PairParams<double> p64, acc_t* force, acc_t* torque,
                               acc_t* energy, acc_t* pot, int all_general) {
    if (maxtiles <= 0) return;
    hipLaunchKernelGGL(k_electrostatics_pot<R>, dim3(maxtiles), dim3(kElecThreads), 0, s, t, bmask, a, mu, p, pos64,
                       lab64, p64, force, torque, energy, pot, all_general);
}

#define MPID_INSTANTIATE(R)                                                                                        \
    template void launch_electrostatics_pairs<R>(hipStream_t, int, int, int, const TileList&, const int*,          \
                                                 const unsigned long long*, PairAtoms<R>, const R*, PairParams<R>,  \
                                                 const double4*, const double*, PairParams<double>, acc_t*, acc_t*, \
                                                 acc_t*);                                                          \
    template void launch_cov_fixed_field<R>(hipStream_t, int, PairAtoms<R>, PairParams<R>, acc_t*);                \
    template void launch_cov_induced_field<R>(hipStream_t, int, PairAtoms<R>, const R*, PairParams<R>, int,        \
                                              acc_t*);                                                            \
    template void launch_cov_electrostatics_pot<R>(hipStream_t, int, PairAtoms<R>, const R*, PairParams<R>,        \
                                                   acc_t*, acc_t*, acc_t*, acc_t*);                                 \
    template void launch_cov_thole<R>(hipStream_t, int, PairAtoms<R>, const R*, PairParams<R>, acc_t*, acc_t*,      \
                                      acc_t*);                                                                      \
    template void launch_electrostatics_pot<R>(hipStream_t, int, const TileList&, const unsigned long long*,        \
                                               PairAtoms<R>, const R*, PairParams<R>, const double4*, const double*, \
                                               PairParams<double>, acc_t*, acc_t*, acc_t*, acc_t*, int);
MPID_INSTANTIATE(float)
MPID_INSTANTIATE(double)
#undef MPID_INSTANTIATE

}  // namespace mpid
