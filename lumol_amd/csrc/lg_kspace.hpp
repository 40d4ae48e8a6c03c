// lg_kspace.hpp -- Ewald k-space on the matrix cores, by octants.
//
// The k set of the reference (lumol-core/src/energy/global/ewald.rs:130-183)
// is symmetric under sign changes of iky and ikz but for its edges, and
//     e^{i k.r} = (cx + i sx) (cy +- i sy) (cz +- i sz)
// for the up to four members (p, +-q, +-r) of an octant (p = ikx >= 0,
// q = |iky|, r = |ikz|).  The structure factors of all four are sign
// combinations of eight real sums
//     T[ab][c] = sum_i q_i X_a(p) Y_b(q) Z_c(r),   a, b, c in {cos, sin},
// 8 multiply-adds per four k-vectors where the complex recursion along ikz
// took 28 operations, and as a real matrix product over atoms
//     T[(p, q), ab][r, c] = sum_i (q X_a Y_b)[i] Z[i][r, c]
// they belong on v_mfma 16x16x4.  The k-space forces are the gradient of
//     Phi(r) = sum_k 2 factor_k Re(e^{i k.r} conj rho_k)
//            = sum_{p,q,ab} X_a Y_b  S[(p, q), ab],   S = sum_{r,c} A Z
// with real coefficients A (from rho), again a matrix product (inner
// dimension (r, c), columns = atoms), and D = sum A dZ/dz beside it for the z
// component; X and Y and their derivatives are applied to S and D per pair.
//
// Layouts.  A row tile is four (p, q) pairs x four ab; a column tile eight r
// x {c, s}.  Rows are ordered so that output register v of lane l is ab = v
// of pair l / 16, column l % 16 in both forms (FP32 D[4 (l/16) + v][l%16],
// FP64 D[l/16 + 4 v][l%16]).  Pairs are sorted by their ikz extent, so that
// pairs with short rows share tiles and skip the columns they do not have.
#pragma once

#include "lg_device.hpp"

namespace lg {

typedef float oct_f4 __attribute__((ext_vector_type(4)));
typedef double oct_d4 __attribute__((ext_vector_type(4)));
template <typename T> struct OctT;
template <> struct OctT<float> {
    typedef oct_f4 acc;
    typedef float2 v2;
    // operand A: lane i + 16 k holds row i; row i = 4 pair + ab
    static __device__ __forceinline__ int row_pair(int i) { return i >> 2; }
    static __device__ __forceinline__ int row_ab(int i) { return i & 3; }
    static __host__ __device__ __forceinline__ int row_of(int pair, int ab) { return pair * 4 + ab; }
};
template <> struct OctT<double> {
    typedef oct_d4 acc;
    typedef double2 v2;
    // row i = 4 ab + pair
    static __device__ __forceinline__ int row_pair(int i) { return i & 3; }
    static __device__ __forceinline__ int row_ab(int i) { return i >> 2; }
    static __host__ __device__ __forceinline__ int row_of(int pair, int ab) { return ab * 4 + pair; }
};
__device__ __forceinline__ oct_f4 oct_mfma(float a, float b, oct_f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ oct_d4 oct_mfma(double a, double b, oct_d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Largest kmax of the octant form: the phase rows of 16 atoms fit the LDS of
// its launches with room to spare (FP64, kmax 64: 404 rows of 17 x 8 B = 55 KB).
// Beyond it (half a million k-vectors) the row kernels run, as they do for few
// atoms from kmax 33 on (oct_pays).
constexpr int kOctMaxK = 64;

// (cos, sin) of 2 pi u, u in turns: the reduction to an eighth of a turn is
// exact, and both Taylor sums there (to the 18th and 19th order of |x| <= pi /
// 4, truncation below 1e-19) are within an ulp or two.  Half the instructions
// of the library's function, whose reduction covers every argument in
// radians, and few registers.
__device__ __forceinline__ void oct_cis(double u, double& c, double& s) {
    const double t = u - rint(u), q = rint(4.0 * t);
    const double x = 2.0 * kPi * (t - 0.25 * q), y = x * x;
    double pc = -1.0 / 6402373705728000.0;  // -1 / 18!
    pc = pc * y + 1.0 / 20922789888000.0;
    pc = pc * y - 1.0 / 87178291200.0;
    pc = pc * y + 1.0 / 479001600.0;
    pc = pc * y - 1.0 / 3628800.0;
    pc = pc * y + 1.0 / 40320.0;
    pc = pc * y - 1.0 / 720.0;
    pc = pc * y + 1.0 / 24.0;
    pc = pc * y - 0.5;
    pc = pc * y + 1.0;
    double ps = -1.0 / 121645100408832000.0;  // -1 / 19!
    ps = ps * y + 1.0 / 355687428096000.0;
    ps = ps * y - 1.0 / 1307674368000.0;
    ps = ps * y + 1.0 / 6227020800.0;
    ps = ps * y - 1.0 / 39916800.0;
    ps = ps * y + 1.0 / 362880.0;
    ps = ps * y - 1.0 / 5040.0;
    ps = ps * y + 1.0 / 120.0;
    ps = ps * y - 1.0 / 6.0;
    ps = (ps * y) * x + x;
    const int k = (int)q & 3;
    const double a = (k & 1) ? ps : pc, b = (k & 1) ? pc : ps;
    c = (k == 1 || k == 2) ? -a : a;
    s = (k & 2) ? -b : b;
}

// f e^{2 pi i n u} for n = n0 .. n1 - 1 by products with e^{2 pi i u}
// (ewald.rs:646-661).
template <typename F>
__device__ __forceinline__ void oct_phases(double f, double u, int n0, int n1, F store) {
    double s1, c1, ex, ey;
    oct_cis(u, c1, s1);
    oct_cis(n0 * u, ex, ey);
    ex *= f;
    ey *= f;
#pragma unroll 2
    for (int n = n0; n < n1; n++) {
        store(n, ex, ey);
        const double rx = ex * c1 - ey * s1, ry = ex * s1 + ey * c1;
        ex = rx;
        ey = ry;
    }
}

// ---- rho(k) -------------------------------------------------------------------------
// A work item of a wave: four output tiles.  shape 0: row tiles rt[0], rt[1]
// x column tiles ct, ct + 1; shape 1: row tiles rt[0..3] x column tile ct.
// Either way four matrix instructions per four atoms, 6 or 9 LDS reads.
struct OctItem {
    int rt[4];
    int ct, shape;
};

struct OctRho {
    const double4* pos;  // positions, charge in w
    int n;
    double inv[3];       // 1 / L per axis
    int kmax, zcols;     // zcols: columns of the Z rows (16 per column tile)
    const OctItem* items;
    const int4* rows;    // per item and matrix row (16): X row | Y row << 16 of its four row tiles
    const int* mask;     // per item and lane: which of the four tiles the lane stores
    int nitems, ngroups, ipg, asplit;  // items per group; waves that share an item's atoms
    int nchunks, width;                // atoms per chunk (block)
    double4* partial;                  // [chunk][4 nitems][64 lanes] (ab = x, y, z, w)
};

// Phase rows in LDS, row-major over the C atoms (a multiple of 16) of a
// stage: X 2 n + {c, s} (times the charge), then Y, then Z (zcols columns).
// The row pitch, twice an odd number of 4-byte words or an odd number of
// 8-byte ones, spreads the lanes of a matrix operand (16 rows x 4 atoms, 32
// lanes of 4 bytes or 16 of 8 at a time) over all banks.
template <typename T>
__host__ __device__ __forceinline__ int oct_pitch(int C) { return sizeof(T) == 4 ? C + 2 : C + 1; }
__host__ __device__ __forceinline__ int oct_rows(int kmax, int zcols) {
    return 4 * (kmax + 1) + (zcols > 2 * (kmax + 1) ? zcols : 2 * (kmax + 1));
}
template <typename T>
__host__ __device__ __forceinline__ size_t oct_lds(int kmax, int zcols, int C) {
    return size_t(oct_rows(kmax, zcols)) * oct_pitch<T>(C) * sizeof(T);
}
constexpr size_t kOctRed = 32768;  // of the rows' LDS, for the sums over asplit

// The phase rows of C atoms, formed by the 512 threads in FP64 by the
// reference's recursion and rounded once in the mixed form.  pos(at):
// position and charge of atom `at` < na (others stand at 0 with no charge up
// to the next multiple of 16).  A barrier has to follow.
template <typename T, typename F>
__device__ __forceinline__ void oct_stage_rows(T* sm, const double* inv3, int kmax, int zcols, int C, int na, F pos) {
    const int P = oct_pitch<T>(C);
    // tasks (segment of n, axis, atom)
    const int K1 = kmax + 1, top = (na + 15) & ~15;
    const int nseg = max(1, min(512 / (3 * top), (K1 + 3) / 4)), len = (K1 + nseg - 1) / nseg;
    for (int t = threadIdx.x; t < 3 * top * nseg; t += 512) {
        const int q = t / top, at = t - q * top, seg = q / 3, axis = q - 3 * seg;
        double4 p = make_double4(0.0, 0.0, 0.0, 0.0);
        if (at < na) p = pos(at);
        const double x = axis == 0 ? p.x : (axis == 1 ? p.y : p.z);
        const double f = axis == 0 ? p.w : 1.0, inv = axis == 0 ? inv3[0] : (axis == 1 ? inv3[1] : inv3[2]);
        T* col = sm + axis * 2 * K1 * P + at;
        oct_phases(f, inv * x, seg * len, min(seg * len + len, K1), [&](int n, double ex, double ey) {
            col[2 * n * P] = (T)ex;
            col[(2 * n + 1) * P] = (T)ey;
        });
        if (axis == 2 && seg == 0)
            for (int c = 2 * K1; c < zcols; c++) col[c * P] = 0;
    }
}

// The rho partials of chunk `chunk` for the items of group `grp`: per stage
// of SA atoms (the rows are formed in `sm`, or stand there already when
// `staged`: one stage), each of the 8 waves sums its item.  Mixed form: FP32
// sums of 32 atoms, whatever the stages, added in FP64.  na atoms in the
// chunk; pos(at).
template <typename T, typename F>
__device__ __forceinline__ void oct_rho_group(const OctRho& a, int SA, int grp, int chunk, int na, bool staged, T* sm,
                                              F pos) {
    typedef typename OctT<T>::acc acc_t;
    const int P = oct_pitch<T>(SA);
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wi = w / a.asplit, ws = w - wi * a.asplit;
    const int item = grp * a.ipg + wi;
    const bool live = wi < a.ipg && item < a.nitems;
    const int i = lane & 15, k = lane >> 4;
    const int4 rw = a.rows[(live ? item : 0) * 16 + i];
    const int mask = a.mask[(live ? item : 0) * 64 + lane];
    const int ct = a.items[live ? item : 0].ct, shape = a.items[live ? item : 0].shape;
    const int ox[4] = {(rw.x & 0xffff) * P + k, (rw.y & 0xffff) * P + k, (rw.z & 0xffff) * P + k,
                       (rw.w & 0xffff) * P + k};
    const int oy[4] = {(rw.x >> 16) * P + k, (rw.y >> 16) * P + k, (rw.z >> 16) * P + k, (rw.w >> 16) * P + k};
    const int oz = (4 * (a.kmax + 1) + ct * 16 + i) * P + k, oz1 = oz + 16 * P;
    acc_t acc[4];
    oct_d4 sum[4];  // mixed form: the FP64 sums of the FP32 ones
#pragma unroll
    for (int u = 0; u < 4; u++) {
        acc[u] = acc_t{0, 0, 0, 0};
        sum[u] = oct_d4{0, 0, 0, 0};
    }
    auto flush = [&]() {
#pragma unroll
        for (int u = 0; u < 4; u++) {
#pragma unroll
            for (int v = 0; v < 4; v++) sum[u][v] += (double)acc[u][v];
            acc[u] = acc_t{0, 0, 0, 0};
        }
    };
    int held = 0;  // trips in the FP32 sums, over the stages
    for (int s0 = 0; s0 < na; s0 += SA) {
        const int ns = min(SA, na - s0);
        if (!staged) {
            if (s0 > 0) __syncthreads();  // the previous stage is summed
            oct_stage_rows<T>(sm, a.inv, a.kmax, a.zcols, SA, ns, [&](int at) { return pos(s0 + at); });
            __syncthreads();
        }
        if (live) {  // uniform over the wave
            // eight atoms per trip (more in flight would spill)
            const int Q = ((ns + 15) & ~15) >> 3, q0 = Q * ws / a.asplit, q1 = Q * (ws + 1) / a.asplit;
            auto trips = [&](auto step) {
                for (int q = q0; q < q1; q++) {
                    step(sm + 8 * q);
                    step(sm + 8 * q + 4);
                    if (sizeof(T) == 4 && (++held & 3) == 0) flush();
                }
            };
            if (shape == 0)
                trips([&](const T* base) {
                    const T A0 = base[ox[0]] * base[oy[0]], A1 = base[ox[1]] * base[oy[1]];
                    const T B0 = base[oz], B1 = base[oz1];
                    acc[0] = oct_mfma(A0, B0, acc[0]);
                    acc[1] = oct_mfma(A0, B1, acc[1]);
                    acc[2] = oct_mfma(A1, B0, acc[2]);
                    acc[3] = oct_mfma(A1, B1, acc[3]);
                });
            else
                trips([&](const T* base) {
                    const T B = base[oz];
#pragma unroll
                    for (int u = 0; u < 4; u++) acc[u] = oct_mfma(base[ox[u]] * base[oy[u]], B, acc[u]);
                });
        }
    }
    if constexpr (sizeof(T) == 4) {
        flush();
    } else {
#pragma unroll
        for (int u = 0; u < 4; u++) sum[u] = acc[u];
    }
    // the waves that share an item add up in wave order (in the rows' LDS:
    // asplit > 1 only with one group or with rows formed anew per group)
    double* red = reinterpret_cast<double*>(sm) + (size_t)wi * 16 * 64;
    for (int r = 1; r < a.asplit; r++) {  // uniform; asplit > 1 only with ipg <= 4
        __syncthreads();
        if (live && ws == r)
#pragma unroll
            for (int u = 0; u < 4; u++)
#pragma unroll
                for (int v = 0; v < 4; v++) red[(u * 4 + v) * 64 + lane] = sum[u][v];
        __syncthreads();
        if (live && ws == 0)
#pragma unroll
            for (int u = 0; u < 4; u++)
#pragma unroll
                for (int v = 0; v < 4; v++) sum[u][v] += red[(u * 4 + v) * 64 + lane];
    }
    if (live && ws == 0) {
        double4* out = a.partial + ((size_t)chunk * 4 * a.nitems + 4 * item) * 64 + lane;
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (mask >> u & 1) out[u * 64] = make_double4(sum[u][0], sum[u][1], sum[u][2], sum[u][3]);
    }
}

// ---- reduction ----------------------------------------------------------------------
// Sum of the partials over the chunks in a fixed order, the structure
// factors of the octant members, their energy and virial, and the force
// coefficients A.  Block (256 threads) = one pair of one output tile (16
// columns), 16 threads per column over the chunks c = g mod 16.
struct OctReduce {
    const double4* partial;
    int nchunks, nslots;
    const int4* slots;    // output tile: slot, row tile, column tile
    const int* kmap;      // [(tile, pair), column][sign of iky]: k-vector or -1
    int nk, nst;          // nst: steps of four columns per row tile of coef
    double2* rho;
    const double* efac;
    const double* vfac;
    double* epart;
    float* coef32;        // [row tile][step][64 lanes], one of the two
    double* coef64;
};

// lds: 8 KB.
template <bool kEnergy>
__device__ __forceinline__ void oct_reduce_block(const OctReduce& a, int blk, unsigned char* lds) {
    double4(*part)[16] = reinterpret_cast<double4(*)[16]>(lds);
    const int g = threadIdx.x >> 4, col = threadIdx.x & 15;
    const int4 sl = a.slots[blk >> 2];
    const int pair = blk & 3;
    const int2 km = reinterpret_cast<const int2*>(a.kmap)[blk * 16 + col];
    {
        // the cos and sin columns of an r that has k-vectors
        const int own = km.x >= 0 || km.y >= 0, need = own | __shfl_xor(own, 1, 64);
        const double4* src = a.partial + (size_t)sl.x * 64 + pair * 16 + col;
        double4 t = make_double4(0.0, 0.0, 0.0, 0.0);
#pragma unroll 4
        for (int c = need ? g : a.nchunks; c < a.nchunks; c += 16) {
            const double4 p = src[(size_t)c * a.nslots * 64];
            t.x += p.x;
            t.y += p.y;
            t.z += p.z;
            t.w += p.w;
        }
        part[g][col] = t;
    }
    __syncthreads();
    if (threadIdx.x >= 64) return;
    double v[7] = {0, 0, 0, 0, 0, 0, 0};
    if (threadIdx.x < 16) {
        double4 t = part[0][col];
        for (int q = 1; q < 16; q++) {
            const double4 p = part[q][col];
            t.x += p.x;
            t.y += p.y;
            t.z += p.z;
            t.w += p.w;
        }
        part[0][col] = t;
    }
    __builtin_amdgcn_wave_barrier();
    if (threadIdx.x < 16) {
        // even columns: ikz = +r, odd: ikz = -r; both read the cos and sin sums
        const double4 c = part[0][col & ~1], s = part[0][col | 1];
        const double sz = (col & 1) ? -1.0 : 1.0;
        double ac[4] = {0, 0, 0, 0}, as[4] = {0, 0, 0, 0};  // cc, cs, sc, ss
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int k = h == 0 ? km.x : km.y;
            if (k >= 0) {
                const double sy = h == 0 ? 1.0 : -1.0;
                const double re = c.x - sy * c.w - sz * (s.z + sy * s.y);
                const double im = c.z + sy * c.y + sz * (s.x - sy * s.w);
                a.rho[k] = make_double2(re, im);
                const double f = a.efac[k], gr = 2.0 * f * re, gi = 2.0 * f * im;
                ac[0] += gr;
                ac[1] += sy * gi;
                ac[2] += gi;
                ac[3] -= sy * gr;
                as[0] += sz * gi;
                as[1] -= sy * sz * gr;
                as[2] -= sz * gr;
                as[3] -= sy * sz * gi;
                if (kEnergy) {
                    const double n2 = re * re + im * im;
                    v[0] += f * n2;
                    for (int x = 0; x < 6; x++) v[1 + x] += n2 * a.vfac[(size_t)x * a.nk + k];
                }
            }
        }
        // the column's own coefficients: cos from both signs for an even
        // column, sin for an odd one
        const int cc = sl.z * 16 + col, st = cc >> 2, kk = cc & 3;
        const size_t at = ((size_t)sl.y * a.nst + st) * 64 + 16 * kk;
#pragma unroll
        for (int x = 0; x < 4; x++) {
            const double oc = ac[x] + __shfl_xor(ac[x], 1, 64), os = as[x] + __shfl_xor(as[x], 1, 64);
            const double val = (col & 1) ? os : oc;
            if (a.coef32)
                a.coef32[at + OctT<float>::row_of(pair, x)] = (float)val;
            else
                a.coef64[at + OctT<double>::row_of(pair, x)] = val;
        }
    }
    if (kEnergy) {
        for (int x = 0; x < 7; x++) {
            double sum = wave_sum(v[x]);
            if (threadIdx.x == 0) a.epart[blk * 7 + x] = sum;
        }
    }
}

// ---- forces -------------------------------------------------------------------------
struct OctForce {
    double kg[3];       // 2 pi / L
    const void* coef;   // [row tile][nst][64 lanes] of T
    const int* pairs;   // p | q << 16, four per row tile
    const int* steps;   // steps of four columns per row tile (<= nst)
    int nrt, nst;
};

// k-space forces of the C atoms whose rows stand in `sm` (oct_stage_rows), by
// 8 waves.  Leaves in res[d * C + atom] the sums q_i sum_k Im(e^{i k.r} conj
// rho_k) 2 factor_k k (ewald.rs:699-719 but for 1 / (4 pi eps0)); a barrier
// ends it.  The units of work (16 atoms, row tile) are dealt to the waves in
// contiguous ranges, atoms outermost, so any number of 16-atom groups keeps
// all of them busy; a wave adds up its row tiles per group and the groups'
// parts are added in wave order.  A row tile's coefficients are read in lane
// order, one coalesced load per two matrix instructions, one unit ahead; the
// Z operands of the group and their z derivatives stay in registers.  NST:
// steps of four columns (0: any number, the operands read at every step).
constexpr int kOctMaxGroups = 16;
template <typename T, int NST>
struct OctUnit {  // a row tile's coefficients, steps and pair of this lane
    T cf[NST > 0 ? NST : 1];
    int ns, pk;
};
template <typename T, int NST>
__device__ __forceinline__ void oct_load_unit(const OctForce& a, int rt, OctUnit<T, NST>& u) {
    const int lane = threadIdx.x & 63;
    if constexpr (NST > 0) {
        const T* coef = reinterpret_cast<const T*>(a.coef) + (size_t)rt * a.nst * 64 + lane;
#pragma unroll
        for (int q = 0; q < NST; q++) u.cf[q] = coef[q * 64];
    }
    u.ns = a.steps[rt];
    u.pk = a.pairs[rt * 4 + (lane >> 4)];
}
__device__ __forceinline__ int oct_unit0(int units, int w) { return units * w / 8; }

template <typename T, int NST>
__device__ __forceinline__ void oct_force_sums(const OctForce& a, int kmax, int C, const T* sm,
                                               double (*red)[3][3][16], double* res, OctUnit<T, NST> nxt) {
    typedef typename OctT<T>::acc acc_t;
    const int P = oct_pitch<T>(C), G = C >> 4, nrt = a.nrt;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int k = lane >> 4;
    const int K1 = kmax + 1;
    const int u0 = oct_unit0(G * nrt, w), u1 = oct_unit0(G * nrt, w + 1), g0 = u0 / nrt;
    double fx = 0.0, fy = 0.0, fz = 0.0;
    int g = g0, rt = u0 - g0 * nrt, gz = -1;
    T z[NST > 0 ? NST : 1], dz[NST > 0 ? NST : 1];
    for (int u = u0; u < u1; u++) {
        const OctUnit<T, NST> cur = nxt;
        const int next = rt + 1 < nrt ? rt + 1 : 0;
        oct_load_unit<T, NST>(a, next, nxt);
        const T* row = sm + 16 * g + (lane & 15);
        const T* zr = row + (4 * K1 + k) * P;
        // operand B: column kk = 4 st + k of the atom: r = 2 st + k / 2, cos or sin
        auto zop = [&](int st, T& zz, T& dd) {
            zz = zr[4 * st * P];
            const T o = zr[(4 * st + ((k & 1) ? -1 : 1)) * P];
            dd = (T)(2 * st + (k >> 1)) * ((k & 1) ? o : -o);
        };
        acc_t S = {0, 0, 0, 0}, D = {0, 0, 0, 0};
        if constexpr (NST > 0) {
            if (g != gz) {  // uniform
#pragma unroll
                for (int st = 0; st < NST; st++) zop(st, z[st], dz[st]);
                gz = g;
            }
#pragma unroll
            for (int st = 0; st < NST; st++)
                if (st < cur.ns) {  // uniform
                    S = oct_mfma(cur.cf[st], z[st], S);
                    D = oct_mfma(cur.cf[st], dz[st], D);
                }
        } else {
            const T* coef = reinterpret_cast<const T*>(a.coef) + (size_t)rt * a.nst * 64 + lane;
            for (int st = 0; st < cur.ns; st++) {
                const T c = coef[st * 64];
                T zz, dd;
                zop(st, zz, dd);
                S = oct_mfma(c, zz, S);
                D = oct_mfma(c, dd, D);
            }
        }
        // this lane: pair k of the tile; registers cc, cs, sc, ss
        const int p = cur.pk & 0xffff, q = cur.pk >> 16;
        const T Xc = row[2 * p * P], Xs = row[(2 * p + 1) * P];
        const T Yc = row[(2 * K1 + 2 * q) * P], Ys = row[(2 * K1 + 2 * q + 1) * P];
        const T uu = Yc * S[0] + Ys * S[1], v = Yc * S[2] + Ys * S[3];
        const T uy = Yc * S[1] - Ys * S[0], vy = Yc * S[3] - Ys * S[2];
        const T ud = Yc * D[0] + Ys * D[1], vd = Yc * D[2] + Ys * D[3];
        // -grad Phi: X' = p (-s, c), Y' = q (-s, c)
        fx += (double)((T)p * (Xs * uu - Xc * v));
        fy -= (double)((T)q * (Xc * uy + Xs * vy));
        fz -= (double)(Xc * ud + Xs * vd);
        rt = next;
        if (rt == 0 || u + 1 == u1) {  // uniform: the group's last unit of this wave
            double f[3] = {fx, fy, fz};
#pragma unroll
            for (int d = 0; d < 3; d++) {
                f[d] += __shfl_xor(f[d], 16, 64);
                f[d] += __shfl_xor(f[d], 32, 64);
                if (lane < 16) red[w][g - g0][d][lane] = f[d];
            }
            fx = fy = fz = 0.0;
            g++;
        }
    }
    __syncthreads();
    for (int t = tid; t < 3 * C; t += 512) {
        const int d = t / C, i = t - d * C, gi = i >> 4;
        double s = 0.0;
        for (int v = 0; v < 8; v++) {
            const int b0 = oct_unit0(G * nrt, v), b1 = oct_unit0(G * nrt, v + 1), f0 = b0 / nrt;
            if (b0 < b1 && f0 <= gi && gi <= (b1 - 1) / nrt) s += red[v][gi - f0][d][i & 15];
        }
        res[t] = a.kg[d] * s;
    }
    __syncthreads();
}

}  // namespace lg
