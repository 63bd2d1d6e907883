// Whole chains of slice products in one launch, on strips of 16 or 32 columns.
//
// A suffix chain S_t = D_t A S_{t+1} multiplies from the left, so each column of S evolves by
// itself; a right chain R_tau = R_{tau-1} D_tau A evolves each row of R by itself.  A workgroup
// therefore owns 16 CT columns of S (rows of R) of one chain, a strip X[c][i] (c: column of S or
// row of R), and runs all its slices without meeting another workgroup: X_new[c][i] = sum_k
// X[c][k] A[k][i] (A is symmetric), scaled by phases along i.  One launch per chain instead of one
// per slice; the strip stays in LDS between two slices, and a right chain's products never reach
// memory (its force diagonal is formed from the accumulators).
//
// A wave owns RT tiles of 16 columns i for 16 rows c: the strip is the A operand of the 16x16x4
// MFMA, the slice matrix the B operand, and lane (lk, lr) = (lane / 16, lane % 16) ends with
// X_new[acc_row(lk, r)][lr], r = 0..3.  So a phase is one value per lane and tile, and the diagonal's
// sum over c runs over a lane's own four entries and two cross-lane steps.  Operands are read in
// units of 8 (FP64) or 16 (FP32) k, 16 bytes per lane: the strip from LDS in operand order
// ([unit][plane][column tile][lane], the lanes' slots XOR-swizzled so that the stores of the
// transposed accumulators spread over the banks), A from L2 in the same order (chain_pack_kernel),
// PF units ahead of its use; the ring runs on into the next slice, over its barriers and stores.
// NU > 0: A held in registers for the whole chain (n <= 128, where a slice is too short to hide
// the L2 latency).
//
// What bounds it: the matrix cores.  256 chains of 32 slices at n = 288 take 11.2 ms (68.0 TFLOP/s of
// the 76.5 that a bare FP64 MFMA loop reaches; one launch per slice: 12.2 ms) and 6.8 ms for the FP32
// right chains (115 of 155 TFLOP/s; 8.7 ms).  With few chains the slices in sequence bound it: 2.6 us
// per slice at n = 72 (13 us as a launch of its own), 23 us at n = 288.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "gemm.hpp"

namespace isle {

constexpr int CHAIN_MAX_RES = 128;  // largest order with A held in registers

// One unit of k: 16 bytes per lane of each operand, KS MFMA steps.
template <typename T>
struct ChainUnit;
template <>
struct ChainUnit<double> {
    typedef double vec __attribute__((ext_vector_type(2)));
    static constexpr int KS = 2, PER_TILE = 2;
};
template <>
struct ChainUnit<float> {
    typedef float vec __attribute__((ext_vector_type(4)));
    static constexpr int KS = 4, PER_TILE = 1;
};

inline int chain_tiles(int n) { return (n + 15) / 16; }
// units of k that hold rows of the matrix, and the units of all its tiles
template <typename T>
__host__ __device__ inline int chain_units(int n) {
    return ChainUnit<T>::PER_TILE == 2 ? (n + 7) / 8 : (n + 15) / 16;
}
template <typename T>
inline size_t chain_packed_elems(int n) {
    return (size_t)chain_tiles(n) * chain_units<T>(n) * 64 * (16 / sizeof(T));
}
// LDS: the strip (both planes of every tile), then the slice's factors
template <typename T>
inline size_t chain_lds(int n, int ct) {
    return (size_t)chain_tiles(n) * (ChainUnit<T>::PER_TILE * 2 * 64 * 16 * ct + 2 * 16 * sizeof(T));
}
// Orders that the strip kernels take: an FP64 strip has to fit the 160 KB LDS of a CU, and the
// tiles of a wave its registers (8 waves of four tiles).
constexpr int CHAIN_MAX_N = 512;
inline bool chain_fits(int n) { return n <= CHAIN_MAX_N; }

// k of element e of lane group lk in unit u.  FP64 in the order of four consecutive k per MFMA step:
// the order in which gemm_rcd_kernel and gemm_kernel sum, so the products agree with theirs to the
// last bit; FP32 as gemm_rck_kernel.
template <typename T>
__host__ __device__ inline int chain_k(int u, int lk, int e) {
    return sizeof(T) == 8 ? 8 * u + 4 * e + lk : 16 * u + 4 * lk + e;
}

// out[tile][unit][lane][e] = A[chain_k(unit, lk, e)][16 tile + lr], 0 outside
template <typename T>
__global__ __launch_bounds__(256) void chain_pack_kernel(const double* __restrict__ a, int n, T* __restrict__ out,
                                                         long total) {
    constexpr int E = 16 / sizeof(T);
    const int units = chain_units<T>(n);
    for (long o = blockIdx.x * 256L + threadIdx.x; o < total; o += (long)gridDim.x * 256) {
        const int e = (int)(o % E), lane = (int)(o / E % 64);
        const long tu = o / E / 64;
        const int k = chain_k<T>((int)(tu % units), lane >> 4, e), i = 16 * (int)(tu / units) + (lane & 15);
        out[o] = i < n && k < n ? (T)a[(long)k * n + i] : T(0);
    }
}

// Suffix chain of one group of slices:  S_f = D_f A, then S_t = D_t A S_{t - dir} for the slices
// after f in direction dir (-1: from the group's last slice to its first).  pre: the phases on the
// other side, S_f = A D_f, S_t = A D_t S_{t - dir}; stored transposed these are, A being symmetric,
// the prefix products D_f A D_{f + dir} A ... D_t A.
struct SuffixItem {
    const double* packed;       // A in chain_pack_kernel's order
    const double* a;            // A, n x n row-major
    const double* d_re;         // phases of slice 0, slice t at + t n
    const double* d_im;
    double* out;                // S_f transposed: re plane, im plane n n after it; each next one at
    long step;                  // + step; the last one is stored as it is, not transposed
    int first, dir, count;      // slice f, -1 or +1, slices in the group
    int all;                    // 1: store every S_t; 0: store the last one only (at out)
    int pre;
    int keep = 0;               // 1: the last one transposed like the others
};

// Right chain of one group:  R_s = K D_s A, R_t = R_{t-1} D_t A, and the force diagonal
// f[t]_i = sum_c R_t[c][i] Suf_{t+1}[i][c] (t < e), f[e]_i = R_e[i][i], as partial sums over 16 c.
template <typename T>
struct RightItem {
    const T* packed;
    const double* k_re;         // K, row stride ldk, times sign
    const double* k_im;
    long ldk;
    double sign;
    const double* d0_re;        // FP64 phases of slice s (applied to K before rounding to T)
    const double* d0_im;
    const T* d_re;              // phases of slice 0 in T, slice t at + t n
    const T* d_im;
    const double* suf;          // Suf_{s+1} transposed: re plane, im plane n n after it; Suf_{s+1+q}
    long step;                  // at + q step; readable for 32 n doubles beyond the last plane
    double* part;               // [count][tiles][n] complex partial sums
    int s, count;
};

// p[lane offset in bytes] with p uniform over the wave: one address register for all accesses
template <typename T>
__device__ __forceinline__ T ld_lane(const T* p, unsigned bytes) {
    return ld_global(reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + bytes));
}
template <typename T>
__device__ __forceinline__ void st_lane(T* p, unsigned bytes, T v) {
    st_global(reinterpret_cast<T*>(reinterpret_cast<char*>(p) + bytes), v);
}
// row of accumulator entry r at lane group lk = acc_row<T>(lk, 0) + r chain_rstep
template <typename T>
constexpr int chain_rstep() {
    return sizeof(T) == 8 ? 4 : 1;
}

__device__ __forceinline__ void chain_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <typename T>
__device__ __forceinline__ typename Acc4<T>::type chain_zero() {
    typename Acc4<T>::type v = {0, 0, 0, 0};
    return v;
}

// Slot of row c in lane group lk of a unit: rows XORed with 4 lk (FP64) or lk (FP32), so that the
// stores of an accumulator entry (16 columns of 4 rows per instruction) spread over all banks.
template <typename T>
__device__ __forceinline__ int chain_slot(int lk, int c) {
    return lk * 16 + (c ^ (sizeof(T) == 8 ? 4 * lk : lk));
}

// The MFMA loop of one slice: acc = X A for this wave's RT tiles.  NU > 0: A in registers; NU == 0:
// streamed through a ring of PF units (slot q of the ring ends a slice with unit q).
template <typename T, int RT, int NU, int CT>
struct ChainLoop {
    typedef typename ChainUnit<T>::vec vec;
    typedef typename Acc4<T>::type V4;
    static constexpr int KS = ChainUnit<T>::KS;
    static constexpr int PF = NU > 0 ? NU : 2;
    vec a[PF][RT];
    const vec* ap[RT];  // operand of unit 0 of each tile (uniform over the wave)
    unsigned off;       // this lane's bytes in a unit's operand
    int units;

    __device__ __forceinline__ void init(const T* packed, int tile0, int ntiles, int nunits, int lane) {
        units = nunits;
        off = 16u * (unsigned)lane;
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            const int t = min(tile0 + i, ntiles - 1);  // surplus tiles repeat the last one, unstored
            ap[i] = reinterpret_cast<const vec*>(packed) + (long)t * units * 64;
        }
#pragma unroll
        for (int u = 0; u < PF; ++u) load(u, min(u, units - 1));
    }
    __device__ __forceinline__ void load(int q, int u) {
        unsigned o = off;
        asm volatile("" : "+v"(o));  // a scalar base and this offset, no 64-bit address kept per tile
#pragma unroll
        for (int i = 0; i < RT; ++i) a[q][i] = ld_lane(ap[i] + u * 64, o);
    }
    __device__ __forceinline__ void step(const vec (&av)[RT], const vec* x, V4 (&re)[RT], V4 (&im)[RT]) {
        const vec xr = x[0], xi = x[64 * CT];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                re[i] = mfma16(xr[ks], av[i][ks], re[i]);
                im[i] = mfma16(xi[ks], av[i][ks], im[i]);
            }
    }
    // x: this lane's slot of its column tile in unit 0
    __device__ __forceinline__ void run(const vec* x, V4 (&re)[RT], V4 (&im)[RT]) {
#pragma unroll
        for (int i = 0; i < RT; ++i) re[i] = im[i] = chain_zero<T>();
        if constexpr (NU > 0) {
#pragma unroll
            for (int u = 0; u < NU; ++u) step(a[u], x + u * 128 * CT, re, im);
        } else {
            int u = 0;
            for (; u + PF <= units; u += PF) {
#pragma unroll
                for (int q = 0; q < PF; ++q) {
                    step(a[q], x + (u + q) * 128 * CT, re, im);
                    load(q, u + q + PF < units ? u + q + PF : q);
                    __builtin_amdgcn_sched_barrier(0);  // the loads leave here, PF - 1 units before their use
                }
            }
#pragma unroll
            for (int q = 0; q < PF - 1; ++q)
                if (u + q < units) {
                    step(a[q], x + (u + q) * 128 * CT, re, im);
                    load(q, q);
                }
        }
    }
};

// This wave's entries of tile `tile` into the strip, at the slots that chain_k gives their columns.
// base: the column tile's slots of unit 0.
template <typename T, int CT>
__device__ __forceinline__ void chain_put(T* base, int tile, int lane, const typename Acc4<T>::type& re,
                                          const typename Acc4<T>::type& im) {
    constexpr int E = 16 / sizeof(T), UE = 128 * CT * E;  // elements of a unit (both planes)
    const int lr = lane & 15, lk = lane >> 4;
    const int u = tile * ChainUnit<T>::PER_TILE + lr / (4 * E);
    const int g = E == 2 ? lr & 3 : lr >> 2, e = E == 2 ? (lr >> 2) & 1 : lr & 3;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        T* p = base + u * UE + chain_slot<T>(g, acc_row<T>(lk, r)) * E + e;
        p[0] = re[r];
        p[64 * CT * E] = im[r];
    }
}

// The two factor planes of a slice on their way into LDS
template <typename T, int MAXR>
struct ChainFactors {
    T v[MAXR];
    __device__ __forceinline__ void load(const T* re, const T* im, int n, int tid, int nth) {
#pragma unroll
        for (int q = 0; q < MAXR; ++q) {
            const int e = tid + q * nth;
            v[q] = e < n ? ld_global(re + e) : (e < 2 * n ? ld_global(im + (e - n)) : T(0));
        }
    }
    __device__ __forceinline__ void put(T* fac, int n, int np, int tid, int nth) const {
#pragma unroll
        for (int q = 0; q < MAXR; ++q) {
            const int e = tid + q * nth;
            if (e < n)
                fac[e] = v[q];
            else if (e < 2 * n)
                fac[np + (e - n)] = v[q];
        }
    }
};

// Most threads of a workgroup with RT tiles per wave and CT column tiles (chain_dispatch keeps to
// them): what the registers of the streamed forms leave room for.
template <int RT, int NU, int CT>
constexpr int chain_threads() {
    return NU > 0 ? 512 : CT == 2 ? 768 : RT == 1 ? 1024 : RT == 2 ? 768 : 512;
}

// Rounds of a block of 64 ceil(tiles / RT) threads over 2 n <= 32 tiles values
template <int RT>
constexpr int chain_rounds() {
    return (RT + 1) / 2;
}

// Sum over the four lane groups of a wave (lanes l, l ^ 16, l ^ 32, l ^ 48)
__device__ __forceinline__ double chain_sum4(double v) {
    const long long b = __double_as_longlong(v);
    auto l = __builtin_amdgcn_permlane32_swap((unsigned)b, (unsigned)b, false, false);
    auto h = __builtin_amdgcn_permlane32_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
    v = __longlong_as_double(((long long)h[0] << 32) | l[0]) + __longlong_as_double(((long long)h[1] << 32) | l[1]);
    const long long c = __double_as_longlong(v);
    l = __builtin_amdgcn_permlane16_swap((unsigned)c, (unsigned)c, false, false);
    h = __builtin_amdgcn_permlane16_swap((unsigned)(c >> 32), (unsigned)(c >> 32), false, false);
    return __longlong_as_double(((long long)h[0] << 32) | l[0]) + __longlong_as_double(((long long)h[1] << 32) | l[1]);
}

template <int RT, int NU, int CT>
__global__ __launch_bounds__((chain_threads<RT, NU, CT>()), 1)
void suffix_chain_kernel(const SuffixItem* __restrict__ items, int n, int ntiles) {
    typedef ChainUnit<double>::vec vec;
    extern __shared__ __align__(16) unsigned char chain_raw[];
    double* strip = reinterpret_cast<double*>(chain_raw);
    double* fac = strip + ntiles * 512 * CT;
    const int np = ntiles * 16, strips = (ntiles + CT - 1) / CT;
    const SuffixItem it = items[blockIdx.x / strips];
    const int tid = threadIdx.x, nth = blockDim.x, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), tile0 = wave / CT * RT;
    const int c0 = ((int)(blockIdx.x % strips) * CT + wave % CT) * 16;  // first of this wave's rows c
    double* mine = strip + (wave % CT) * 128;
    const vec* x = reinterpret_cast<const vec*>(mine) + chain_slot<double>(lk, lr);
    const long nn = (long)n * n;
    const unsigned off = 8u * (unsigned)((c0 + lk) * n + lr);  // element (c0 + lk, lr) of a plane
    ChainLoop<double, RT, NU, CT> loop;
    loop.init(it.packed, tile0, ntiles, chain_units<double>(n), lane);
    for (int e = tid; e < 2 * np; e += nth) fac[e] = 0.0;
    dbl4 re[RT], im[RT];
    ChainFactors<double, chain_rounds<RT>()> fv;
    // the factors of step q: slice first + q dir, with pre the next one (none in the last step)
    const long dn = (long)it.dir * n;
    const double *dr = it.d_re + (long)(it.first + it.pre * it.dir) * n, *di = dr + (it.d_im - it.d_re);
    const int nfac = it.count - it.pre;
    if (nfac > 0) fv.load(dr, di, n, tid, nth);
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {  // the chain starts from A itself
            const int c = c0 + 4 * r + lk, j = (tile0 + i) * 16 + lr;
            const bool in = c < n && j < n;
            const double v = in ? ld_global(it.a + (long)c * n + j) : 0.0;
            re[i][r] = in && it.pre ? v * ld_global(it.d_re + (long)it.first * n + c) : v;
            im[i][r] = in && it.pre ? v * ld_global(it.d_im + (long)it.first * n + c) : 0.0;
        }
    double* out = it.out;
    chain_barrier();
    if (nfac > 0) fv.put(fac, n, np, tid, nth);
    if (nfac > 1) fv.load(dr + dn, di + dn, n, tid, nth);
    chain_barrier();
    for (int q = 0;; ++q) {  // fac: the factors of step q
        const bool last = q == it.count - 1;
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            const int tile = tile0 + i;
            if (tile >= ntiles) continue;
            const int j = tile * 16 + lr;
            const double fr = q < nfac ? fac[j] : 1.0, fi = q < nfac ? fac[np + j] : 0.0;
            dbl4 vr, vi;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                vr[r] = j < n ? re[i][r] * fr - im[i][r] * fi : 0.0;
                vi[r] = j < n ? re[i][r] * fi + im[i][r] * fr : 0.0;
            }
            if (!last) {
                chain_put<double, CT>(mine, tile, lane, vr, vi);
                if (it.all) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        double* o = out + (tile * 16 + 4 * r * n);
                        if (c0 + 4 * r + lk < n && j < n) {
                            st_lane(o, off, it.pre ? re[i][r] : vr[r]);
                            st_lane(o + nn, off, it.pre ? im[i][r] : vi[r]);
                        }
                    }
                }
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int c = c0 + 4 * r + lk;
                    if (c < n && j < n) {
                        const long o = it.keep ? (long)c * n + j : (long)j * n + c;
                        st_global(out + o, vr[r]);
                        st_global(out + nn + o, vi[r]);
                    }
                }
            }
        }
        if (last) return;
        if (it.all) out += it.step;
        chain_barrier();  // the strip is complete, the factors are read
        if (q + 1 < nfac) fv.put(fac, n, np, tid, nth);
        if (q + 2 < nfac) fv.load(dr + (q + 2) * dn, di + (q + 2) * dn, n, tid, nth);
        loop.run(x, re, im);
        chain_barrier();  // every wave has read the strip
    }
}

template <typename T, int RT, int NU, int CT>
__global__ __launch_bounds__((chain_threads<RT, NU, CT>()), 1)
void right_chain_kernel(const RightItem<T>* __restrict__ items, int n, int ntiles) {
    typedef typename ChainUnit<T>::vec vec;
    typedef typename Acc4<T>::type V4;
    constexpr int E = 16 / sizeof(T);
    extern __shared__ __align__(16) unsigned char chain_raw[];
    T* strip = reinterpret_cast<T*>(chain_raw);
    T* fac = strip + ntiles * (ChainUnit<T>::PER_TILE * 128 * E) * CT;
    const int np = ntiles * 16, strips = (ntiles + CT - 1) / CT;
    const RightItem<T> it = items[blockIdx.x / strips];
    const int tid = threadIdx.x, nth = blockDim.x, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), tile0 = wave / CT * RT;
    const int ctile = (int)(blockIdx.x % strips) * CT + wave % CT, c0 = ctile * 16;
    T* mine = strip + (wave % CT) * 64 * E;
    const vec* x = reinterpret_cast<const vec*>(mine) + chain_slot<T>(lk, lr);
    const long nn = (long)n * n;
    const int lrow = acc_row<T>(lk, 0);
    const unsigned off = 8u * (unsigned)((c0 + lrow) * n + lr);  // element (c0 + lrow, lr) of a plane
    ChainLoop<T, RT, NU, CT> loop;
    loop.init(it.packed, tile0, ntiles, chain_units<T>(n), lane);
    for (int e = tid; e < 2 * np; e += nth) fac[e] = T(0);
    ChainFactors<T, chain_rounds<RT>()> fv;  // the factors of the next slice
    if (it.count > 1) fv.load(it.d_re + (long)(it.s + 1) * n, it.d_im + (long)(it.s + 1) * n, n, tid, nth);
    const double* suf = it.suf;
    double lre[RT][4], lim[RT][4];  // the left factor's entries of a step, in flight during its product
    auto load_left = [&](int i) {  // beyond row or column n: masked below
        const int tile = min(tile0 + i, ntiles - 1);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const double* l = suf + (tile * 16 + chain_rstep<T>() * r * n);
            lre[i][r] = ld_lane(l, off);
            lim[i][r] = ld_lane(l + nn, off);
        }
    };
    V4 re[RT], im[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        const int tile = tile0 + i, j = tile * 16 + lr;
        V4 vr, vi;
        const double dr = j < n ? ld_global(it.d0_re + j) : 0.0, di = j < n ? ld_global(it.d0_im + j) : 0.0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {  // K D_s
            const int c = c0 + acc_row<T>(lk, r);
            const bool in = c < n && j < n;
            const long o = in ? (long)c * it.ldk + j : 0;
            const double kr = in ? it.sign * ld_global(it.k_re + o) : 0.0;
            const double ki = in ? it.sign * ld_global(it.k_im + o) : 0.0;
            vr[r] = (T)(kr * dr - ki * di);
            vi[r] = (T)(kr * di + ki * dr);
        }
        if (tile < ntiles) chain_put<T, CT>(mine, tile, lane, vr, vi);
        if (it.count > 1) load_left(i);
    }
    double* part = it.part + (long)ctile * n * 2;
    const long part_step = (long)ntiles * n * 2;
    for (int q = 0; q < it.count; ++q) {
        const bool last = q == it.count - 1;
        chain_barrier();  // the strip is complete, the factors are read
        if (!last) fv.put(fac, n, np, tid, nth);
        if (q + 2 < it.count)
            fv.load(it.d_re + (long)(it.s + q + 2) * n, it.d_im + (long)(it.s + q + 2) * n, n, tid, nth);
        loop.run(x, re, im);
        chain_barrier();  // every wave has read the strip
        suf += it.step;
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            const int tile = tile0 + i, j = tile * 16 + lr;
            if (tile >= ntiles) continue;
            double sr = 0, si = 0;
            if (last) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const bool d = c0 + acc_row<T>(lk, r) == j;
                    sr += d ? (double)re[i][r] : 0.0;
                    si += d ? (double)im[i][r] : 0.0;
                }
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const bool in = c0 + acc_row<T>(lk, r) < n && j < n;
                    const double xr = re[i][r], xi = im[i][r];
                    const double a = in ? lre[i][r] : 0.0, b = in ? lim[i][r] : 0.0;
                    sr = fma(a, xr, fma(-b, xi, sr));
                    si = fma(a, xi, fma(b, xr, si));
                }
                if (q + 2 < it.count) load_left(i);
            }
            sr = chain_sum4(sr);
            si = chain_sum4(si);
            if (lk == 0 && j < n && ctile < ntiles) {
                typedef double dbl2 __attribute__((ext_vector_type(2)));
                st_global(reinterpret_cast<dbl2*>(part + 2 * j), dbl2{sr, si});
            }
            if (!last) {
                const T dr = fac[j], di = fac[np + j];
                V4 vr, vi;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    vr[r] = j < n ? re[i][r] * dr - im[i][r] * di : T(0);
                    vi[r] = j < n ? re[i][r] * di + im[i][r] * dr : T(0);
                }
                chain_put<T, CT>(mine, tile, lane, vr, vi);
            }
        }
        part += part_step;
    }
}

// f(RT, NU, CT, waves) with U = the units of n
template <int U, typename F>
inline void chain_resident(int u, int nw, F&& f) {
    if (u == U)
        f(std::integral_constant<int, 1>{}, std::integral_constant<int, U>{}, std::integral_constant<int, 1>{}, nw);
    else if constexpr (U > 1)
        chain_resident<U - 1>(u, nw, f);
}

// The streamed forms: tiles per wave RT, column tiles per strip CT, most waves of a workgroup.  ({3, 1} costs more
// than one of the others, or as much on fewer waves, at every order from 129 to 512.)
struct ChainShape {
    int rt, ct, waves;
};
constexpr ChainShape CHAIN_SHAPES[] = {{1, 1, 16}, {2, 1, 12}, {4, 1, 8}, {5, 1, 8}, {3, 2, 12}};

// Tile products of the busiest SIMD of a CU per slice, the strips of nitems chains dealt to the CUs in
// rounds: workgroups that share a CU put their first waves on the same SIMDs, so its tiles are those of
// ceil(waves / 4) waves however many workgroups there are.  At n = 288 (18 tiles) 5 tiles with one
// column tile on 4 waves (6 waves of 3 tiles: 6), 9 with two on 12 waves: 256 chains of 32 slices take
// 12.1 ms with {5, 1}, 16.0 with {3, 1}, 11.2 with {3, 2}; two chains of 96 slices 2.21, 2.55, 3.69 ms.
inline long chain_cost(const ChainShape& sh, int ntiles, int nitems, int cus) {
    const int nw = (ntiles + sh.rt - 1) / sh.rt * sh.ct;
    const long wgs = (long)((ntiles + sh.ct - 1) / sh.ct) * nitems;
    return (wgs + cus - 1) / cus * ((nw + 3) / 4 * sh.rt);
}
template <typename T>
inline int chain_shape(int n, int nitems, int cus) {
    const int nt = chain_tiles(n);
    int best = -1, waves = 0;
    long cost = 0;
    for (int i = 0; i < 5; ++i) {
        const ChainShape& sh = CHAIN_SHAPES[i];
        const int nw = (nt + sh.rt - 1) / sh.rt * sh.ct;
        if (nw > sh.waves || chain_lds<T>(n, sh.ct) > 160 * 1024) continue;
        const long c = chain_cost(sh, nt, nitems, cus);
        if (best < 0 || c < cost || (c == cost && nw > waves)) {  // ties: more waves hide more latency
            best = i;
            cost = c;
            waves = nw;
        }
    }
    return best;
}
constexpr int CHAIN_CUS = 256;

// Calls f(RT, NU, CT, waves) with the form of order n for nitems chains: A in registers up to
// CHAIN_MAX_RES (one tile per wave, NU = the units of n), else streamed.
template <typename T, typename F>
inline void chain_dispatch(int n, int nitems, F&& f) {
    const int nt = chain_tiles(n);
    if (n <= CHAIN_MAX_RES) return chain_resident<CHAIN_MAX_RES / 16 * ChainUnit<T>::PER_TILE>(chain_units<T>(n), nt, f);
    const int i = chain_shape<T>(n, nitems, CHAIN_CUS);
    const int nw = (nt + CHAIN_SHAPES[i].rt - 1) / CHAIN_SHAPES[i].rt * CHAIN_SHAPES[i].ct;
    const std::integral_constant<int, 0> st;
    const std::integral_constant<int, 1> c1;
    switch (i) {
    case 0: return f(std::integral_constant<int, 1>{}, st, c1, nw);
    case 1: return f(std::integral_constant<int, 2>{}, st, c1, nw);
    case 2: return f(std::integral_constant<int, 4>{}, st, c1, nw);
    case 3: return f(std::integral_constant<int, 5>{}, st, c1, nw);
    default: return f(std::integral_constant<int, 3>{}, st, std::integral_constant<int, 2>{}, nw);
    }
}

template <typename T, int CT, typename Kern, typename Item>
inline void launch_chain(Kern kern, const Item* d_items, int nitems, int n, int nw, hipStream_t s) {
    const size_t lds = chain_lds<T>(n, CT);
    ISLE_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                 (int)lds));
    const int nt = chain_tiles(n);
    hipLaunchKernelGGL(kern, dim3((unsigned)((nt + CT - 1) / CT * nitems)), dim3(64 * nw), lds, s, d_items, n, nt);
    ISLE_HIP(hipGetLastError());
}

inline void launch_suffix_chain(const SuffixItem* d_items, int nitems, int n, hipStream_t s) {
    chain_dispatch<double>(n, nitems, [&](auto rt, auto nu, auto ct, int nw) {
        constexpr int RT = decltype(rt)::value, NU = decltype(nu)::value, CT = decltype(ct)::value;
        launch_chain<double, CT>(suffix_chain_kernel<RT, NU, CT>, d_items, nitems, n, nw, s);
    });
}

template <typename T>
inline void launch_right_chain(const RightItem<T>* d_items, int nitems, int n, hipStream_t s) {
    chain_dispatch<T>(n, nitems, [&](auto rt, auto nu, auto ct, int nw) {
        constexpr int RT = decltype(rt)::value, NU = decltype(nu)::value, CT = decltype(ct)::value;
        launch_chain<T, CT>(right_chain_kernel<T, RT, NU, CT>, d_items, nitems, n, nw, s);
    });
}

}  // namespace isle
