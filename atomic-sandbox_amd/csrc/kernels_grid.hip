// gfx950 kernels on the dense n^3 grid: the block stencil H.X, reductions, the tall-skinny Gram S^T U, block
// linear combinations, density accumulation, LSDA, nuclear potential, orbital guess, DIIS mix and HF forces.
// All kernels are written for 64-wide wavefronts; reductions are deterministic (fixed partial counts, fixed order).
#include "gram_plan.hpp"
#include "lira_internal.hpp"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <type_traits>
#include <vector>

namespace lira {

void check_hip(hipError_t e, const char *what) {
    if (e != hipSuccess) throw DeviceError(std::string(what) + ": " + hipGetErrorString(e));
}

void DevBuf::alloc(size_t b) {
    release();
    if (b == 0) b = 256;
    LIRA_HIP(hipMalloc(&ptr, b));
    bytes = b;
}

void DevBuf::release() {
    if (ptr) (void)hipFree(ptr);
    ptr = nullptr;
    bytes = 0;
}

// 8th-order second-derivative coefficients c1..c4 (qm/src/stencil.rs:24), c0 = -205/72 = -2 sum c_m. The kernels use
// their partial sums in their own precision (StCoef below): a bare double constant would promote an f32 stencil's products
// to f64.
#define C1 (8.0 / 5.0)
#define C2 (-1.0 / 5.0)
#define C3 (8.0 / 315.0)
#define C4 (-1.0 / 560.0)

// ---- buffer addressing of the stencil fields ----
// The stencils read and write whole fields through raw buffer descriptors whose range is one field. A load at a byte
// offset outside [0, range) returns 0 -- the Dirichlet zero of every out-of-box neighbour -- and a store there is
// dropped, so no load or store sits in a branch (a bounds branch around each load forces a wait for every load in
// flight at the join, which would serialise the look-ahead). A lane's (x, y) position gets the byte offset of its row in
// a plane, or BUF_OOB when (x, y) lies outside the box; plane z adds z * plane_bytes in 32-bit unsigned arithmetic, so
// z < 0 wraps to >= 2^31 and z >= n lands at or past the end. Both stay out of range while
// (N + 4 n^2) * sizeof(T) < 2^31, which the host launchers check.
constexpr unsigned BUF_OOB = 0x80000000u;
typedef __amdgpu_buffer_rsrc_t BufRes;
__device__ __forceinline__ BufRes field_res(const void *base, long bytes) {
    // word 3 = 0x00020000: 32-bit data format, no swizzle, raw addressing (the gfx9 family's value). Opaque to the compiler,
    // so that each descriptor keeps its four registers: it shared the equal words 2 and 3 of a kernel's descriptors and
    // moved them at every use (95^3 x 16 f32 31.4 us, 31.0 without).
    int range = (int)bytes, format = 0x00020000;
    asm volatile("" : "+s"(range), "+s"(format));
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, range, format);
}
__device__ __forceinline__ unsigned row_off(int xx, int yy, int n, int esize) {
    return (xx >= 0 && xx < n && yy >= 0 && yy < n) ? (unsigned)(xx + n * yy) * (unsigned)esize : BUF_OOB;
}
template <typename T> __device__ __forceinline__ T bload(BufRes r, unsigned off);
template <> __device__ __forceinline__ float bload<float>(BufRes r, unsigned off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
template <> __device__ __forceinline__ double bload<double>(BufRes r, unsigned off) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}
// aux 2 = nontemporal: the stencil output streams out and should not evict the inputs still in use
template <typename T> __device__ __forceinline__ void bstore_nt(T v, BufRes r, unsigned off);
template <> __device__ __forceinline__ void bstore_nt<float>(float v, BufRes r, unsigned off) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, off, 0, 2);
}
template <> __device__ __forceinline__ void bstore_nt<double>(double v, BufRes r, unsigned off) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), r, off, 0, 2);
}

// ------------------------------------------------------------------------------------------ stencil ----
// 2.5-D z-streaming: a workgroup owns a TX x TYL tile of (x, y) columns of one band and a chunk of z planes; a lane
// owns VX consecutive x points of one row (16 bytes: float4 / double2) and streams them along z. The z neighbours stay
// in registers, the x / y neighbours of the current plane come from a double-buffered LDS tile with a 4-point halo (one
// barrier per plane).
//
// The second derivative along an axis is taken from first differences D_j = f_{j+1} - f_j:
//   sum_m c_m (f_m - 2 f_0 + f_{-m}) = sum_{j=0..3} K_j (D_j - D_{-1-j}),  K_j = sum_{m>j} c_m.
// A difference of neighbouring values of a smooth field is exact or nearly so in its own precision, and the sum of
// second differences never carries the large central term, so the f32 stencil keeps its accuracy (2-norm error of H.X
// against 64 bits on orbital-like bands, 95^3: 4e-8 .. 7e-8). Neighbouring outputs share their D's: along z they stay in
// registers (four below the plane, four of the planes ahead), along x a lane's VX points share VX + 7, and each axis
// costs 8 more operations per point: 40 VALU operations per f32 point, against 56 of the pair form c_m [(f_m - f_0) +
// (f_{-m} - f_0)] that this replaces. Without packed FP32 instructions an f32 operation issues at the f64 rate (39 T
// lane-operations/s), so at 192^3 x 64 the pair form alone cost 0.65 ms of VALU issue against 0.63 ms for the bytes at the
// copy rate.
//
// XCD-aware workgroup order. The dispatcher hands consecutive workgroup ids to the 8 XCDs round-robin (id mod 8);
// each XCD has its own L2. The stencil launches a 1-D grid and gives XCD x the contiguous logical range
// [x P, (x + 1) P) of (band, z chunk, tile) work items, tiles fastest: the tiles of one band (whose halos overlap) and
// neighbouring bands (which share V) then run together on one XCD and meet in its L2.
struct StWork {
    int tile_x, tile_y, band, zchunk;
    bool valid;
};
// order 0: tiles fastest, then z chunks, then bands; G >= 2: bands in groups of G fastest, then tiles, then z chunks,
// then groups: the G bands of a tile share V in L2 while neighbouring tiles (the halos) run side by side. Bands padded
// to a multiple of G are skipped.
__device__ __forceinline__ StWork st_decode(int ntx, int nty, int nzc, int nb, int order) {
    const int tiles = ntx * nty;
    const int nbp = order >= 2 ? ((nb + order - 1) / order) * order : nb;
    const int total = tiles * nzc * nbp;
    const int per = (total + 7) / 8;
    const int lin = blockIdx.x;
    const int L = (lin & 7) * per + (lin >> 3);
    StWork w;
    const int group = order >= 2 ? order : 1;
    const int gi = L % group;
    int rest = L / group;
    const int tile = rest % tiles;
    rest /= tiles;
    w.zchunk = rest % nzc;
    w.band = (rest / nzc) * group + gi;
    w.valid = L < total && w.band < nb;
    w.tile_x = tile % ntx;
    w.tile_y = tile / ntx;
    return w;
}
static inline unsigned st_grid(int ntx, int nty, int nzc, int nb, int order) {
    const long nbp = order >= 2 ? ((nb + order - 1) / order) * order : nb;
    const long total = (long)ntx * nty * nzc * nbp;
    return (unsigned)(8 * ((total + 7) / 8));
}

// Compile-time plane unrolling: f(integral_constant<int, S>) for S = 0 .. W-1 (every register slot index a constant)
template <int S, int W> struct PlaneUnroll {
    template <typename F> __device__ __forceinline__ static void run(F &f) {
        f(std::integral_constant<int, S>{});
        PlaneUnroll<S + 1, W>::run(f);
    }
};
template <int W> struct PlaneUnroll<W, W> {
    template <typename F> __device__ __forceinline__ static void run(F &) {}
};

// native 16-byte vectors: VX = 4 f32 or 2 f64 points
template <typename T> struct Vec16;
template <> struct Vec16<float> {
    typedef float type __attribute__((ext_vector_type(4)));
    static constexpr int N = 4;
};
template <> struct Vec16<double> {
    typedef double type __attribute__((ext_vector_type(2)));
    static constexpr int N = 2;
};
// 16-byte buffer load / nontemporal store of one vector at any element alignment; the range check is per dword
template <typename T> __device__ __forceinline__ typename Vec16<T>::type bloadv(BufRes r, unsigned off) {
    return __builtin_bit_cast(typename Vec16<T>::type, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
template <typename V> __device__ __forceinline__ void bstorev_nt(V v, BufRes r, unsigned off) {
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), r, off, 0, 2);
}

constexpr int ST_AHEAD = 6;  // a lane loads its plane z + ST_AHEAD at plane z
// factor K_j, K_j = sum_{m > j} c_m, in the kernel's precision; factor is -1/2 / h^2, or scale / h^2. A sum (2j + 1) k_j
// that is off by d scales every kinetic energy by 1 + d, so a total energy is off by d times it, and in f32 the k_j rounded
// one by one give d up to 1e-7. k_0 and k_1 are rounded; k_2 and k_3 are small, so finely spaced in f32, and make up what
// these lost in that sum and in the 4th moment: d is below 1e-9, the 4th moment's error below 1e-8.
template <typename T> struct StCoef {
    T k[4];
};
template <typename T> static StCoef<T> st_coef(double factor) {
    const double K[4] = {factor * (C1 + C2 + C3 + C4), factor * (C2 + C3 + C4), factor * (C3 + C4), factor * C4};
    StCoef<T> c;
    for (int j = 0; j < 4; j++) c.k[j] = (T)K[j];
    if (!std::isfinite(c.k[0])) return c;
    const double e0 = K[0] - (double)c.k[0], e1 = K[1] - (double)c.k[1];
    const double m2 = e0 + 3.0 * e1, m4 = e0 + 15.0 * e1;  // (j + 1)^p - j^p: 1, 3, 5, 7 and 1, 15, 65, 175
    const double x3 = (m4 - 13.0 * m2) / 84.0, x2 = (m2 - 7.0 * x3) / 5.0;
    c.k[2] = (T)(K[2] + x2);
    c.k[3] = (T)(K[3] + (m2 + 5.0 * (K[2] - (double)c.k[2])) / 7.0);
    return c;
}

// Register state of a lane: F holds its vector on planes z .. z + 5 (plane p in slot (p - z0) mod 8; step z loads plane
// z + 6), D the differences D_{z-4} .. D_{z-1} (D_j in slot (j - z0) mod 4; step z replaces D_{z-4} by D_z), and hq /
// vq / rq its halo vectors, V and R, loaded two planes ahead. The z loop is unrolled by 8 so every slot is a compile-time
// constant: registers rotate by name, and a load is only waited for when its plane is used. Keeping D_z .. D_{z+3} as
// well would save three operations per point but 16 registers: at three waves per SIMD (168 registers) the f32 Jacobi
// sweep then spills (95^3 x 8: 24.9 us, 19.6 us without them). The f64 sweep on rows that are no whole vectors is past
// that limit as it is, by 7 or 8 registers.
template <typename T, int HV> struct StRegs {
    typedef typename Vec16<T>::type V;
    V F[8], D[4];
    V hq[2][HV];
    V vq[2], rq[2];
};

template <typename T, int HV> struct StCtx {
    typedef typename Vec16<T>::type V;
    BufRes bx, bo, bv, br;  // x and out of this band, V, R of this band
    unsigned pb;            // bytes per plane
    unsigned co;            // this lane's vector: byte offset in a plane, or BUF_OOB
    unsigned ho[HV];        // its halo vectors, or BUF_OOB
    int hl[HV];             // their element offset in an LDS plane, -1: none
    int hnv[HV];            // points of them inside the box (the rest belong to the next row)
    int nv;                 // points of the lane's vector inside the box
    int lo;                 // the lane's element offset in an LDS plane
    int n, zlim;            // planes at or past zlim are not loaded
    StCoef<T> cf;
    T omega, diag_t, lamb;
    // plane zz at byte offset off; a plane past the last one the chunk needs reads plane n: out of range, 0
    __device__ V ld(BufRes r, unsigned off, int zz, int lim) const {
        return bloadv<T>(r, off + (unsigned)(zz < lim ? zz : n) * pb);
    }
};

template <typename V, int VX> __device__ __forceinline__ V st_mask(V v, int nv) {
#pragma unroll
    for (int i = 0; i < VX; i++) v[i] = i < nv ? v[i] : 0;
    return v;
}

// omega / d for d >= 0.1: a reciprocal estimate, the quotient and one residual correction
__device__ __forceinline__ float st_quot(float a, float d) {
    const float r = __builtin_amdgcn_rcpf(d), q = a * r;
    return __builtin_fmaf(__builtin_fmaf(-d, q, a), r, q);
}
__device__ __forceinline__ double st_quot(double a, double d) { return a / d; }
__device__ __forceinline__ float st_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double st_fma(double a, double b, double c) { return __builtin_fma(a, b, c); }

// one plane z of the stream; S = (z - z0) mod 8
template <typename T, int MODE, int TXL, int TYL, bool XT, bool RAG, int HV, int S>
__device__ __forceinline__ void st_plane(StRegs<T, HV> &R, const StCtx<T, HV> &c, T *tl, int z, int z1) {
    typedef typename Vec16<T>::type V;
    constexpr int VX = Vec16<T>::N;
    constexpr int LXP = TXL * VX + 8;
    R.F[(S + ST_AHEAD) & 7] = c.ld(c.bx, c.co, z + ST_AHEAD, c.zlim);
    const V ce = RAG ? st_mask<V, VX>(R.F[S], c.nv) : R.F[S];
    *reinterpret_cast<V *>(tl + c.lo) = ce;
#pragma unroll
    for (int k = 0; k < HV; k++)
        if (c.hl[k] >= 0)
            *reinterpret_cast<V *>(tl + c.hl[k]) = XT && RAG ? st_mask<V, VX>(R.hq[S & 1][k], c.hnv[k]) : R.hq[S & 1][k];
#pragma unroll
    for (int k = 0; k < HV; k++) R.hq[S & 1][k] = c.ld(c.bx, c.ho[k], z + 2, z1);
    __syncthreads();
    // The second differences e_j = D_j - D_{-1-j} of each axis: those of j = 3, 2, 1 (coefficients up to K0 / 8) go into acc
    // as they come, the j = 0 ones are summed over the axes and added last, so the large partial sums are rounded three
    // times in all.
    V acc, e0;
    auto add = [&](V e, T k) {
#pragma unroll
        for (int i = 0; i < VX; i++) acc[i] = st_fma(e[i], k, acc[i]);
    };
    // z
    {
        V dn[4];
#pragma unroll
        for (int j = 0; j < 4; j++) dn[j] = R.F[(S + j + 1) & 7] - R.F[(S + j) & 7];
        acc = (dn[3] - R.D[S & 3]) * c.cf.k[3];
        add(dn[2] - R.D[(S + 1) & 3], c.cf.k[2]);
        add(dn[1] - R.D[(S + 2) & 3], c.cf.k[1]);
        e0 = dn[0] - R.D[(S + 3) & 3];
        R.D[S & 3] = dn[0];
    }
    // y: the eight rows about this one
    {
        V m[5], p[5];
        m[0] = p[0] = ce;
#pragma unroll
        for (int q = 1; q <= 4; q++) {
            m[q] = *reinterpret_cast<const V *>(tl + c.lo - q * LXP);
            p[q] = *reinterpret_cast<const V *>(tl + c.lo + q * LXP);
        }
        add((p[4] - p[3]) - (m[3] - m[4]), c.cf.k[3]);
        add((p[3] - p[2]) - (m[2] - m[3]), c.cf.k[2]);
        add((p[2] - p[1]) - (m[1] - m[2]), c.cf.k[1]);
        e0 += (p[1] - p[0]) - (m[0] - m[1]);
    }
    // x: the VX + 8 points of this row about the lane's, their differences shared by its points
    {
        T w[VX + 8], d[VX + 7];
#pragma unroll
        for (int b = 0; b < 4 / VX; b++) {
            const V l = *reinterpret_cast<const V *>(tl + c.lo - 4 + VX * b);
            const V r = *reinterpret_cast<const V *>(tl + c.lo + VX + VX * b);
#pragma unroll
            for (int i = 0; i < VX; i++) {
                w[VX * b + i] = l[i];
                w[4 + VX + VX * b + i] = r[i];
            }
        }
#pragma unroll
        for (int i = 0; i < VX; i++) w[4 + i] = ce[i];
#pragma unroll
        for (int i = 0; i < VX + 7; i++) d[i] = w[i + 1] - w[i];
#pragma unroll
        for (int j = 3; j >= 1; j--)
#pragma unroll
            for (int i = 0; i < VX; i++) acc[i] = st_fma(d[4 + i + j] - d[3 + i - j], c.cf.k[j], acc[i]);
#pragma unroll
        for (int i = 0; i < VX; i++) e0[i] += d[4 + i] - d[3 + i];
    }
    add(e0, c.cf.k[0]);
    // the kinetic term is rounded and the potential's product is not: near the nuclei the two nearly cancel, and the product
    // is the larger one (f32 error of H.X against 64 bits over 40 drawn fields, to that of the pair form c_m [(f_m - f_0) +
    // (f_{-m} - f_0)]: 0.73 .. 1.00 of it, 0.87 in the mean; with the product rounded instead up to 1.4)
    V o;
#pragma unroll
    for (int i = 0; i < VX; i++) {
        if (MODE == ST_LAP) {
            o[i] = acc[i];
        } else if (MODE == ST_HAM) {
            o[i] = st_fma(R.vq[S & 1][i], ce[i], acc[i]);
        } else {
            const T t = R.vq[S & 1][i] - c.lamb;
            const T hw = st_fma(t, ce[i], acc[i]);
            T d = c.diag_t + t;
            d = d > T(0.1) ? d : T(0.1);
            o[i] = st_fma(st_quot(c.omega, d), R.rq[S & 1][i] - hw, ce[i]);
        }
    }
    if (MODE != ST_LAP) R.vq[S & 1] = c.ld(c.bv, c.co, z + 2, z1);
    if (MODE == ST_JAC) R.rq[S & 1] = c.ld(c.br, c.co, z + 2, z1);
    // a lane outside the box has offset BUF_OOB: its store is dropped; the row's last vector may be partly inside
    const unsigned so = c.co + (unsigned)z * c.pb;
    if (!RAG || c.nv >= VX) {
        bstorev_nt(o, c.bo, so);
    } else {
#pragma unroll
        for (int i = 0; i < VX - 1; i++)
            if (i < c.nv) bstore_nt<T>(o[i], c.bo, so + i * (unsigned)sizeof(T));
    }
}

// TXL lanes in x (TX = TXL VX columns), TYL rows. XT: several tiles in x (their x halos are loaded; with one tile the
// x neighbours outside it are outside the box and its LDS halo columns stay 0). RAG: n is no multiple of VX, so a row's
// last vector holds points of the next row, which are masked (as neighbours) and not stored.
template <typename T, int MODE, int TXL, int TYL, bool XT, bool RAG>
__global__ __launch_bounds__(TXL *TYL) __attribute__((amdgpu_waves_per_eu(3))) void k_stencil(const T *__restrict__ x, T *__restrict__ out,
                                                      const T *__restrict__ v, const T *__restrict__ r,
                                                      const double *__restrict__ lam, int n, long N, int zc, int nb,
                                                      int order, StCoef<T> cf, T omega, T diag_t, const T *__restrict__ x2,
                                                      T *__restrict__ out2, int nb1) {
    typedef typename Vec16<T>::type V;
    constexpr int VX = Vec16<T>::N, TX = TXL * VX, LXP = TX + 8, THREADS = TXL * TYL;
    constexpr int XV = 4 / VX;  // x-halo vectors per row and side
    constexpr int YH = 8 * TXL, XH = XT ? 2 * XV * TYL : 0, HV = (YH + XH + THREADS - 1) / THREADS;
    static_assert(THREADS % 64 == 0, "whole waves");
    __shared__ __align__(16) T tile[2][(TYL + 8) * LXP];
    const int t = threadIdx.x, tx = t % TXL, ty = t / TXL;
    const int nzc = (n + zc - 1) / zc;
    const StWork wk = st_decode((n + TX - 1) / TX, (n + TYL - 1) / TYL, nzc, nb, order);
    if (!wk.valid) return;
    const int x0 = wk.tile_x * TX, y0 = wk.tile_y * TYL, band = wk.band;
    const int z0 = wk.zchunk * zc, z1 = min(n, z0 + zc);
    const long fb = N * (long)sizeof(T);
    StCtx<T, HV> c;
    c.bx = field_res(band < nb1 ? x + (long)band * N : x2 + (long)(band - nb1) * N, fb);
    c.bo = field_res(band < nb1 ? out + (long)band * N : out2 + (long)(band - nb1) * N, fb);
    c.bv = field_res(MODE == ST_LAP ? x : v, MODE == ST_LAP ? 0 : fb);
    c.br = field_res(MODE == ST_JAC ? r + (long)band * N : x, MODE == ST_JAC ? fb : 0);
    c.lamb = MODE == ST_JAC ? (T)lam[band] : T(0);
    c.n = n;
    c.zlim = z1 + 4;
    c.pb = (unsigned)((long)n * n * (long)sizeof(T));
    const int gx = x0 + VX * tx;
    c.co = row_off(gx, y0 + ty, n, (int)sizeof(T));
    c.nv = n - gx;
    c.lo = (ty + 4) * LXP + 4 + VX * tx;
    c.cf = cf;
    c.omega = omega;
    c.diag_t = diag_t;
    // halo vectors: the 4 rows above and below the tile, then (XT) each row's 4 points left and right of it
#pragma unroll
    for (int k = 0; k < HV; k++) {
        const int e = t + k * THREADS;
        int hgx = -1, hgy = -1;
        c.hl[k] = -1;
        if (e < YH) {
            const int row = e / TXL, col = e % TXL, ly = row < 4 ? row : TYL + row;
            hgx = x0 + VX * col;
            hgy = y0 - 4 + ly;
            c.hl[k] = ly * LXP + 4 + VX * col;
        } else if (XT && e < YH + XH) {
            const int q = e - YH, row = q / (2 * XV), s = q % (2 * XV);
            const int lx = s < XV ? VX * s : 4 + TX + VX * (s - XV);
            hgx = x0 - 4 + lx;
            hgy = y0 + row;
            c.hl[k] = (row + 4) * LXP + lx;
        }
        c.ho[k] = row_off(hgx, hgy, n, (int)sizeof(T));
        c.hnv[k] = n - hgx;
    }
    if (!XT)
        for (int e = t; e < 2 * 8 * TYL; e += THREADS) {
            const int b = e / (8 * TYL), q = e % (8 * TYL), row = q >> 3, s = q & 7;
            tile[b][(row + 4) * LXP + (s < 4 ? s : TX + s)] = T(0);
        }
    StRegs<T, HV> R;
    {
        V p[4];
#pragma unroll
        for (int q = 0; q < 4; q++) p[q] = c.ld(c.bx, c.co, z0 - 4 + q, c.zlim);
#pragma unroll
        for (int q = 0; q < ST_AHEAD; q++) R.F[q] = c.ld(c.bx, c.co, z0 + q, c.zlim);
#pragma unroll
        for (int s = 0; s < 2; s++) {
#pragma unroll
            for (int k = 0; k < HV; k++) R.hq[s][k] = c.ld(c.bx, c.ho[k], z0 + s, z1);
            if (MODE != ST_LAP) R.vq[s] = c.ld(c.bv, c.co, z0 + s, z1);
            if (MODE == ST_JAC) R.rq[s] = c.ld(c.br, c.co, z0 + s, z1);
        }
#pragma unroll
        for (int q = 0; q < 3; q++) R.D[q] = p[q + 1] - p[q];  // D_{z0-4+q}
        R.D[3] = R.F[0] - p[3];
    }
    // consecutive planes alternate the two LDS buffers (plane p uses buffer (p - z0) & 1): one barrier per plane then
    // separates every write of a buffer from the previous reads of it
    int z = z0;
    for (; z + 8 <= z1; z += 8) {
        auto step = [&](auto sc) {
            constexpr int S = decltype(sc)::value;
            st_plane<T, MODE, TXL, TYL, XT, RAG, HV, S>(R, c, tile[S & 1], z + S, z1);
        };
        PlaneUnroll<0, 8>::run(step);
    }
    // remainder (< 8 planes) with the same slot sequence
    auto tail = [&](auto sc) {
        constexpr int S = decltype(sc)::value;
        if (z + S < z1) st_plane<T, MODE, TXL, TYL, XT, RAG, HV, S>(R, c, tile[S & 1], z + S, z1);
    };
    PlaneUnroll<0, 7>::run(tail);
}

struct StVariant {
    int tx;     // tile width in points
    int zc;     // planes per chunk; 0: whole columns, -1: chunks that load the CUs evenly
    int order;  // XCD work order: 0 tiles fastest, G >= 2 bands in groups of G fastest
    const char *name;
};
static const StVariant ST_VARIANTS[] = {
    {32, -1, 0, "32-wide tile, balanced z chunks"},
    {32, 0, 0, "32-wide tile, full z column"},
    {32, 32, 0, "32-wide tile, z chunks of 32"},
    {32, 16, 0, "32-wide tile, z chunks of 16"},
    {32, 8, 0, "32-wide tile, z chunks of 8"},
    {64, -1, 0, "64-wide tile, balanced z chunks"},
    {64, 0, 0, "64-wide tile, full z column"},
    {64, 32, 0, "64-wide tile, z chunks of 32"},
    {64, 16, 0, "64-wide tile, z chunks of 16"},
    {64, 8, 0, "64-wide tile, z chunks of 8"},
    {64, 0, 4, "64-wide tile, full z column, bands in groups of 4"},
    {64, 24, 4, "64-wide tile, z chunks of 24, bands in groups of 4"},
    {96, -1, 0, "96-wide tile, balanced z chunks"},
    {96, 0, 0, "96-wide tile, full z column"},
    {96, 32, 0, "96-wide tile, z chunks of 32"},
    {96, 16, 0, "96-wide tile, z chunks of 16"},
    {96, 8, 0, "96-wide tile, z chunks of 8"},
    {128, -1, 0, "128-wide tile, balanced z chunks"},
    {128, 0, 0, "128-wide tile, full z column"},
    {128, 32, 0, "128-wide tile, z chunks of 32"},
    {128, 16, 0, "128-wide tile, z chunks of 16"},
    {128, 8, 0, "128-wide tile, z chunks of 8"},
    {192, -1, 0, "192-wide tile, balanced z chunks"},
    {192, 0, 0, "192-wide tile, full z column"},
    {192, 32, 0, "192-wide tile, z chunks of 32"},
    {192, 16, 0, "192-wide tile, z chunks of 16"},
    {192, 8, 0, "192-wide tile, z chunks of 8"},
    {192, 0, 4, "192-wide tile, full z column, bands in groups of 4"},
    {192, 24, 4, "192-wide tile, z chunks of 24, bands in groups of 4"},
};
static int g_default_variant[2] = {-1, -1};

int stencil_variants() { return (int)(sizeof(ST_VARIANTS) / sizeof(ST_VARIANTS[0])); }
const char *stencil_variant_name(int v) { return (v >= 0 && v < stencil_variants()) ? ST_VARIANTS[v].name : "auto"; }
void stencil_set_default_variant(int dtype_size, int variant) { g_default_variant[dtype_size == 8 ? 1 : 0] = variant; }

// rows and waves of the tile of each width (the TXL x TYL of stencil_dispatch)
static int st_rows(int tx, int esize) { return esize == 4 ? (tx == 32 ? 32 : tx == 192 ? 8 : 16) : (tx <= 64 ? 16 : 8); }
static int st_waves(int tx, int esize) { return tx / (16 / esize) * st_rows(tx, esize) / 64; }

// The balanced chunk: a chunk of zc planes streams zc + 8, and the launch takes as long as its fullest CU. With w waves
// on a CU a plane step took about max(7, w) in one unit (0.09 us) wherever it was measured (95^3 f32, 96-wide tiles: 7
// bands, 252 blocks of 6 waves in chunks of 16, 13.9 us; 504 blocks in chunks of 8, 16.8 us; 336 in chunks of 12,
// > 17.4 us; 16 bands, 480 blocks in chunks of 19, 31.2 us; 576 in chunks of 16, 37.1 us). f32 tiles on rows that do not
// fit one tile keep chunks of at most 16 planes, whose tiles meet in the L2s (160^3 x 46 sweep: 477 us, 490 in chunks of
// 32).
static int st_chunk(int tx, int n, int nb, int esize) {
    const int rows = st_rows(tx, esize), waves = st_waves(tx, esize);
    const long cols = (long)((n + tx - 1) / tx) * ((n + rows - 1) / rows) * nb;
    int best = n, zc = esize == 4 && n > 128 && tx < n ? std::min(n, 16) : n;
    double best_cost = 1e300;
    do {
        const int nzc = (n + zc - 1) / zc;
        zc = (n + nzc - 1) / nzc;
        const double per_cu = (double)((cols * nzc + 255) / 256);
        const double cost = (zc + 8) * std::max(7.0, per_cu * waves);
        if (cost < best_cost) {
            best_cost = cost;
            best = zc;
        }
        zc--;
    } while (zc >= 2);
    return best;
}

// The tile when no tuned choice exists: the narrowest one that takes whole rows up to 128 points (no x halos), in f32
// also 192-wide rows that fill it; 64-wide otherwise; in balanced chunks. Over 72 shapes (25^3 .. 256^3, 1 .. 64 bands,
// three modes, both types) its time was 1.03 of the best variant's in the geometric mean, and on single shapes up to 1.24
// (72^3 x 10 f64; 40^3 x 24 f64 1.16, 176^3 x 4 f32 1.14, 64^3 x 32 f32 1.13, 160^3 x 12 f32 1.10): the solver, and a
// caller of lira_autotune_stencil, time the variants on their own shape.
static int pick_variant(int n, int esize) {
    const int tx = n <= 64 ? 64 : n <= 96 ? 96 : n <= 128 ? 128 : esize == 4 && n > 176 && n <= 192 ? 192 : 64;
    for (int v = 0; v < stencil_variants(); v++)
        if (ST_VARIANTS[v].tx == tx && ST_VARIANTS[v].zc == -1) return v;
    return 0;
}

template <typename T, int MODE, int TXL, int TYL, bool XT>
static void launch_stencil(const StencilParams &p, int zc, int order, const T *x, T *out, const T *v, const T *r,
                           const double *lam, hipStream_t s) {
    constexpr int VX = Vec16<T>::N, TX = TXL * VX;
    const int n = p.n;
    const long N = (long)n * n * n;
    if (zc < 0) zc = st_chunk(TX, n, p.nb, (int)sizeof(T));
    if (zc == 0 || zc > n) zc = n;
    const int nzc = (n + zc - 1) / zc;
    const dim3 grid(st_grid((n + TX - 1) / TX, (n + TYL - 1) / TYL, nzc, p.nb, order)), block(TXL * TYL);
    const double inv_h2 = 1.0 / (p.h * p.h);
    const StCoef<T> cf = st_coef<T>(MODE == ST_LAP ? p.scale * inv_h2 : -0.5 * inv_h2);
    const int nb1 = p.nb1 < 0 ? p.nb : p.nb1;
#define LIRA_GO(RAG_)                                                                                                   \
    hipLaunchKernelGGL((k_stencil<T, MODE, TXL, TYL, XT, RAG_>), grid, block, 0, s, x, out, v, r, lam, n, N, zc, p.nb, \
                       order, cf, (T)p.omega, (T)p.diag_t, static_cast<const T *>(p.x2), static_cast<T *>(p.out2), nb1)
    if (n % VX) LIRA_GO(true);
    else LIRA_GO(false);
#undef LIRA_GO
    LIRA_HIP(hipGetLastError());
}

// the tile of each width: TXL lanes x TYL rows
template <typename T, int MODE>
static void stencil_dispatch(const StVariant &sv, const StencilParams &p, const T *x, T *out, const T *v, const T *r,
                             const double *lam, hipStream_t s) {
#define LIRA_ST(TXL_, TYL_, XT_) launch_stencil<T, MODE, TXL_, TYL_, XT_>(p, sv.zc, sv.order, x, out, v, r, lam, s)
    if constexpr (sizeof(T) == 4) {
        if (sv.tx == 32) LIRA_ST(8, 32, true);
        else if (sv.tx == 64) LIRA_ST(16, 16, true);
        else if (sv.tx == 96) LIRA_ST(24, 16, false);
        else if (sv.tx == 128) LIRA_ST(32, 16, false);
        else LIRA_ST(48, 8, false);
    } else {
        if (sv.tx == 32) LIRA_ST(16, 16, true);
        else if (sv.tx == 64) LIRA_ST(32, 16, true);
        else if (sv.tx == 96) LIRA_ST(48, 8, false);
        else LIRA_ST(64, 8, false);
    }
#undef LIRA_ST
}

// a tile of 96 or more columns takes the whole row
bool stencil_variant_usable(int variant, int n, int dtype_size) {
    if (variant < 0 || variant >= stencil_variants()) return false;
    const int tx = ST_VARIANTS[variant].tx;
    return tx <= 64 || (n <= tx && (tx < 192 || dtype_size == 4));
}

template <typename T>
void stencil(int mode, const StencilParams &p, const T *x, T *out, const T *v, const T *r, const double *lam,
             hipStream_t s, int variant) {
    if (p.nb <= 0) return;
    if (x == out) throw InvalidError("stencil: output aliases the input");
    if (p.nb1 >= 0 && p.nb1 < p.nb) {
        if (!p.x2 || !p.out2 || p.x2 == p.out2 || mode == ST_JAC)
            throw InvalidError("stencil: bad second band segment");
    }
    if (!stencil_buffer_ok(p.n, (int)sizeof(T)))
        throw InvalidError("stencil: grid too large for 32-bit field offsets ((n^3 + 4 n^2) values must stay below "
                           "2^31 bytes)");
    if (variant < 0) variant = g_default_variant[sizeof(T) == 8 ? 1 : 0];
    if (!stencil_variant_usable(variant, p.n, (int)sizeof(T))) variant = pick_variant(p.n, (int)sizeof(T));
    const StVariant &sv = ST_VARIANTS[variant];
    if (mode == ST_LAP) stencil_dispatch<T, ST_LAP>(sv, p, x, out, v, r, lam, s);
    else if (mode == ST_HAM) stencil_dispatch<T, ST_HAM>(sv, p, x, out, v, r, lam, s);
    else stencil_dispatch<T, ST_JAC>(sv, p, x, out, v, r, lam, s);
}


// ------------------------------------------------------------------------------------------ reductions ----
__device__ inline double block_sum256(double v, double *sh) {
    sh[threadIdx.x] = v;
    __syncthreads();
#pragma unroll
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    double r = sh[0];
    __syncthreads();
    return r;
}

__device__ inline double block_max256(double v, double *sh) {
    sh[threadIdx.x] = v;
    __syncthreads();
#pragma unroll
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sh[threadIdx.x] = fmax(sh[threadIdx.x], sh[threadIdx.x + w]);
        __syncthreads();
    }
    double r = sh[0];
    __syncthreads();
    return r;
}

template <typename T>
__global__ __launch_bounds__(256) void k_reduce(RedJobs<T> jobs, long N, int n, double *partials) {
    __shared__ double sh[256];
    const int j = blockIdx.y;
    const int kind = jobs.kind[j];
    const T *a = jobs.a[j];
    const T *b = jobs.b[j];
    double acc = 0.0;
    const long stride = (long)gridDim.x * 256;
    if (kind == RED_DOT) {
        for (long p = blockIdx.x * 256L + threadIdx.x; p < N; p += stride) acc += (double)a[p] * (double)b[p];
    } else if (kind == RED_SUM) {
        for (long p = blockIdx.x * 256L + threadIdx.x; p < N; p += stride) acc += (double)a[p];
    } else if (kind == RED_ABSDIFF) {
        for (long p = blockIdx.x * 256L + threadIdx.x; p < N; p += stride) acc += fabs((double)a[p] - (double)b[p]);
    } else if (kind == RED_FACEMAX) {
        const long nn = (long)n * n;
        for (long p = blockIdx.x * 256L + threadIdx.x; p < N; p += stride) {
            const long k = p / nn, rem = p - k * nn, jj = rem / n, i = rem - jj * n;
            if (i == 0 || jj == 0 || k == 0 || i == n - 1 || jj == n - 1 || k == n - 1) acc = fmax(acc, fabs((double)a[p]));
        }
    } else {
        for (long p = blockIdx.x * 256L + threadIdx.x; p < N; p += stride) acc = fmax(acc, fabs((double)a[p]));
    }
    const bool is_max = kind == RED_FACEMAX || kind == RED_MAX_ABS;
    const double r = is_max ? block_max256(acc, sh) : block_sum256(acc, sh);
    if (threadIdx.x == 0) partials[(long)j * RED_BLOCKS + blockIdx.x] = r;
}

struct KindList {
    int kind[MAX_JOBS];
};

__global__ __launch_bounds__(256) void k_reduce_finish(KindList kinds, const double *partials, double *out,
                                                        double scale) {
    __shared__ double sh[256];
    const int j = blockIdx.x;
    const bool is_max = kinds.kind[j] == RED_FACEMAX || kinds.kind[j] == RED_MAX_ABS;
    double acc = 0.0;
    for (int p = threadIdx.x; p < RED_BLOCKS; p += 256) {
        const double v = partials[(long)j * RED_BLOCKS + p];
        acc = is_max ? fmax(acc, v) : acc + v;
    }
    const double r = is_max ? block_max256(acc, sh) : block_sum256(acc, sh);
    if (threadIdx.x == 0) out[j] = is_max ? r : r * scale;
}

template <typename T>
void reduce_jobs(const RedJobs<T> &jobs, int n, double scale, double *partials, double *out, hipStream_t s) {
    if (jobs.count <= 0) return;
    if (jobs.count > MAX_JOBS) throw InvalidError("reduce_jobs: too many jobs");
    const long N = (long)n * n * n;
    hipLaunchKernelGGL(k_reduce<T>, dim3(RED_BLOCKS, jobs.count), dim3(256), 0, s, jobs, N, n, partials);
    LIRA_HIP(hipGetLastError());
    KindList kl;
    for (int j = 0; j < MAX_JOBS; j++) kl.kind[j] = j < jobs.count ? jobs.kind[j] : RED_SUM;
    hipLaunchKernelGGL(k_reduce_finish, dim3(jobs.count), dim3(256), 0, s, kl, partials, out, scale);
    LIRA_HIP(hipGetLastError());
}

// ------------------------------------------------------------------------------------------- Gram ----
// A load through a pointer the compiler cannot place (one read from an LDS table of column bases) becomes a flat
// load, which also counts against the LDS wait counter: every wait for an LDS read would then wait for the loads in
// flight as well. Column data is always global memory, so these loads name that address space.
template <typename T> __device__ __forceinline__ T gload(const T *p) {
    return *(const __attribute__((address_space(1))) T *)p;
}

struct ColPtrs {
    const void *base[MAX_SEGS];
    int start[MAX_SEGS + 1];
    int nseg;
};

// column col's base address on the host (the same arithmetic as col_base)
static const void *col_host(const ColPtrs &c, int col, long N, int esize) {
    int s = 0;
    for (int i = 1; i < c.nseg; i++)
        if (col >= c.start[i]) s = i;
    return static_cast<const char *>(c.base[s]) + (size_t)(col - c.start[s]) * (size_t)N * (size_t)esize;
}

__device__ inline const void *col_base(const ColPtrs &c, int col, long N, int esize) {
    int s = 0;
#pragma unroll
    for (int i = 1; i < MAX_SEGS; i++)
        if (i < c.nseg && col >= c.start[i]) s = i;
    return static_cast<const char *>(c.base[s]) + (size_t)(col - c.start[s]) * (size_t)N * (size_t)esize;
}

// G = scale S^T U on the f64 matrix cores: v_mfma_f64_16x16x4f64 with A = 16 S columns x 4 points, B = 4 points x 16 U
// columns (lane l holds A[l % 16][l / 16] and B[l / 16][l % 16]; the 16 x 16 result lands as D[l / 16 + 4 r][l % 16] in
// register r, measured on gfx950). Inputs convert to f64 exactly, so the products are exact and the accumulation is f64
// in every precision mode.
//
// The operands go from memory to the matrix cores without LDS. The order in which points enter the sum is free, so a lane
// loads 16 bytes of consecutive points and feeds one of them to each MFMA (GramLoad); A and B share that layout, so a
// column block that is both (S^T S, SHARE) is loaded once. A wave holds RB x CB output blocks: per 16 points RB + CB
// blocks loaded and converted against 4 RB CB MFMAs (64 cycles each), one unit of points in flight while the
// previous one is multiplied. The waves of a workgroup take interleaved units of its chunk of points and their blocks
// are summed in wave order; the workgroups that share a chunk run next to each other on one XCD, so its columns
// come from that L2. (Before, each wave staged its columns through LDS as f64 with a pointer lookup per load: 24 x 48
// columns on 95^3 f32 60 us, 138 x 276 on 160^3 11 ms.)
typedef double lira_d4 __attribute__((ext_vector_type(4)));

// What a lane loads of one 16-column block, and operand j of its unit: a value of column l % 16, at the same point in every
// block.
// QUAD: four points (16 bytes in f32, 32 in f64) of column l % 16, 4 (l / 16) .. + 3 of 16, H times. One instruction takes
// 64 bytes of each of 16 columns.
template <typename T, int H, int LOADS> struct GramLoad;
template <typename T, int H> struct GramLoad<T, H, GRAM_QUAD> {
    typedef T Q __attribute__((ext_vector_type(4), aligned(sizeof(T))));
    static constexpr int COLS = 1, P = 4 * H;
    Q v[H];
    __device__ static int column(int lane, int) { return lane & 15; }
    __device__ static int point(int lane, int j) { return 16 * (j / 4) + 4 * (lane >> 4) + j % 4; }
    __device__ static int source(int) { return 0; }
    __device__ void load(const T *const *c, long p, int lane) {
#pragma unroll
        for (int h = 0; h < H; h++) v[h] = *(const __attribute__((address_space(1))) Q *)(c[0] + p + point(lane, 4 * h));
    }
    __device__ void set(int j, T x) { v[j / 4][j % 4] = x; }
    __device__ double operand(int j) const { return (double)v[j / 4][j % 4]; }
};
// PAIR: 16 bytes of columns l % 8 and l % 8 + 8, at piece l / 8 of 128 bytes, H times. One instruction takes 128 bytes of
// each of 8 columns, so the columns cost half as many requests and address translations; lanes l and l ^ 8 of a
// row of 16 then exchange the halves that are not their column's (a move each, no select: the other banks keep theirs).
// f64, kernels of both loads: 24 x 48 on 95^3 86 -> 75 us, on 128^3 222 -> 171 (173 with the LDS kernel before), on 192^3
// 733 -> 523 (539); 32 x 64 on 128^3 318 -> 223. Where the columns stay in the 256 MiB cache it gains nothing. With two
// loads of a column in flight (PAIR2) 32 x 64 on 192^3 755 -> 700 us, on 256^3 2303 -> 1641, but on 95^3 91 -> 97.
// f32, where both take 64 or 128 bytes of a column: it gains where a stride of a multiple of 8 MiB puts all columns on the
// same channels (32 x 64 on 128^3 176 -> 139 us, on 256^3 1611 -> 1000) and costs elsewhere (on 95^3 57 -> 62).
template <typename T, int H> struct GramLoad<T, H, GRAM_PAIR> {
    static constexpr int COLS = 2, VX = 16 / (int)sizeof(T), P = 2 * VX * H;
    typedef T V __attribute__((ext_vector_type(VX), aligned(sizeof(T))));
    V v[2 * H];  // per depth the first column's points, then the second's
    __device__ static int column(int lane, int i) { return (lane & 7) + 8 * i; }
    __device__ static int point(int lane, int j) { return 8 * VX * (j / (2 * VX)) + VX * (lane >> 3) + j % VX; }
    __device__ static int source(int j) { return j / VX % 2; }
    __device__ void load(const T *const *c, long p, int lane) {
#pragma unroll
        for (int i = 0; i < 2 * H; i++)
            v[i] = *(const __attribute__((address_space(1))) V *)(c[i % 2] + p + point(lane, VX * i));
    }
    __device__ void set(int j, T x) { v[j / VX][j % VX] = x; }
    // lanes of BANKS (four lanes each) take `from` of the lane eight over, the others `keep`
    template <int BANKS> __device__ static int cross(int keep, int from) {
        return __builtin_amdgcn_update_dpp(keep, from, 0x128, 0xf, BANKS, false);  // row_ror:8
    }
    template <int BANKS> __device__ static float cross(float keep, float from) {
        return __builtin_bit_cast(float, cross<BANKS>(__builtin_bit_cast(int, keep), __builtin_bit_cast(int, from)));
    }
    template <int BANKS> __device__ static double cross(double keep, double from) {
        const int2 k = __builtin_bit_cast(int2, keep), f = __builtin_bit_cast(int2, from);
        return __builtin_bit_cast(double, int2{cross<BANKS>(k.x, f.x), cross<BANKS>(k.y, f.y)});
    }
    __device__ double operand(int j) const {
        const int i = j / VX, e = j % VX;
        return (double)(i % 2 == 0 ? cross<0xc>(T(v[i][e]), T(v[i + 1][e])) : cross<0x3>(T(v[i][e]), T(v[i - 1][e])));
    }
};
template <typename T, int H> struct GramLoad<T, H, GRAM_PAIR2> : GramLoad<T, H, GRAM_PAIR> {};

// With sym (U's first m columns are S's), the 16 x 16 blocks of S^T S strictly below its diagonal are skipped
// (gram_mirrored): k_gram_finish reads their values from the transposed block, the same sum of the same exact products.
__host__ __device__ inline bool gram_mirrored(int sym, int m, int i, int j) {
    const int rb = i >> 4, cb = j >> 4;
    return sym && cb < rb && 16 * (cb + 1) <= m;
}

template <typename T, int RB, int CB, bool SHARE, int LOADS>
__global__ __launch_bounds__(64 * gram_waves(RB, CB, SHARE), gram_waves(RB, CB, SHARE) == 16 ? 4 : 2) void k_gram(
    ColPtrs S, ColPtrs U, int m, int q, long N, long chunk, int chunks, int nc, int nsub, double *partials, int sym) {
    constexpr int H = gram_depth(RB, CB, sizeof(T), LOADS), W = gram_waves(RB, CB, SHARE);
    typedef GramLoad<T, H, LOADS> Load;
    constexpr int UP = gram_unit(H, sizeof(T), LOADS);  // points of a wave's unit
    static_assert(UP == 4 * Load::P, "four lanes of a column hold a unit");
    constexpr int NB = gram_loaded(RB, CB, SHARE);  // column blocks loaded
    __shared__ double red[W][256];
    const int total = chunks * nsub, per = (total + 7) / 8;
    const int L = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || L >= total) return;
    const int ch = L / nsub, sub = L - ch * nsub, bi = sub / nc, bj = sub - bi * nc;
    const int i0 = bi * RB * 16, j0 = bj * CB * 16;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int c16 = lane & 15, k4 = lane >> 4;
    // the output blocks this tile computes; a tile with none returns here, before any barrier
    unsigned live = 0;
#pragma unroll
    for (int a = 0; a < RB; a++)
#pragma unroll
        for (int b = 0; b < CB; b++)
            if (i0 + 16 * a < m && j0 + 16 * b < q && !gram_mirrored(sym, m, i0 + 16 * a, j0 + 16 * b))
                live |= 1u << (a * CB + b);
    if (live == 0) return;
    // this lane's columns of each block; past the last column it reads that one (its outputs are not stored)
    const T *col[NB][Load::COLS];
#pragma unroll
    for (int i = 0; i < Load::COLS; i++) {
        const int c = Load::column(lane, i);
#pragma unroll
        for (int b = 0; b < CB; b++)
            col[b][i] = static_cast<const T *>(col_base(U, min(j0 + 16 * b + c, q - 1), N, sizeof(T)));
        if constexpr (!SHARE) {
#pragma unroll
            for (int a = 0; a < RB; a++)
                col[CB + a][i] = static_cast<const T *>(col_base(S, min(i0 + 16 * a + c, m - 1), N, sizeof(T)));
        }
    }
    lira_d4 acc[RB][CB];
#pragma unroll
    for (int a = 0; a < RB; a++)
#pragma unroll
        for (int b = 0; b < CB; b++) acc[a][b] = lira_d4{0.0, 0.0, 0.0, 0.0};
    const long p_begin = (long)ch * chunk, p_end = min(N, p_begin + chunk);
    const long units = p_end > p_begin ? (p_end - p_begin) / UP : 0;  // whole units; the rest is the last chunk's tail
    // the products of one unit; ALL: every block of the tile is live. (A SHARE tile is the whole product, so its dead
    // blocks are those with b < a, known here.)
    auto multiply = [&](const Load(&v)[NB], auto all) {
#pragma unroll
        for (int j = 0; j < Load::P; j++) {
            double x[NB];
#pragma unroll
            for (int b = 0; b < NB; b++) x[b] = v[b].operand(j);
#pragma unroll
            for (int a = 0; a < RB; a++)
#pragma unroll
                for (int b = SHARE ? a : 0; b < CB; b++)
                    if (SHARE || decltype(all)::value || (live >> (a * CB + b)) & 1u)
                        acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[SHARE ? a : CB + a], x[b], acc[a][b], 0, 0, 0);
        }
    };
    auto run = [&](auto all) {
        if (units > 0) {
            // every load is issued unconditionally (a load under a branch would be waited for at the join): past the
            // wave's last unit it reads the chunk's last unit again, which is not multiplied
            auto fetch = [&](long u, Load(&v)[NB]) {
                const long p = p_begin + min(u, units - 1) * UP;
#pragma unroll
                for (int b = 0; b < NB; b++) v[b].load(col[b], p, lane);
            };
            Load va[NB], vb[NB];
            long u = wave;
            fetch(u, va);
            for (; u + W < units; u += 2 * W) {
                fetch(u + W, vb);
                multiply(va, all);
                fetch(u + 2 * W, va);
                multiply(vb, all);
            }
            if (u < units) multiply(va, all);
        }
        const long pt = p_begin + units * UP;
        if (pt < p_end && wave == (int)(units % W)) {  // the tail, fewer than UP points: guarded loads
            Load v[NB];
#pragma unroll
            for (int b = 0; b < NB; b++)
#pragma unroll
                for (int j = 0; j < Load::P; j++) {
                    const long p = pt + Load::point(lane, j);
                    v[b].set(j, p < p_end ? gload(col[b][Load::source(j)] + p) : T(0));
                }
            multiply(v, all);
        }
    };
    if (SHARE || live == (1u << (RB * CB)) - 1u) run(std::true_type{});
    else run(std::false_type{});
    // sum the waves' accumulators in wave order through LDS, one block per pass
    double *dst = partials + (long)ch * m * q;
#pragma unroll
    for (int a = 0; a < RB; a++)
#pragma unroll
        for (int b = 0; b < CB; b++) {
            if (!((live >> (a * CB + b)) & 1u)) continue;  // uniform over the workgroup
            __syncthreads();
#pragma unroll
            for (int r = 0; r < 4; r++) red[wave][r * 64 + lane] = acc[a][b][r];
            __syncthreads();
            if (wave < 4) {  // wave r sums register r
                double sum = red[0][threadIdx.x];
#pragma unroll
                for (int w = 1; w < W; w++) sum += red[w][threadIdx.x];
                const int i = i0 + a * 16 + k4 + 4 * wave, j = j0 + b * 16 + c16;
                if (i < m && j < q) dst[(long)i * q + j] = sum;
            }
        }
}

// sums the per-chunk partials of every output in a fixed order: 16 consecutive outputs per workgroup (a chunk's 16 are one
// 128-byte segment), 64 threads per output each summing a strided subset of the chunks, then a fixed tree
__global__ __launch_bounds__(1024) void k_gram_finish(const double *partials, int chunks, int m, int q, double scale,
                                                      double *G, int sym) {
    __shared__ double sh[64][17];
    const int o16 = threadIdx.x & 15, cl = threadIdx.x >> 4;
    const long mq = (long)m * q;
    const long out = blockIdx.x * 16L + o16;
    // a skipped block's output is summed from its transposed entry (i, j) -> (j, i)
    long src = out;
    if (out < mq) {
        const int i = (int)(out / q), j = (int)(out - (long)i * q);
        if (gram_mirrored(sym, m, i, j)) src = (long)j * q + i;
    }
    double acc = 0.0;
    if (out < mq) {
        int c = cl;
        for (; c + 3 * 64 < chunks; c += 4 * 64) {  // four loads in flight
            double v[4];
#pragma unroll
            for (int u = 0; u < 4; u++) v[u] = partials[(long)(c + 64 * u) * mq + src];
#pragma unroll
            for (int u = 0; u < 4; u++) acc += v[u];
        }
        for (; c < chunks; c += 64) acc += partials[(long)c * mq + src];
    }
    sh[cl][o16] = acc;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        __syncthreads();
        if (cl < off) sh[cl][o16] += sh[cl + off][o16];
    }
    if (cl == 0 && out < mq) G[out] = sh[0][o16] * scale;
}

static ColPtrs to_ptrs(const Cols &c) {
    ColPtrs p{};
    p.nseg = c.nseg;
    int acc = 0;
    for (int i = 0; i < c.nseg; i++) {
        p.base[i] = c.seg[i].base;
        p.start[i] = acc;
        acc += c.seg[i].count;
    }
    p.start[c.nseg] = acc;
    return p;
}

template <typename T, int RB, int CB, bool SHARE>
static void launch_gram(const GramPlan &g, const ColPtrs &sp, const ColPtrs &up, int m, int q, long N, double *partials,
                        int sym, hipStream_t s) {
    const int total = g.chunks * g.nr * g.nc;
    const dim3 grid((unsigned)(8 * ((total + 7) / 8))), block(64 * gram_waves(RB, CB, SHARE));
    auto go = [&](auto loads) {
        constexpr int L = decltype(loads)::value;
        if constexpr (gram_has(RB, CB, SHARE, sizeof(T), L)) {
            if (g.loads == L)
                hipLaunchKernelGGL((k_gram<T, RB, CB, SHARE, L>), grid, block, 0, s, sp, up, m, q, N, g.chunk, g.chunks, g.nc,
                                   g.nr * g.nc, partials, sym);
        }
    };
    go(std::integral_constant<int, GRAM_QUAD>{});
    go(std::integral_constant<int, GRAM_PAIR>{});
    go(std::integral_constant<int, GRAM_PAIR2>{});
}

template <typename T>
void gram(const Cols &S, const Cols &U, long N, double scale, double *partials, size_t partial_cap, double *G,
          hipStream_t s) {
    const int m = S.total(), q = U.total();
    if (m == 0 || q == 0) return;
    // U begins with S's m columns (LOBPCG's U = [S, R, HW, HP]): S^T S is symmetric and its lower blocks are mirrored
    const ColPtrs sp = to_ptrs(S), up = to_ptrs(U);
    int sym = q >= m ? 1 : 0;
    for (int j = 0; j < m && sym; j++)
        if (col_host(sp, j, N, sizeof(T)) != col_host(up, j, N, sizeof(T))) sym = 0;
    const GramPlan g = gram_plan(m, q, N, (int)sizeof(T), sym != 0);
    if ((size_t)g.chunks * m * q > partial_cap) throw InvalidError("gram: partial buffer too small");
#define LIRA_GRAM(R_, C_)                                                                                              \
    if (g.RB == R_ && g.CB == C_) {                                                                                    \
        if constexpr (R_ <= C_) {                                                                                      \
            if (g.share) launch_gram<T, R_, C_, true>(g, sp, up, m, q, N, partials, sym, s);                             \
        }                                                                                                              \
        if constexpr (sizeof(T) == 4 || C_ <= 4) {                                                                     \
            if (!g.share) launch_gram<T, R_, C_, false>(g, sp, up, m, q, N, partials, sym, s);                           \
        }                                                                                                              \
    }
    LIRA_GRAM(1, 1) LIRA_GRAM(1, 2) LIRA_GRAM(1, 3) LIRA_GRAM(1, 4) LIRA_GRAM(1, 5) LIRA_GRAM(1, 6)
    LIRA_GRAM(2, 1) LIRA_GRAM(2, 2) LIRA_GRAM(2, 3) LIRA_GRAM(2, 4) LIRA_GRAM(2, 5) LIRA_GRAM(2, 6)
    LIRA_GRAM(3, 1) LIRA_GRAM(3, 2) LIRA_GRAM(3, 3) LIRA_GRAM(3, 4) LIRA_GRAM(3, 5) LIRA_GRAM(3, 6)
#undef LIRA_GRAM
    LIRA_HIP(hipGetLastError());
    const long mq = (long)m * q;
    hipLaunchKernelGGL(k_gram_finish, dim3((unsigned)((mq + 15) / 16)), dim3(1024), 0, s, partials, g.chunks, m, q, scale, G,
                       sym);
    LIRA_HIP(hipGetLastError());
}

// ------------------------------------------------------------------------------------------ lincomb ----
// Y_j = sum_i S_i C_ij: one thread per point holds QB outputs in f64 registers; grid.y covers q in groups of QB.
// C arrives padded (lincomb_rows(m) rows, lincomb_ldc(q) columns, zeros beyond m x q), so every loop below has a
// compile-time trip count and no bounds branch: each row's QB coefficients are wave-uniform and come in a few wide
// scalar loads, and every FMA takes one as its scalar operand. Padded rows read column 0 (their coefficients are 0).
constexpr int LC_MAX_M = 384;  // input columns of one lincomb: [X, W, P] of blocks up to 128 columns
constexpr int LC_GROUP = 8;    // input columns loaded together

static int lincomb_qb(int q) {
    // the output group QB: the smallest of 8, 16, 24, 32 that splits q into equal-count launches
    const int groups = (q + 31) / 32;
    const int per = (q + groups - 1) / groups;
    return per <= 8 ? 8 : per <= 16 ? 16 : per <= 24 ? 24 : 32;
}
int lincomb_rows(int m) { return (m + LC_GROUP - 1) / LC_GROUP * LC_GROUP; }
int lincomb_ldc(int q) {
    const int qb = lincomb_qb(q);
    return (q + qb - 1) / qb * qb;
}

template <typename T, int QB>
__global__ __launch_bounds__(256) void k_lincomb(ColPtrs S, int m, int mp, const double *__restrict__ C, int ldc,
                                                 int q, T *__restrict__ Y, int qsplit, T *__restrict__ Y2, long N) {
    __shared__ const T *cols[LC_MAX_M];
    const int j0 = blockIdx.y * QB;
    for (int i = threadIdx.x; i < mp; i += 256)
        cols[i] = static_cast<const T *>(col_base(S, i < m ? i : 0, N, sizeof(T)));
    __syncthreads();
    const long p = blockIdx.x * 256L + threadIdx.x;
    if (p >= N) return;
    double acc[QB];
#pragma unroll
    for (int c = 0; c < QB; c++) acc[c] = 0.0;
    for (int i0 = 0; i0 < mp; i0 += LC_GROUP) {
        // the group's loads are independent and issued together
        double sv[LC_GROUP];
#pragma unroll
        for (int u = 0; u < LC_GROUP; u++) sv[u] = (double)gload(cols[i0 + u] + p);
#pragma unroll
        for (int u = 0; u < LC_GROUP; u++) {
            const double *__restrict__ row = C + (long)(i0 + u) * ldc + j0;
#pragma unroll
            for (int c = 0; c < QB; c++) acc[c] += sv[u] * row[c];
        }
    }
#pragma unroll
    for (int c = 0; c < QB; c++) {
        const int j = j0 + c;
        if (j < q) {
            T *dst = j < qsplit ? Y + (long)j * N : Y2 + (long)(j - qsplit) * N;
            dst[p] = (T)acc[c];
        }
    }
}

template <typename T>
void lincomb(const Cols &S, const double *C, int ldc, int q, T *Y, long N, hipStream_t s, int qsplit, T *Y2) {
    const int m = S.total();
    if (q <= 0) return;
    if (m > LC_MAX_M) throw InvalidError("lincomb: more than " + std::to_string(LC_MAX_M) + " input columns");
    if (ldc != lincomb_ldc(q)) throw InvalidError("lincomb: coefficients not padded to lincomb_ldc(q) columns");
    if (qsplit < 0 || qsplit > q) qsplit = q;
    const unsigned gx = (unsigned)((N + 255) / 256);
    const int qb = lincomb_qb(q), mp = lincomb_rows(m);
    const ColPtrs sp = to_ptrs(S);
    const dim3 grid(gx, (unsigned)(ldc / qb));
#define LIRA_LC(QB_) hipLaunchKernelGGL((k_lincomb<T, QB_>), grid, dim3(256), 0, s, sp, m, mp, C, ldc, q, Y, qsplit, Y2, N)
    if (qb == 8) LIRA_LC(8);
    else if (qb == 16) LIRA_LC(16);
    else if (qb == 24) LIRA_LC(24);
    else LIRA_LC(32);
#undef LIRA_LC
    LIRA_HIP(hipGetLastError());
}

// ----------------------------------------------------------------------------------------- pointwise ----
#define LIRA_GRID1(N) dim3((unsigned)(((N) + 255) / 256)), dim3(256)

template <typename T> __global__ void k_fill(T *y, long n, T a) {
    const long i = blockIdx.x * 256L + threadIdx.x;
    if (i < n) y[i] = a;
}
template <typename T> void fill(T *y, long count, double a, hipStream_t s) {
    if (count <= 0) return;
    hipLaunchKernelGGL(k_fill<T>, LIRA_GRID1(count), 0, s, y, count, (T)a);
    LIRA_HIP(hipGetLastError());
}

template <typename T> __global__ void k_axpy(T *y, const T *x, long n, T a) {
    const long i = blockIdx.x * 256L + threadIdx.x;
    if (i < n) y[i] += a * x[i];
}
template <typename T> void axpy(T *y, const T *x, long count, double a, hipStream_t s) {
    hipLaunchKernelGGL(k_axpy<T>, LIRA_GRID1(count), 0, s, y, x, count, (T)a);
    LIRA_HIP(hipGetLastError());
}

template <typename T>
__global__ void k_residual(T *r, const T *hx, const T *x, const double *theta, int nb, long N) {
    const long i = blockIdx.x * 256L + threadIdx.x;
    const int b = blockIdx.y;
    if (i >= N) return;
    const long id = (long)b * N + i;
    r[id] = (T)((double)hx[id] - theta[b] * (double)x[id]);
}
template <typename T> void residual(T *r, const T *hx, const T *x, const double *theta, int nb, long N, hipStream_t s) {
    if (nb <= 0) return;
    hipLaunchKernelGGL(k_residual<T>, dim3((unsigned)((N + 255) / 256), nb), dim3(256), 0, s, r, hx, x, theta, nb, N);
    LIRA_HIP(hipGetLastError());
}

// R = HX - theta X, the preconditioner's first pass W = R / max(diag_t + V - lam, 0.1) and the partial sums of |r_b|^2 in
// one pass (k_residual's formula; the partials are those that k_reduce would
// form from R, block by block and in its order, so the norms keep their bits). Bound by memory: a k_reduce of its own
// read R again. 95^3 x 8, f32: 31.3 us for this kernel and the reduction before, 20.8 us as one. RU points of a thread
// are loaded together, as many as keep the block's loads in flight.
template <typename T>
__global__ __launch_bounds__(256) void k_residual_precond(T *r, T *w, const T *hx, const T *x, const double *theta,
                                                          const T *v, const double *lam, T diag_t, long N,
                                                          double *partials) {
    constexpr int RU = 4;
    __shared__ double sh[256];
    const int b = blockIdx.y;
    const T *hb = hx + (long)b * N, *xb = x + (long)b * N;
    T *rb = r + (long)b * N, *wb = w + (long)b * N;
    const double th = theta[b];
    const T shift = (T)lam[b];
    const long stride = (long)RED_BLOCKS * 256;
    double acc = 0.0;
    auto point = [&](long p, T hv, T xv, T vv) {
        const T rv = (T)((double)hv - th * (double)xv);
        T d = diag_t + vv - shift;
        d = d > T(0.1) ? d : T(0.1);
        rb[p] = rv;
        wb[p] = rv / d;
        acc += (double)rv * (double)rv;
    };
    long p = blockIdx.x * 256L + threadIdx.x;
    for (; p + (RU - 1) * stride < N; p += RU * stride) {
        T hv[RU], xv[RU], vv[RU];
#pragma unroll
        for (int u = 0; u < RU; u++) {
            hv[u] = hb[p + u * stride];
            xv[u] = xb[p + u * stride];
            vv[u] = v[p + u * stride];
        }
#pragma unroll
        for (int u = 0; u < RU; u++) point(p + u * stride, hv[u], xv[u], vv[u]);
    }
    for (; p < N; p += stride) point(p, hb[p], xb[p], v[p]);
    const double sum = block_sum256(acc, sh);
    if (threadIdx.x == 0) partials[(long)b * RED_BLOCKS + blockIdx.x] = sum;
}
template <typename T>
void residual_precond(T *r, T *w, const T *hx, const T *x, const double *theta, const T *v, const double *lam,
                      double diag_t, int nb, long N, double scale, double *partials, double *norms, hipStream_t s) {
    for (int b0 = 0; b0 < nb; b0 += MAX_JOBS) {
        const int cnt = nb - b0 < MAX_JOBS ? nb - b0 : MAX_JOBS;
        const long off = (long)b0 * N;
        hipLaunchKernelGGL(k_residual_precond<T>, dim3(RED_BLOCKS, cnt), dim3(256), 0, s, r + off, w + off, hx + off,
                           x + off, theta + b0, v, lam + b0, (T)diag_t, N, partials);
        LIRA_HIP(hipGetLastError());
        KindList kl;
        for (int j = 0; j < MAX_JOBS; j++) kl.kind[j] = RED_DOT;
        hipLaunchKernelGGL(k_reduce_finish, dim3(cnt), dim3(256), 0, s, kl, partials, norms + b0, scale);
        LIRA_HIP(hipGetLastError());
    }
}

template <typename T> __global__ void k_density(T *rho, const T *psi, const double *f, int nb, long N) {
    const long i = blockIdx.x * 256L + threadIdx.x;
    if (i >= N) return;
    double acc = 0.0;
    for (int b = 0; b < nb; b++) {
        const double fb = f[b];
        if (fb == 0.0) continue;
        const double p = (double)psi[(long)b * N + i];
        acc += fb * p * p;
    }
    rho[i] = (T)acc;
}
template <typename T> void density(T *rho, const T *psi, const double *f, int nb, long N, hipStream_t s) {
    hipLaunchKernelGGL(k_density<T>, LIRA_GRID1(N), 0, s, rho, psi, f, nb, N);
    LIRA_HIP(hipGetLastError());
}

template <typename T> __global__ void k_sum3(T *o, const T *a, const T *b, const T *c, long N) {
    const long i = blockIdx.x * 256L + threadIdx.x;
    if (i < N) o[i] = (T)(((double)a[i] + (double)b[i]) + (double)c[i]);
}
template <typename T> void sum3(T *out, const T *a, const T *b, const T *c, long N, hipStream_t s) {
    hipLaunchKernelGGL(k_sum3<T>, LIRA_GRID1(N), 0, s, out, a, b, c, N);
    LIRA_HIP(hipGetLastError());
}
template <typename T> __global__ void k_add2(T *o, const T *a, const T *b, long N) {
    const long i = blockIdx.x * 256L + threadIdx.x;
    if (i < N) o[i] = a[i] + b[i];
}
template <typename T> void add2(T *out, const T *a, const T *b, long N, hipStream_t s) {
    hipLaunchKernelGGL(k_add2<T>, LIRA_GRID1(N), 0, s, out, a, b, N);
    LIRA_HIP(hipGetLastError());
}
template <typename T> __global__ void k_sub2(T *o, const T *a, const T *b, long N) {
    const long i = blockIdx.x * 256L + threadIdx.x;
    if (i < N) o[i] = a[i] - b[i];
}
template <typename T> void sub2(T *out, const T *a, const T *b, long N, hipStream_t s) {
    hipLaunchKernelGGL(k_sub2<T>, LIRA_GRID1(N), 0, s, out, a, b, N);
    LIRA_HIP(hipGetLastError());
}
template <typename T> void copy(T *out, const T *a, long N, hipStream_t s) {
    LIRA_HIP(hipMemcpyAsync(out, a, (size_t)N * sizeof(T), hipMemcpyDeviceToDevice, s));
}
template <typename Td, typename Ts> __global__ void k_convert(Td *o, const Ts *a, long N) {
    const long i = blockIdx.x * 256L + threadIdx.x;
    if (i < N) o[i] = (Td)a[i];
}
template <typename Td, typename Ts> void convert(Td *out, const Ts *a, long N, hipStream_t s) {
    hipLaunchKernelGGL((k_convert<Td, Ts>), LIRA_GRID1(N), 0, s, out, a, N);
    LIRA_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------------------------- LSDA ----
// Dirac exchange + PW92 correlation (qm/src/xc.rs:78-187), evaluated in f64 at every point: the formulas of exc_point,
// with the roots, logarithms and quotients in the forms that they need. The kernel is bound by f64 issue (4 cycles per
// instruction and wave): with the library's cbrt, log and sqrt and IEEE division a point took 664 f64 instructions, here
// 273. Each form starts from a hardware estimate and ends with one step of third order, whose last operation is an fma:
// relative errors below 1 ulp. 95^3 f32: 23.5 -> 11.8 us a call; the f64 kernel alone 27.6 -> 14.3 us. Mean errors against
// 113-bit arithmetic over n of 1e-2 .. 1e5, in units of 2^-53, here and with exc_point's forms: e 0.76 and 0.81, v_up 1.32
// and 1.32, v_down 0.76 and 0.76; at low densities both are set by the rounding of 1 + 1 / q1.

// 1/x: y (1 + e + e^2), e = 1 - x y (the estimates of this and the next are good to some 2^-24)
__device__ inline double rcp64(double x) {
    const double y = __builtin_amdgcn_rcp(x), e = fma(-x, y, 1.0);
    return fma(y, fma(e, e, e), y);
}

// x^{-1/2}: y (1 - e)^{-1/2}, e = 1 - x y^2
__device__ inline double rsqrt64(double x) {
    const double y = __builtin_amdgcn_rsq(x), e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
}

// m^{1/3} for a normal f32-range m: with r ~ m^{-1/3}, c = m r^2 and e = 1 - c r, it is c (1 - e)^{-2/3}
__device__ inline double cbrt_of(double m, double r) {
    const double c = m * (r * r), e = fma(-c, r, 1.0);
    return fma(c * e, fma(e, 5.0 / 9.0, 2.0 / 3.0), c);
}
__device__ inline double cbrt_seed(double m) {
    return (double)__builtin_amdgcn_exp2f(__builtin_amdgcn_logf((float)m) * (-1.0f / 3.0f));
}
// x = m 2^{3k} with m within 2^{+-3}: the seed's f32 range, for any positive finite x
__device__ inline double cbrt_scale(double x, int &k) {
    k = (__builtin_amdgcn_frexp_exp(x) * 21846) >> 16;
    return __builtin_amdgcn_ldexp(x, -3 * k);
}
__device__ inline double cbrt64(double x) {  // x >= 0
    int k;
    const double m = cbrt_scale(x, k);
    return x > 0.0 ? __builtin_amdgcn_ldexp(cbrt_of(m, cbrt_seed(m)), k) : x;
}
// cbrt of 0 or 2^-54 .. 2, which needs no scaling
__device__ inline double cbrt_unit(double x) { return x > 0.0 ? cbrt_of(x, cbrt_seed(x)) : x; }
__device__ inline double rcbrt64(double x) {  // x > 0
    int k;
    const double m = cbrt_scale(x, k), r = cbrt_seed(m), e = fma(-(m * (r * r)), r, 1.0);
    return __builtin_amdgcn_ldexp(fma(r * e, fma(e, 2.0 / 9.0, 1.0 / 3.0), r), -k);
}

// ln(a), a >= 1: with a = 2^j m, m in [sqrt(1/2), sqrt 2), it is j ln 2 + 2 atanh((m - 1) / (m + 1)). |s| is at most
// 3 - 2 sqrt 2, so the series' first term left out is 3e-17 of its sum; m - 1 is exact.
__device__ inline double log64(double a) {
    double m = __builtin_amdgcn_frexp_mant(a);
    const bool low = m < 0.70710678118654752;
    const int j = __builtin_amdgcn_frexp_exp(a) - (low ? 1 : 0);
    m = low ? m + m : m;
    const double s = (m - 1.0) * rcp64(m + 1.0), t = s * s;
    double p = 1.0 / 19.0;
    p = fma(p, t, 1.0 / 17.0);
    p = fma(p, t, 1.0 / 15.0);
    p = fma(p, t, 1.0 / 13.0);
    p = fma(p, t, 1.0 / 11.0);
    p = fma(p, t, 1.0 / 9.0);
    p = fma(p, t, 1.0 / 7.0);
    p = fma(p, t, 1.0 / 5.0);
    p = fma(p, t, 1.0 / 3.0);
    const double s2 = 2.0 * s;
    return fma((double)j, 0.6931471805599453, fma(s2 * t, p, s2));
}

// PW92's G(rs) and dG/drs, given srs = sqrt(rs) and its inverse
__device__ inline void pw92_point(double rs, double srs, double isr, double a, double a1, double b1, double b2,
                                  double b3, double b4, double &g, double &dg) {
    const double q0 = -2.0 * a * (1.0 + a1 * rs);
    const double q1 = 2.0 * a * (srs * (b1 + rs * b3) + rs * (b2 + rs * b4));
    const double q1p = a * (b1 * isr + 2.0 * b2 + 3.0 * b3 * srs + 4.0 * b4 * rs);
    const double ln = log64(1.0 + rcp64(q1));
    g = q0 * ln;
    dg = -2.0 * a * a1 * ln - q0 * q1p * rcp64(fma(q1, q1, q1));
}

__device__ inline void lsda_point(double nu, double nd, double &e, double &vu, double &vd) {
    nu = nu > 0.0 ? nu : 0.0;
    nd = nd > 0.0 ? nd : 0.0;
    const double n = nu + nd;
    if (n < 1e-20) {
        e = vu = vd = 0.0;
        return;
    }
    const double third = 1.0 / 3.0;
    const double cnu = cbrt64(nu), cnd = cbrt64(nd);
    const double ex = -0.9305257363491001 * (nu * cnu + nd * cnd);     // (3/4) (6 / pi)^{1/3}
    const double vxu = -1.2407009817988 * cnu, vxd = -1.2407009817988 * cnd;
    const double rs = 0.6203504908994 * rcbrt64(n);                  // (3 / (4 pi n))^{1/3}
    const double isr = rsqrt64(rs), srs = rs * isr;
    const double in = rcp64(n), z0 = (nu - nd) * in;
    double z = fma(fma(-n, z0, nu - nd), in, z0);  // correctly rounded: exactly +-1 at full polarisation, where 1 -+ z
                                                   // under a cube root must be 0
    z = z < -1.0 ? -1.0 : (z > 1.0 ? 1.0 : z);
    double ec0, dec0, ec1, dec1, mac, dmac;
    pw92_point(rs, srs, isr, 0.031091, 0.21370, 7.5957, 3.5876, 1.6382, 0.49294, ec0, dec0);
    pw92_point(rs, srs, isr, 0.015545, 0.20548, 14.1189, 6.1977, 3.3662, 0.62517, ec1, dec1);
    pw92_point(rs, srs, isr, 0.016887, 0.11125, 10.357, 3.6231, 0.88026, 0.49671, mac, dmac);
    const double ac = -mac, dac = -dmac;
    const double opz = cbrt_unit(1.0 + z), omz = cbrt_unit(1.0 - z);
    const double f0 = (1.0 + z) * opz + (1.0 - z) * omz - 2.0;
    const double f = fma(f0, 1.9236610509315364, f0 * -6.729470784749165e-17);  // f0 / (2^{4/3} - 2), the constant to 100 bits
    const double fp = 2.564881401242048 * (opz - omz);  // 4/3 (opz - omz) / (2^{4/3} - 2)
    const double IFPP0 = 1.0 / 1.709921;
    const double z3 = z * z * z, z4 = z3 * z;
    const double ec = ec0 + ac * f * IFPP0 * (1.0 - z4) + (ec1 - ec0) * f * z4;
    const double decdrs = dec0 + dac * f * IFPP0 * (1.0 - z4) + (dec1 - dec0) * f * z4;
    const double decdz = ac * IFPP0 * (fp * (1.0 - z4) - 4.0 * z3 * f) + (ec1 - ec0) * (fp * z4 + 4.0 * z3 * f);
    const double common = ec - rs * third * decdrs;
    e = ex + n * ec;
    vu = vxu + common - (z - 1.0) * decdz;
    vd = vxd + common - (z + 1.0) * decdz;
}

template <typename T> __global__ void k_xc(const T *nu, const T *nd, T *e, T *vu, T *vd, long N, const T *pc) {
    const long i = blockIdx.x * 256L + threadIdx.x;
    if (i >= N) return;
    double ee, a, b;
    // with a partial core the LSDA sees n_sigma = rho_sigma + rho_pc / 2 (qm/src/scf.rs:757-769)
    const double c = pc ? 0.5 * (double)pc[i] : 0.0;
    lsda_point((double)nu[i] + c, (double)nd[i] + c, ee, a, b);
    e[i] = (T)ee;
    vu[i] = (T)a;
    vd[i] = (T)b;
}
template <typename T> void xc_lsda(const T *nu, const T *nd, T *e, T *vu, T *vd, long N, hipStream_t s, const T *pc) {
    hipLaunchKernelGGL(k_xc<T>, LIRA_GRID1(N), 0, s, nu, nd, e, vu, vd, N, pc);
    LIRA_HIP(hipGetLastError());
}

// rho_in = max(2 rho_t - rho_{t-1}, 0): the density extrapolation of a warm start (crates/qm-gpu/src/scf.rs:1146-1162)
template <typename T> __global__ void k_extrapolate(T *out, const T *a, const T *b, long N) {
    const long i = blockIdx.x * 256L + threadIdx.x;
    if (i >= N) return;
    const double v = 2.0 * (double)a[i] - (double)b[i];
    out[i] = (T)(v > 0.0 ? v : 0.0);
}
template <typename T> void extrapolate(T *out, const T *a, const T *b, long N, hipStream_t s) {
    hipLaunchKernelGGL(k_extrapolate<T>, LIRA_GRID1(N), 0, s, out, a, b, N);
    LIRA_HIP(hipGetLastError());
}

// y *= num / den when both are > 0 (the per-channel charge renormalisation of the mixed density to the output's
// integral, crates/qm-gpu/src/scf.rs:1574-1582): the ratio in f64, rounded to T, applied in T
template <typename T> __global__ void k_scale_ratio(T *y, long N, const double *num, const double *den) {
    const long i = blockIdx.x * 256L + threadIdx.x;
    if (i >= N) return;
    const double a = *num, b = *den;
    if (!(a > 0.0 && b > 0.0)) return;
    y[i] = y[i] * (T)(a / b);
}
template <typename T> void scale_ratio(T *y, long N, const double *num, const double *den, hipStream_t s) {
    hipLaunchKernelGGL(k_scale_ratio<T>, LIRA_GRID1(N), 0, s, y, N, num, den);
    LIRA_HIP(hipGetLastError());
}

// (u + d)(p) by trilinear interpolation: the cell and fractions of qm::Grid::trilinear_cell in f64, neighbours beyond an
// upper face read 0, blended a (1 - t) + b t along x, then y, then z (crates/qm/src/grid.rs:54-86)
template <typename T>
__global__ void k_sample(const T *u, const T *d, int n, double h, const double *pts, int count, double *out) {
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q >= count) return;
    const double o = -((double)n - 1.0) * h / 2.0;
    long cell[3];
    double t[3];
    for (int a = 0; a < 3; a++) {
        const double x = (pts[3 * q + a] - o) / h;
        if (!(x >= 0.0 && x <= (double)(n - 1))) {
            out[q] = 0.0;
            return;
        }
        const double i0 = floor(x);
        cell[a] = (long)i0;
        t[a] = x - i0;
    }
    auto at = [&](int di, int dj, int dk) {
        const long a = cell[0] + di, b = cell[1] + dj, c = cell[2] + dk;
        if (a < n && b < n && c < n) {
            const long id = a + (long)n * (b + (long)n * c);
            return (double)u[id] + (double)d[id];
        }
        return 0.0;
    };
    auto lerp = [](double a, double b, double tt) { return a * (1.0 - tt) + b * tt; };
    auto xl = [&](int dj, int dk) { return lerp(at(0, dj, dk), at(1, dj, dk), t[0]); };
    auto yl = [&](int dk) { return lerp(xl(0, dk), xl(1, dk), t[1]); };
    out[q] = lerp(yl(0), yl(1), t[2]);
}
template <typename T>
void sample_density(const T *u, const T *d, int n, double h, const double *pts, int count, double *out,
                    hipStream_t s) {
    if (count <= 0) return;
    hipLaunchKernelGGL(k_sample<T>, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, s, u, d, n, h, pts, count, out);
    LIRA_HIP(hipGetLastError());
}

// --------------------------------------------------------------------------------------------- nuclei ----
template <typename T>
__global__ void k_nuclear(T *out, int n, double h, const double *pos, const double *zf, int nat, double sigma) {
    const long N = (long)n * n * n;
    const long i = blockIdx.x * 256L + threadIdx.x;
    if (i >= N) return;
    const long nn = (long)n * n;
    const long k = i / nn, rem = i - k * nn, j = rem / n, ii = rem - j * n;
    const double o = -((double)n - 1.0) * h / 2.0;
    const double x = o + (double)ii * h, y = o + (double)j * h, z = o + (double)k * h;
    const double s2 = sigma * sqrt(2.0), on_site = sqrt(2.0 / M_PI) / sigma;
    double acc = 0.0;
    for (int a = 0; a < nat; a++) {
        const double dx = x - pos[3 * a], dy = y - pos[3 * a + 1], dz = z - pos[3 * a + 2];
        const double d = sqrt(dx * dx + dy * dy + dz * dz);
        acc += d < 1e-10 ? -zf[a] * on_site : -zf[a] * erf(d / s2) / d;
    }
    out[i] = (T)acc;
}
template <typename T>
void nuclear_potential(T *out, int n, double h, const double *pos, const double *zf, int nat, double sigma,
                       hipStream_t s) {
    const long N = (long)n * n * n;
    hipLaunchKernelGGL(k_nuclear<T>, LIRA_GRID1(N), 0, s, out, n, h, pos, zf, nat, sigma);
    LIRA_HIP(hipGetLastError());
}

template <typename T>
__global__ void k_deposit(T *out, int n, double h, const double *pos, const double *zf, int nat, double sigma,
                          double scale) {
    const long N = (long)n * n * n;
    const long i = blockIdx.x * 256L + threadIdx.x;
    if (i >= N) return;
    const long nn = (long)n * n;
    const long k = i / nn, rem = i - k * nn, j = rem / n, ii = rem - j * n;
    const double o = -((double)n - 1.0) * h / 2.0;
    const double x = o + (double)ii * h, y = o + (double)j * h, z = o + (double)k * h;
    const double norm = 1.0 / pow(2.0 * M_PI * sigma * sigma, 1.5), inv = 1.0 / (2.0 * sigma * sigma);
    double acc = 0.0;
    for (int a = 0; a < nat; a++) {
        const double dx = x - pos[3 * a], dy = y - pos[3 * a + 1], dz = z - pos[3 * a + 2];
        acc += zf[a] * norm * exp(-(dx * dx + dy * dy + dz * dz) * inv);
    }
    out[i] = (T)(acc * scale);
}
template <typename T>
void deposit_charge(T *out, int n, double h, const double *pos, const double *zf, int nat, double sigma, double scale,
                    hipStream_t s) {
    const long N = (long)n * n * n;
    hipLaunchKernelGGL(k_deposit<T>, LIRA_GRID1(N), 0, s, out, n, h, pos, zf, nat, sigma, scale);
    LIRA_HIP(hipGetLastError());
}

// The LCG x -> a x + c (mod 2^64) advanced t steps: (A_t, C_t) with x_t = A_t x_0 + C_t, by binary powering.
__device__ inline void lcg_jump(uint64_t t, uint64_t &A, uint64_t &Cc) {
    uint64_t a = 6364136223846793005ULL, c = 1442695040888963407ULL;
    A = 1;
    Cc = 0;
    while (t) {
        if (t & 1) {
            A = A * a;
            Cc = Cc * a + c;
        }
        c = c * a + c;
        a = a * a;
        t >>= 1;
    }
}

constexpr int IO_RUN = 64;
template <typename T>
__global__ void k_initial(T *out, int n, double h, const double *pos, int nat, int k, uint64_t seed0) {
    const long N = (long)n * n * n;
    const long total = N * k;
    const long e0 = (blockIdx.x * 256L + threadIdx.x) * IO_RUN;
    if (e0 >= total) return;
    uint64_t A, Cc;
    lcg_jump((uint64_t)e0, A, Cc);
    uint64_t seed = A * seed0 + Cc;
    const double o = -((double)n - 1.0) * h / 2.0;
    const long nn = (long)n * n;
    for (long e = e0; e < min(total, e0 + IO_RUN); e++) {
        seed = seed * 6364136223846793005ULL + 1442695040888963407ULL;
        const double u = (double)(seed >> 11) / 9007199254740992.0;
        const long i = e % N;
        const long kk = i / nn, rem = i - kk * nn, j = rem / n, ii = rem - j * n;
        const double x = o + (double)ii * h, y = o + (double)j * h, z = o + (double)kk * h;
        double env = 0.0;
        for (int a = 0; a < nat; a++) {
            const double dx = x - pos[3 * a], dy = y - pos[3 * a + 1], dz = z - pos[3 * a + 2];
            env += exp(-(dx * dx + dy * dy + dz * dz) / 4.0);
        }
        out[e] = (T)((u + 0.5) * env);
    }
}
template <typename T>
void initial_orbitals(T *out, int n, double h, const double *pos, int nat, int k, uint64_t seed0, hipStream_t s) {
    const long total = (long)n * n * n * k;
    const long threads = (total + IO_RUN - 1) / IO_RUN;
    hipLaunchKernelGGL(k_initial<T>, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, out, n, h, pos, nat, k,
                       seed0);
    LIRA_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------------------------- DIIS ----
constexpr int DIIS_MAX = 16;
template <typename T> struct PtrList {
    const T *p[DIIS_MAX];
};
template <typename T>
__global__ void k_diis_mix(T *out, PtrList<T> rho, PtrList<T> res, const double *c, int m, double alpha, long N) {
    const long i = blockIdx.x * 256L + threadIdx.x;
    if (i >= N) return;
    double acc = 0.0;
    for (int q = 0; q < m; q++) acc += c[q] * ((double)rho.p[q][i] + alpha * (double)res.p[q][i]);
    out[i] = (T)(acc > 0.0 ? acc : 0.0);
}
template <typename T>
void diis_mix(T *out, const T *const *rho, const T *const *res, const double *c, int m, double alpha, long N,
              hipStream_t s) {
    if (m > DIIS_MAX) throw InvalidError("diis_mix: history too long");
    PtrList<T> a{}, b{};
    for (int q = 0; q < m; q++) {
        a.p[q] = rho[q];
        b.p[q] = res[q];
    }
    hipLaunchKernelGGL(k_diis_mix<T>, LIRA_GRID1(N), 0, s, out, a, b, c, m, alpha, N);
    LIRA_HIP(hipGetLastError());
}

// -------------------------------------------------------------------------------------------- forces ----
template <typename T>
__global__ __launch_bounds__(256) void k_hf_forces(const T *rho, int n, double h, const double *pos, const double *zf,
                                                   double sigma, double *partials) {
    __shared__ double sh[256];
    const int I = blockIdx.y;
    const long N = (long)n * n * n, nn = (long)n * n;
    const double o = -((double)n - 1.0) * h / 2.0;
    const double a = sigma * sqrt(2.0);
    const double px = pos[3 * I], py = pos[3 * I + 1], pz = pos[3 * I + 2], z = zf[I];
    double f0 = 0.0, f1 = 0.0, f2 = 0.0;
    for (long p = blockIdx.x * 256L + threadIdx.x; p < N; p += (long)gridDim.x * 256) {
        const long k = p / nn, rem = p - k * nn, j = rem / n, i = rem - j * n;
        const double dx = o + (double)i * h - px, dy = o + (double)j * h - py, dz = o + (double)k * h - pz;
        const double d = sqrt(dx * dx + dy * dy + dz * dz);
        if (d < 1e-8) continue;
        const double u = d / a;
        const double gp = ((2.0 / sqrt(M_PI)) * u * exp(-u * u) - erf(u)) / (d * d);
        const double w = (double)rho[p] * (-z * gp / d);
        f0 += w * dx;
        f1 += w * dy;
        f2 += w * dz;
    }
    const double r0 = block_sum256(f0, sh), r1 = block_sum256(f1, sh), r2 = block_sum256(f2, sh);
    if (threadIdx.x == 0) {
        partials[((long)I * 3 + 0) * RED_BLOCKS + blockIdx.x] = r0;
        partials[((long)I * 3 + 1) * RED_BLOCKS + blockIdx.x] = r1;
        partials[((long)I * 3 + 2) * RED_BLOCKS + blockIdx.x] = r2;
    }
}

__global__ __launch_bounds__(256) void k_sum_partials(const double *partials, double *out, double scale) {
    __shared__ double sh[256];
    double acc = 0.0;
    for (int p = threadIdx.x; p < RED_BLOCKS; p += 256) acc += partials[(long)blockIdx.x * RED_BLOCKS + p];
    const double r = block_sum256(acc, sh);
    if (threadIdx.x == 0) out[blockIdx.x] = r * scale;
}

template <typename T>
void hf_forces(const T *rho, int n, double h, const double *pos, const double *zf, int nat, double sigma,
               double *partials, double *out, hipStream_t s) {
    if (nat <= 0) return;
    hipLaunchKernelGGL(k_hf_forces<T>, dim3(RED_BLOCKS, nat), dim3(256), 0, s, rho, n, h, pos, zf, sigma, partials);
    LIRA_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_sum_partials, dim3(3 * nat), dim3(256), 0, s, partials, out, h * h * h);
    LIRA_HIP(hipGetLastError());
}

// ------------------------------------------------------------------------------- explicit instances ----
#define LIRA_INST(T)                                                                                                  \
    template void stencil<T>(int, const StencilParams &, const T *, T *, const T *, const T *, const double *,       \
                             hipStream_t, int);                                                                       \
    template void reduce_jobs<T>(const RedJobs<T> &, int, double, double *, double *, hipStream_t);                 \
    template void gram<T>(const Cols &, const Cols &, long, double, double *, size_t, double *, hipStream_t);       \
    template void residual_precond<T>(T *, T *, const T *, const T *, const double *, const T *, const double *,     \
                                      double, int, long, double, double *, double *, hipStream_t);                    \
    template void lincomb<T>(const Cols &, const double *, int, int, T *, long, hipStream_t, int, T *);                       \
    template void fill<T>(T *, long, double, hipStream_t);                                                           \
    template void axpy<T>(T *, const T *, long, double, hipStream_t);                                                \
    template void residual<T>(T *, const T *, const T *, const double *, int, long, hipStream_t);                    \
    template void density<T>(T *, const T *, const double *, int, long, hipStream_t);                                \
    template void sum3<T>(T *, const T *, const T *, const T *, long, hipStream_t);                                  \
    template void add2<T>(T *, const T *, const T *, long, hipStream_t);                                             \
    template void sub2<T>(T *, const T *, const T *, long, hipStream_t);                                             \
    template void copy<T>(T *, const T *, long, hipStream_t);                                                        \
    template void xc_lsda<T>(const T *, const T *, T *, T *, T *, long, hipStream_t, const T *);                                \
    template void nuclear_potential<T>(T *, int, double, const double *, const double *, int, double, hipStream_t); \
    template void deposit_charge<T>(T *, int, double, const double *, const double *, int, double, double,          \
                                    hipStream_t);                                                                     \
    template void initial_orbitals<T>(T *, int, double, const double *, int, int, uint64_t, hipStream_t);            \
    template void diis_mix<T>(T *, const T *const *, const T *const *, const double *, int, double, long,            \
                              hipStream_t);                                                                           \
    template void hf_forces<T>(const T *, int, double, const double *, const double *, int, double, double *,        \
                               double *, hipStream_t);                                                                \
    template void extrapolate<T>(T *, const T *, const T *, long, hipStream_t);                                      \
    template void scale_ratio<T>(T *, long, const double *, const double *, hipStream_t);                             \
    template void sample_density<T>(const T *, const T *, int, double, const double *, int, double *, hipStream_t);
LIRA_INST(float)
LIRA_INST(double)
template void convert<float, double>(float *, const double *, long, hipStream_t);
template void convert<double, float>(double *, const float *, long, hipStream_t);
template void convert<double, double>(double *, const double *, long, hipStream_t);
template void convert<float, float>(float *, const float *, long, hipStream_t);

}  // namespace lira
