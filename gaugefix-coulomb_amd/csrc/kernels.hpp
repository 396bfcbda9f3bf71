// kernels.hpp -- HIP kernels of the Coulomb gauge-fixing engine (gfx950).
//
// Device state of one lattice (V = ns^3 nt sites, Vh = V/2 per parity):
//   cfg : AoS FP64, the reference's U image (4V matrices, site-major, mu=T,Z,Y,X)
//   u0  : SoA spatial links of the configuration being fixed
//   g   : SoA gauge transformation
// u0 and g hold SU(3) matrices as their first two rows (6 complex numbers; an
// FP64 u0 link as five, see u0 fields below); row 2 = conj(r0 x r1) is rebuilt
// in registers on every load.  One tiled field
// (see field_size below) per parity p and, for u0, direction i = Z,Y,X:
//   u0 field p*3 + i,   g field p.
// Within a parity the index is h = lex >> 1 with lex = ((t ns + z) ns + y) ns + x
// (ns even), so the y/z neighbours of a site sit at a constant offset +-ns/2,
// +-ns^2/2 in the other parity's field and the x neighbours at h or h+-1; a
// timeslice t is the range [t ns^3/2, (t+1) ns^3/2) of h.
//
// The sweep keeps the reference's state in factored form: the current links are
// U_i(n) = G(n) u0_i(n) G(n+i)^dagger, so a half-sweep only rewrites G on the
// active parity while u0 stays read-only.  w(n) = sum_i U_i(n) + U_i(n-i)^dagger
// (src/gauge_fixing.c:493-531) becomes w(n) = G(n) W(n) with
// W(n) = sum_i [u0_i(n) G(n+i)^dagger + u0_i(n-i)^dagger G(n-i)^dagger].
//
// The axial frame.  The links G(n) u_i(n) G(n+i)^dagger are, with any field
// h(n) of SU(3) matrices, also G'(n) u0_i(n) G'(n+i)^dagger with
// u0_i(n) = h(n) u_i(n) h(n+i)^dagger and G' = G h^dagger, and since an update
// multiplies G from the left it acts on G' in the same way.  FP64 sweeps take
// for h the ordered product of the Z links in the site's column below it,
// h(z+1) = h(z) u_Z(z): then u0_Z = 1 except on the plane z = ns - 1, where it
// is the product of the whole column.  A sweep reads four links per site
// instead of six (320 instead of 480 B of u0 per update) and forms four
// products instead of six; only the sites of the two planes next to the wrap
// read a Z link.  G = G' h is formed at the end of a fix (k_frame_end).  The
// sweeps are bound by the rate of their bytes and next by instructions: 768 ->
// 608 B and 2414 -> about 2080 VALU instructions per update took the 48^3 x 96
// FP64 fix from 0.652 to 0.547 s; 32^3 x 64 from 131 to 110 ms, 8^3 x 16 from
// 9.4 to 7.9 ms.  (With the update as it stands, 1895 instructions and 639 B of
// L2 misses per update, the fix takes 0.513 s, of which entering and leaving the
// frame are 3.1 ms.)
// Two kinds of sweeps keep the configuration's own frame.  The FP32 phase of a
// mixed fix: the rounding of its sweeps is carried to the result in the
// directions that do not change the gauge condition, 1e-6 to 1e-5 of G as a
// rule but 1e-3 on the odd timeslice (1.3e-4 of G), and another frame would give
// another one.  And links that are not near SU(3) (near_su3), which the products
// up a column would spread.
#pragma once

#include "su3.hpp"

namespace gfc {

constexpr int kBlock = 256;
constexpr int kPlanes = 6;  // planes of a tile: complex numbers of a two-row matrix

// Kernels and device helpers have internal linkage: each translation unit
// that launches them (engine.hip, server.hip) carries its own code object.
namespace {

// Loads that stream (read once per sweep of a lattice larger than the
// Infinity Cache) carry the non-temporal hint so that the L2 keeps the
// neighbour G matrices, which six sites read.
typedef double dvec2 __attribute__((ext_vector_type(2)));
typedef float fvec2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ cplx<double> ld_stream(const cplx<double> *p) {
    dvec2 v = __builtin_nontemporal_load(reinterpret_cast<const dvec2 *>(p));
    return c_make<double>(v.x, v.y);
}
__device__ __forceinline__ cplx<float> ld_stream(const cplx<float> *p) {
    fvec2 v = __builtin_nontemporal_load(reinterpret_cast<const fvec2 *>(p));
    return c_make<float>(v.x, v.y);
}
__device__ __forceinline__ void st_stream(cplx<double> *p, const cplx<double> &c) {
    dvec2 v = {c.re, c.im};
    __builtin_nontemporal_store(v, reinterpret_cast<dvec2 *>(p));
}
__device__ __forceinline__ void st_stream(cplx<float> *p, const cplx<float> &c) {
    fvec2 v = {c.re, c.im};
    __builtin_nontemporal_store(v, reinterpret_cast<fvec2 *>(p));
}

// Tiled layout of a matrix field over n parity sites: the six stored complex
// numbers of 32 consecutive sites form one 6 x 32 tile, element k of site h at
// (h / 32) 192 + h % 32 + 32 k.  One 32-bit offset (on a uniform base) plus immediate
// steps of 32 elements addresses a whole matrix, and 32 lanes with
// consecutive h read 32 consecutive numbers.  A field holds field_size(n)
// complex numbers (n rounded up to whole tiles) and must stay below 4 GiB.
constexpr int kTile = 32;

__host__ __device__ constexpr int64_t field_size(int64_t n) {
    return (n + kTile - 1) / kTile * kTile * kPlanes;
}

// (FP64: h < 2^26, so the tile number takes a full-rate 24-bit product)
template <typename T>
__device__ __forceinline__ uint32_t tile_bytes_of(int h, int planes) {
    if constexpr (sizeof(T) == sizeof(double))
        return __umul24((unsigned)(h >> 5), (unsigned)(kTile * planes * sizeof(cplx<T>))) +
               (uint32_t)(h & (kTile - 1)) * (uint32_t)sizeof(cplx<T>);
    else
        return ((uint32_t)(h >> 5) * (uint32_t)(kTile * planes) + (uint32_t)(h & (kTile - 1))) *
               (uint32_t)sizeof(cplx<T>);
}

template <typename T>
__device__ __forceinline__ const cplx<T> *elem_ptr(const cplx<T> *field, uint32_t byte_off,
                                                   int k) {
    return reinterpret_cast<const cplx<T> *>(reinterpret_cast<const char *>(field) +
                                             (uint64_t)byte_off + k * kTile * sizeof(cplx<T>));
}
template <typename T>
__device__ __forceinline__ cplx<T> *elem_ptr(cplx<T> *field, uint32_t byte_off, int k) {
    return reinterpret_cast<cplx<T> *>(reinterpret_cast<char *>(field) + (uint64_t)byte_off +
                                       k * kTile * sizeof(cplx<T>));
}

template <typename T>
__device__ __forceinline__ uint32_t tile_bytes(int h) {
    return tile_bytes_of<T>(h, kPlanes);
}

// u0 fields.  The sweeps read all six u0 links of a site per update, two
// thirds of their bytes, and they are bound by bytes; so an FP64 u0 matrix
// keeps five complex numbers: row 0, and the two elements of row 1 that do not
// sit under row 0's element of largest modulus (its pivot).  The pivot's row-1
// element follows from the orthogonality of the rows (u0_unpack), to a few
// ulps of the projected input.  FP32 u0 keeps both rows (six numbers): the
// FP32 sweep is also at its VALU limit.  G keeps both rows too: stored in five
// numbers it made the 48^3 x 96 FP64 fix 6% slower (the unpacking sits on the
// neighbour loads' path).  Tiles hold U0Planes<T>::n planes of
// 32 sites; the allocation keeps six planes per field (it also stages FP32
// input on upload).
template <typename T>
struct U0Planes {
    static constexpr int n = kPlanes;
};
template <>
struct U0Planes<double> {
    static constexpr int n = 5;
};

template <typename T>
__host__ __device__ constexpr int64_t u0_field_size(int64_t n) {
    return (n + kTile - 1) / kTile * kTile * U0Planes<T>::n;
}

template <typename T>
__device__ __forceinline__ uint32_t u0_tile_bytes(int h) {
    return tile_bytes_of<T>(h, U0Planes<T>::n);
}

// Field of the spatial links u0_i on parity p; field of G on parity p.
template <typename T>
__device__ __forceinline__ const cplx<T> *u0_field(const cplx<T> *u0, int Vh, int p, int i) {
    return u0 + (p * 3 + i) * u0_field_size<T>(Vh);
}
template <typename T>
__device__ __forceinline__ cplx<T> *u0_field(cplx<T> *u0, int Vh, int p, int i) {
    return u0 + (p * 3 + i) * u0_field_size<T>(Vh);
}
// In the axial frame: field of the links u0_i on parity p, i = 1 (Y), 2 (X);
// of the Z links of the plane z = ns - 1 on parity p, by their index in the
// plane, t ns^2/2 + y ns/2 + x/2 (Vh / ns sites); and of h^dagger on parity p,
// kept for the way out of the frame.
template <typename C>
__device__ __forceinline__ C *axial_field(C *u0, int Vh, int p, int i) {
    return u0 + (p * 2 + i - 1) * u0_field_size<double>(Vh);
}
template <typename C>
__device__ __forceinline__ C *axial_wrap(C *u0, int Vh, int ns, int p) {
    return u0 + 4 * u0_field_size<double>(Vh) + p * u0_field_size<double>(Vh / ns);
}
template <typename C>
__device__ __forceinline__ C *axial_h(C *u0, int Vh, int ns, int p) {
    return axial_wrap(u0, Vh, ns, 2) + p * field_size(Vh);
}
// Numbers of the u0 allocation: the six fields of links in the configuration's
// frame at six planes each (which also stage FP32 input), or those of the axial
// frame, 32 to 37 planes of Vh numbers (more than 36 for ns = 2 and lattices
// of a few tiles).
__host__ __device__ constexpr int64_t u0_alloc_size(int64_t Vh, int ns) {
    const int64_t own = 6 * field_size(Vh);
    const int64_t axial = 4 * u0_field_size<double>(Vh) + 2 * u0_field_size<double>(Vh / ns) +
                          2 * field_size(Vh);
    return own > axial ? own : axial;
}
template <typename T>
__device__ __forceinline__ const cplx<T> *g_field(const cplx<T> *g, int Vh, int p) {
    return g + p * field_size(Vh);
}
template <typename T>
__device__ __forceinline__ cplx<T> *g_field(cplx<T> *g, int Vh, int p) {
    return g + p * field_size(Vh);
}

// SU(3) matrix from its two stored rows.
template <bool STREAM, typename T>
__device__ __forceinline__ void load_su3(mat3<T> &m, const cplx<T> *__restrict__ field, int h) {
    const uint32_t off = tile_bytes<T>(h);
#pragma unroll
    for (int k = 0; k < kPlanes; k++)
        m.e[k] = STREAM ? ld_stream(elem_ptr(field, off, k)) : *elem_ptr(field, off, k);
    m_fill_row2(m);
}

// The two stored rows only (row 2 left unset).
template <bool STREAM, typename T>
__device__ __forceinline__ void load_rows01(mat3<T> &m, const cplx<T> *__restrict__ field, int h) {
    const uint32_t off = tile_bytes<T>(h);
#pragma unroll
    for (int k = 0; k < kPlanes; k++)
        m.e[k] = STREAM ? ld_stream(elem_ptr(field, off, k)) : *elem_ptr(field, off, k);
}

// Index of row 0's element of largest modulus (ties to the lower index); the
// products are explicit FMAs, so a builder and a reader compute the same bits.
__device__ __forceinline__ int u0_pivot(const cplx<double> *r0) {
    const double n0 = __builtin_fma(r0[0].re, r0[0].re, r0[0].im * r0[0].im);
    const double n1 = __builtin_fma(r0[1].re, r0[1].re, r0[1].im * r0[1].im);
    const double n2 = __builtin_fma(r0[2].re, r0[2].re, r0[2].im * r0[2].im);
    return (n0 >= n1 && n0 >= n2) ? 0 : (n1 >= n2 ? 1 : 2);
}

// Rows 0 and 1 of an FP64 u0 matrix from its five stored numbers e[0..4]:
// row 0 = e[0..2]; row 1 = e[3], e[4] in the two non-pivot columns, and in the
// pivot column k the element x with sum_j r0_j conj(r1_j) = 0, i.e.
// x = -conj(S) r0_k / |r0_k|^2, S = sum_{j != k} r0_j conj(r1_j).  |r0_k|^2 is
// at least 1/3, so the division (a reciprocal, rcp_nr) is well conditioned.
__device__ __forceinline__ cplx<double> csel(bool c, cplx<double> x, cplx<double> y) {
    return c_make<double>(c ? x.re : y.re, c ? x.im : y.im);
}

__device__ __forceinline__ void u0_unpack(mat3<double> &m, const cplx<double> *e) {
    const int k = u0_pivot(e);
    const cplx<double> e0 = e[0], e1 = e[1], e2 = e[2], s0 = e[3], s1 = e[4];
    const cplx<double> r = csel(k == 0, e0, csel(k == 1, e1, e2));
    const cplx<double> a = csel(k == 0, e1, e0);  // row 0 over the first stored element
    const cplx<double> b = csel(k == 2, e1, e2);  // ... and over the second
    // S = a conj(s0) + b conj(s1)
    const double sre = __builtin_fma(a.re, s0.re, __builtin_fma(a.im, s0.im,
                       __builtin_fma(b.re, s1.re, b.im * s1.im)));
    const double sim = __builtin_fma(a.im, s0.re, -__builtin_fma(a.re, s0.im,
                       -__builtin_fma(b.im, s1.re, -(b.re * s1.im))));
    const double nr = __builtin_fma(r.re, r.re, r.im * r.im);
    const double inv = rcp_nr(nr);
    const cplx<double> x = c_make<double>(-__builtin_fma(sre, r.re, sim * r.im) * inv,
                                          -__builtin_fma(sre, r.im, -(sim * r.re)) * inv);
    m.e[0] = e0;
    m.e[1] = e1;
    m.e[2] = e2;
    m.e[3] = csel(k == 0, x, s0);
    m.e[4] = csel(k == 0, s0, csel(k == 1, x, s1));
    m.e[5] = csel(k == 2, x, s1);
}

// The N stored numbers of a matrix at byte offset off of a field, as loaded.
template <bool STREAM, typename T, int N>
__device__ __forceinline__ void load_raw(cplx<T> (&e)[N], const cplx<T> *__restrict__ field,
                                         uint32_t off) {
#pragma unroll
    for (int k = 0; k < N; k++)
        e[k] = STREAM ? ld_stream(elem_ptr(field, off, k)) : *elem_ptr(field, off, k);
}

// Rows 0 and 1 (row 2 left unset) from the stored numbers of a G matrix ...
template <typename T>
__device__ __forceinline__ void rows01(mat3<T> &m, const cplx<T> (&e)[kPlanes]) {
#pragma unroll
    for (int k = 0; k < kPlanes; k++) m.e[k] = e[k];
}

// ... and of a u0 matrix.
template <typename T>
__device__ __forceinline__ void u0_rows01(mat3<T> &m, const cplx<T> (&e)[U0Planes<T>::n]) {
    if constexpr (U0Planes<T>::n == kPlanes)
        rows01(m, e);
    else
        u0_unpack(m, e);
}

// Rows 0 and 1 of a u0 matrix (row 2 left unset).
template <bool STREAM, typename T>
__device__ __forceinline__ void load_u0_rows01(mat3<T> &m, const cplx<T> *__restrict__ field,
                                               int h) {
    cplx<T> e[U0Planes<T>::n];
    load_raw<STREAM>(e, field, u0_tile_bytes<T>(h));
    u0_rows01(m, e);
}

// A u0 matrix in FP64 (rows 0 and 1 as stored, row 2 rebuilt).
template <typename T>
__device__ __forceinline__ void load_u0_d(mat3<double> &m, const cplx<T> *__restrict__ field,
                                          int h) {
    mat3<T> t;
    load_u0_rows01<false>(t, field, h);
#pragma unroll
    for (int k = 0; k < kPlanes; k++) m.e[k] = c_make<double>((double)t.e[k].re, (double)t.e[k].im);
    m_fill_row2(m);
}

template <bool STREAM, typename T>
__device__ __forceinline__ void store_su3(const mat3<T> &m, cplx<T> *__restrict__ field, int h) {
    const uint32_t off = tile_bytes<T>(h);
#pragma unroll
    for (int k = 0; k < kPlanes; k++) {
        if (STREAM)
            st_stream(elem_ptr(field, off, k), m.e[k]);
        else
            *elem_ptr(field, off, k) = m.e[k];
    }
}

// The reunitarization of G (reunitarizeField, src/fields.c:144-187) always
// projects in FP64: an FP32 G (the FP32 phase of the mixed mode) is promoted,
// projected and rounded back.  The projection reads rows 0 and 1 only.
__device__ __forceinline__ void project_g(mat3<double> &m) { m_project_su3(m); }
__device__ __forceinline__ void project_g(mat3<float> &m) {
    mat3<double> d;
#pragma unroll
    for (int k = 0; k < kPlanes; k++) d.e[k] = c_make<double>(m.e[k].re, m.e[k].im);
    m_project_su3<double>(d);  // the rounding it always had: FP32 results hang on it
#pragma unroll
    for (int k = 0; k < kPlanes; k++) m.e[k] = c_make<float>((float)d.e[k].re, (float)d.e[k].im);
}

// Site geometry of parity index h on parity p.
struct Site {
    int x, y, z, t, xh, row;
};

__device__ __forceinline__ Site site_of(int h, int p, int ns) {
    const int nh = ns >> 1;
    Site s;
    s.xh = h % nh;
    int r = h / nh;
    s.y = r % ns;
    r /= ns;
    s.z = r % ns;
    s.t = r / ns;
    s.x = 2 * s.xh + ((s.y + s.z + s.t + p) & 1);
    s.row = h - s.xh;
    return s;
}

// Division of numbers below 2^26 by a fixed divisor d: n / d = n m >> s with
// m = ceil(2^s / d), s = 26 + ceil(log2 d) (exact: m d - 2^s < d <= 2^(s - 26)).
struct Divisor {
    uint32_t d, m, s;
};

inline Divisor make_divisor(uint32_t d) {
    uint32_t l = 0;
    while ((1u << l) < d) l++;
    return {d, (uint32_t)((((uint64_t)1 << (26 + l)) + d - 1) / d), 26 + l};
}

__device__ __forceinline__ uint32_t divide(uint32_t n, const Divisor &v) {
    return (uint32_t)(((uint64_t)n * v.m) >> v.s);
}

// Extents of a lattice as the sweeps' index arithmetic uses them.
struct Extents {
    int ns, Vh;
    Divisor nh, n;  // ns / 2, ns
};

inline Extents make_extents(int ns, int Vh) {
    return {ns, Vh, make_divisor((uint32_t)ns / 2), make_divisor((uint32_t)ns)};
}

// n / d and n % d for n below 2^16 and d = inv^-1 below 2^15, in FP32:
// (n + 1/2) / d is 1 / (2 d) or more from a whole number, further than its
// rounding (3 2^-24 n / d).
__device__ __forceinline__ int small_div(int &n, int d, float inv) {
    const int q = (int)(((float)n + 0.5f) * inv);
    n -= __mul24(q, d);
    return q;
}

// site_of for the workgroups of a sweep: the first index of a workgroup, which
// is uniform, is split by whole-number products on the scalar unit, and a
// lane's offset of at most 255 carried over with small quotients (three 32-bit
// divisions per lane took 75 vector instructions, 15 of them quarter-rate
// products, of about 2050 in the FP32 update).
__device__ __forceinline__ Site site_in_block(uint32_t first, int lane, int p, const Extents &x) {
    const int ns = x.ns, nh = ns >> 1;
    const uint32_t r0 = divide(first, x.nh), z0 = divide(r0, x.n), t0 = divide(z0, x.n);
    const float inv_nh = __builtin_amdgcn_rcpf((float)nh), inv_n = 0.5f * inv_nh;
    Site s;
    s.xh = (int)(first - r0 * x.nh.d) + lane;
    s.y = (int)(r0 - z0 * x.n.d) + small_div(s.xh, nh, inv_nh);
    s.z = (int)(z0 - t0 * x.n.d) + small_div(s.y, ns, inv_n);
    s.t = (int)t0 + small_div(s.z, ns, inv_n);
    s.x = 2 * s.xh + ((s.y + s.z + s.t + p) & 1);
    s.row = (int)first + lane - s.xh;
    return s;
}

// Parity indices (in the other parity) of the six spatial neighbours, in the
// direction order i = 0 (Z), 1 (Y), 2 (X).
struct Nbr {
    int fwd[3], bwd[3];
};

__device__ __forceinline__ Nbr neighbours(const Site &s, int h, int ns) {
    const int nh = ns >> 1, sz = ns * nh;
    Nbr n;
    n.fwd[0] = h + (s.z + 1 == ns ? -(ns - 1) * sz : sz);
    n.bwd[0] = h + (s.z == 0 ? (ns - 1) * sz : -sz);
    n.fwd[1] = h + (s.y + 1 == ns ? -(ns - 1) * nh : nh);
    n.bwd[1] = h + (s.y == 0 ? (ns - 1) * nh : -nh);
    n.fwd[2] = s.row + ((s.x + 1 == ns ? 0 : s.x + 1) >> 1);
    n.bwd[2] = s.row + ((s.x == 0 ? ns - 1 : s.x - 1) >> 1);
    return n;
}

// W += u0_Z(n) G(n+z)^dagger + u0_Z(n-z)^dagger G(n-z)^dagger in the axial
// frame, gf = G(n+z) and gb = G(n-z) with all three rows.  u0_Z is 1 but on the plane z = ns - 1,
// which only the sites of that plane and of z = 0 meet: one plane is ns^2 / 2
// consecutive parity indices, so most waves skip both branches.
template <bool STREAM>
__device__ __forceinline__ void axial_z(mat3<double> &W, const cplx<double> *__restrict__ u0,
                                        const Site &s, int ns, int Vh, int p,
                                        const mat3<double> &gf, const mat3<double> &gb) {
    const int hw = s.t * (ns * (ns >> 1)) + s.y * (ns >> 1) + s.xh;
    if (s.z + 1 == ns) {
        mat3<double> u;
        load_u0_rows01<STREAM>(u, axial_wrap(u0, Vh, ns, p), hw);
        m_mac_nd_su3(W, u, gf);
    } else {
        m_add_dagger(W, gf);
    }
    if (s.z == 0) {
        mat3<double> u;
        load_u0_rows01<STREAM>(u, axial_wrap(u0, Vh, ns, 1 - p), hw);
        m_fill_row2(u);
        m_mac_dagger_su3(W, gb, u);
    } else {
        m_add_dagger(W, gb);
    }
}

// ---------------------------------------------------------------------------
// The site update of parity index h = first + lane on parity p: reads the u0
// links (in the axial frame 4, and a Z link next to the wrap; else 6), 6
// neighbour G and G(n); writes G(n).  Shared by the single-lattice and the
// batched (serving) kernels, so a site computes the same bits in both.
// POUT projects the new G(n) onto SU(3) (in FP64, project_g) before storing
// it: the same bits as a reunitarization of this parity's G right after the
// sweep, since the projection reads rows 0 and 1 only.  PIN projects G(n)
// right after loading it and rebuilds its third row from the projected rows,
// as a store and reload would: the same bits as a reunitarization of this
// parity's G before the sweep (nothing else reads it in between).  STREAM
// reads u0 and G(n) with non-temporal loads (data read once per sweep);
// without it they are cached, for sweeps whose data stays in the Infinity
// Cache from one half-sweep to the next.
//
// In the configuration's own frame: the four matrices of a direction are loaded
// together, one memory round trip per direction rather than the
// compiler's two.
template <typename T, bool POUT, bool STREAM, bool PIN>
__device__ __forceinline__ void sweep_own(const cplx<T> *__restrict__ u0,
                                          cplx<T> *__restrict__ g, int ns, int Vh, int p,
                                          T omega, int hits, int h) {
    const Site s = site_of(h, p, ns);
    const Nbr nb = neighbours(s, h, ns);
    const cplx<T> *gq = g_field(static_cast<const cplx<T> *>(g), Vh, 1 - p);  // other parity
    cplx<T> *gp = g_field(g, Vh, p);
    // with PIN, G(n) is loaded and projected first and its rows 0 and 1 kept
    // through the W products (loaded later, next to its use, the projection
    // makes the compiler hold twice the registers)
    mat3<T> gn;
    if (PIN) {
        load_rows01<STREAM>(gn, static_cast<const cplx<T> *>(gp), h);
        project_g(gn);
        __builtin_amdgcn_sched_barrier(0);
    }
    // the products are SU(3): rows 0, 1 from the stored rows of the left
    // factor, row 2 by closure (m_mac_nd_su3, m_mac_dagger_su3).  The matrices
    // of a direction are loaded together, one memory round trip per direction
    // rather than the compiler's two (48^3 x 96: FP64 fix 1%, mixed 2% faster).
    mat3<T> W;
    m_zero(W);
#pragma unroll
    for (int i = 0; i < 3; i++) {
        constexpr int NU = U0Planes<T>::n;
        cplx<T> ruf[NU], rub[NU], rgf[kPlanes], rgb[kPlanes];
        load_raw<STREAM>(ruf, u0_field(u0, Vh, p, i), u0_tile_bytes<T>(h));
        load_raw<false>(rgf, gq, tile_bytes<T>(nb.fwd[i]));
        load_raw<STREAM>(rub, u0_field(u0, Vh, 1 - p, i), u0_tile_bytes<T>(nb.bwd[i]));
        load_raw<false>(rgb, gq, tile_bytes<T>(nb.bwd[i]));
        __builtin_amdgcn_sched_barrier(0);
        mat3<T> uf, gf, ub, gb;
        u0_rows01(uf, ruf);
        rows01(gf, rgf);
        m_fill_row2(gf);
        m_mac_nd_su3(W, uf, gf);  // u0_i(n) G(n+i)^dagger
        u0_rows01(ub, rub);
        m_fill_row2(ub);
        rows01(gb, rgb);
        m_mac_dagger_su3(W, gb, ub);  // (G(n-i) u0_i(n-i))^dagger
    }
    if (PIN)
        m_fill_row2(gn);  // the third row a store and reload would give
    else
        load_su3<STREAM>(gn, static_cast<const cplx<T> *>(gp), h);
    mat3<T> w, upd, out;
    m_mul(gn, W, w);
    la_or_update(w, hits, omega, upd);
    m_mul(upd, gn, out);
    if (POUT) project_g(out);
    store_su3<true>(out, gp, h);
}

// FP64, in the axial frame: the matrices of Z and Y come in one memory round
// trip, those of X and G(n) in another, in 214 registers (2 waves per SIMD).
// us per half-sweep at 64^3 x 128 / 48^3 x 96 / 32^3 x 64 / 24^3 x 48: 1475 /
// 479 / 92 / 31.4; with a round trip per direction in 168 registers (3 waves),
// three integer divisions per lane, and the compiler's contraction and branches
// in the local update 1600 / 498 / 96.5 / 33.3.  Of the same update, X's loads
// ahead of Y's products cost 0.3 to 2% and all loads first (one wave per SIMD)
// 35 to 50%.
struct AxialDir {
    cplx<double> uf[5], gf[kPlanes], ub[5], gb[kPlanes];
};

// W += u0_i(n) G(n+i)^dagger + u0_i(n-i)^dagger G(n-i)^dagger
__device__ __forceinline__ void axial_dir(mat3<double> &W, const AxialDir &r) {
    mat3<double> u, m;
    u0_rows01(u, r.uf);
    rows01(m, r.gf);
    m_fill_row2(m);
    m_mac_nd_su3(W, u, m);
    u0_rows01(u, r.ub);
    m_fill_row2(u);
    rows01(m, r.gb);
    m_mac_dagger_su3(W, m, u);  // (G(n-i) u0_i(n-i))^dagger
}

template <bool POUT, bool STREAM, bool PIN>
__device__ __forceinline__ void sweep_axial(const cplx<double> *__restrict__ u0,
                                            cplx<double> *__restrict__ g, const Extents &x, int p,
                                            double omega, int hits, int first, int lane) {
    typedef cplx<double> C;
    const int ns = x.ns, Vh = x.Vh, h = first + lane;
    const Site s = site_in_block((uint32_t)first, lane, p, x);
    const Nbr nb = neighbours(s, h, ns);
    const C *gq = g_field(static_cast<const C *>(g), Vh, 1 - p);  // other parity
    C *gp = g_field(g, Vh, p);
    mat3<double> gn;
    if (PIN) {
        load_rows01<STREAM>(gn, static_cast<const C *>(gp), h);
        project_g(gn);
        __builtin_amdgcn_sched_barrier(0);
    }
    auto load_dir = [&](AxialDir &r, int i) {
        load_raw<STREAM>(r.uf, axial_field(u0, Vh, p, i), u0_tile_bytes<double>(h));
        load_raw<false>(r.gf, gq, tile_bytes<double>(nb.fwd[i]));
        load_raw<STREAM>(r.ub, axial_field(u0, Vh, 1 - p, i), u0_tile_bytes<double>(nb.bwd[i]));
        load_raw<false>(r.gb, gq, tile_bytes<double>(nb.bwd[i]));
    };
    mat3<double> W, gf, gb;
    m_zero(W);
    load_rows01<false>(gf, gq, nb.fwd[0]);
    load_rows01<false>(gb, gq, nb.bwd[0]);
    AxialDir y, r;
    load_dir(y, 1);
    __builtin_amdgcn_sched_barrier(0);
    m_fill_row2(gf);
    m_fill_row2(gb);
    axial_z<STREAM>(W, u0, s, ns, Vh, p, gf, gb);
    __builtin_amdgcn_sched_barrier(0);
    axial_dir(W, y);
    load_dir(r, 2);
    if (!PIN) load_rows01<STREAM>(gn, static_cast<const C *>(gp), h);
    __builtin_amdgcn_sched_barrier(0);
    axial_dir(W, r);
    m_fill_row2(gn);  // with PIN, the third row a store and reload would give
    mat3<double> w, upd, out;
    m_mul(gn, W, w);
    la_or_update(w, hits, omega, upd);
    m_mul(upd, gn, out);
    if (POUT) project_g(out);
    store_su3<true>(out, gp, h);
}

// OWN: FP64 too in the configuration's own frame.
template <typename T, bool POUT = false, bool STREAM = true, bool PIN = false, bool OWN = false>
__device__ __forceinline__ void sweep_site(const cplx<T> *__restrict__ u0,
                                           cplx<T> *__restrict__ g, const Extents &x, int p,
                                           T omega, int hits, int first, int lane) {
    if constexpr (sizeof(T) == sizeof(double) && !OWN)
        sweep_axial<POUT, STREAM, PIN>(u0, g, x, p, omega, hits, first, lane);
    else
        sweep_own<T, POUT, STREAM, PIN>(u0, g, x.ns, x.Vh, p, omega, hits, first + lane);
}

// Workgroup order.  The hardware hands workgroup i of a launch to XCD i % 8,
// and each XCD has its own L2.  xcd_order renumbers the workgroups so that,
// in rounds of 8 x 64 workgroups, each XCD takes one contiguous run of the
// round (a launch of at most 512 workgroups: one contiguous eighth of it).
// The z-neighbour G of a site, ns^2 / 2 sites away (4.5 workgroups at 48^3),
// are then mostly in the same L2.  A bijection of [0, n).  The sweeps with
// cached loads use it: measured at 48^3 x 96 with cache-resident waves of
// single-timeslice launches (216 workgroups), an FP64 half-sweep is 11%
// faster and an FP32 one 10%.  The streaming sweeps keep the plain order,
// under which all XCDs stream one stretch of sites together (with xcd_order
// they were 1-2% slower; an XCD per contiguous eighth of a whole-lattice
// launch, 5% slower).
__device__ __forceinline__ unsigned xcd_order(unsigned i, unsigned n) {
    constexpr unsigned kXcd = 8, kRound = kXcd * 64;
    const unsigned base = i / kRound * kRound;
    const unsigned m = n - base < kRound ? n - base : kRound;  // workgroups in i's round
    const unsigned j = i - base, q = m / kXcd, r = m % kXcd, x = j % kXcd;
    return base + x * q + (x < r ? x : r) + j / kXcd;
}

// Whether G is reunitarized after half-sweep s (1, 2, ...): every R, and in the
// axial frame every kFrameReunit at least.  In exact arithmetic these more
// projections do nothing; here G drifts off SU(3) by its rounding, and with it a
// timeslice turns as a whole, a direction no gauge condition holds.  In the
// frame that drift is another one, by parameters 0.7 to 1.5 times that in the
// configuration's own: relative error of G against 80-bit arithmetic after 240
// half-sweeps at 14^3 x 12 with one / two hits (omega 1.7, R = 250), own frame
// 7.8e-15 / 7.9e-15, axial 8.6e-15 / 10.5e-15, axial with this 4.3e-15 / 2.5e-15
// (every 25: 2.6e-15 / 2.0e-15, but served lattices, which are projected one
// launch each, take 20% longer at 8^3 x 16).
constexpr unsigned kFrameReunit = 50;

__host__ __device__ inline bool reunit_due(unsigned s, unsigned R, bool frame) {
    return s % R == 0 || (frame && R > kFrameReunit && s % kFrameReunit == 0);
}

// One red/black half-sweep on parity p over parity indices [h0, h0 + count), in
// as many workgroups as count takes.  A small lattice's launch is a chain that
// begins with its arguments, so those that every sweep needs first lie in their
// first 64 bytes, and the number of workgroups is computed rather than read from
// behind them (FP32, us per half-sweep: 8^3 x 16 7.5 -> 7.2, 16^3 x 32 7.65 ->
// 7.35).
template <typename T, bool POUT = false, bool STREAM = true, bool PIN = false, bool OWN = false>
__global__ __launch_bounds__(kBlock) void k_sweep(const cplx<T> *__restrict__ u0,
                                                  cplx<T> *__restrict__ g, int p, T omega,
                                                  int hits, int h0, int count, Extents x) {
    const unsigned nb = ((unsigned)count + kBlock - 1) / kBlock;  // the launch's workgroups
    const unsigned b = STREAM ? blockIdx.x : xcd_order(blockIdx.x, nb);
    const int lane = (int)threadIdx.x;
    if ((int)(b * kBlock) + lane >= count) return;
    sweep_site<T, POUT, STREAM, PIN, OWN>(u0, g, x, p, omega, hits, h0 + (int)(b * kBlock), lane);
}

// Half-sweeps [from, to) of a small lattice in FP64, one workgroup per
// timeslice and one thread per site of each parity (S = ns^3 / 2 <= N sites):
// timeslices do not interact, so a workgroup runs through all the sweeps by
// itself, its G in LDS, with a workgroup barrier where the other path has a
// launch boundary.  Reunitarizations after the sweeps s + 1 < end for which
// they are due, as in the timeslice-blocked sweeps; the same bits.
//
// Bound by one wave's chain of instructions: a half-sweep launch of 8^3 x 16
// lasts 6.9 us from one to the next whatever its loads and code size, a
// half-sweep here 4.7 us; 8^3 x 2048 47 and 36 us, 10^3 x 256 12.8 and 9.5.
// (Loading the next sweep's links before the local update: 5.0 us, and with 512
// threads the registers spill.)
template <int N>
__global__ __launch_bounds__(N) void k_sweep_slices(const cplx<double> *__restrict__ u0,
                                                    cplx<double> *__restrict__ g, Extents x,
                                                    double omega, int hits, int from, int to,
                                                    int end, unsigned R) {
    typedef cplx<double> C;
    __shared__ C sh[2][N * kPlanes];
    const int ns = x.ns, Vh = x.Vh, S = ns * ns * (ns >> 1), lane = (int)threadIdx.x;
    const int first = (int)blockIdx.x * S, h = first + lane;
    const bool on = lane < S;
    auto copy = [&](bool in) {
        if (!on) return;
#pragma unroll
        for (int p = 0; p < 2; p++) {
            mat3<double> m;
            load_rows01<false>(m, in ? g_field(static_cast<const C *>(g), Vh, p)
                                     : static_cast<const C *>(sh[p]), in ? h : lane);
            store_su3<false>(m, in ? sh[p] : g_field(g, Vh, p), in ? lane : h);
        }
    };
    copy(true);
    __syncthreads();
    for (int k = from; k < to; k++) {
        const int p = k & 1;
        if (on) {
            const Site s = site_in_block((uint32_t)first, lane, p, x);
            const Nbr nb = neighbours(s, h, ns);
            const C *gq = sh[1 - p];
            AxialDir d[2];
#pragma unroll
            for (int i = 1; i < 3; i++) {
                load_raw<false>(d[i - 1].uf, axial_field(u0, Vh, p, i), u0_tile_bytes<double>(h));
                load_raw<false>(d[i - 1].ub, axial_field(u0, Vh, 1 - p, i),
                                u0_tile_bytes<double>(nb.bwd[i]));
            }
            mat3<double> W, gf, gb, gn, w, upd, out;
            m_zero(W);
            load_rows01<false>(gf, gq, nb.fwd[0] - first);
            load_rows01<false>(gb, gq, nb.bwd[0] - first);
            m_fill_row2(gf);
            m_fill_row2(gb);
            axial_z<false>(W, u0, s, ns, Vh, p, gf, gb);
#pragma unroll
            for (int i = 1; i < 3; i++) {
                load_raw<false>(d[i - 1].gf, gq, tile_bytes<double>(nb.fwd[i] - first));
                load_raw<false>(d[i - 1].gb, gq, tile_bytes<double>(nb.bwd[i] - first));
                axial_dir(W, d[i - 1]);
            }
            load_su3<false>(gn, static_cast<const C *>(sh[p]), lane);
            m_mul(gn, W, w);
            la_or_update(w, hits, omega, upd);
            m_mul(upd, gn, out);
            store_su3<false>(out, sh[p], lane);
        }
        __syncthreads();
        if (k + 1 < end && reunit_due((unsigned)(k + 1), R, true)) {
            if (on) {
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    mat3<double> m;
                    load_rows01<false>(m, static_cast<const C *>(sh[q]), lane);
                    project_g(m);
                    store_su3<false>(m, sh[q], lane);
                }
            }
            __syncthreads();
        }
    }
    copy(false);
}

// ---------------------------------------------------------------------------
// Per-site G kernels: one thread per site of the parities [p0, p0 + np),
// idx in [0, np Vh), parity p = p0 + idx / Vh.

// G <- identity (setFieldToIdentity, src/fields.c:64-100).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_g_identity(cplx<T> *__restrict__ g, int Vh) {
    const int idx = blockIdx.x * kBlock + threadIdx.x;
    if (idx >= 2 * Vh) return;
    const int p = idx >= Vh, h = idx - p * Vh;
    mat3<T> m;
    m_identity(m);
    store_su3<false>(m, g_field(g, Vh, p), h);
}

// Projects G onto SU(3) at parity index h of parity p.
template <typename T>
__device__ __forceinline__ void reunit_site(cplx<T> *__restrict__ g, int Vh, int p, int h) {
    cplx<T> *base = g_field(g, Vh, p);
    const uint32_t off = tile_bytes<T>(h);
    mat3<T> m;
#pragma unroll
    for (int k = 0; k < kPlanes; k++) m.e[k] = *elem_ptr(base, off, k);
    project_g(m);
    store_su3<false>(m, base, h);
}

// Parity indices [h0, h0 + count) of parities [p0, p0 + np).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_g_reunit(cplx<T> *__restrict__ g, int Vh, int p0,
                                                     int np, int h0, int count) {
    const int idx = blockIdx.x * kBlock + threadIdx.x;
    if (idx >= np * count) return;
    reunit_site<T>(g, Vh, p0 + idx / count, h0 + idx % count);
}

// FP32 -> FP64 hand-off of G: rows 0, 1 of the FP32 G promoted and projected
// in FP64, then, with FRAME, taken into the axial frame, where g holds h^dagger
// (k_frame_begin).
template <bool FRAME>
__global__ __launch_bounds__(kBlock) void k_g_promote(const cplx<float> *__restrict__ gf,
                                                      cplx<double> *__restrict__ g, int Vh) {
    const int idx = blockIdx.x * kBlock + threadIdx.x;
    if (idx >= 2 * Vh) return;
    const int p = idx >= Vh, h = idx - p * Vh;
    const cplx<float> *src = g_field(gf, Vh, p);
    const uint32_t off = tile_bytes<float>(h);
    mat3<double> m, hd, out;
#pragma unroll
    for (int k = 0; k < kPlanes; k++) {
        cplx<float> v = *elem_ptr(src, off, k);
        m.e[k] = c_make<double>(v.re, v.im);
    }
    m_project_su3(m);
    if (FRAME) {
        load_su3<false>(hd, g_field(static_cast<const cplx<double> *>(g), Vh, p), h);
        m_mul(m, hd, out);
    } else {
        out = m;
    }
    store_su3<false>(out, g_field(g, Vh, p), h);
}

// Stores a u0 matrix of type T from its rows 0 and 1 in FP64.
template <typename T>
__device__ __forceinline__ void store_u0(const mat3<double> &m, cplx<T> *__restrict__ field,
                                         int h) {
    cplx<double> e[kPlanes];
#pragma unroll
    for (int k = 0; k < kPlanes; k++) e[k] = m.e[k];
    if constexpr (U0Planes<T>::n == 5) {
        // row 1 without the element under row 0's pivot (u0_unpack)
        const int piv = u0_pivot(e);
        const cplx<double> s0 = csel(piv == 0, e[4], e[3]);
        const cplx<double> s1 = csel(piv == 2, e[4], e[5]);
        e[3] = s0;
        e[4] = s1;
    }
    const uint32_t off = u0_tile_bytes<T>(h);
#pragma unroll
    for (int k = 0; k < U0Planes<T>::n; k++)
        *elem_ptr(field, off, k) = c_make<T>((T)e[k].re, (T)e[k].im);
}

// The axial frame of a column (t, y, x): one thread walks its sites z = 0 ..
// ns - 1 with d(z) = h(z)^dagger, d(0) = 1 and d(z+1) = u_Z(z)^dagger d(z), one
// rounding per step, and calls visit(z, d); returns the adjoint of the Z link
// of the plane z = ns - 1 in the frame.  The next site's link is loaded while
// this one's product is formed.
template <typename Visit>
__device__ __forceinline__ mat3<double> walk_column(const cplx<double> *__restrict__ cfg, int ns,
                                                    int64_t lex0, Visit visit) {
    const int64_t stride = (int64_t)ns * ns * 36;  // numbers from one z to the next
    const cplx<double> *src = cfg + lex0 * 36 + 9;
    mat3<double> d, u, next, zero;
    m_zero(zero);
    m_identity(d);
#pragma unroll
    for (int k = 0; k < 9; k++) next.e[k] = src[k];
    for (int z = 0; z < ns; z++) {
        u = next;
        if (z + 1 < ns) {
            src += stride;
#pragma unroll
            for (int k = 0; k < 9; k++) next.e[k] = src[k];
        }
        visit(z, d);
        mat3<double> hi, lo;
        m_mul2<2>(m_dagger(u), zero, d, hi, lo);
        m_polish_su3(hi, lo, d);
    }
    return d;
}

// Column index of a thread -> its y, x, t and the site index of its z = 0.
struct Column {
    int x, y, t;
    int64_t lex0;
};

__device__ __forceinline__ Column column_of(int c, int ns) {
    Column q;
    q.x = c % ns;
    const int r = c / ns;
    q.y = r % ns;
    q.t = r / ns;
    q.lex0 = ((int64_t)q.t * ns * ns + q.y) * ns + q.x;
    return q;
}

// G = 1 in the axial frame: G' = h^dagger, and the Z links of the plane
// z = ns - 1.  One thread per column, ncol = ns^2 nt columns.
__global__ __launch_bounds__(64) void k_frame_begin(const cplx<double> *__restrict__ cfg,
                                                    cplx<double> *__restrict__ u0,
                                                    cplx<double> *__restrict__ g, int ns, int Vh,
                                                    int ncol) {
    const int c = blockIdx.x * 64 + threadIdx.x;
    if (c >= ncol) return;
    const Column q = column_of(c, ns);
    const mat3<double> w = walk_column(cfg, ns, q.lex0, [&](int z, const mat3<double> &d) {
        const int p = (q.x + q.y + z + q.t) & 1;
        store_su3<false>(d, g_field(g, Vh, p), (int)((q.lex0 + (int64_t)z * ns * ns) >> 1));
    });
    const int p = (q.x + q.y + ns - 1 + q.t) & 1;
    const int hw = (q.t * ns + q.y) * (ns >> 1) + (q.x >> 1);
    store_u0(m_dagger(w), axial_wrap(u0, Vh, ns, p), hw);
}

// End of a fix: G = G' h, projected onto SU(3) if `project` (the last
// reunitarization of G).  One thread per site; bound by its three matrices.
__global__ __launch_bounds__(kBlock) void k_frame_end(const cplx<double> *__restrict__ u0,
                                                      cplx<double> *__restrict__ g, int ns,
                                                      int Vh, bool project) {
    const int idx = blockIdx.x * kBlock + threadIdx.x;
    if (idx >= 2 * Vh) return;
    const int p = idx >= Vh, h = idx - p * Vh;
    cplx<double> *field = g_field(g, Vh, p);
    mat3<double> gp, d, zero, out, lo;
    m_zero(zero);
    load_su3<false>(gp, static_cast<const cplx<double> *>(field), h);
    load_rows01<false>(d, axial_h(u0, Vh, ns, p), h);
    m_close_row2(d);
    m_mul2<2>(gp, zero, m_dagger(d), out, lo);
#pragma unroll
    for (int k = 0; k < kPlanes; k++)
        out.e[k] = c_make<double>(out.e[k].re + lo.e[k].re, out.e[k].im + lo.e[k].im);
    if (project) m_project_su3(out);
    store_su3<false>(out, field, h);
}

// The Y and X links of cfg (AoS FP64) in the axial frame, u0_i(n) =
// h(n) u_i(n) h(n+i)^dagger with h = G'^dagger (k_frame_begin), and h^dagger for
// k_frame_end, which walked the columns a second time before (a fix of one
// half-sweep at 8^3 x 16 / 16^3 x 32 / 48^3 x 96: 114 -> 83, 226 -> 163, 7840 ->
// 7400 us).  One thread per site.
__global__ __launch_bounds__(kBlock) void k_axial_u0(const cplx<double> *__restrict__ cfg,
                                                     const cplx<double> *__restrict__ g,
                                                     cplx<double> *__restrict__ u0, int ns,
                                                     int Vh) {
    const int idx = blockIdx.x * kBlock + threadIdx.x;
    if (idx >= 2 * Vh) return;
    const int p = idx >= Vh, h = idx - p * Vh;
    const Site s = site_of(h, p, ns);
    const Nbr nb = neighbours(s, h, ns);
    const int64_t lex = (int64_t)2 * s.row + s.x;
    mat3<double> gn;
    load_su3<false>(gn, g_field(g, Vh, p), h);
    store_su3<true>(gn, axial_h(u0, Vh, ns, p), h);
#pragma unroll
    for (int i = 1; i < 3; i++) {
        const cplx<double> *src = cfg + (lex * 4 + 1 + i) * 9;
        mat3<double> u, gm, zero, a, alo, out, lo;
        m_zero(zero);
#pragma unroll
        for (int k = 0; k < 9; k++) u.e[k] = src[k];
        load_su3<false>(gm, g_field(g, Vh, 1 - p), nb.fwd[i]);
        m_mul2<2>(m_dagger(gn), zero, u, a, alo);
        m_mul2<2>(a, alo, gm, out, lo);
        m_polish_su3(out, lo, out);
        store_u0(out, axial_field(u0, Vh, p, i), h);
    }
}

// Whether a matrix is one of SU(3) to within 1e-6, some ten times what storing
// it in FP32 makes of it.  The axial frame multiplies links up a column and
// keeps the nearest SU(3) matrices; links further off are swept in the
// configuration's own frame, where each stands for itself, as its first two
// rows.  (No number is not near.)
__device__ __forceinline__ bool near_su3(const mat3<double> &u) {
    mat3<double> c = u;
    m_fill_row2(c);
    cplx<double> s = c_make<double>(0, 0);
    double d = fmax(fabs(row_norm(u.e) - 1), fabs(row_norm(u.e + 3) - 1));
    bool ok = true;
#pragma unroll
    for (int b = 0; b < 3; b++) {
        c_mac_cb(s, u.e[b], u.e[3 + b]);
        const cplx<double> r = c_make<double>(u.e[6 + b].re - c.e[6 + b].re,
                                              u.e[6 + b].im - c.e[6 + b].im);
        ok = ok && fabs(r.re) < 1e-6 && fabs(r.im) < 1e-6;
    }
    return ok && d < 1e-6 && fabs(s.re) < 1e-6 && fabs(s.im) < 1e-6;
}

// cfg (AoS FP64) spatial links -> u0 fields in FP64 and, unless u0f is null,
// FP32 in the configuration's own frame; *off, if given, is set to 1 when a
// link is not near SU(3).
__global__ __launch_bounds__(kBlock) void k_build_u0(const cplx<double> *__restrict__ cfg,
                                                     cplx<double> *__restrict__ u0,
                                                     cplx<float> *__restrict__ u0f, int ns,
                                                     int Vh, int *off) {
    const int idx = blockIdx.x * kBlock + threadIdx.x;
    if (idx >= 2 * Vh) return;
    const int p = idx >= Vh, h = idx - p * Vh;
    const Site s = site_of(h, p, ns);
    const int64_t lex = (int64_t)2 * s.row + s.x;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const cplx<double> *src = cfg + (lex * 4 + 1 + i) * 9;
        mat3<double> m;
#pragma unroll
        for (int k = 0; k < 9; k++) m.e[k] = src[k];
        if (off && !near_su3(m)) *off = 1;
        store_u0(m, u0_field(u0, Vh, p, i), h);
        if (u0f) store_u0(m, u0_field(u0f, Vh, p, i), h);
    }
}

// tile[k] = src[at(k)] for 64 P pieces of 16 bytes, n of them valid, moved
// straight to LDS, 64 pieces by a wave's load, all of them in flight together
// (through registers, a piece at a time, they arrived one after the other:
// 4.6 instead of 3.3 ms for the plaquettes of 48^3 x 96).  Pieces from n on get
// src[at(0)].  Complete on return; the tile must have been read before.  With
// ALIGNED = false src need only lie at a double's alignment, and its pieces go
// through registers.
template <int P, bool ALIGNED = true, typename At>
__device__ __forceinline__ void stage_tile(double2 *tile, const double2 *src, int n, At at) {
    typedef __attribute__((address_space(3))) void *lds_ptr;
    typedef const __attribute__((address_space(1))) void *global_ptr;
    static_assert(kBlock == 256, "four waves");
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
#pragma unroll
    for (int j = 0; j < (P + 3) / 4; j++) {
        const int c = wave + 4 * j, k = c * 64 + ((int)threadIdx.x & 63);
        if (c >= P) continue;
        const double2 *from = src + at(k < n ? k : 0);
        if constexpr (ALIGNED) {
            __builtin_amdgcn_global_load_lds((global_ptr)from, (lds_ptr)(tile + c * 64), 16, 0, 0);
        } else {
            const double *d = reinterpret_cast<const double *>(from);
            tile[k] = double2{d[0], d[1]};
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
}

// n AoS FP64 matrices from base to LDS and back, in consecutive 16-byte pieces.
__device__ __forceinline__ void stage_links(double2 *sh, const double2 *base, int n) {
    stage_tile<36>(sh, base, n * 9, [](int k) { return k; });
}
__device__ __forceinline__ void unstage_links(double2 *base, const double2 *sh, int n) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 9; j++) {
        const int k = j * kBlock + (int)threadIdx.x;
        if (k < n * 9) base[k] = sh[k];
    }
}

// cfg <- G(n) cfg G(n+mu)^dagger for all four directions
// (applyGaugeTransformationU, src/fields.c:375-435); with PROJECT every link
// is then projected onto SU(3), the reunitarization of U that ends a
// converged gaugefixOverrelaxation (src/gauge_fixing.c:822).  One thread per
// link, 64 sites (256 links, 36 KiB) per workgroup: the links are read from
// and written back to the AoS array through LDS in consecutive 16-byte
// pieces, so that every wave's loads and stores cover whole cache lines (one
// thread per site reading its 576 bytes directly left the accesses of a wave
// 576 bytes apart).  48^3 x 96: 4.7 ms so, 2.77 staged through registers, 2.49
// with the pieces straight to LDS and the two G under way before them.
template <bool PROJECT>
__global__ __launch_bounds__(kBlock) void k_materialize(cplx<double> *__restrict__ cfg,
                                                        const cplx<double> *__restrict__ g,
                                                        int ns, int nt, int Vh) {
    __shared__ double2 sh[kBlock * 9];
    const int64_t link0 = (int64_t)blockIdx.x * kBlock;
    const int nl = (int)min<int64_t>(kBlock, 8 * (int64_t)Vh - link0);  // links here
    double2 *base = reinterpret_cast<double2 *>(cfg) + link0 * 9;
    const bool on = (int)threadIdx.x < nl;
    mat3<double> gn, gm;
    if (on) {
        const int64_t link = link0 + threadIdx.x;
        const int64_t lex = link >> 2;
        const int mu = (int)(link & 3);
        const int x = (int)(lex % ns);
        int64_t r = lex / ns;
        const int y = (int)(r % ns);
        r /= ns;
        const int z = (int)(r % ns);
        const int t = (int)(r / ns);
        const int p = (x + y + z + t) & 1;
        int c[4] = {t, z, y, x};
        c[mu] += 1;
        if (c[mu] == (mu == 0 ? nt : ns)) c[mu] = 0;
        const int64_t ln = (((int64_t)c[0] * ns + c[1]) * ns + c[2]) * ns + c[3];
        load_su3<false>(gn, g_field(g, Vh, p), (int)(lex >> 1));
        load_su3<false>(gm, g_field(g, Vh, 1 - p), (int)(ln >> 1));
    }
    stage_links(sh, base, nl);
    if (on) {
        mat3<double> u, tmp, out;
        double2 *mine = sh + threadIdx.x * 9;
#pragma unroll
        for (int k = 0; k < 9; k++) u.e[k] = c_make<double>(mine[k].x, mine[k].y);
        m_mul(gn, u, tmp);
        m_mul_nd(tmp, gm, out);
        if (PROJECT) m_project_su3(out);
#pragma unroll
        for (int k = 0; k < 9; k++) mine[k] = double2{out.e[k].re, out.e[k].im};
    }
    unstage_links(base, sh, nl);
}

// Projects n AoS FP64 matrices onto SU(3); sets *flag when a row was null
// (reunitarizeField's -1).  One thread per matrix, staged as in k_materialize:
// bound by reading and writing the array (48^3 x 96, 12.2 GB: 2.46 -> 2.34 ms,
// 16^3 x 32 55 -> 45 us with the call, against nine 16-byte accesses of a thread
// 144 bytes from its neighbours').
__global__ __launch_bounds__(kBlock) void k_reunit_aos(cplx<double> *__restrict__ m_,
                                                       int64_t n, int *flag) {
    __shared__ double2 sh[kBlock * 9];
    const int64_t link0 = (int64_t)blockIdx.x * kBlock;
    const int nl = (int)min<int64_t>(kBlock, n - link0);  // matrices here
    double2 *base = reinterpret_cast<double2 *>(m_) + link0 * 9;
    stage_links(sh, base, nl);
    if ((int)threadIdx.x < nl) {
        double2 *mine = sh + threadIdx.x * 9;
        mat3<double> m;
#pragma unroll
        for (int k = 0; k < 9; k++) m.e[k] = c_make<double>(mine[k].x, mine[k].y);
        if (!m_project_su3(m)) atomicOr(flag, 1);
#pragma unroll
        for (int k = 0; k < 9; k++) mine[k] = double2{m.e[k].re, m.e[k].im};
    }
    unstage_links(base, sh, nl);
}

__global__ __launch_bounds__(kBlock) void k_f32_to_f64(const float *__restrict__ in,
                                                       double *__restrict__ out, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) out[i] = (double)in[i];
}

// SoA G (FP64) -> AoS image (site-major, full 3x3).
__global__ __launch_bounds__(kBlock) void k_g_to_aos(const cplx<double> *__restrict__ g,
                                                     cplx<double> *__restrict__ out, int ns,
                                                     int Vh) {
    const int64_t lex = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (lex >= 2 * (int64_t)Vh) return;
    const int x = (int)(lex % ns);
    int64_t r = lex / ns;
    const int y = (int)(r % ns);
    r /= ns;
    const int z = (int)(r % ns);
    const int t = (int)(r / ns);
    const int p = (x + y + z + t) & 1;
    mat3<double> m;
    load_su3<false>(m, g_field(g, Vh, p), (int)(lex >> 1));
#pragma unroll
    for (int k = 0; k < 9; k++) out[lex * 9 + k] = m.e[k];
}

// ---------------------------------------------------------------------------
// Observables.  Per site: D = sum_i [(U_i(n) - U_i(n)^dag) - (U_i(n-i) - U_i(n-i)^dag)]
// made traceless, div A = -(i/2) D (divergenceA/calculateA,
// src/four_potential.c:35-113); e2 density = sum_a c_a^2 with the Gell-Mann
// components of decomposeAlgebraSU3 (src/SU3_ops.c:1055-1107); theta density
// = Re Tr(divA divA^dag) (calculateTheta, src/gauge_fixing.c:341-384); and
// Re Tr sum_i U_i(n) for F (calculateF, :289-337).  All arithmetic in FP64.

struct Obs {
    double e2, theta, f;
};

__device__ __forceinline__ void accum_link(mat3<double> &D, const mat3<double> &u, double sgn) {
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++) {
            const cplx<double> uab = u.e[3 * a + b], uba = u.e[3 * b + a];
            D.e[3 * a + b].re += sgn * (uab.re - uba.re);
            D.e[3 * a + b].im += sgn * (uab.im + uba.im);
        }
}

__device__ __forceinline__ Obs site_obs(mat3<double> &D, double f) {
    const double tr = (D.e[0].im + D.e[4].im + D.e[8].im) / 3.0;
    D.e[0].im -= tr;
    D.e[4].im -= tr;
    D.e[8].im -= tr;
    // A = -(i/2) D : A.re = D.im / 2, A.im = -D.re / 2
    mat3<double> A;
#pragma unroll
    for (int k = 0; k < 9; k++) A.e[k] = c_make<double>(0.5 * D.e[k].im, -0.5 * D.e[k].re);
    double c[8];
    c[0] = A.e[1].re + A.e[3].re;
    c[1] = -A.e[1].im + A.e[3].im;
    c[2] = A.e[0].re - A.e[4].re;
    c[3] = A.e[2].re + A.e[6].re;
    c[4] = -A.e[2].im + A.e[6].im;
    c[5] = A.e[5].re + A.e[7].re;
    c[6] = -A.e[5].im + A.e[7].im;
    c[7] = (A.e[0].re + A.e[4].re - 2.0 * A.e[8].re) * 0.57735026918962573;
    Obs o;
    o.e2 = 0;
#pragma unroll
    for (int a = 0; a < 8; a++) o.e2 += c[a] * c[a];
    o.theta = 0;
#pragma unroll
    for (int k = 0; k < 9; k++) o.theta += A.e[k].re * A.e[k].re + A.e[k].im * A.e[k].im;
    o.f = f;
    return o;
}

template <typename T>
__device__ __forceinline__ void load_su3_d(mat3<double> &m, const cplx<T> *__restrict__ field,
                                           int h) {
    const uint32_t off = tile_bytes<T>(h);
#pragma unroll
    for (int k = 0; k < kPlanes; k++) {
        const cplx<T> v = *elem_ptr(field, off, k);
        m.e[k] = c_make<double>((double)v.re, (double)v.im);
    }
    m_fill_row2(m);
}

// Deterministic block reduction of three doubles; writes part[3*block + j].
__device__ __forceinline__ void block_reduce3(Obs o, double *__restrict__ part, unsigned blk) {
    __shared__ double sh[3][kBlock / 64];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        o.e2 += __shfl_xor(o.e2, off, 64);
        o.theta += __shfl_xor(o.theta, off, 64);
        o.f += __shfl_xor(o.f, off, 64);
    }
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) {
        sh[0][wv] = o.e2;
        sh[1][wv] = o.theta;
        sh[2][wv] = o.f;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        double s = 0;
#pragma unroll
        for (int w = 0; w < kBlock / 64; w++) s += sh[threadIdx.x][w];
        part[3 * blk + threadIdx.x] = s;
    }
}

// Observables of the factored state at site index idx in [0, 2 Vh) (parity
// idx >= Vh); u0 in FP64 (in the axial frame with an FP64 G unless OWN, in the
// configuration's own with an FP32 one), arithmetic in FP64.  They come
// from the site's w = G(n) W(n), formed as the sweep forms it:
// w = sum_i [U_i(n) + U_i(n-i)^dagger], so w - w^dagger is the divergence
// sum_i [(U - U^dagger)_i(n) - (U - U^dagger)_i(n-i)] that e2 and theta
// measure (calculateA, divergenceA: src/four_potential.c), and
// Re Tr w / 2 summed over all sites is the sum over links of Re Tr U that F
// measures (calculateF, src/gauge_fixing.c).  Seven products (five in the axial
// frame) instead of the twelve of forming every link.
template <typename TG, bool OWN = false>
__device__ __forceinline__ Obs obs_site(const cplx<double> *__restrict__ u0,
                                        const cplx<TG> *__restrict__ g, int ns, int Vh,
                                        int idx) {
    Obs o = {0, 0, 0};
    if (idx < 2 * Vh) {
        const int p = idx >= Vh, h = idx - p * Vh;
        const Site s = site_of(h, p, ns);
        const Nbr nb = neighbours(s, h, ns);
        const cplx<TG> *gq = g_field(g, Vh, 1 - p);
        mat3<double> W;
        m_zero(W);
        constexpr bool axial = sizeof(TG) == sizeof(double) && !OWN;
        if constexpr (axial) {
            mat3<double> gf, gb;
            load_su3_d(gf, gq, nb.fwd[0]);
            load_su3_d(gb, gq, nb.bwd[0]);
            axial_z<false>(W, u0, s, ns, Vh, p, gf, gb);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = axial ? 1 : 0; i < 3; i++) {
            mat3<double> uf, gf, ub, gb;
            load_u0_d(uf, axial ? axial_field(u0, Vh, p, i) : u0_field(u0, Vh, p, i), h);
            load_su3_d(gf, gq, nb.fwd[i]);
            load_u0_d(ub, axial ? axial_field(u0, Vh, 1 - p, i) : u0_field(u0, Vh, 1 - p, i),
                      nb.bwd[i]);
            load_su3_d(gb, gq, nb.bwd[i]);
            m_mac_nd_su3(W, uf, gf);      // u0_i(n) G(n+i)^dagger
            m_mac_dagger_su3(W, gb, ub);  // (G(n-i) u0_i(n-i))^dagger
            // one direction's loads at a time (hoisting all of them took 2
            // waves/SIMD)
            __builtin_amdgcn_sched_barrier(0);
        }
        mat3<double> gn, w, D;
        load_su3_d(gn, g_field(g, Vh, p), h);
        m_mul(gn, W, w);
        m_zero(D);
        accum_link(D, w, 1.0);
        o = site_obs(D, 0.5 * (w.e[0].re + w.e[4].re + w.e[8].re));
    }
    return o;
}

// The b-th block of n to be worked on, in the order of the site index: the
// first and the second half of the blocks, i.e. the two parities of the same
// sites, in turn.  A link is read as a site's forward link by one parity and as
// a backward link by the other; in index order the second read came when the
// first was long out of the caches (us at 48^3 x 96 with an FP32 / FP64 G: 1020
// / 1240 -> 717 / 867).
__host__ __device__ inline unsigned parity_order(unsigned b, unsigned n) {
    return (b & 1) ? (n + 1) / 2 + b / 2 : b / 2;
}

// One thread per site, both parities; per-block partial sums in part, in
// site order.  The workgroups run in XCD-contiguous order (xcd_order), so that
// the neighbour G and backward u0 links a site reads were mostly brought into
// its XCD's L2 by the sites next to it.
template <typename TG, bool OWN = false>
__global__ __launch_bounds__(kBlock, 3) void k_obs_factored(const cplx<double> *__restrict__ u0,
                                                            const cplx<TG> *__restrict__ g,
                                                            int ns, int Vh,
                                                            double *__restrict__ part) {
    const unsigned b = parity_order(xcd_order(blockIdx.x, gridDim.x), gridDim.x);
    const int idx = (int)(b * kBlock + threadIdx.x);
    block_reduce3(obs_site<TG, OWN>(u0, g, ns, Vh, idx), part, b);
}

// The sums of each timeslice t (one workgroup), out[3 t + j]: partials
// t bps + [0, bps) of either parity, which begin at 0 and half.
__global__ __launch_bounds__(kBlock) void k_slice_sums(const double *__restrict__ part, int half,
                                                       int bps, double *__restrict__ out) {
    Obs o = {0, 0, 0};
    for (int k = threadIdx.x; k < 2 * bps; k += kBlock) {
        const double *v = part + 3 * ((k < bps ? k : half + k - bps) + (int64_t)blockIdx.x * bps);
        o.e2 += v[0];
        o.theta += v[1];
        o.f += v[2];
    }
    block_reduce3(o, out, blockIdx.x);
}

// The kernels over an AoS configuration.  A thread reading the 144 bytes of a
// matrix by itself leaves the lanes of a load 144 to 576 bytes apart, a cache
// line each, and the kernel waits for the address units; so the links of 64
// sites are brought into LDS in consecutive 16-byte pieces, and four threads
// work on a site, one per direction.  48^3 x 96: residues 2.15 -> 1.19 ms,
// plaquettes 4.86 -> 3.3 ms (the configuration's 6.1 GB take 0.98 ms at 6.25
// TB/s; the plaquettes read 16 links per site, the T neighbours' and part of
// the Z neighbours' from beyond the L2).
constexpr int kAosSites = 64;

// Matrix of nine pieces in LDS.
__device__ __forceinline__ void lds_mat(mat3<double> &m, const double2 *__restrict__ s) {
#pragma unroll
    for (int k = 0; k < 9; k++) m.e[k] = c_make<double>(s[k].x, s[k].y);
}

// The value of the lane whose number differs in the bits X (1 to 3).
template <int X>
__device__ __forceinline__ double quad_xor(double v) {
    constexpr int ctrl = X == 1 ? 0xB1 : X == 2 ? 0x4E : 0x1B;  // quad_perm
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, ctrl, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), ctrl, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) |
                                            (unsigned)lo));
}

// Groups of kAosSites sites a workgroup takes: four, so that its partial sums
// are those of kBlock sites, or for a small lattice, whose workgroups do not
// fill the GPU, one.
inline int aos_groups(int64_t V) { return V <= 1024 * kBlock ? 1 : kBlock / kAosSites; }
inline unsigned aos_blocks(int64_t V) {
    const int64_t sites = (int64_t)aos_groups(V) * kAosSites;
    return (unsigned)((V + sites - 1) / sites);
}

// First site of the q-th of workgroup b's groups: runs of 64 workgroups (one
// XCD's, xcd_order) go through their groups side by side, 4096 consecutive
// sites at a time, so that a site's Y and Z neighbours are read by the same XCD
// at about the same time.
__device__ __forceinline__ int aos_group(unsigned b, unsigned nb, int q, int groups) {
    const unsigned run = b / 64, m = min(64u, nb - run * 64);
    return (int)(run * 64 * (unsigned)groups + (unsigned)q * m + b % 64) * kAosSites;
}

// lex index of the site one step from lex in direction mu, forward or backward.
__device__ __forceinline__ int aos_neighbour(int lex, int mu, bool fwd, int ns, int nt) {
    int c[4];  // t, z, y, x
    c[3] = lex % ns;
    int r = lex / ns;
    c[2] = r % ns;
    r /= ns;
    c[1] = r % ns;
    c[0] = r / ns;
#pragma unroll
    for (int k = 0; k < 4; k++)
        if (k == mu) {
            const int n = k == 0 ? nt : ns;
            c[k] = fwd ? (c[k] + 1 == n ? 0 : c[k] + 1) : (c[k] == 0 ? n - 1 : c[k] - 1);
        }
    return ((c[0] * ns + c[1]) * ns + c[2]) * ns + c[3];
}

// Observables of an AoS FP64 configuration.  Thread i (1 to 3) of a site adds
// its direction's U_i(n) - U_i(n-i); thread 0 takes the sum.  With CHECK, *off
// is set to 1 when a spatial link is not near SU(3).
template <bool CHECK = false, bool ALIGNED = true>
__global__ __launch_bounds__(kBlock) void k_obs_aos(const cplx<double> *__restrict__ cfg, int ns,
                                                    int64_t V, int groups,
                                                    double *__restrict__ part, int *off) {
    __shared__ double2 tile[kAosSites * 27];
    __shared__ int nbr[kAosSites * 3];
    const double2 *src = reinterpret_cast<const double2 *>(cfg);
    const unsigned b = xcd_order(blockIdx.x, gridDim.x);
    const int site = threadIdx.x >> 2, i = threadIdx.x & 3, n = (int)V;
    Obs o = {0, 0, 0};
#pragma unroll 1
    for (int q = 0; q < groups; q++) {
        const int lex0 = aos_group(b, gridDim.x, q, groups), count = min(kAosSites, n - lex0);
        if (count <= 0) break;
        const bool on = i > 0 && site < count;
        const double2 *mine = tile + site * 27 + (i - 1) * 9;
        mat3<double> u, v;
        if (on) nbr[site * 3 + i - 1] = aos_neighbour(lex0 + site, i, false, ns, 1 << 30);
        stage_tile<27, ALIGNED>(tile, src, count * 27,
                                [&](int k) { return (int64_t)lex0 * 36 + 9 + k + k / 27 * 9; });
        if (on) {
            lds_mat(u, mine);
            if (CHECK && !near_su3(u)) *off = 1;
        }
        __syncthreads();
        stage_tile<27, ALIGNED>(tile, src, count * 27,
                                [&](int k) { return (int64_t)nbr[k / 9] * 36 + 9 + k % 27; });
        // D = sum_i (E_i - E_i^dagger), E_i = U_i(n) - U_i(n-i): the imaginary
        // parts of its diagonal, D01, D02, D12, and Re Tr U
        double d[10];
#pragma unroll
        for (int k = 0; k < 10; k++) d[k] = 0;
        if (on) {
            lds_mat(v, mine);
            d[9] = u.e[0].re + u.e[4].re + u.e[8].re;
#pragma unroll
            for (int k = 0; k < 9; k++)
                u.e[k] = c_make<double>(u.e[k].re - v.e[k].re, u.e[k].im - v.e[k].im);
            d[0] = 2 * u.e[0].im;
            d[1] = 2 * u.e[4].im;
            d[2] = 2 * u.e[8].im;
            d[3] = u.e[1].re - u.e[3].re;
            d[4] = u.e[1].im + u.e[3].im;
            d[5] = u.e[2].re - u.e[6].re;
            d[6] = u.e[2].im + u.e[6].im;
            d[7] = u.e[5].re - u.e[7].re;
            d[8] = u.e[5].im + u.e[7].im;
        }
#pragma unroll
        for (int k = 0; k < 10; k++) d[k] += quad_xor<1>(d[k]);
#pragma unroll
        for (int k = 0; k < 10; k++) d[k] += quad_xor<2>(d[k]);
        if (i == 0 && site < count) {
            mat3<double> D;
            D.e[0] = c_make<double>(0, d[0]);
            D.e[4] = c_make<double>(0, d[1]);
            D.e[8] = c_make<double>(0, d[2]);
            D.e[1] = c_make<double>(d[3], d[4]);
            D.e[3] = c_make<double>(-d[3], d[4]);
            D.e[2] = c_make<double>(d[5], d[6]);
            D.e[6] = c_make<double>(-d[5], d[6]);
            D.e[5] = c_make<double>(d[7], d[8]);
            D.e[7] = c_make<double>(-d[7], d[8]);
            const Obs s = site_obs(D, d[9]);
            o.e2 += s.e2;
            o.theta += s.theta;
            o.f += s.f;
        }
        __syncthreads();
    }
    block_reduce3(o, part, b);
}

// Re Tr of the plaquette in the plane of directions r (this thread) and
// d = r ^ X (the thread X lanes over): a = U_d(n) U_r(n+d) here and
// U_r(n) U_d(n+r) there, Re Tr(a_here a_there^dagger).
template <int X>
__device__ __forceinline__ double plaquette_trace(const mat3<double> &a) {
    double tr = 0;
#pragma unroll
    for (int k = 0; k < 9; k++) {
        tr = __builtin_fma(a.e[k].re, quad_xor<X>(a.e[k].re), tr);
        tr = __builtin_fma(a.e[k].im, quad_xor<X>(a.e[k].im), tr);
    }
    return tr;
}

// Plaquettes of an AoS FP64 configuration (TrPlaquette, src/measurement.c:38-84):
// Re Tr[U_mu(n) U_nu(n+mu) U_mu(n+nu)^dag U_nu(n)^dag] / 3, spatial planes
// (XY, XZ, YZ) into slot 0 and temporal planes (TZ, TY, TX) into slot 1.
// Thread r of a site meets each other direction d = r ^ X once, X = 1, 2, 3;
// both threads of a plane find its trace, and each counts half.
template <bool ALIGNED = true>
__global__ __launch_bounds__(kBlock) void k_plaquette_aos(const cplx<double> *__restrict__ cfg,
                                                          int ns, int nt, int64_t V, int groups,
                                                          double *__restrict__ part) {
    __shared__ double2 tile[kAosSites * 36];
    __shared__ int nbr[kAosSites * 4];
    const double2 *src = reinterpret_cast<const double2 *>(cfg);
    const unsigned b = xcd_order(blockIdx.x, gridDim.x);
    const int site = threadIdx.x >> 2, r = threadIdx.x & 3, n = (int)V;
    Obs o = {0, 0, 0};
#pragma unroll 1
    for (int q = 0; q < groups; q++) {
        const int lex0 = aos_group(b, gridDim.x, q, groups), count = min(kAosSites, n - lex0);
        if (count <= 0) break;
        if (site < count) nbr[threadIdx.x] = aos_neighbour(lex0 + site, r, true, ns, nt);
        stage_tile<36, ALIGNED>(tile, src, count * 36,
                                [&](int k) { return (int64_t)lex0 * 36 + k; });
        mat3<double> own;  // U_r(n)
        m_zero(own);
        if (site < count) lds_mat(own, tile + threadIdx.x * 9);
#pragma unroll
        for (int X = 1; X < 4; X++) {
            __syncthreads();  // the tile has been read
            stage_tile<36, ALIGNED>(tile, src, count * 36,
                                    [&](int k) { return (int64_t)nbr[(k / 9) ^ X] * 36 + k % 36; });
            mat3<double> u, v, a;
#pragma unroll
            for (int k = 0; k < 9; k++)
                u.e[k] = X == 1   ? c_make<double>(quad_xor<1>(own.e[k].re), quad_xor<1>(own.e[k].im))
                         : X == 2 ? c_make<double>(quad_xor<2>(own.e[k].re), quad_xor<2>(own.e[k].im))
                                  : c_make<double>(quad_xor<3>(own.e[k].re), quad_xor<3>(own.e[k].im));
            m_zero(v);
            if (site < count) lds_mat(v, tile + threadIdx.x * 9);
            m_mul(u, v, a);
            double tr = (X == 1   ? plaquette_trace<1>(a)
                         : X == 2 ? plaquette_trace<2>(a)
                                  : plaquette_trace<3>(a)) / 6.0;
            // formed here: the compiler would keep the three products for later
            asm volatile("" : "+v"(tr));
            if (r == 0 || (r ^ X) == 0)
                o.theta += tr;
            else
                o.e2 += tr;
        }
        __syncthreads();
    }
    block_reduce3(o, part, b);
}

// Streaming copy of n 16-byte elements (bandwidth probe / counter calibration).
__global__ __launch_bounds__(kBlock) void k_copy16(const double2 *__restrict__ in,
                                                   double2 *__restrict__ out, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) out[i] = in[i];
}

// Read-rate probe: `passes` reads of gridDim.x contiguous chunks of `chunk`
// 16-byte elements, eight loads in flight per lane.  In pass p workgroup b
// reads chunk (b + p) mod gridDim.x, so no workgroup reads the same bytes twice
// in a row and the next reader of a chunk runs on another XCD: every pass
// streams the buffer from where it resides (the Infinity Cache up to 256 MiB,
// HBM above), not from an L2.  The sum is stored only if it takes a value a
// zeroed buffer cannot give.
__global__ __launch_bounds__(kBlock) void k_read16(const double2 *__restrict__ in, int64_t chunk,
                                                   int passes, double2 *__restrict__ sink) {
    constexpr int kInFlight = 8;
    double2 acc = {0.0, 0.0};
    for (int p = 0; p < passes; p++) {
        asm volatile("" ::: "memory");  // every pass loads again
        const double2 *c = in + (int64_t)((blockIdx.x + (unsigned)p) % gridDim.x) * chunk;
        int64_t j = threadIdx.x;
        for (; j + (kInFlight - 1) * kBlock < chunk; j += kInFlight * kBlock) {
            double2 v[kInFlight];
#pragma unroll
            for (int u = 0; u < kInFlight; u++) v[u] = c[j + u * kBlock];
#pragma unroll
            for (int u = 0; u < kInFlight; u++) acc += v[u];
        }
        for (; j < chunk; j += kBlock) acc += c[j];
    }
    if (acc.x == 1.2345e-300) sink[(int64_t)blockIdx.x * kBlock + threadIdx.x] = acc;
}

// Sums part[3*b + j] over b in fixed order with one block; out[j].  A thread
// adds every 256th partial one after the other; eight are loaded at a time, as
// one load in flight per thread made this latency alone (48^3 x 96, 41472
// partials: 72 -> 21 us).
__device__ __forceinline__ void reduce_parts(const double *__restrict__ part, int nblocks,
                                             double *__restrict__ out) {
    constexpr int kLoads = 8;
    Obs o = {0, 0, 0};
    int b = threadIdx.x;
    for (; b + (kLoads - 1) * kBlock < nblocks; b += kLoads * kBlock) {
        double v[kLoads][3];
#pragma unroll
        for (int k = 0; k < kLoads; k++)
#pragma unroll
            for (int j = 0; j < 3; j++) v[k][j] = part[3 * (b + k * kBlock) + j];
#pragma unroll
        for (int k = 0; k < kLoads; k++) {
            o.e2 += v[k][0];
            o.theta += v[k][1];
            o.f += v[k][2];
        }
    }
    for (; b < nblocks; b += kBlock) {
        o.e2 += part[3 * b];
        o.theta += part[3 * b + 1];
        o.f += part[3 * b + 2];
    }
    block_reduce3(o, out, 0);
}

__global__ __launch_bounds__(kBlock) void k_reduce_final(const double *__restrict__ part,
                                                         int nblocks, double *__restrict__ out) {
    reduce_parts(part, nblocks, out);
}

// ---------------------------------------------------------------------------
// Batched kernels for the serving scheduler: many lattices per launch.  A
// work item is one 256-site chunk of one lattice; the per-site code is the
// same device function as in the single-lattice kernels, and reductions use
// the same block decomposition and order, so every lattice gets the same
// bits alone or packed with others.

struct BatchJob {
    const void *u0;   // cplx<T> planes of the lattice's u0 (T = sweep launch type)
    void *g;          // cplx<T> planes of its G (T = sweep launch type)
    const void *u0d;  // FP64 u0 (observables always read FP64 links)
    const void *gd;   // FP64 G, for FP64-state observables
    const void *gf;   // FP32 G (MIXED only, else null), for FP32-state observables
    double omega;
    Extents x;
    int hits;
    int part_off;     // first partial-sum slot of this lattice (observables)
};

// One workgroup per item = (job index, first parity index, parity, unused).
// (Looping a workgroup over several items measured 17% slower.)  STREAM and OWN
// as in sweep_site.
template <typename T, bool STREAM = true, bool OWN = false>
__global__ __launch_bounds__(kBlock) void k_sweep_batch(const BatchJob *__restrict__ jobs,
                                                        const int4 *__restrict__ items,
                                                        int nitems) {
    const int i = (int)(STREAM ? blockIdx.x : xcd_order(blockIdx.x, gridDim.x));
    if (i >= nitems) return;
    const int4 it = items[i];
    const BatchJob J = jobs[it.x];
    const int lane = (int)threadIdx.x;
    if (it.y + lane < J.x.Vh)
        sweep_site<T, false, STREAM, false, OWN>(static_cast<const cplx<T> *>(J.u0),
                                                 static_cast<cplx<T> *>(J.g), J.x, it.z,
                                                 (T)J.omega, J.hits, it.y, lane);
}

// item = (job index, block index within the lattice's [0, 2 Vh) range, fp32 G?, _)
__global__ __launch_bounds__(kBlock) void k_obs_batch(const BatchJob *__restrict__ jobs,
                                                      const int4 *__restrict__ items,
                                                      double *__restrict__ part) {
    const int4 it = items[xcd_order(blockIdx.x, gridDim.x)];
    const BatchJob J = jobs[it.x];
    const int idx = it.y * kBlock + (int)threadIdx.x;
    const cplx<double> *u0 = static_cast<const cplx<double> *>(J.u0d);
    Obs o = it.z ? obs_site<float>(u0, static_cast<const cplx<float> *>(J.gf), J.x.ns,
                                           J.x.Vh, idx)
                 : obs_site<double>(u0, static_cast<const cplx<double> *>(J.gd), J.x.ns,
                                            J.x.Vh, idx);
    block_reduce3(o, part + 3 * (int64_t)J.part_off, it.y);
}

// One block per evaluated lattice: jobs[sel[k]] partials -> out[3k + j].
__global__ __launch_bounds__(kBlock) void k_reduce_batch(const BatchJob *__restrict__ jobs,
                                                         const int *__restrict__ sel,
                                                         const double *__restrict__ part,
                                                         double *__restrict__ out) {
    const BatchJob J = jobs[sel[blockIdx.x]];
    const int nb = (2 * J.x.Vh + kBlock - 1) / kBlock;
    reduce_parts(part + 3 * (int64_t)J.part_off, nb, out + 3 * blockIdx.x);
}

// ---------------------------------------------------------------------------
// Device-side synthetic configuration: the same construction as the host
// generator (host_gen.c: splitmix64 draws, Box-Muller normals, Gram-Schmidt
// Haar SU(3), exp(i eps H) by scaling and squaring of a 16-term Taylor
// polynomial, U_mu(n) = g(n) exp(i eps H_mu(n)) g(n+mu)^dagger).  The device
// libm and FMA contraction make it agree with the host one to rounding, not
// bit for bit; the serving scheduler uses it to synthesise request inputs.

__device__ __forceinline__ uint64_t gen_mix64(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

__device__ __forceinline__ void gen_normals(uint64_t base, uint64_t site, unsigned k,
                                            double &a, double &b) {
    const uint64_t gold = 0x9E3779B97F4A7C15ULL;
    const uint64_t z1 = gen_mix64(base + (site * 64 + k + 1) * gold);
    const uint64_t z2 = gen_mix64(base + (site * 64 + k + 2) * gold);
    const double u1 = (double)((z1 >> 11) + 1) * 0x1.0p-53;
    const double u2 = (double)((z2 >> 11) + 1) * 0x1.0p-53;
    const double r = sqrt(-2.0 * log(u1));
    double sn, cs;
    sincos(6.283185307179586 * u2, &sn, &cs);
    a = r * cs;
    b = r * sn;
}

__device__ void gen_haar(uint64_t base, uint64_t site, mat3<double> &g) {
    double v[18];
#pragma unroll
    for (unsigned k = 0; k < 18; k += 2) gen_normals(base, site, k, v[k], v[k + 1]);
#pragma unroll
    for (int k = 0; k < 9; k++) g.e[k] = c_make<double>(v[2 * k], v[2 * k + 1]);
#pragma unroll
    for (int i = 0; i < 3; i++) {
#pragma unroll
        for (int q = 0; q < i; q++) {
            cplx<double> ip = c_make<double>(0, 0);
#pragma unroll
            for (int j = 0; j < 3; j++) c_mac_cb(ip, g.e[3 * i + j], g.e[3 * q + j]);
            // ip = <r_q, r_i> = sum conj(r_q) r_i
#pragma unroll
            for (int j = 0; j < 3; j++) {
                const cplx<double> rq = g.e[3 * q + j];
                g.e[3 * i + j].re -= ip.re * rq.re - ip.im * rq.im;
                g.e[3 * i + j].im -= ip.re * rq.im + ip.im * rq.re;
            }
        }
        double n = 0;
#pragma unroll
        for (int j = 0; j < 3; j++) n += g.e[3 * i + j].re * g.e[3 * i + j].re +
                                         g.e[3 * i + j].im * g.e[3 * i + j].im;
        n = 1.0 / sqrt(n);
#pragma unroll
        for (int j = 0; j < 3; j++) g.e[3 * i + j] = c_make(g.e[3 * i + j].re * n, g.e[3 * i + j].im * n);
    }
    const cplx<double> d = m_det(g);
    double sn, cs;
    sincos(-atan2(d.im, d.re) / 3.0, &sn, &cs);
#pragma unroll
    for (int k = 0; k < 9; k++)
        g.e[k] = c_make(g.e[k].re * cs - g.e[k].im * sn, g.e[k].re * sn + g.e[k].im * cs);
}

__device__ void gen_expi(uint64_t base, uint64_t site, int mu, double eps, mat3<double> &E) {
    double d[10];
    const unsigned k0 = 18 + 10 * (unsigned)mu;
#pragma unroll
    for (unsigned k = 0; k < 10; k += 2) gen_normals(base, site, k0 + k, d[k], d[k + 1]);
    const double s2 = 0.7071067811865476;
    const double mean = (d[0] + d[1] + d[2]) / 3.0;
    mat3<double> H;
    H.e[0] = c_make(d[0] - mean, 0.0);
    H.e[4] = c_make(d[1] - mean, 0.0);
    H.e[8] = c_make(d[2] - mean, 0.0);
    H.e[1] = c_make(d[3] * s2, d[4] * s2);
    H.e[2] = c_make(d[5] * s2, d[6] * s2);
    H.e[5] = c_make(d[7] * s2, d[8] * s2);
    H.e[3] = c_make(H.e[1].re, -H.e[1].im);
    H.e[6] = c_make(H.e[2].re, -H.e[2].im);
    H.e[7] = c_make(H.e[5].re, -H.e[5].im);
    double nrm = 0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        double rs = 0;
#pragma unroll
        for (int j = 0; j < 3; j++) rs += hypot(H.e[3 * i + j].re, H.e[3 * i + j].im);
        nrm = rs > nrm ? rs : nrm;
    }
    nrm *= fabs(eps);
    int sq = 0;
    while (nrm > 0.5 && sq < 64) {
        nrm *= 0.5;
        sq++;
    }
    const double scale = ldexp(eps, -sq);
    mat3<double> A, T;
    // A = i scale H
#pragma unroll
    for (int k = 0; k < 9; k++) A.e[k] = c_make(-scale * H.e[k].im, scale * H.e[k].re);
    m_identity(E);
    for (int n = 16; n >= 1; n--) {
        m_mul(A, E, T);
#pragma unroll
        for (int k = 0; k < 9; k++)
            E.e[k] = c_make(T.e[k].re / n + ((k % 4 == 0) ? 1.0 : 0.0), T.e[k].im / n);
    }
    for (int s = 0; s < sq; s++) {
        m_mul(E, E, T);
        E = T;
    }
    m_project_su3(E);
}

// g(n) for every site into tmp (AoS, 9 complex per site).
__global__ __launch_bounds__(kBlock) void k_gen_haar(uint64_t base, int64_t V,
                                                     cplx<double> *__restrict__ tmp) {
    const int64_t s = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (s >= V) return;
    mat3<double> g;
    gen_haar(base, (uint64_t)s, g);
#pragma unroll
    for (int k = 0; k < 9; k++) tmp[s * 9 + k] = g.e[k];
}

__global__ __launch_bounds__(kBlock) void k_gen_links(uint64_t base, double eps, int ns, int nt,
                                                      const cplx<double> *__restrict__ tmp,
                                                      cplx<double> *__restrict__ cfg) {
    const int64_t s = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const int64_t V = (int64_t)ns * ns * ns * nt;
    if (s >= V) return;
    const int x = (int)(s % ns), y = (int)((s / ns) % ns), z = (int)((s / ns / ns) % ns);
    const int t = (int)(s / ((int64_t)ns * ns * ns));
    mat3<double> gs;
#pragma unroll
    for (int k = 0; k < 9; k++) gs.e[k] = tmp[s * 9 + k];
    for (int mu = 0; mu < 4; mu++) {
        int c[4] = {t, z, y, x};
        c[mu] += 1;
        if (c[mu] == (mu == 0 ? nt : ns)) c[mu] = 0;
        const int64_t sn = (((int64_t)c[0] * ns + c[1]) * ns + c[2]) * ns + c[3];
        mat3<double> X, T1, gn, out;
        gen_expi(base, (uint64_t)s, mu, eps, X);
#pragma unroll
        for (int k = 0; k < 9; k++) gn.e[k] = tmp[sn * 9 + k];
        m_mul(gs, X, T1);
        m_mul_nd(T1, gn, out);
#pragma unroll
        for (int k = 0; k < 9; k++) cfg[(s * 4 + mu) * 9 + k] = out.e[k];
    }
}

}  // namespace
}  // namespace gfc
