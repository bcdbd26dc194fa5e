// Forward trace and backward re-trace kernels.
//
// Four ways to the sixteen nearest hits of a ray, which all give the same hits bit for bit:
//   bundle walk (bundle.inc)  images: a wave carries an 8x8 tile of rays; its lanes take boxes, then quads, against
//                             the planes around the whole tile, and what survives is tested exactly, a ray per lane
//   row walk (row.inc)        ray lists, small images, reflections: sixteen lanes per ray
//   per-lane walk             tiles handed over by the bundle walk, and rays that go apart in the kernels that carry
//                             the hand-over or trace without a record: a ray per lane, each on its own
//   packet walk               the backward trace without a hit record: a wave goes down with all its rays at once
// Tiles keep the buffer of a ray in a lane's registers, rows across sixteen lanes; compositing follows chunk by chunk.
// Replaces the raygen / any-hit programs of the reference (optix_tracer/forward.cu, optix_tracer/backward.cu).
//
// Arithmetic that feeds a decision (hit test, hit order, uv, alpha, transmittance, reflection)
// is plain fp32 evaluated as written: this file is compiled with -ffp-contract=off, rsqrt is
// 1/sqrt with IEEE division and square root, and exp is the fixed polynomial below.  Only the
// gradient algebra, which feeds no decision, allows fused multiply-adds.
#include "dst_internal.h"

#include <algorithm>

namespace {

constexpr int kChunk = 16;
constexpr float kInfDepth = 1e16f;
constexpr double kStepEps = 0.00001;
constexpr int kMaxContrib = 256;
constexpr float kStartOffset = 0.06f;
constexpr float kNear = 0.2f;
constexpr float kFar = 100.0f;   // reference auxiliary.h:20-21
constexpr float kTmin = 0.0001f;
constexpr int kWavesPerBlock = 4;
#ifndef DST_FWD_WPB
#define DST_FWD_WPB 1
#endif
constexpr int kFwdWavesPerBlock = DST_FWD_WPB;   // 1 or kWavesPerBlock
#ifndef DST_BWD_WAVES
#define DST_BWD_WAVES 2
#endif
#ifndef DST_STRIP_FWD
#define DST_STRIP_FWD 8   // width of the column strips the blocks of an image grid are walked in (0: row-major)
#endif
#ifndef DST_STRIP_BWD
#define DST_STRIP_BWD 8
#endif
constexpr uint32_t kOrderMinBlocks = 1536;   // replay: blocks are taken longest first on grids of at least three rounds of
                                             // blocks (512 fit the chip at once).  Training steps with / without: 8160 blocks
                                             // (1080p room) 10.74 / 10.91 ms, 2500 (800x800 sphere) 3.70 / 3.78; at 405 blocks
                                             // (233x417) no difference beyond the noise, and one kernel less
constexpr uint32_t kStripMinBlocks = 4096;   // forward: strips only for grids of at least this many blocks (see launch())

__device__ const float SH0 = 0.28209479177387814f;
__device__ const float SH1 = 0.4886025119029199f;
__device__ const float SH2[5] = {1.0925484305920792f, -1.0925484305920792f, 0.31539156525252005f,
                                 -1.0925484305920792f, 0.5462742152960396f};
__device__ const float SH3[7] = {-0.5900435899266435f, 2.890611442640554f, -0.4570457994644658f,
                                 0.3731763325901154f, -0.4570457994644658f, 1.445305721320277f,
                                 -0.5900435899266435f};

struct F3 { float x, y, z; };
// Lanes for which `b` holds (the compare result itself becomes the mask: no 0/1 detour through a register).
__device__ __forceinline__ uint64_t wave_ballot(bool b) { return __builtin_amdgcn_ballot_w64(b); }
__device__ __forceinline__ F3 f3(float x, float y, float z) { return F3{x, y, z}; }
__device__ __forceinline__ F3 operator+(F3 a, F3 b) { return F3{a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ F3 operator-(F3 a, F3 b) { return F3{a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ F3 operator-(F3 a) { return F3{-a.x, -a.y, -a.z}; }
__device__ __forceinline__ F3 operator*(F3 a, float s) { return F3{a.x * s, a.y * s, a.z * s}; }
__device__ __forceinline__ F3 operator*(float s, F3 a) { return F3{s * a.x, s * a.y, s * a.z}; }
__device__ __forceinline__ F3 operator/(F3 a, float s) { return F3{a.x / s, a.y / s, a.z / s}; }
__device__ __forceinline__ float dot(F3 a, F3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ F3 cross(F3 a, F3 b) {
    return F3{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ float length(F3 a) { return __builtin_sqrtf(dot(a, a)); }
__device__ __forceinline__ F3 ld3(const float *p) { return F3{p[0], p[1], p[2]}; }

// exp for x <= 0 (any x works): Cody-Waite reduction, degree-6 polynomial, exponent patched in.
__device__ __forceinline__ float exp_det(float x) {
    if (!(x >= -87.0f)) return 0.0f;
    if (x > 88.0f) x = 88.0f;
    float kf = __builtin_rintf(x * 1.44269504088896341f);
    float r = (x - kf * 0.693359375f) - kf * -2.12194440e-4f;
    float z = r * r;
    float p = 1.9875691500e-4f;
    p = p * r + 1.3981999507e-3f;
    p = p * r + 8.3334519073e-3f;
    p = p * r + 4.1665795894e-2f;
    p = p * r + 1.6666665459e-1f;
    p = p * r + 5.0000001201e-1f;
    p = p * z + r;
    p = p + 1.0f;
    return __uint_as_float(__float_as_uint(p) + ((uint32_t)((int32_t)kf << 23)));
}

// quaternion (w,x,y,z) -> rows: tangent u, tangent v, normal (reference auxiliary.h:403-429)
__device__ __forceinline__ void quat_rows(const float q0, const float q1, const float q2, const float q3, F3 (&R)[3]) {
    float s = 1.0f / __builtin_sqrtf(q3 * q3 + q0 * q0 + q1 * q1 + q2 * q2);
    float w = q0 * s, x = q1 * s, y = q2 * s, z = q3 * s;
    R[0] = f3(1.f - 2.f * (y * y + z * z), 2.f * (x * y + w * z), 2.f * (x * z - w * y));
    R[1] = f3(2.f * (x * y - w * z), 1.f - 2.f * (x * x + z * z), 2.f * (y * z + w * x));
    R[2] = f3(2.f * (x * z + w * y), 2.f * (y * z - w * x), 1.f - 2.f * (x * x + y * y));
}

// Surfel record (DstParams.scratch): what the evaluation of a hit takes from its surfel's parameters alone, made once a
// call by the operations a hit would make it with (so with the same bits): rotation rows, minus the first two's products
// with the mean, opacity, scales and their reciprocals.  A hit then reads one line of 64 bytes instead of one in each of four
// tensors, and is spared a square root, a division and some eighty other instructions.  Tiles of a 1080p room 3640 -> 3462 us,
// of an 800x800 sphere 1954 -> 1873, reflections by rows 11.35 -> 11.01 ms and 2438 -> 2373 us; the records of a million
// surfels take 30 us.  (The same for the replay, with the corners and the quaternion, 128 bytes: 5621 -> 5576 us + 96 for
// making them, 8754 -> 8656 + 48: no gain.)
struct alignas(64) DstSurfel {
    float r0[3], tx;
    float r1[3], ty;
    float r2[3], opac;
    float sx, sy, isx, isy;
};
static_assert(sizeof(DstSurfel) == 64, "one cache line's half");

// a / b, rounded once as the division operator does, given r = 1 / b rounded once: the first correction leaves a quotient
// within an ulp, and one corrected from there by its exact remainder is the rounded one (Markstein, IBM J. Res. Dev. 34,
// 1990).  Holds while nothing under- or overflows on the way.  A record's r is no number where b is outside 2^+-40, and
// a too large makes the result none either: callers divide where the squares of the two quotients do not add up to a
// number.  A quotient below 2^-40 may be off by an ulp, which the splat's exponent does not see (1 + x for |x| < 2^-25).
__device__ __forceinline__ float div_by(float a, float b, float r) {
    const float q0 = a * r;
    const float q1 = __builtin_fmaf(__builtin_fmaf(-b, q0, a), r, q0);
    return __builtin_fmaf(__builtin_fmaf(-b, q1, a), r, q1);
}

// Where a surfel's SH coefficients come from: the caller's fp32 tensor, or (DST_FLAG_SH_HALF) its binary16 copy,
// widened to fp32 as it is read - the arithmetic after that is the same fp32 sequence either way.
struct ShF32 {
    const float *p;
    __device__ __forceinline__ float operator()(int k) const { return p[k]; }
};
struct ShF16 {
    const uint16_t *p;
    __device__ __forceinline__ float operator()(int k) const { return (float)__builtin_bit_cast(_Float16, p[k]); }
};
// The first `n_halves` binary16 coefficients of a surfel as 16-byte loads (rows of 16 coefficients x 3 channels are 96
// bytes, so every row starts on a 16-byte boundary when the tensor does), kept in registers.
struct ShF16Row {
    uint32_t w[24];
    __device__ __forceinline__ void load(const uint16_t *row, int n_halves) {
        const uint4 *src = reinterpret_cast<const uint4 *>(row);
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            if (8 * k < n_halves) {
                const uint4 v = src[k];
                w[4 * k] = v.x; w[4 * k + 1] = v.y; w[4 * k + 2] = v.z; w[4 * k + 3] = v.w;
            } else {
                w[4 * k] = w[4 * k + 1] = w[4 * k + 2] = w[4 * k + 3] = 0u;
            }
        }
    }
    __device__ __forceinline__ float operator()(int k) const {
        const uint32_t word = w[k >> 1];
        return (float)__builtin_bit_cast(_Float16, (uint16_t)((k & 1) ? (word >> 16) : (word & 0xFFFFu)));
    }
};

// SH colour of one surfel in direction d (reference forward.cu:18-58); clamp flags for backward.
template <class SH>
__device__ __forceinline__ F3 sh_color(int deg, const SH &sh, F3 d, bool (&neg)[3]) {
#define SHC(j) f3(sh(3 * (j)), sh(3 * (j) + 1), sh(3 * (j) + 2))
    F3 r = SH0 * SHC(0);
    if (deg > 0) {
        float x = d.x, y = d.y, z = d.z;
        r = r - SH1 * y * SHC(1) + SH1 * z * SHC(2) - SH1 * x * SHC(3);
        if (deg > 1) {
            float xx = x * x, yy = y * y, zz = z * z, xy = x * y, yz = y * z, xz = x * z;
            r = r + SH2[0] * xy * SHC(4) + SH2[1] * yz * SHC(5) + SH2[2] * (2.0f * zz - xx - yy) * SHC(6) +
                SH2[3] * xz * SHC(7) + SH2[4] * (xx - yy) * SHC(8);
            if (deg > 2) {
                r = r + SH3[0] * y * (3.0f * xx - yy) * SHC(9) + SH3[1] * xy * z * SHC(10) +
                    SH3[2] * y * (4.0f * zz - xx - yy) * SHC(11) +
                    SH3[3] * z * (2.0f * zz - 3.0f * xx - 3.0f * yy) * SHC(12) +
                    SH3[4] * x * (4.0f * zz - xx - yy) * SHC(13) + SH3[5] * z * (xx - yy) * SHC(14) +
                    SH3[6] * x * (xx - 3.0f * yy) * SHC(15);
            }
        }
    }
#undef SHC
    r = f3(r.x + 0.5f, r.y + 0.5f, r.z + 0.5f);
    neg[0] = r.x < 0.f;
    neg[1] = r.y < 0.f;
    neg[2] = r.z < 0.f;
    return f3(r.x > 0.f ? r.x : 0.f, r.y > 0.f ? r.y : 0.f, r.z > 0.f ? r.z : 0.f);
}
// The colour from the binary16 copy of the coefficients (DST_FLAG_SH_HALF).
__device__ __forceinline__ F3 sh_color_half(const DstParams &p, int g, F3 d, bool (&neg)[3]) {
    const uint16_t *row = p.shs_half + (size_t)g * p.M * 3;
    if ((p.M & 7) == 0 && p.M <= 16 && (reinterpret_cast<uintptr_t>(p.shs_half) & 15u) == 0u) {
        ShF16Row r;
        r.load(row, 3 * (p.D + 1) * (p.D + 1));
        return sh_color(p.D, r, d, neg);
    }
    return sh_color(p.D, ShF16{row}, d, neg);
}

// ---- ray / quad -----------------------------------------------------------------------------------------
// Products feeding a difference or a running sum are fused here BY DEFINITION (explicit fma, one rounding);
// the CPU statement of the same test uses the same calls, so both sides produce the same bits.
__device__ __forceinline__ F3 cross_f(F3 x, F3 y) {
    return F3{__builtin_fmaf(x.y, y.z, -(x.z * y.y)), __builtin_fmaf(x.z, y.x, -(x.x * y.z)),
              __builtin_fmaf(x.x, y.y, -(x.y * y.x))};
}
__device__ __forceinline__ float dot_f(F3 a, F3 b) {
    return __builtin_fmaf(a.z, b.z, __builtin_fmaf(a.y, b.y, a.x * b.x));
}
__device__ __forceinline__ bool same_sign(float a, float b, float c) {
    return (a >= 0.f && b >= 0.f && c >= 0.f) || (a <= 0.f && b <= 0.f && c <= 0.f);
}
// Quad = triangles ABC and BCD, given as the leaf record holds it: corner A, edge vectors AB, AC, AD, normals
// n0 = AB x AC, n1 = (C-B) x (D-B), n2 = AC x AD, c1 = n1.AB.  The signed volumes d.((P-o) x (Q-o)) of the edge tests
// are formed from one cross product with the ray, m = d x (A-o), and the edge vectors:
//     d.((A+P'-o) x (A+Q'-o)) = (Q'-P').m + d.(P' x Q'),
// so that nothing is multiplied that is as long as the way from the origin to the quad except in m itself (with the
// corners relative to the origin in every product, a ray passing half a millimetre-sized quad outside it counted as
// a hit from a few metres away).  Then t = n.(v1-o) / n.d on the plane of the triangle that was hit.
__device__ __forceinline__ bool ray_quad(F3 o, F3 d, F3 A, F3 AB, F3 AC, F3 AD, F3 n0, F3 n1, F3 n2, float c1, float &t,
                                         uint32_t &tri) {
    const F3 a = A - o;
    const F3 m = cross_f(d, a);
    const float X = dot_f(AB, m), Y = dot_f(AC, m), Z = dot_f(AD, m);
    const float q0 = dot_f(n0, d), q1 = dot_f(n1, d), q2 = dot_f(n2, d);
    const float u2 = X, u1 = -Y, u0 = (Y - X) + q0;          // edges AB, CA, BC
    const bool in0 = same_sign(u0, u1, u2);
    const float w0 = (Z - Y) + q2;                            // edge CD
    const float w1 = (X - Z) + ((q1 - q0) - q2);              // edge DB (AD x AB = n1 - n0 - n2)
    const bool in1 = same_sign(w0, w1, u0);
    if (!(in0 || in1)) return false;
    tri = in0 ? 0u : 1u;
    const float pa = dot_f(in0 ? n0 : n1, a);
    const float p = in0 ? pa : pa + c1;                       // n1.(B-o) = n1.(A-o) + n1.AB
    const float q = in0 ? q0 : q1;
    t = p / q;
    return (t > 0.0f) && (t < kInfDepth);
}

// v_writelane_b32: value (uniform) into lane `lane` (uniform) of `old`; the compiler offers no builtin for it.
__device__ int dst_writelane(int value, int lane, int old) __asm("llvm.amdgcn.writelane.i32");

// The kernel's parameter block where the hardware put it.  Read through a pointer the compiler cannot follow
// (fresh_params), the block's pointers are scalar loads at their place of use, in every step of a loop anew; read
// through the kernel's argument they are loaded once, far too many for the scalar registers, and every use in a loop
// brings them back from lanes of a vector register, one vector instruction per word: a quarter of the compositing
// loop's instructions.
typedef const __attribute__((address_space(4))) DstParams *const_params;
__device__ __forceinline__ const_params fresh_params() {
    const_params p = (const_params)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}

// ---- wave-uniform fetches ---------------------------------------------------------------------------------
typedef const __attribute__((address_space(4))) uint32_t *const_u32_ptr;
typedef __attribute__((address_space(3))) uint32_t *lds_u32;
typedef __attribute__((address_space(3))) double *lds_f64;
template <int N>
__device__ __forceinline__ void load_uniform(const void *p, uint32_t (&out)[N]) {
    const_u32_ptr c = (const_u32_ptr)(uintptr_t)p;
#pragma unroll
    for (int k = 0; k < N; ++k) out[k] = c[k];
}

typedef float v4f __attribute__((ext_vector_type(4)));
// Two consecutive 64-byte records (the stand-ins of a leaf group's two quads), or one 96-byte quad record, in one
// trip: left to itself the compiler splits these fetches and waits for the first part before asking for the rest.
typedef uint32_t u32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ void load_record_pair(const void *p, u32x16 &a, u32x16 &b) {
    asm volatile("s_load_dwordx16 %0, %2, 0x0\n\ts_load_dwordx16 %1, %2, 0x40\n\ts_waitcnt lgkmcnt(0)"
                 : "=&s"(a), "=&s"(b)
                 : "s"(p)
                 : "memory");
}
typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ void load_quad_record(const void *p, u32x16 &a, u32x8 &b) {
    asm volatile("s_load_dwordx16 %0, %2, 0x0\n\ts_load_dwordx8 %1, %2, 0x40\n\ts_waitcnt lgkmcnt(0)"
                 : "=&s"(a), "=&s"(b)
                 : "s"(p)
                 : "memory");
}
// bits = 2 * bits + (mask != 0): one compare and one add-with-carry per lane mask.
__device__ __forceinline__ uint32_t shift_in_any(uint32_t bits, uint64_t mask) {
    asm("s_cmp_lg_u64 %1, 0\n\ts_addc_u32 %0, %0, %0" : "+s"(bits) : "s"(mask) : "scc");
    return bits;
}
// A whole traversal node in one trip, and one wait for all of it.
__device__ __forceinline__ void load_node(const void *node, u32x16 &a, u32x16 &b) { load_record_pair(node, a, b); }

struct RaySlab {   // per-lane precomputation for the conservative slab test
    float ix, iy, iz;     // 1/d, with tiny components pushed away from zero
    float nx, ny, nz;     // -o * (1/d)
    float wx, wy, wz;     // interval widening per axis
    float max_abs;        // largest vertex coordinate of the scene (uniform)
};

__device__ __forceinline__ float safe_inv(float d) {
    float a = __builtin_fabsf(d);
    float v = (a < 1e-20f) ? __builtin_copysignf(1e-20f, d) : d;   // NaN passes through
    return 1.0f / v;
}

// (`reach`: how large the numbers are that the ray's origin was made from, where it has been moved up along the ray.)
__device__ __forceinline__ RaySlab make_slab(F3 o, F3 d, float max_abs, float reach = 0.f) {
    RaySlab s;
    s.ix = safe_inv(d.x);
    s.iy = safe_inv(d.y);
    s.iz = safe_inv(d.z);
    s.nx = -o.x * s.ix;
    s.ny = -o.y * s.iy;
    s.nz = -o.z * s.iz;
    // The quad test works in origin-relative fp32 coordinates, so it can accept a ray that passes
    // a few ulps of (|o| + |vertex|) outside the quad; boxes are widened by well above that: by 4e-6 |o| here,
    // and by 4e-6 of the quad's own largest coordinate where the boxes are made (lbvh.hip, kBoxPad).
    float oa = __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(o.x), reach), __builtin_fmaxf(__builtin_fabsf(o.y), __builtin_fabsf(o.z)));
    s.max_abs = max_abs;
    float pad = 4e-6f * oa;
    s.wx = pad * __builtin_fabsf(s.ix);
    s.wy = pad * __builtin_fabsf(s.iy);
    s.wz = pad * __builtin_fabsf(s.iz);
    return s;
}

// Conservative slab test for a packet whose lanes all have the same direction signs: the near and far plane of
// each axis are then the same box faces for all lanes, picked once per wave, and the widening folds into the
// offsets.  The box is hit iff the entry distance tn <= min(exit distance, tmax); tmax < 0 disables a lane.
struct RaySlabFast {
    float ix, iy, iz;
    float cnx, cny, cnz;   // -o/d - widening: added to (near face)/d
    float cfx, cfy, cfz;   // -o/d + widening: added to (far face)/d
};
// Returns the lanes that hit as a mask (the compare writes the wave mask directly).
__device__ __forceinline__ uint64_t slab_hit_fast(const RaySlabFast &s, float nx, float ny, float nz, float fx,
                                                  float fy, float fz, float tmax, float &tn) {
    const float a = __builtin_fmaf(nx, s.ix, s.cnx), b = __builtin_fmaf(ny, s.iy, s.cny),
                c = __builtin_fmaf(nz, s.iz, s.cnz);
    const float e = __builtin_fmaf(fx, s.ix, s.cfx), f = __builtin_fmaf(fy, s.iy, s.cfy),
                g = __builtin_fmaf(fz, s.iz, s.cfz);
    tn = __builtin_fmaxf(__builtin_fmaxf(a, b), __builtin_fmaxf(c, 0.0f));
    const float tf = __builtin_fminf(__builtin_fminf(e, f), __builtin_fminf(g, tmax));
    return __builtin_amdgcn_fcmpf(tn, tf, 5);   // 5 = ordered <=
}

// The 16 nearest hits of a lane, ascending.  One entry = (bits of t) << 32 | idx: t is positive, so the
// unsigned 64-bit order is the (t, idx) lexicographic order and the content does not depend on the order in
// which the BVH delivers candidates (ties in t resolve to ascending primitive index).
struct KBuf {
    uint64_t e[kChunk];
};
__device__ __forceinline__ uint64_t kb_pack(float t, uint32_t idx) { return ((uint64_t)__float_as_uint(t) << 32) | idx; }
__device__ __forceinline__ float kb_t(uint64_t e) { return __uint_as_float((uint32_t)(e >> 32)); }
__device__ __forceinline__ uint32_t kb_idx(uint64_t e) { return (uint32_t)e; }

__device__ __forceinline__ void kbuf_reset(KBuf &b) {
#pragma unroll
    for (int k = 0; k < kChunk; ++k) b.e[k] = kb_pack(kInfDepth, 0u);
}

// Entries as doubles: an entry's upper word is the bits of a float between 0 and kInfDepth, so as a double it is a
// finite number of the same sign whose order is that of the 64-bit integers (no NaN, and nothing that a double-precision
// comparison would take for equal); kNoEntry is larger than all of them.  64-bit integer comparisons and selects cost
// seven instructions per slot of a sorted insertion, minimum and maximum of doubles two.
constexpr uint64_t kNoEntry = 0x7F000000FFFFFFFFull;
__device__ __forceinline__ bool kb_less(uint64_t a, uint64_t b) {
    return __builtin_bit_cast(double, a) < __builtin_bit_cast(double, b);
}
__device__ __forceinline__ uint64_t kb_min(uint64_t a, uint64_t b) {   // (written out: no canonicalising of operands)
    uint64_t r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ uint64_t kb_max(uint64_t a, uint64_t b) {
    uint64_t r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// Sorted insert in place: slot k becomes the middle one of its entry, the entry above and the new one.
__device__ __forceinline__ void kbuf_insert(KBuf &b, uint64_t x_in, bool on) {
    const uint64_t x = on ? x_in : kNoEntry;   // a lane that inserts nothing offers what leaves every slot as it is
    // (two slots at a time: a double-precision result is not ready for the very next instruction)
#pragma unroll
    for (int k = kChunk - 1; k >= 1; k -= 2) {
        const uint64_t m1 = kb_min(b.e[k], x), m0 = kb_min(b.e[k - 1], x);
        b.e[k] = kb_max(b.e[k - 1], m1);
        b.e[k - 1] = k >= 2 ? kb_max(b.e[k - 2], m0) : m0;
    }
}

#ifdef DST_STATS
struct WaveStats { unsigned long long nodes, leaves, t_trav, t_comp, chunks, leaf_any, t_plan, t_hb, steps; };
#define STAT(x) x
#define WSP , ws
#else
#define STAT(x)
#define WSP
#endif

// Per-lane constants of the conservative stand-in for the quad test (DstLeafPre).  With S = |o|_max + the largest
// coordinate of the quad: the stand-in's distance along the ray is off by at most about 3.4e-5 S/|d| + 1e-5 |t| when
// |n.d| >= 0.05 |d| (flatter rays skip the stand-in), its hit point by 7e-5 S; the margins below are twice that.
struct RayPre {
    float padw;     // in-plane slack, world units
    float tp;       // slack on the distance along the ray
    float graze;    // |n.d| below this: too flat for the stand-in
    float inv_dl;   // 1 / |d|
};
__device__ __forceinline__ RayPre make_pre(F3 o, F3 d, float max_abs) {
    RayPre r;
    const float oa = __builtin_fmaxf(__builtin_fabsf(o.x), __builtin_fmaxf(__builtin_fabsf(o.y), __builtin_fabsf(o.z)));
    const float S = oa;   // the ray's share; the quad's own coordinates are in its limits already (lbvh.hip, make_leaf)
    const float dl = __builtin_sqrtf(d.x * d.x + d.y * d.y + d.z * d.z);
    r.inv_dl = 1.0f / dl;
    r.padw = 1.5e-4f * S;
    r.tp = 1e-4f * S * r.inv_dl;
    r.graze = 0.05f * dl;
    return r;
}

// The stand-in test of one quad for all lanes (about 28 instructions), as a lane mask: bit clear = that lane's ray
// cannot pass the exact test (lanes that are switched off come back set or clear; the caller masks them).
__device__ __forceinline__ uint64_t quad_may_hit(const u32x16 &Q, const RayPre &rp, F3 o, F3 d, float tmax) {
#define QF(k) __uint_as_float(Q[k])
    const float hx = QF(0) - o.x, hy = QF(1) - o.y, hz = QF(2) - o.z;
    const float qd = __builtin_fmaf(QF(5), d.z, __builtin_fmaf(QF(4), d.y, QF(3) * d.x));
    const float ph = __builtin_fmaf(QF(5), hz, __builtin_fmaf(QF(4), hy, QF(3) * hx));
    const float t = ph * __builtin_amdgcn_rcpf(qd);
    const float wx = __builtin_fmaf(t, d.x, -hx), wy = __builtin_fmaf(t, d.y, -hy), wz = __builtin_fmaf(t, d.z, -hz);
    const float s = __builtin_fmaf(QF(8), wz, __builtin_fmaf(QF(7), wy, QF(6) * wx));
    const float r = __builtin_fmaf(QF(11), wz, __builtin_fmaf(QF(10), wy, QF(9) * wx));
    const float m = __builtin_fmaxf(__builtin_fabsf(s), __builtin_fabsf(r));
    const float lim = __builtin_fmaf(rp.padw, QF(12), QF(13));
    const float tpq = __builtin_fmaf(QF(14), rp.inv_dl, rp.tp);
    // every comparison is written so that a NaN keeps the ray in; the lane masks are combined without branches
    const uint64_t flat = wave_ballot(__builtin_fabsf(qd) < rp.graze);
    const uint64_t out_base = wave_ballot(m > lim) | wave_ballot(t < -tpq);
    const uint64_t out_t = wave_ballot(__builtin_fmaf(t, 0.9999f, -tpq) > tmax);
#undef QF
    return flat | ~(out_base | out_t);
}

// The exact test of one quad record for all lanes; hits are admitted into the lanes' buffers.
__device__ __forceinline__ void quad_exact(const u32x16 &La, const u32x8 &Lb, F3 o, F3 d, bool active, KBuf &buf, uint32_t &cnt
#ifdef DST_STATS
                                           , WaveStats &ws
#endif
) {
    STAT(ws.t_plan++;)
#define LW(k) ((k) < 16 ? La[(k) & 15] : Lb[((k) - 16) & 7])
#define LF3(k) f3(__uint_as_float(LW(k)), __uint_as_float(LW((k) + 1)), __uint_as_float(LW((k) + 2)))
    float t = 0.f;
    uint32_t tri = 0u;
    const bool hit = active && ray_quad(o, d, LF3(0), LF3(3), LF3(6), LF3(9), LF3(16), LF3(12), LF3(19),
                                        __uint_as_float(LW(22)), t, tri);
#undef LF3
    const uint64_t x = kb_pack(t, 2u * LW(15) + tri);
#undef LW
    const bool adm = hit && (kb_less(x, buf.e[kChunk - 1]));
    if (wave_ballot(adm) != 0ull) {
        STAT(ws.leaf_any++;)
        cnt += adm ? 1u : 0u;
        kbuf_insert(buf, x, adm);
    }
}

// A leaf group (up to DST_GROUP quads, consecutive records) against all lanes' rays.  The stand-in records of
// two quads are fetched together, then the exact records of those that some lane's ray may hit, again together:
// one trip to memory per stage instead of one per quad.
__device__ __forceinline__ void test_group(const DstAccelView &acc, uint32_t first, uint32_t count, const RayPre &rp,
                                           F3 o, F3 d, bool active, KBuf &buf, uint32_t &cnt
#ifdef DST_STATS
                                           , WaveStats &ws
#endif
) {
    uint32_t q0 = 0;   // count >= 1
#pragma unroll 1
    do {
        const bool two = q0 + 1u < count;
        // the record after the last quad of the structure exists (the array has one spare record)
        u32x16 Q0, Q1;
        load_record_pair(&acc.pre[first + q0], Q0, Q1);
        STAT(ws.leaves += two ? 2 : 1;)
        const float tmax = kb_t(buf.e[kChunk - 1]);
        const uint64_t live = wave_ballot(active);
        const uint64_t k0 = quad_may_hit(Q0, rp, o, d, tmax) & live;
        const uint64_t k1 = two ? (quad_may_hit(Q1, rp, o, d, tmax) & live) : 0ull;
        uint32_t todo = (k0 != 0ull ? 1u : 0u) | (k1 != 0ull ? 2u : 0u);
#pragma unroll 1
        while (todo != 0u) {
            const uint32_t k = (todo & 1u) ? 0u : 1u;
            todo &= ~(1u << k);
            u32x16 La;
            u32x8 Lb;
            load_quad_record(&acc.leaves[first + q0 + k], La, Lb);
            quad_exact(La, Lb, o, d, active, buf, cnt WSP);
        }
        q0 += 2;
    } while (DST_GROUP > 2 && q0 < count);   // groups of at most two quads: one pass, no loop
}

// One traversal for the whole wave: every active lane ends with its own 16 nearest hits (t relative
// to its origin, 0 < t < 1e16) and the number of admissions.  Wave-uniform control flow: nodes and quads
// are fetched once per wave, the stack is two VGPRs addressed by lane.  128 entries are enough by construction:
// a step defers at most three children, and the builder only hands over hierarchies whose wide nodes are at most 42
// levels deep (grandchildren nodes over a binary hierarchy of at most 62 levels, whose depth the Morton keys bound or
// the build measures; nodes that open one level at a time only over hierarchies measured to be at most 42 deep).  A
// stack that is full all the same loses the entry (no fault; checked on the builder's side, not here).
// All active lanes share the direction signs `sgn` (bit a set = axis a negative), see slab_hit_fast.
// (The backward trace without a hit record: its LDS is taken by the gradient table, which leaves none for the lists
// of the bundle walk.)
__device__ __forceinline__ void packet_walk(const DstAccelView &acc, const RaySlab &slab, uint32_t sgn, F3 o, F3 d,
                                            bool active, KBuf &buf, uint32_t &cnt
#ifdef DST_STATS
                                            , WaveStats &ws
#endif
) {
    const RayPre rp = make_pre(o, d, slab.max_abs);
    RaySlabFast fs;
    fs.ix = slab.ix; fs.iy = slab.iy; fs.iz = slab.iz;
    fs.cnx = slab.nx - slab.wx; fs.cny = slab.ny - slab.wy; fs.cnz = slab.nz - slab.wz;
    fs.cfx = slab.nx + slab.wx; fs.cfy = slab.ny + slab.wy; fs.cfz = slab.nz + slab.wz;
    const bool sx = (sgn & 1u) != 0u, sy = (sgn & 2u) != 0u, sz = (sgn & 4u) != 0u;
    uint32_t stack0 = 0u, stack1 = 0u;
    int sp = 0;
    // A well-formed hierarchy is walked in at most one step per node and per leaf group; the cap makes the
    // loops finite whatever the memory holds.  Two loops: the inner one goes down through nodes and never touches
    // the hit buffer, the outer one tests a leaf group and pops (with one loop around both, the compiler kept two
    // copies of the buffer's 32 registers and moved them back and forth at every leaf group).
    constexpr uint32_t kEnd = 0xFFFFFFFFu;   // not a reference: leaf bit set, impossible position
    uint32_t budget = 2u * acc.n_leaves + 8u;
    auto pop = [&]() -> uint32_t {
        if (sp == 0) return kEnd;
        --sp;
        const uint32_t a = __builtin_amdgcn_readlane(stack0, sp & 63), b = __builtin_amdgcn_readlane(stack1, sp & 63);
        return sp < 64 ? a : b;
    };
    uint32_t ref = acc.root;
    for (;;) {
        while ((ref & DST_LEAF_BIT) == 0u) {
            if (budget == 0u || ref + 1u >= acc.n_leaves) {   // spent, or not a node of this hierarchy
                ref = kEnd;
                break;
            }
            --budget;
            const char *node = reinterpret_cast<const char *>(&acc.wide[ref]);
            STAT(ws.nodes++;)
            const float tmax = active ? kb_t(buf.e[kChunk - 1]) : -1.0f;
            uint32_t tail[4];
            uint32_t hit = 0u;                     // bit k: some lane enters child k
            {
                u32x16 n0, n1;                     // children 0 and 1, children 2 and 3
                load_node(node, n0, n1);
#pragma unroll
                for (int k = DST_WIDE - 1; k >= 0; --k) {   // last child first: its bit is shifted up the furthest
                    auto word = [&](int w) { return __uint_as_float(k < 2 ? n0[8 * k + w] : n1[8 * (k - 2) + w]); };
                    tail[k] = __float_as_uint(word(3));
                    float tn;   // (the box of an unused slot is empty)
                    hit = shift_in_any(hit, slab_hit_fast(fs, sx ? word(4) : word(0), sy ? word(5) : word(1), sz ? word(6) : word(2),
                                                          sx ? word(0) : word(4), sy ? word(1) : word(5), sz ? word(2) : word(6), tmax, tn));
                }
            }
            if (hit != 0u) {
                // Children are taken in stored order: the first one that is hit next, the others deferred (last
                // first).  Ordering them by entry distance was measured: 3 % fewer visits, but the scalar work of
                // the sort costs more than those visits.
                const uint32_t rest = hit & (hit - 1u);   // the hit children after the first one (never child 0)
                if (__builtin_expect(sp + 3 <= DST_WAVE, 1)) {
                    // Without branches: each candidate is written at the top of the stack and the top moves up only
                    // if the child was hit (an entry above the top is dead, so a write there does no harm).
                    stack0 = (uint32_t)dst_writelane((int)tail[3], sp, (int)stack0);
                    sp += (int)((rest >> 3) & 1u);
                    stack0 = (uint32_t)dst_writelane((int)tail[2], sp, (int)stack0);
                    sp += (int)((rest >> 2) & 1u);
                    stack0 = (uint32_t)dst_writelane((int)tail[1], sp, (int)stack0);
                    sp += (int)((rest >> 1) & 1u);
                } else {
#define DST_PUSH(v)                                                                                          \
    {                                                                                                        \
        if (sp < 64) stack0 = (uint32_t)dst_writelane((int)(v), sp, (int)stack0);               \
        else stack1 = (uint32_t)dst_writelane((int)(v), sp - 64, (int)stack1);                  \
        sp = min(sp + 1, 2 * DST_WAVE - 1);                                                                  \
    }
                    if (rest & 8u) DST_PUSH(tail[3])
                    if (rest & 4u) DST_PUSH(tail[2])
                    if (rest & 2u) DST_PUSH(tail[1])
#undef DST_PUSH
                }
                ref = (hit & 1u) ? tail[0] : ((hit & 2u) ? tail[1] : ((hit & 4u) ? tail[2] : tail[3]));
            } else {
                ref = pop();
            }
        }
        if (ref == kEnd || budget == 0u) break;
        --budget;
        const uint32_t first = ref & DST_REF_FIRST_MASK, count = ((ref >> 28) & 7u) + 1u;
        if (first + count > acc.n_leaves) break;   // not a leaf group of this hierarchy
        test_group(acc, first, count, rp, o, d, active, buf, cnt WSP);
        ref = pop();
    }
}

// ---- per-lane walk ------------------------------------------------------------------------------------------
// For rays that share neither origin nor direction (reflection rays off rough geometry, arbitrary ray lists) a
// packet visits the union of 64 unrelated paths with one useful lane each.  Here every lane walks the hierarchy
// on its own: own stack (private memory), own node and quad fetches through the vector path, same slab and
// quad tests, same buffer.  The buffer's content does not depend on the order of arrival, so both walks give
// the same result bit for bit; the choice between them only changes the time.
#ifndef DST_PACKET_DIR_SPREAD
#define DST_PACKET_DIR_SPREAD 0.02f   // measured: 0.06 makes packets of lidar rays that are metres apart at their hits
#endif
#ifndef DST_PACKET_ORG_SPREAD
#define DST_PACKET_ORG_SPREAD 0.02f
#endif
constexpr float kPacketDirSpread = DST_PACKET_DIR_SPREAD;   // largest direction difference (relative) inside a packet
constexpr float kPacketOrgSpread = DST_PACKET_ORG_SPREAD;   // largest origin difference, relative to the scene extent
constexpr int kLaneStack = 2 * 64;        // as deep as the packet's two lane-indexed registers
constexpr uint32_t kWalkDone = 0xFFFFFFFFu;   // not a reference: leaf bit set with an impossible position
// A real call on purpose: inlined, its register needs would spill the bundle walk that nearly every wave takes.
// The walk is a real function, so the compiler cannot see where its pointers lead: say it (global memory, LDS).
typedef const __attribute__((address_space(1))) float *global_f32;
typedef const __attribute__((address_space(1))) uint32_t *global_u32;
#define LD3(p, k) f3((p)[(k)], (p)[(k) + 1], (p)[(k) + 2])
// (Four waves per SIMD, DST_MIXED_WAVES, spill some hundred registers around this call: 20,000 unrelated rays among
// small quads take 813 us at four, 791 at three, 734 at two waves.  The row walk takes 290 for the same list.)
// `shelf`: optional LDS for the first kLaneShelf stack entries of every lane ([entry][lane], conflict-free);
// deeper entries, or all of them without a shelf, live in private memory.
constexpr int kLaneShelf = 32;
struct LaneWalkAccel { const DstLeaf *leaves; const DstWideNode *wide; uint32_t n_leaves, root; };   // by value: registers
static_assert(DST_GROUP <= 2, "the per-lane walk fetches a leaf group as at most two quad records");
static_assert(sizeof(DstWideNode) == 128 && sizeof(DstLeaf) == 96, "the per-lane walk reads both as 16-byte words");
// A value that is the same in every lane, moved to a scalar register (arguments of a real call arrive in vector ones).
template <class T>
__device__ __forceinline__ T *uniform_ptr(T *p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return reinterpret_cast<T *>(((uint64_t)hi << 32) | lo);
}
__device__ __attribute__((noinline)) void lane_walk(const LaneWalkAccel acc_in, const RaySlab &slab, F3 o, F3 d,
                                                    bool active, KBuf &buf_mem, uint32_t &cnt_mem, uint32_t *shelf_in) {
    const LaneWalkAccel acc = {uniform_ptr(acc_in.leaves), uniform_ptr(acc_in.wide),
                               (uint32_t)__builtin_amdgcn_readfirstlane(acc_in.n_leaves),
                               (uint32_t)__builtin_amdgcn_readfirstlane(acc_in.root)};
    uint32_t *const shelf = uniform_ptr(shelf_in);
    // The caller's buffer is in memory (its address crosses the call): work on a register copy and store it once
    // at the end.  Left in memory, every leaf test re-read its 128 bytes per lane and every admission re-wrote them.
    KBuf buf = buf_mem;
    uint32_t cnt = cnt_mem;
    RaySlabFast fs;
    fs.ix = slab.ix; fs.iy = slab.iy; fs.iz = slab.iz;
    fs.cnx = slab.nx - slab.wx; fs.cny = slab.ny - slab.wy; fs.cnz = slab.nz - slab.wz;
    fs.cfx = slab.nx + slab.wx; fs.cfy = slab.ny + slab.wy; fs.cfz = slab.nz + slab.wz;
    const bool neg_x = slab.ix < 0.f, neg_y = slab.iy < 0.f, neg_z = slab.iz < 0.f;
    uint32_t stack[kLaneStack];
    int sp = 0;
    uint32_t ref = active ? acc.root : kWalkDone;
    uint32_t budget = 2u * acc.n_leaves + 8u;   // a well-formed hierarchy needs fewer steps; bounds the loop regardless
    // A step of a lane is one dependent trip to memory: the lane's node (128 bytes) or its leaf group (two quad
    // records of 96 bytes, consecutive, the first 64 of each) is requested whole - eight to ten 16-byte loads from one base address, whatever
    // the lane is at - before anything is tested, so that lanes at nodes and lanes at leaf groups wait together,
    // once.  (Left to the compiler, a quad came in three trips - the first words, then the rest behind the first edge
    // test, then the surfel id behind the hit - and the lanes at leaf groups took theirs after the lanes at nodes had
    // finished theirs.)
    typedef const __attribute__((address_space(1))) v4f *global_v4f;
#pragma unroll 1
    while (wave_ballot(ref != kWalkDone) != 0ull) {
        if (ref == kWalkDone) continue;
        uint32_t next = kWalkDone;
        bool have_next = false;
        const bool is_leaf = (ref & DST_LEAF_BIT) != 0u;
        const uint32_t first = ref & DST_REF_FIRST_MASK, count = ((ref >> 28) & 7u) + 1u;
        const bool good = is_leaf ? (first < acc.n_leaves) : (ref + 1u < acc.n_leaves);
        if (good) {
            const bool two = is_leaf && count > 1u && first + 1u < acc.n_leaves;
            const global_v4f src = is_leaf ? (global_v4f)reinterpret_cast<const v4f *>(&acc.leaves[first])
                                           : (global_v4f)reinterpret_cast<const v4f *>(&acc.wide[ref]);
            // a node is 8 x 16 bytes; of a quad's record the first 4 words of 16 bytes are read (a leaf group of one quad
            // asks for 8 as well: the array has spare records behind its last quad), the second quad's are words 6 to 9
            v4f r0 = src[0], r1 = src[1], r2 = src[2], r3 = src[3], r4 = src[4], r5 = src[5], r6 = src[6], r7 = src[7];
            v4f r8 = {0.f, 0.f, 0.f, 0.f}, r9 = {0.f, 0.f, 0.f, 0.f};
            if (two) {
                r8 = src[8];
                r9 = src[9];
            }
            // every value is in its registers here: nothing of the above may be requested later, behind a test
            asm volatile("" : "+v"(r0), "+v"(r1), "+v"(r2), "+v"(r3), "+v"(r4));
            asm volatile("" : "+v"(r5), "+v"(r6), "+v"(r7), "+v"(r8), "+v"(r9));
            if (is_leaf) {
                // the first 64 bytes of a record: A, AB, AC, AD, n1 (three floats each), surfel id; n0, n2 and c1 are
                // formed as the builder forms them for the record's other 32 bytes
#define DST_LANE_QUAD(w0, w1, w2, w3)                                                                                  \
    {                                                                                                                  \
        float t = 0.f;                                                                                                 \
        uint32_t tri = 0u;                                                                                             \
        const F3 AB = f3(w0.w, w1.x, w1.y), AC = f3(w1.z, w1.w, w2.x), AD = f3(w2.y, w2.z, w2.w), n1 = f3(w3.x, w3.y, w3.z); \
        const bool hit = ray_quad(o, d, f3(w0.x, w0.y, w0.z), AB, AC, AD, cross_f(AB, AC), n1, cross_f(AC, AD),        \
                                  dot_f(n1, AB), t, tri);                                                              \
        const uint64_t x = kb_pack(t, 2u * __float_as_uint(w3.w) + tri);                                               \
        if (hit && (kb_less(x, buf.e[kChunk - 1]))) {                                                                          \
            cnt += 1u;                                                                                                 \
            kbuf_insert(buf, x, true);                                                                                 \
        }                                                                                                              \
    }
                DST_LANE_QUAD(r0, r1, r2, r3)
                if (two) DST_LANE_QUAD(r6, r7, r8, r9)
#undef DST_LANE_QUAD
                // (groups of more than two quads do not occur: DST_GROUP = 2; a longer one would lose its tail)
            } else {
                // a child is two words: low corner and reference, high corner and whether the slot is used
                const float tmax = kb_t(buf.e[kChunk - 1]);
                uint32_t key[DST_WIDE], cref[DST_WIDE];
#pragma unroll
                for (int k = 0; k < DST_WIDE; ++k) {
                    const v4f lo = k == 0 ? r0 : (k == 1 ? r2 : (k == 2 ? r4 : r6)), hi = k == 0 ? r1 : (k == 1 ? r3 : (k == 2 ? r5 : r7));
                    float tn;
                    const uint64_t h = slab_hit_fast(fs, neg_x ? hi.x : lo.x, neg_y ? hi.y : lo.y, neg_z ? hi.z : lo.z,
                                                     neg_x ? lo.x : hi.x, neg_y ? lo.y : hi.y, neg_z ? lo.z : hi.z, tmax, tn);
                    const bool mine = ((h >> __lane_id()) & 1ull) != 0ull && __float_as_uint(hi.w) != 0u;
                    key[k] = mine ? __float_as_uint(tn) : 0xFFFFFFFFu;   // entry distance (non-negative: bits order like the value)
                    cref[k] = __float_as_uint(lo.w);
                }
#define CSWAP(a, b)                                                            \
    {                                                                          \
        const bool sw_ = key[b] < key[a];                                      \
        const uint32_t ka_ = sw_ ? key[b] : key[a], kb_ = sw_ ? key[a] : key[b]; \
        const uint32_t ra_ = sw_ ? cref[b] : cref[a], rb_ = sw_ ? cref[a] : cref[b]; \
        key[a] = ka_; key[b] = kb_; cref[a] = ra_; cref[b] = rb_;              \
    }
                CSWAP(0, 1) CSWAP(2, 3) CSWAP(0, 2) CSWAP(1, 3) CSWAP(1, 2)
#undef CSWAP
                // defer the farther children (farthest first), go on with the nearest
#pragma unroll
                for (int k = DST_WIDE - 1; k >= 1; --k) {
                    if (key[k] != 0xFFFFFFFFu && sp < kLaneStack) {
                        if (shelf != nullptr && sp < kLaneShelf) ((lds_u32)shelf)[sp * DST_WAVE + (int)__lane_id()] = cref[k];
                        else stack[sp] = cref[k];
                        ++sp;
                    }
                }
                if (key[0] != 0xFFFFFFFFu) {
                    next = cref[0];
                    have_next = true;
                }
            }
        }
        if (!have_next && sp > 0) {
            --sp;
            next = (shelf != nullptr && sp < kLaneShelf) ? ((lds_u32)shelf)[sp * DST_WAVE + (int)__lane_id()] : stack[sp];
        }
        ref = (--budget == 0u) ? kWalkDone : next;
    }
    buf_mem = buf;
    cnt_mem = cnt;
}

#include "bundle.inc"

// One walk for the rays of this wave, or one per lane (kernels that carry both)?  Walking together pays off when the rays
// run side by side: every live ray is compared with the first live one (origins as given by the caller, not advanced
// along the ray).
__device__ __forceinline__ bool rays_run_together(F3 o, F3 d, bool active, float max_abs) {
    const uint64_t live = wave_ballot(active);
    if (live == 0ull) return true;
    const int lead = __builtin_ctzll(live);
    const F3 o0 = f3(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(o.x), lead)),
                     __int_as_float(__builtin_amdgcn_readlane(__float_as_int(o.y), lead)),
                     __int_as_float(__builtin_amdgcn_readlane(__float_as_int(o.z), lead)));
    const F3 d0 = f3(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(d.x), lead)),
                     __int_as_float(__builtin_amdgcn_readlane(__float_as_int(d.y), lead)),
                     __int_as_float(__builtin_amdgcn_readlane(__float_as_int(d.z), lead)));
    const float dd = __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(d.x - d0.x), __builtin_fabsf(d.y - d0.y)),
                                     __builtin_fabsf(d.z - d0.z));
    const float od = __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(o.x - o0.x), __builtin_fabsf(o.y - o0.y)),
                                     __builtin_fabsf(o.z - o0.z));
    const float dl = __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(d0.x), __builtin_fabsf(d0.y)),
                                     __builtin_fabsf(d0.z));
    const bool apart = active && (!(dd <= kPacketDirSpread * dl) || !(od <= kPacketOrgSpread * max_abs));
    return wave_ballot(apart) == 0ull;
}

// `bw`: the bundle walk's state (forward), carried from chunk to chunk of a bounce.
template <bool BWD, bool MIXED, bool SHELF, bool HAND>
__device__ __forceinline__ void wave_knn(const DstAccelView &acc, float max_abs, F3 ro, F3 o, F3 d, float pay, bool active,
                                         KBuf &buf, uint32_t &cnt, bool as_packet, BundleWalk &bw, uint32_t *shelf
#ifdef DST_STATS
                                         , WaveStats &ws
#endif
) {
    const uint64_t live = wave_ballot(active);
    if (live == 0ull) return;
    if (MIXED && !as_packet) {
        const RaySlab slab = make_slab(o, d, max_abs);
        KBuf mine = buf;   // a copy the call may keep in memory; the caller's buffer stays in registers
        uint32_t n = cnt;
        // forward kernels (one wave per workgroup, no other LDS) give the walk an LDS shelf for its stacks
        const LaneWalkAccel view = {acc.leaves, acc.wide, acc.n_leaves, acc.root};
        lane_walk(view, slab, o, d, active, mine, n, SHELF ? shelf : nullptr);
        buf = mine;
        cnt = n;
        return;
    }
    if constexpr (!BWD) {
        bundle_knn<HAND>(acc, max_abs, ro, o, d, pay, active, buf, cnt, bw WSP);
    } else {
        // The walk assumes one set of direction signs per packet (the near face of every box is then the same for
        // all lanes).  A wave whose rays straddle an axis plane (about 1 % of the tiles of a pinhole image) is
        // walked once per sign class present, each time with the lanes of that class only.
        const RaySlab slab = make_slab(o, d, max_abs);
        const uint32_t my_sgn = (slab.ix < 0.f ? 1u : 0u) | (slab.iy < 0.f ? 2u : 0u) | (slab.iz < 0.f ? 4u : 0u);
        uint64_t todo = live;
        while (todo != 0ull) {
            const uint32_t sgn = __builtin_amdgcn_readlane(my_sgn, __builtin_ctzll(todo));
            const bool mine = active && my_sgn == sgn;
            todo &= ~wave_ballot(mine);
            packet_walk(acc, slab, sgn, o, d, mine, buf, cnt WSP);
        }
    }
}

__device__ __forceinline__ void aadd(float *p, float v) { unsafeAtomicAdd(p, v); }

// ---- per-block gradient table (backward) ---------------------------------------------------------------
// The 16x16 pixel tile of a block keeps hitting the same few hundred surfels, so the per-surfel gradients
// are first summed in an LDS hash table (one row of columns per surfel, LDS atomics) and written to
// global memory once per surfel and block when the block ends.  A surfel that finds no free row within a
// few probes goes straight to global atomics, so the table can never be wrong, only less effective.
#ifndef DST_TABLE_FLUSH_NUM
#define DST_TABLE_FLUSH_NUM 2   // the table is emptied between rounds once this many eighths of its rows are in use
                                // (a fuller table sends more hits past it, straight to memory.  Replay at 2 / 3 / 5 / 7
                                // eighths: 1080p room 5.11 / 5.20 / 5.35 / 5.66 ms, 800x800 sphere 1.38 / 1.37 / 1.36 / 1.40,
                                // two reflections 8.52 / 8.66 / 9.32 / 11.25)
#endif
constexpr uint32_t kEmptyKey = 0xFFFFFFFFu;
// Row columns: colour 0-2, opacity 3, scales 4-5, rotation 6-9, mean 10-12, densification mean 13-15, SH coefficient
// j channel c at 16+16c+j (16..63: what sixteen lanes add together lies together), aux 64..64+AUXM-1.
constexpr int kColColor = 0, kColOpac = 3, kColScale = 4, kColRot = 6, kColMean = 10, kColGrad = 13, kColSh = 16,
              kColAux = 64;
// The sums are doubles (deterministic mode: 64-bit fixed point).  Not for their precision: an LDS addition of floats
// takes its lanes one after the other (measured: 3 cycles a lane, 192 for a wave, whatever the addresses), one of
// doubles or of integers takes 8.
template <int AUXM> struct RowLayout {
    static constexpr int cols = kColAux + AUXM;
    static constexpr int stride = cols | 1;     // 8-byte words of a table row; odd: rows spread over all LDS banks
    // A wave's staging area in words: a hit's columns (GradSink), or sixteen sums a channel of four rays (row.inc).
    static constexpr int stage = DST_WAVE * 17 > 4 * (7 + AUXM) * 20 ? DST_WAVE * 17 : 4 * (7 + AUXM) * 20;
    // Rows of the block's table, and behind them one for each row of sixteen lanes that takes what belongs nowhere: what
    // DST_BWD_WAVES blocks (two: 112 rows with two auxiliary channels) leave each other of a CU's 160 KB, which is given out
    // in pieces of 1280 bytes.
    static constexpr int spare = 4;
    static constexpr int rows = (((128 / DST_BWD_WAVES) * 1280 - kWavesPerBlock * stage * 4 - 1024) / (8 * stride) - spare) / 4 * 4;
    static constexpr int words = (rows + spare) * stride;
    // Where column `col` of surfel g lies in the caller's rows of P surfels: 64 columns a row, so that the sixteen lanes of
    // an addition share a cache line of 64 bytes, and the auxiliary channels behind all of them.
    static __device__ __forceinline__ size_t word(int32_t P, uint32_t g, int col) {
        return col < kColAux ? (size_t)g * kColAux + col : (size_t)P * kColAux + (size_t)g * AUXM + (col - kColAux);
    }
};

// ---- deterministic mode: sums in 64-bit fixed point ------------------------------------------------------
// Integer addition is exact, so a sum of fixed-point numbers does not depend on the order of its terms: every
// atomically accumulated value (LDS table, global memory) is converted first.  2^-36 units for the geometric
// columns (scale, rotation, mean, densification: range +-6.7e7), 2^-40 for the others and for the blending
// weights (+-4.2e6); a value outside the range saturates.  The closing kernels count the sums they find in the outer
// half of the range (one saturated term puts a sum there), so that a scene too large for the mode is noticed.
constexpr int kDetShiftGeo = 36, kDetShiftOther = 40;
__device__ __forceinline__ bool det_out_of_range(long long q) { return q >= (1LL << 61) || q <= -(1LL << 61); }
__device__ __forceinline__ int det_shift(int col) { return (col >= kColScale && col < kColSh) ? kDetShiftGeo : kDetShiftOther; }
__device__ __forceinline__ long long to_fixed(float v, int shift) {
    float x = __builtin_ldexpf(v, shift);                       // exact scaling
    x = __builtin_fminf(__builtin_fmaxf(x, -4.6e18f), 4.6e18f);   // |x| < 2^62; NaN becomes a bound
    return (long long)x;
}
__device__ __forceinline__ float from_fixed(long long q, int shift) { return (float)__builtin_ldexp((double)q, -shift); }

// (P: DstParams, wherever it lies.)
// Address in the caller's gradient tensors of column `col` of surfel g (nullptr: nothing to write).
template <int AUXM, class P>
__device__ __forceinline__ float *tensor_address(const P &p, uint32_t g, int col) {
    if (col < kColOpac) return p.dL_dcolors + 3 * (size_t)g + col;
    if (col < kColScale) return p.dL_dopacities + g;
    if (col < kColRot) return p.dL_dscales + 2 * (size_t)g + (col - kColScale);
    if (col < kColMean) return p.dL_drotations + 4 * (size_t)g + (col - kColRot);
    if (col < kColGrad) return p.dL_dmeans3D + 3 * (size_t)g + (col - kColMean);
    if (col < kColSh) return p.dL_dgrads3D + 3 * (size_t)g + (col - kColGrad);
    if (col >= kColAux) {
        const int ch = col - kColAux;
        return (p.others_precomp != nullptr && ch < p.aux) ? p.dL_dothers + (size_t)p.aux * g + ch : nullptr;
    }
    const int c = (col - kColSh) >> 4, j = (col - kColSh) & 15;
    return (p.colors_precomp == nullptr && j < p.M) ? p.dL_dshs + (size_t)g * p.M * 3 + 3 * j + c : nullptr;
}
// Is column `col` in use?  (no auxiliary input: no aux columns; colours given: no SH columns; SH degree < 3: fewer)
template <int AUXM, class P>
__device__ __forceinline__ bool column_live(const P &p, int col) {
    if (col < kColSh) return true;
    if (col >= kColAux) return p.others_precomp != nullptr && col - kColAux < p.aux;
    return p.colors_precomp == nullptr && ((col - kColSh) & 15) < p.M;
}
// Where the kernels add column `col` of surfel g: the row of g in the caller's gradient rows if there are any
// (all columns of a surfel side by side; a closing kernel adds the rows to the tensors), else the tensors.
template <int AUXM, class P>
__device__ __forceinline__ float *grad_address(const P &p, uint32_t g, int col) {
    if (p.grad_rows == nullptr) return tensor_address<AUXM>(p, g, col);
    return column_live<AUXM>(p, col) ? p.grad_rows + RowLayout<AUXM>::word(p.P, g, col) : nullptr;
}

// Sum of v over the 64 lanes; every lane must be active.
__device__ __forceinline__ float wave_sum_f32(float v) {
#define DST_DPP_ADD(ctrl, rmask)                                                                              \
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, rmask, 0xf, true))
    DST_DPP_ADD(0x111, 0xf);   // row_shr:1
    DST_DPP_ADD(0x112, 0xf);   // row_shr:2
    DST_DPP_ADD(0x114, 0xf);   // row_shr:4
    DST_DPP_ADD(0x118, 0xf);   // row_shr:8   -> lane 15 of each row holds the row total
    DST_DPP_ADD(0x142, 0xa);   // row_bcast:15 into rows 1 and 3
    DST_DPP_ADD(0x143, 0xc);   // row_bcast:31 into rows 2 and 3 -> lane 63 holds the wave total
#undef DST_DPP_ADD
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));   // the builtin moves bits of an int
}

// base[key] += v for every lane with `on`, wave-uniform call.  Neighbouring rays mostly composite the same surfel
// in the same step, and atomics of one instruction to one address are served one after the other, so the lanes
// of the most frequent keys are summed across the wave and their first lane adds the total.
__device__ __forceinline__ void wave_add_grouped(float *base, unsigned long long *det, bool on, uint32_t key, float v) {
    auto add = [&](uint32_t k, float x) {
        if (det != nullptr) atomicAdd(det + k, (unsigned long long)to_fixed(x, kDetShiftOther));
        else aadd(base + k, x);
    };
    const uint32_t lane = __lane_id();
    uint64_t rem = wave_ballot(on);
#pragma unroll 1
    for (int tries = 0; tries < 6 && rem != 0ull; ++tries) {
        const int first = __builtin_ctzll(rem);
        const uint32_t k0 = __builtin_amdgcn_readlane(key, first);
        const bool same = on && key == k0;
        const uint64_t grp = wave_ballot(same);
        if (__popcll(grp) >= 3) {
            const float s = wave_sum_f32(same ? v : 0.f);
            if (lane == (uint32_t)first) add(k0, s);
            on = on && !same;
        }
        rem &= ~grp;
    }
    if (on) add(key, v);
}

// The blending weights of an image wave (forward, training): a wave composites the same two hundred or so surfels over
// and over (64 neighbouring rays, some 37 hits each), so their weights are first summed in a small hash table in LDS
// (surfel id -> running sum, LDS atomics on doubles: those on floats take a lane at a time) and go to memory once per surfel and wave when the wave ends - a sixteenth of
// the global atomics.  A surfel that finds no slot within a few probes adds straight to memory.
constexpr int kWetSlotsLog2 = 8, kWetSlots = 1 << kWetSlotsLog2, kWetProbes = 4;
__device__ __forceinline__ void wet_add(uint32_t *keys, double *vals, float *a_weights, bool on, uint32_t g, float w) {
    if (!on) return;
    uint32_t slot = (g * 2654435761u) >> (32 - kWetSlotsLog2);
#pragma unroll 1
    for (int probe = 0; probe < kWetProbes; ++probe) {
        uint32_t k = __hip_atomic_load(keys + slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (k == 0xFFFFFFFFu) {
            uint32_t expected = 0xFFFFFFFFu;
            __hip_atomic_compare_exchange_strong(keys + slot, &expected, g, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_WORKGROUP);
            k = expected == 0xFFFFFFFFu ? g : expected;
        }
        if (k == g) {
            __hip_atomic_fetch_add(vals + slot, (double)w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            return;
        }
        slot = (slot + 1u) & (uint32_t)(kWetSlots - 1);
    }
    aadd(a_weights + g, w);
}

// Find or claim the table row of surfel g; -1 if none is free where it looks.  keys[rows] counts the rows claimed since
// the table was last emptied.  The rows are looked at four at a time, in the two groups that the surfel may lie in: two trips
// to LDS, and one more for a claim.  (Figures: table_flush.)
template <int ROWS>
__device__ __forceinline__ int table_slot(uint32_t *keys, uint32_t g) {
    static_assert(ROWS % 4 == 0, "groups of four rows");
    uint32_t group = __umulhi(g * 2654435761u, (uint32_t)ROWS / 4u);
#pragma unroll 1
    for (int look = 0; look < 2; ++look) {
        const lds_u32 at = (lds_u32)keys + 4u * group;
#pragma unroll 1
        for (;;) {
            typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
            const u32x4 k = *(volatile __attribute__((address_space(3))) u32x4 *)at;
            // the place of the surfel, or of the first free row (rows fill up from the front, so it lies behind all others)
            const uint32_t j = (k.x == g || k.x == kEmptyKey) ? 0u : (k.y == g || k.y == kEmptyKey) ? 1u : (k.z == g || k.z == kEmptyKey) ? 2u : 3u;
            const uint32_t found = j == 0u ? k.x : j == 1u ? k.y : j == 2u ? k.z : k.w;
            if (found == g) return (int)(4u * group + j);
            if (found != kEmptyKey) break;   // a full group
            uint32_t expected = kEmptyKey;
            __hip_atomic_compare_exchange_strong((uint32_t *)(at + j), &expected, g, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_WORKGROUP);
            if (expected == kEmptyKey) {
                __hip_atomic_fetch_add(keys + ROWS, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                return (int)(4u * group + j);
            }
            if (expected == g) return (int)(4u * group + j);   // (another lane's claim; otherwise a row fewer is free: again)
        }
        group = group + 1u == (uint32_t)ROWS / 4u ? 0u : group + 1u;
    }
    return -1;
}

// The SH basis in direction d up to degree `deg`, zero beyond (gradient algebra; reference backward.cu:68-166).
__device__ __forceinline__ void sh_basis(int deg, F3 d, float (&basis)[16]) {
#pragma clang fp contract(fast)
    const float x = d.x, y = d.y, z = d.z;
#pragma unroll
    for (int j = 0; j < 16; ++j) basis[j] = 0.f;
    basis[0] = SH0;
    if (deg > 0) {
        basis[1] = -SH1 * y;
        basis[2] = SH1 * z;
        basis[3] = -SH1 * x;
        if (deg > 1) {
            const float xx = x * x, yy = y * y, zz = z * z, xy = x * y, yz = y * z, xz = x * z;
            basis[4] = SH2[0] * xy;
            basis[5] = SH2[1] * yz;
            basis[6] = SH2[2] * (2.f * zz - xx - yy);
            basis[7] = SH2[3] * xz;
            basis[8] = SH2[4] * (xx - yy);
            if (deg > 2) {
                basis[9] = SH3[0] * y * (3.f * xx - yy);
                basis[10] = SH3[1] * xy * z;
                basis[11] = SH3[2] * y * (4.f * zz - xx - yy);
                basis[12] = SH3[3] * z * (2.f * zz - 3.f * xx - 3.f * yy);
                basis[13] = SH3[4] * x * (4.f * zz - xx - yy);
                basis[14] = SH3[5] * z * (xx - yy);
                basis[15] = SH3[6] * x * (xx - 3.f * yy);
            }
        }
    }
}

// Value of lane m of this lane's row of sixteen.
template <int M>
__device__ __forceinline__ uint32_t row_bcast(uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x150 + M, 0xf, 0xf, true); }
template <int M>
__device__ __forceinline__ float row_bcast(float v) { return __uint_as_float(row_bcast<M>(__float_as_uint(v))); }

// One hit's columns to memory, for the lanes with `on`: lane%16 has the geometric column of that number and the three
// channels of that SH coefficient.  The slow way, column by column: for the
// deterministic mode, and for callers without gradient rows.
template <int AUXM, bool DET>
__device__ __attribute__((noinline)) void put_columns(const DstParams *p_in, uint32_t g, bool on, float geo, F3 sh) {
    const DstParams &p = *uniform_ptr(p_in);
    const int i = (int)(__lane_id() & 15u);
    auto put = [&](int col, float v) {
        if (DET) {
            if (column_live<AUXM>(p, col))
                atomicAdd(p.det_workspace + RowLayout<AUXM>::word(p.P, g, col), (unsigned long long)to_fixed(v, det_shift(col)));
        } else {
            float *dst = grad_address<AUXM>(p, g, col);
            if (dst != nullptr) aadd(dst, v);
        }
    };
    if (!on) return;
    if (geo != 0.f) put(i, geo);
    if (sh.x != 0.f) put(kColSh + i, sh.x);
    if (sh.y != 0.f) put(kColSh + 16 + i, sh.y);
    if (sh.z != 0.f) put(kColSh + 32 + i, sh.z);
}

// Where one step's per-surfel gradients go: into the block's table, row of the hit's surfel, columns 0..15 geometry,
// 16..63 SH (basis_j(ray) * colour gradient_c), 64.. auxiliary channels.  A row of sixteen lanes takes the hits of its
// own sixteen rays one after the other, a lane per column (and per SH coefficient): four hits at a time, sixteen
// rounds.  The geometric columns come through LDS ([ray][column], an odd stride); the basis belongs to the ray, so
// each lane keeps its coefficient's values for its row's sixteen rays in registers for the whole bounce, and the hit's
// colour gradient is broadcast along the row by the multiplication itself.  Hits of the same surfel meet in the LDS
// atomics, and it does not matter how many different surfels a step composites.
// (Before, the lanes of a surfel were summed by matrix products over up to sixteen groups a step, the 64 columns staged
// in LDS.  Grouping cost more than it saved: a step of these scenes composites 6 to 20 different surfels, over half the
// steps of two of them more than sixteen, and what did not fit went column by column.)
constexpr int kGeoCols = 16;
template <int AUXM, bool DET>
struct GradSink {
    // basis value of this lane's coefficient for ray M of its row (rows of one ray: the same for all)
    template <int M> static __device__ __forceinline__ float basis_of(const float (&b)[16]) { return b[M]; }
    template <int M> static __device__ __forceinline__ float basis_of(const float &b) { return b; }
    static constexpr int stride = kGeoCols + 1;   // four rays sixteen apart start in different quarters of the banks
    static constexpr int words = DST_WAVE * stride;
    static_assert(words <= RowLayout<AUXM>::stage, "the table's size counts on the staging areas'");
    double *rows;        // the block's table; the rows behind it take what belongs nowhere
    float *stage;        // this wave's staging area
    bool did;            // this lane composited a hit in this step
    uint32_t g;          // its surfel
    int own_slot;        // table row of g, -1: none
    uint64_t wt;         // wave-uniform: lanes whose surfel has no table row (their values go to global memory)

    __device__ __forceinline__ void plan(uint32_t *keys) {
        own_slot = did ? table_slot<RowLayout<AUXM>::rows>(keys, g) : -1;
        wt = wave_ballot(did && own_slot < 0);
    }
    // Column `col` of this lane's hit (every lane; a lane without a hit may pass anything).
    __device__ __forceinline__ void set(int col, float v) const { stage[__lane_id() * stride + col] = v; }

    // v into word `at` of the table's memory; into the word at LDS address `at`.
    __device__ __forceinline__ void put(uint32_t at, int shift, float v) const { put_at((uint32_t)(uintptr_t)(lds_f64)rows + 8u * at, shift, v); }
    static __device__ __forceinline__ void put_at(uint32_t at, int shift, float v) {
        double *const dst = (double *)(lds_f64)at;
        if (DET) __hip_atomic_fetch_add(reinterpret_cast<long long *>(dst), to_fixed(v, shift), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        else __hip_atomic_fetch_add(dst, (double)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }

    // The hits of ray M of each row, a column per lane: `slot` is each ray's table row, `column` this lane's place in a row, both
    // in bytes.  Twelve instructions and no mask: with two waves on a SIMD a wave issues one in five cycles or so, whatever it
    // is, and sixteen rounds a step were two fifths of the replay's time.  (Rows without a hit masked out, reads between the
    // additions: 1080p room 5619 -> 5101 us, 800x800 sphere 1478 -> 1458, two reflections 8748 -> 8790.)
    template <int M, bool SH, class B>
    static __device__ __forceinline__ void round(uint32_t slot, uint32_t column, float geo, const B &basis, F3 gc) {
        const uint32_t at = row_bcast<M>(slot) + column;
        put_at(at, geo_shift(), geo);
        if (SH) {
            const float b = basis_of<M>(basis);
            put_at(at + 8u * kColSh, kDetShiftOther, row_bcast<M>(gc.x) * b);
            put_at(at + 8u * kColSh + 128u, kDetShiftOther, row_bcast<M>(gc.y) * b);
            put_at(at + 8u * kColSh + 256u, kDetShiftOther, row_bcast<M>(gc.z) * b);
        }
    }
    static __device__ __forceinline__ int geo_shift() { return DET ? det_shift((int)(__lane_id() & 15u)) : 0; }
    template <bool SH, class B>
    __device__ __forceinline__ void rounds(uint32_t slot, uint32_t column, const float (&geo)[16], const B &basis, F3 gc) const {
        round<0, SH>(slot, column, geo[0], basis, gc); round<1, SH>(slot, column, geo[1], basis, gc);
        round<2, SH>(slot, column, geo[2], basis, gc); round<3, SH>(slot, column, geo[3], basis, gc);
        round<4, SH>(slot, column, geo[4], basis, gc); round<5, SH>(slot, column, geo[5], basis, gc);
        round<6, SH>(slot, column, geo[6], basis, gc); round<7, SH>(slot, column, geo[7], basis, gc);
        round<8, SH>(slot, column, geo[8], basis, gc); round<9, SH>(slot, column, geo[9], basis, gc);
        round<10, SH>(slot, column, geo[10], basis, gc); round<11, SH>(slot, column, geo[11], basis, gc);
        round<12, SH>(slot, column, geo[12], basis, gc); round<13, SH>(slot, column, geo[13], basis, gc);
        round<14, SH>(slot, column, geo[14], basis, gc); round<15, SH>(slot, column, geo[15], basis, gc);
    }
    // The same for those among them that have no place in the table: to memory.
    template <int M, class B>
    __device__ __forceinline__ void past(const_params p, uint32_t ray0, const B &basis, F3 gc, bool sh) const {
        if (((wt >> M) & 0x0001000100010001ull) == 0ull) return;
        const uint32_t i = __lane_id() & 15u;
        const float geo = stage[ray0 + M * stride], b = basis_of<M>(basis);
        const float x = row_bcast<M>(gc.x) * b, y = row_bcast<M>(gc.y) * b, z = row_bcast<M>(gc.z) * b;
        const uint32_t gm = row_bcast<M>(g);
        const bool on = ((wt >> ((__lane_id() & 48u) + M)) & 1ull) != 0ull;
        float *const grad_rows = p->grad_rows;
        if (DET || grad_rows == nullptr) {
            put_columns<AUXM, DET>((const DstParams *)p, gm, on, geo, sh ? f3(x, y, z) : f3(0, 0, 0));
        } else if (on) {
            float *dst = grad_rows + (size_t)gm * kColAux + i;
            aadd(dst, geo);
            if (sh) {
                aadd(dst + kColSh, x);
                aadd(dst + kColSh + 16, y);
                aadd(dst + kColSh + 32, z);
            }
        }
    }

    // After the columns: everything into the table.  Wave-uniform call.
    template <class B>
    __device__ __forceinline__ void commit(const_params p, const B &basis, F3 gc, bool sh, bool aux, const float (&aux_v)[AUXM]) const {
        const uint32_t lane = __lane_id();
        const uint32_t slot = (own_slot >= 0 ? (uint32_t)own_slot : (uint32_t)RowLayout<AUXM>::rows + (lane >> 4)) * RowLayout<AUXM>::stride;
        const uint32_t ray0 = (lane & 48u) * stride + (lane & 15u);
        if (did && own_slot < 0 && p->grad_touched != nullptr) p->grad_touched[g] = 1u;   // (the table's flush marks its own)
        // All columns are read before the first addition: LDS answers in order, and a read between two rounds would wait for
        // the additions of the round before it.
        float geo[16];
#pragma unroll
        for (int m = 0; m < 16; ++m) geo[m] = stage[ray0 + m * stride];
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t column = (uint32_t)(uintptr_t)(lds_f64)rows + 8u * (lane & 15u);
        if (sh) rounds<true>(8u * slot, column, geo, basis, gc);
        else rounds<false>(8u * slot, column, geo, basis, gc);
        if (wt != 0ull) {
            past<0>(p, ray0, basis, gc, sh); past<1>(p, ray0, basis, gc, sh); past<2>(p, ray0, basis, gc, sh); past<3>(p, ray0, basis, gc, sh);
            past<4>(p, ray0, basis, gc, sh); past<5>(p, ray0, basis, gc, sh); past<6>(p, ray0, basis, gc, sh); past<7>(p, ray0, basis, gc, sh);
            past<8>(p, ray0, basis, gc, sh); past<9>(p, ray0, basis, gc, sh); past<10>(p, ray0, basis, gc, sh); past<11>(p, ray0, basis, gc, sh);
            past<12>(p, ray0, basis, gc, sh); past<13>(p, ray0, basis, gc, sh); past<14>(p, ray0, basis, gc, sh); past<15>(p, ray0, basis, gc, sh);
        }
        if (aux) {   // the few auxiliary channels ray by ray; past the table, a ray's channels together
            if (own_slot >= 0) {
#pragma unroll
                for (int ch = 0; ch < AUXM; ++ch) put(slot + kColAux + ch, kDetShiftOther, aux_v[ch]);
            }
            if (wt != 0ull) {
#pragma unroll
                for (int ch = 0; ch < AUXM; ++ch) set(ch, aux_v[ch]);
                constexpr uint32_t kRays = DST_WAVE / AUXM;   // rays a round takes
                const uint32_t ch = lane % AUXM, k = lane / AUXM;
                uint64_t m = wt;
#pragma unroll 1
                while (m != 0ull) {
                    // lane's ray: the k-th of those left
                    uint64_t mine = m;
                    for (uint32_t q = 0; q < kRays - 1u; ++q)
                        if (q < k) mine &= mine - 1ull;
                    const int src = mine != 0ull ? __builtin_ctzll(mine) : -1;
                    const uint32_t gs = (uint32_t)__builtin_amdgcn_ds_bpermute((src & 63) << 2, (int)g);
                    const float v = stage[(src & 63) * stride + ch];
                    if (src >= 0 && (int)ch < p->aux && v != 0.f) {
                        if (DET) atomicAdd(p->det_workspace + RowLayout<AUXM>::word(p->P, gs, kColAux + (int)ch), (unsigned long long)to_fixed(v, kDetShiftOther));
                        else aadd(p->grad_rows != nullptr ? p->grad_rows + RowLayout<AUXM>::word(p->P, gs, kColAux + (int)ch)
                                                          : p->dL_dothers + (size_t)p->aux * gs + ch, v);
                    }
                    for (uint32_t q = 0; q < kRays; ++q) m &= m - 1ull;
                }
            }
        }
    }
};
// The basis values as GradSink wants them: basis[m] = coefficient lane%16 of ray m of this lane's row.  Once per bounce;
// `stage` is free then.
template <int STRIDE>
__device__ __forceinline__ void sh_operand(float *stage, int deg, F3 rd, float (&basis)[16]) {
    float b[16];
    sh_basis(deg, rd, b);
    const uint32_t lane = __lane_id();
#pragma unroll
    for (int j = 0; j < 16; ++j) stage[lane * STRIDE + j] = b[j];
#pragma unroll
    for (int m = 0; m < 16; ++m) basis[m] = stage[((lane & 48u) + m) * STRIDE + (lane & 15u)];
}

template <int AUXM>
struct BounceIn {  // backward: saved results of the bounce and the gradients flowing into them
    float rgb[3], dpt, acc, nrm[3], aux[AUXM];
    float g_rgb[3], g_dpt, g_acc, g_nrm[3], g_aux[AUXM];
};

template <int AUXM>
struct BounceAcc {
    float C[3], D, N[3], O[AUXM], T;
};

// The SH colour's derivative with respect to the direction it was evaluated for, contracted with the colour
// gradient gc (backward.cu:100-165).
struct LastShHit {
    int g; F3 gc; bool any;
#ifdef DST_STATS
    unsigned long long t0, t_alg, t_sh;
#endif
};
template <class SH>
__device__ __forceinline__ F3 sh_direction_gradient(int deg, const SH &sh, F3 rd, F3 gc) {
#pragma clang fp contract(fast)
    auto S = [&](int j) { return f3(sh(3 * j), sh(3 * j + 1), sh(3 * j + 2)); };
    F3 ddx = f3(0, 0, 0), ddy = f3(0, 0, 0), ddz = f3(0, 0, 0);
    const float x = rd.x, y = rd.y, z = rd.z;
    if (deg > 0) {
        ddx = -SH1 * S(3);
        ddy = -SH1 * S(1);
        ddz = SH1 * S(2);
        if (deg > 1) {
            const float xx = x * x, yy = y * y, zz = z * z, xy = x * y, yz = y * z, xz = x * z;
            ddx = ddx + SH2[0] * y * S(4) + SH2[2] * 2.f * -x * S(6) + SH2[3] * z * S(7) + SH2[4] * 2.f * x * S(8);
            ddy = ddy + SH2[0] * x * S(4) + SH2[1] * z * S(5) + SH2[2] * 2.f * -y * S(6) + SH2[4] * 2.f * -y * S(8);
            ddz = ddz + SH2[1] * y * S(5) + SH2[2] * 4.f * z * S(6) + SH2[3] * x * S(7);
            if (deg > 2) {
                ddx = ddx + (SH3[0] * 6.f * xy) * S(9) + (SH3[1] * yz) * S(10) + (SH3[2] * -2.f * xy) * S(11) +
                      (SH3[3] * -6.f * xz) * S(12) + (SH3[4] * (-3.f * xx + 4.f * zz - yy)) * S(13) +
                      (SH3[5] * 2.f * xz) * S(14) + (SH3[6] * 3.f * (xx - yy)) * S(15);
                ddy = ddy + (SH3[0] * 3.f * (xx - yy)) * S(9) + (SH3[1] * xz) * S(10) +
                      (SH3[2] * (-3.f * yy + 4.f * zz - xx)) * S(11) + (SH3[3] * -6.f * yz) * S(12) +
                      (SH3[4] * -2.f * xy) * S(13) + (SH3[5] * -2.f * yz) * S(14) + (SH3[6] * -6.f * xy) * S(15);
                ddz = ddz + (SH3[1] * xy) * S(10) + (SH3[2] * 8.f * yz) * S(11) +
                      (SH3[3] * 3.f * (2.f * zz - xx - yy)) * S(12) + (SH3[4] * 8.f * xz) * S(13) +
                      (SH3[5] * (xx - yy)) * S(14);
            }
        }
    }
    return f3(dot(ddx, gc), dot(ddy, gc), dot(ddz, gc));
}

// What the gradient of a hit needs of its surfel besides the geometry it was evaluated with: the corners of the triangle that
// was hit, and the auxiliary channels.  Callers ask for it together with that geometry, so that it is there in one trip.  (Asked
// for where they were used, two trips later: replay of two reflections 11.7 -> 9.0 ms with eight channels, of a 1080p room
// 6.04 -> 5.81, rows of 131,072 lidar rays 510 -> 467 us.)
template <int AUXM>
struct HitData {
    F3 v[3];
    float others[AUXM];
    __device__ __forceinline__ void fetch(const const_params p, uint32_t pidx, bool on) {
        v[0] = v[1] = v[2] = f3(0, 0, 0);
#pragma unroll
        for (int ch = 0; ch < AUXM; ++ch) others[ch] = 0.f;
        if (!on) return;
        const float *V = p->vertices + (size_t)(pidx >> 1) * 12 + 3u * (pidx & 1u);
        v[0] = ld3(V);
        v[1] = ld3(V + 3);
        v[2] = ld3(V + 6);
        if (p->others_precomp != nullptr) {
            const float *o = p->others_precomp + (size_t)p->aux * (pidx >> 1);
#pragma unroll
            for (int ch = 0; ch < AUXM; ++ch)
                if (ch < p->aux) others[ch] = o[ch];
        }
    }
};

// Gradient of one composited hit (reference backward.cu:528-640 and 201-287, 68-166).
// Pure gradient algebra: nothing here feeds a decision, so contraction is allowed.
template <int AUXM, class SINK, class B>
__device__ __forceinline__ void hit_backward(const const_params p, const BounceIn<AUXM> &in, const BounceAcc<AUXM> &run,
                                             int g, uint32_t pidx, float Tp, float alpha, float G, float w, float dpt,
                                             F3 xyz, const F3 (&R)[3], float u, float v, float sx, float sy, F3 mean,
                                             float q0, float q1, float q2, float q3, float opac, float nsign,
                                             F3 normal, const float (&col)[3], const bool (&neg)[3], F3 ro, F3 rd,
                                             F3 &g_ro, F3 &g_rd,
                                             const SINK &sink, const B &basis, bool did, LastShHit &last, const HitData<AUXM> &hit) {
#pragma clang fp contract(fast)
    // gradient algebra only: divisions become multiplications by a hardware reciprocal (1 ulp)
    const float num = 1.0f - alpha, inv_num = __builtin_amdgcn_rcpf(num);
    const float T_final = 1.0f - in.acc;
    float g_alpha = 0.f;
    float g_col[3], g_aux_w[AUXM];
#pragma unroll
    for (int ch = 0; ch < 3; ++ch) {
        g_col[ch] = in.g_rgb[ch] * w;
        g_alpha += in.g_rgb[ch] * (Tp * col[ch] - (in.rgb[ch] - run.C[ch]) * inv_num);
        g_alpha += in.g_rgb[ch] * p->background[ch] * (-T_final * inv_num);
    }
#pragma unroll
    for (int ch = 0; ch < AUXM; ++ch) g_aux_w[ch] = 0.f;
    if (p->others_precomp != nullptr) {
#pragma unroll
        for (int ch = 0; ch < AUXM; ++ch) {
            if (ch < p->aux) {
                const float o = hit.others[ch];
                g_aux_w[ch] = in.g_aux[ch] * w;
                g_alpha += in.g_aux[ch] * (Tp * o - (in.aux[ch] - run.O[ch]) * inv_num);
            }
        }
    }
    const float g_D = in.g_dpt * w;
    g_alpha += in.g_dpt * (Tp * dpt - (in.dpt - run.D) * inv_num);
    const F3 g_N = f3(in.g_nrm[0] * w, in.g_nrm[1] * w, in.g_nrm[2] * w);
    g_alpha += in.g_nrm[0] * (Tp * normal.x - (in.nrm[0] - run.N[0]) * inv_num) +
               in.g_nrm[1] * (Tp * normal.y - (in.nrm[1] - run.N[1]) * inv_num) +
               in.g_nrm[2] * (Tp * normal.z - (in.nrm[2] - run.N[2]) * inv_num);
    g_alpha += in.g_acc * (Tp - in.acc * inv_num);   // the reference never accumulates W (backward.cu:568)
    const float g_G = g_alpha * opac;
    const float pc = (opac * G) > 0.99f ? 0.0f : 1.0f;

    // triangle that was hit, with its corner coordinates in splat units (backward.cu:583-602)
    const bool second = (pidx & 1u) != 0u;
    const F3 v1 = hit.v[0], v2 = hit.v[1], v3 = hit.v[2];
    const float k = g_G * pc;
    const float gu = k * -G * u, gv = k * -G * v;
    F3 gR[3];
    const F3 rel = xyz - mean;
    const float inv_sx = __builtin_amdgcn_rcpf(sx), inv_sy = __builtin_amdgcn_rcpf(sy);
    gR[0] = (gu * inv_sx) * rel;
    gR[1] = (gv * inv_sy) * rel;
    gR[2] = g_N * nsign;
    float g_sx = k * (G * u * u * inv_sx), g_sy = k * (G * v * v * inv_sy);
    F3 g_mean = k * (G * (R[0] * (u * inv_sx) + R[1] * (v * inv_sy)));
    const F3 g_xyz = (gu * inv_sx) * R[0] + (gv * inv_sy) * R[1];
    const float g_d = g_D + dot(g_xyz, rd);
    const F3 n = cross(v2 - v1, v3 - v1);
    const F3 c = v1 - ro;
    const float pp = dot(n, c), q = dot(n, rd), inv_q = __builtin_amdgcn_rcpf(q);
    const F3 g_n = (c - (pp * inv_q) * rd) * inv_q;
    if (did) {
        g_ro = g_ro + (g_xyz + (-g_d * inv_q) * n);
        g_rd = g_rd + (g_xyz * dpt + ((g_d * -pp) * (inv_q * inv_q)) * n);
    }
    // The corner gradients (backward.cu:583-602) are g_v1 = g_d (v2-v3) x g_n + (g_d/q) n, g_v2 = g_d (v3-v1) x g_n,
    // g_v3 = g_d (v1-v2) x g_n, and the corners sit at (+-3, +-3) splat units.  Their sums with those weights are
    // taken on the edge vectors first, where they collapse to one edge each: the three cross products nearly
    // cancel for a long thin quad, and summed after the fact they leave mostly rounding.
    //   sum of the corners' gradients          = (g_d/q) n
    //   weighted by the corners' u coordinates = g_d 6 a x g_n + hu (g_d/q) n
    //   weighted by the corners' v coordinates = g_d 6 b x g_n + hv (g_d/q) n
    // with a = v1-v2, b = v1-v3, (hu,hv) = (-3,3) for the first triangle; a = v3-v2, b = v3-v1, (-3,-3) for the second.
    const F3 g_c = (g_d * inv_q) * n;
    const F3 ea = second ? v3 - v2 : v1 - v2, eb = second ? v3 - v1 : v1 - v3;
    const F3 su = (6.f * g_d) * cross(ea, g_n) - 3.f * g_c;
    const F3 sv = (6.f * g_d) * cross(eb, g_n) + (second ? -3.f : 3.f) * g_c;
    gR[0] = gR[0] + sx * su;
    gR[1] = gR[1] + sy * sv;
    g_sx += dot(R[0], su);
    g_sy += dot(R[1], sv);
    g_mean = g_mean + g_c;
    // rotation: vjp of quat_rows without the normalisation Jacobian (auxiliary.h:433-477)
    float g_rot[4];
    {
        float s = __builtin_amdgcn_rsqf(q3 * q3 + q0 * q0 + q1 * q1 + q2 * q2);
        float w_ = q0 * s, x = q1 * s, y = q2 * s, z = q3 * s;
        float r0 = 2.f * (x * (gR[1].z - gR[2].y) + y * (gR[2].x - gR[0].z) + z * (gR[0].y - gR[1].x));
        float r1 = 2.f * (-2.f * x * (gR[1].y + gR[2].z) + y * (gR[0].y + gR[1].x) + z * (gR[0].z + gR[2].x) +
                          w_ * (gR[1].z - gR[2].y));
        float r2 = 2.f * (x * (gR[0].y + gR[1].x) - 2.f * y * (gR[0].x + gR[2].z) + z * (gR[1].z + gR[2].y) +
                          w_ * (gR[2].x - gR[0].z));
        float r3 = 2.f * (x * (gR[0].z + gR[2].x) + y * (gR[1].z + gR[2].y) - 2.f * z * (gR[0].x + gR[1].y) +
                          w_ * (gR[0].y - gR[1].x));
        g_rot[0] = r0; g_rot[1] = r1; g_rot[2] = r2; g_rot[3] = r3;
    }
    STAT(last.t_alg += __builtin_readcyclecounter() - last.t0; last.t0 = __builtin_readcyclecounter();)
    sink.set(kColColor + 0, g_col[0]); sink.set(kColColor + 1, g_col[1]); sink.set(kColColor + 2, g_col[2]);
    sink.set(kColOpac, g_alpha * G * pc);
    sink.set(kColScale + 0, g_sx);
    sink.set(kColScale + 1, g_sy);
    sink.set(kColRot + 0, g_rot[0]); sink.set(kColRot + 1, g_rot[1]); sink.set(kColRot + 2, g_rot[2]); sink.set(kColRot + 3, g_rot[3]);
    sink.set(kColMean + 0, g_mean.x); sink.set(kColMean + 1, g_mean.y); sink.set(kColMean + 2, g_mean.z);
    const float hd = 0.5f * dpt;
    sink.set(kColGrad + 0, g_mean.x * hd); sink.set(kColGrad + 1, g_mean.y * hd); sink.set(kColGrad + 2, g_mean.z * hd);
    const bool sh = p->colors_precomp == nullptr;
    // SH backward (backward.cu:68-166); the direction gradient REPLACES the ray's (backward.cu:165)
    const F3 gc = f3(neg[0] ? 0.f : g_col[0], neg[1] ? 0.f : g_col[1], neg[2] ? 0.f : g_col[2]);
    sink.commit(p, basis, gc, sh, p->others_precomp != nullptr, g_aux_w);
    STAT(last.t_sh += __builtin_readcyclecounter() - last.t0;)
    if (sh) {
        // The reference overwrites the ray-direction gradient with the SH term at every hit (backward.cu:165), so
        // only the last composited hit's term survives: remember it, walk_bounce computes it once per bounce.
        if (did) {
            last.g = g;
            last.gc = gc;
            last.any = true;
        }
    }
}

// ---- hit record: the forward trace can store every chunk's hit buffer, the backward trace then replays
// them instead of walking the BVH again.  Layout of the caller's buffer, in 8-byte words:
//   [0] blocks requested so far (the forward kernel counts on past the capacity, which is how overflow shows)
//   [1] chains that a replay found broken (stays 0 for a record written by a forward trace with a zeroed header)
//   [2] 0, or the count of pieces of a record written ray by ray (row.inc)
//   [3 ...) directory: one uint32 per (wave, bounce slot): low 26 bits = 1 + first block of that wave's bounce (0 =
//           none), high 6 bits = the number of chunks the wave stored for that bounce (what its replay will cost)
//   then `capacity` blocks of kRecBlockWords words: 16x64 entries ([slot][lane]), 64 uint32 counts, next+1, and
//   the colour of every composited hit as the forward evaluated it ([slot][channel][lane] floats; a channel clamped
//   at zero is stored as -0): the replay then neither gathers nor evaluates the 48 SH coefficients per hit again.
constexpr uint32_t kRecDirBlockBits = 26, kRecDirBlockMask = (1u << kRecDirBlockBits) - 1u;
constexpr uint32_t kRecColourWord = kChunk * DST_WAVE + DST_WAVE / 2 + 8;   // first word of the colours
constexpr uint32_t kRecBlockWords = kRecColourWord + kChunk * 3 * DST_WAVE / 2;
// Are images of this many rays small enough to be traced ray by ray?  (Ray lists, th_log2 < 3, always may be.)
#ifndef DST_ROW_MAX_WAVES
#define DST_ROW_MAX_WAVES 400
#endif
__host__ __device__ static inline bool rows_may_trace(uint64_t rays, int th_log2) {
    return th_log2 < 3 || (rays + 63u) / 64u <= DST_ROW_MAX_WAVES;
}
// Words in front of the first block: the three of the header and the directory, of the wave layout (one entry per wave and
// bounce slot) or, on grids that may be traced ray by ray, of the row layout (one per ray and slot, row.inc) if it is longer;
// behind them, for a list, the order its rays were traced in (a backward trace that made it again spent 0.12 ms on 131,072
// rays).
__host__ __device__ static inline uint64_t record_order_at(uint64_t rays, int th_log2, uint32_t slots, uint64_t waves) {
    const uint64_t entries = (rows_may_trace(rays, th_log2) && rays > waves ? rays : waves) * slots;
    return 3u + ((entries + 1u) / 2u + 1u) / 2u * 2u + 1u;   // even: blocks start on 16-byte boundaries where the record does
}
__host__ __device__ static inline uint64_t record_header_words(uint64_t rays, int th_log2, uint32_t slots, uint64_t waves) {
    return record_order_at(rays, th_log2, slots, waves) + (th_log2 == 0 ? ((rays + 1u) / 2u + 1u) / 2u * 2u : 0u);
}
struct RecView {
    uint64_t *base;      // nullptr: not recording / not replaying
    uint64_t *blocks;    // first block
    uint32_t *dir;       // this wave's directory entries (one per bounce slot)
    uint32_t capacity;
};

// Forward: append one chunk of this wave to the record.  `prev` is the wave's previous block in this bounce.
// Returns where the chunk's colours go (nullptr: the record is full).
__device__ __forceinline__ float *rec_store(const RecView &rv, int bounce, uint32_t &prev, const KBuf &buf, uint32_t cnt) {
    const uint32_t lane = __lane_id();
    uint32_t blk = 0;
    if (lane == 0) blk = (uint32_t)atomicAdd((unsigned long long *)rv.base, 1ull);
    blk = __builtin_amdgcn_readfirstlane(blk);
    if (blk >= rv.capacity || blk >= kRecDirBlockMask) return nullptr;   // too small: the host sees the count and the backward pass re-traces
    uint64_t *b = rv.blocks + (size_t)blk * kRecBlockWords;
#pragma unroll
    for (int k = 0; k < kChunk; ++k) __builtin_nontemporal_store(buf.e[k], b + k * DST_WAVE + lane);
    uint32_t *cnts = reinterpret_cast<uint32_t *>(b + kChunk * DST_WAVE);
    cnts[lane] = cnt;
    if (lane == 0) {
        cnts[DST_WAVE] = 0u;   // next: none yet
        if (prev == 0xFFFFFFFFu) rv.dir[bounce] = blk + 1u;
        else reinterpret_cast<uint32_t *>(rv.blocks + (size_t)prev * kRecBlockWords + kChunk * DST_WAVE)[DST_WAVE] = blk + 1u;
    }
    prev = blk;
    return reinterpret_cast<float *>(b + kRecColourWord);
}

// Backward: locate the next chunk of this wave's bounce; its entries are then read one slot at a time.
// Returns nullptr when the chain ends early.
__device__ __forceinline__ const uint64_t *rec_open(const RecView &rv, uint32_t &cur, uint32_t &cnt) {
    if (cur == 0u || cur > rv.capacity) return nullptr;
    const uint32_t lane = __lane_id();
    const uint64_t *b = rv.blocks + (size_t)(cur - 1u) * kRecBlockWords;
    const uint32_t *cnts = reinterpret_cast<const uint32_t *>(b + kChunk * DST_WAVE);
    cnt = cnts[lane];
    cur = __builtin_amdgcn_readfirstlane(cnts[DST_WAVE]);
    return b;
}

// Block-wide: add the table to the caller's gradients and empty it.  A wave takes a row at a time, a lane per column (the
// 64 columns of a surfel go out as four lines of atomics), and of its rows those alone that are in use.
// (A thread per
// word of all rows, in use or not, and one trip after the other for a claim, table_slot: replay of an 800x800 sphere 1444 -> 1360
// us, rows of 131,072 lidar rays 463 -> 417, of 128x128 rays at a cube 80 -> 73.)  The caller puts barriers around it.
template <int AUXM, bool DET>
__device__ __forceinline__ void table_flush(const DstParams &p, uint32_t *keys, double *rows) {
    constexpr uint32_t stride = RowLayout<AUXM>::stride, n_rows = (uint32_t)RowLayout<AUXM>::rows;
    static_assert(n_rows <= kWavesPerBlock * DST_WAVE, "a wave's rows have a lane each");
    uint32_t lane = threadIdx.x % DST_WAVE;
    const uint32_t wave = uni(threadIdx.x / DST_WAVE);
    asm volatile("" : "+v"(lane));   // (addresses are made here, not in front of the loop that calls this now and then)
    const uint32_t mine = lane * kWavesPerBlock + wave, key = mine < n_rows ? keys[mine] : kEmptyKey;
    const bool live = column_live<AUXM>(p, (int)lane), aux = lane < (uint32_t)AUXM && column_live<AUXM>(p, kColAux + (int)lane);
    auto add = [&](uint32_t g, int col, double v) {
        if (DET) {
            const long long q = __builtin_bit_cast(long long, v);
            if (q != 0) atomicAdd(p.det_workspace + RowLayout<AUXM>::word(p.P, g, col), (unsigned long long)q);
        } else if (v != 0.0) {
            aadd(p.grad_rows != nullptr ? p.grad_rows + RowLayout<AUXM>::word(p.P, g, col) : tensor_address<AUXM>(p, g, col), (float)v);
        }
    };
    uint64_t used = wave_ballot(key != kEmptyKey);
#pragma unroll 1
    while (used != 0ull) {
        const int k = __builtin_ctzll(used);
        used &= used - 1ull;
        const uint32_t g = (uint32_t)__builtin_amdgcn_readlane((int)key, k);
        double *const row = rows + ((uint32_t)k * kWavesPerBlock + wave) * stride;
        const double v = row[lane], x = aux ? row[kColAux + lane] : 0.0;
        row[lane] = 0.0;
        if (aux) row[kColAux + lane] = 0.0;
        if (p.grad_touched != nullptr && lane == 0u) p.grad_touched[g] = 1u;
        if (live) add(g, (int)lane, v);
        if (aux) add(g, kColAux + (int)lane, x);
    }
}
template <int AUXM, bool DET>
__device__ __forceinline__ void table_clear_keys(uint32_t *keys) {
    for (int k = threadIdx.x; k <= RowLayout<AUXM>::rows; k += kWavesPerBlock * DST_WAVE)
        keys[k] = (k < RowLayout<AUXM>::rows) ? kEmptyKey : 0u;
}

// One bounce: chunked 16-nearest traversal + front-to-back compositing (reference forward.cu:136-315),
// and for BWD the per-hit gradients of the re-trace (reference backward.cu:332-655).
// `first_walk` (forward): 0, or the number of steps the bundle walk of the bounce's first chunk may take before the
// wave gives its tile up (returns true, nothing written yet: see the tile hand-over in trace_body), or kWalkPerLane:
// every ray of the wave walks on its own whatever the rays look like (the waves that take such tiles over).
// HAND: kernels without the hand-over do not contain its code at all (first_walk is ignored).
constexpr uint32_t kWalkPerLane = 0xFFFFFFFFu;
// PACK (forward): hits are evaluated from the surfels' records.
template <bool BWD, int AUXM, bool REC, bool MIXED, bool DET, bool HAND, bool PACK>
__device__ __forceinline__ bool walk_bounce(const DstParams &p, const DstAccelView &acc, float max_abs, bool lane_on,
                                            F3 ro, F3 rd, float min_depth, BounceAcc<AUXM> &run,
                                            const BounceIn<AUXM> &in, F3 &g_ro, F3 &g_rd, uint32_t &n_proc,
                                            uint32_t &n_con, uint32_t *tab_keys, double *tab_rows, float *stage,
                                            const RecView &rv, int bounce, F3 &dist_acc, uint32_t first_walk
#ifdef DST_STATS
                                            , WaveStats &ws
#endif
) {
    run.C[0] = run.C[1] = run.C[2] = 0.f;
    run.D = 0.f;
    run.N[0] = run.N[1] = run.N[2] = 0.f;
#pragma unroll
    for (int ch = 0; ch < AUXM; ++ch) run.O[ch] = 0.f;
    float pay_dpt = 0.f, dpt = 0.f, Tp = 1.f, Tn = 1.f;
    int last_g = -1, contrib = 0;
    F3 ot = ro;
    bool live = lane_on;
    KBuf buf;
    LastShHit last_sh = {0, f3(0, 0, 0), false};
    STAT(last_sh.t_alg = 0; last_sh.t_sh = 0;)
    // kernels built without the per-lane walk (MIXED false) walk once for every wave
    const bool as_packet = (!MIXED || (REC && BWD)) ? true
                                                    : (HAND && first_walk == kWalkPerLane ? false : rays_run_together(ro, rd, lane_on, max_abs));
    // Forward: one LDS area per wave serves the bundle walk's lists or the per-lane walk's stack shelf (all chunks of a
    // bounce use the same walk, and a bounce starts without a list).
    constexpr bool SHELF = MIXED && !BWD;
    constexpr uint32_t kWaveLds = BWD ? 1u : (SHELF ? (uint32_t)(kLaneShelf * DST_WAVE) : kBwWords);
    static_assert(kBwWords <= (uint32_t)(kLaneShelf * DST_WAVE), "the lists fit where the shelf is");
    __shared__ uint32_t s_walk[BWD ? 1u : (uint32_t)kFwdWavesPerBlock * kWaveLds];
    uint32_t *const wave_lds = s_walk + (BWD ? 0u : (threadIdx.x / DST_WAVE) * kWaveLds);
    BundleWalk bw;
    bw.lds.base = (lds_u32)wave_lds;
    bw.da = bw.uoff = 0.f;
    bw.kept = bw.spent = false;
    bw.limit = (HAND && first_walk != kWalkPerLane) ? first_walk : 0u;
    uint32_t rec_pos = (REC && BWD) ? (rv.dir[bounce] & kRecDirBlockMask) : 0xFFFFFFFFu;   // replay: next block + 1; record: previous block
    // (the re-tracing kernel, short of registers, brings it into place in every step)
    float basis[16];
    constexpr bool KEEP_BASIS = BWD && REC;
    if (KEEP_BASIS && p.colors_precomp == nullptr) sh_operand<GradSink<AUXM, DET>::stride>(stage, p.D, rd, basis);
    uint32_t rec_chunks = 0u;   // forward with a record: chunks stored for this bounce
    for (;;) {
        // Backward: the four waves of the block take their chunks in step, so that between two rounds nobody
        // touches the gradient table and it can be emptied when it fills up.
        const bool wave_live = wave_ballot(live) != 0ull;
        if (BWD) {
            if (__syncthreads_or(wave_live ? 1 : 0) == 0) break;
        } else if (!wave_live) {
            break;
        }
        if (wave_live) do {
        uint32_t cnt = 0;
        STAT(ws.chunks++; unsigned long long c0 = __builtin_readcyclecounter();)
        // Where the compositing loop below takes its entries from: the recorded block, one slot at a time
        // (backward replay: no buffer registers at all), or the register buffer the traversal just filled.
        const uint64_t *rec_block = nullptr;
        float *rec_colours = nullptr;   // forward with a record: where this chunk's hit colours are kept
        const uint32_t lane_ = __lane_id();
        if (REC && BWD) {
            rec_block = rec_open(rv, rec_pos, cnt);
            if (rec_block == nullptr) {   // cannot happen with a complete record: count it where the caller can see it
                if (lane_ == 0) atomicAdd((unsigned long long *)(rv.base + 1), 1ull);
                live = false;
                break;
            }
        } else {
            kbuf_reset(buf);
            wave_knn<BWD, MIXED, SHELF, HAND>(acc, max_abs, ro, ot, rd, pay_dpt, live, buf, cnt, as_packet, bw, wave_lds WSP);
            if constexpr (HAND) {
                if (bw.spent) return true;   // only a bounce's first walk has a limit: nothing has been written yet
                bw.limit = 0u;
            }
            if (REC && !BWD) {
                rec_colours = rec_store(rv, bounce, rec_pos, buf, cnt);
                rec_chunks += rec_colours != nullptr ? 1u : 0u;
            }
        }
        STAT(unsigned long long c1 = __builtin_readcyclecounter(); ws.t_trav += c1 - c0;)
        int here = 0;
        bool stop = false;
        // Compositing and replay run one step ahead of themselves (room view 3.81 -> 3.64 ms, forward of its training step 4.39 ->
        // 4.20; the kernels with the per-lane walk have no registers left for it).  In the replay the entry of step it+1 is
        // fetched while step it evaluates, and its surfel's geometry while step it does its gradient algebra, so a step
        // starts with its operands in registers instead of two dependent trips to memory; forward, the entry is in a
        // register and the geometry is fetched while step it evaluates.
        constexpr bool AHEAD = (REC && BWD) || (!BWD && !MIXED);
        struct Ahead { uint64_t e; float m[3], s[2], q[4], o, c[3]; v4f w[4]; } nx = {0ull, {0.f, 0.f, 0.f}, {1.f, 1.f}, {1.f, 0.f, 0.f, 0.f}, 0.f, {0.f, 0.f, 0.f}, {}};
        auto fetch_geometry = [&](bool want) {
            const const_params kp = fresh_params();
            if (!want) return;
            if constexpr (PACK) {
                const v4f *w = reinterpret_cast<const v4f *>(reinterpret_cast<const DstSurfel *>(kp->scratch) + (kb_idx(nx.e) >> 1));
#pragma unroll
                for (int k = 0; k < 4; ++k) nx.w[k] = w[k];
                return;
            }
            const size_t gn = (size_t)(kb_idx(nx.e) >> 1);
            nx.m[0] = kp->means3D[3 * gn]; nx.m[1] = kp->means3D[3 * gn + 1]; nx.m[2] = kp->means3D[3 * gn + 2];
            nx.s[0] = kp->scales[2 * gn]; nx.s[1] = kp->scales[2 * gn + 1];
            nx.q[0] = kp->rotations[4 * gn]; nx.q[1] = kp->rotations[4 * gn + 1];
            nx.q[2] = kp->rotations[4 * gn + 2]; nx.q[3] = kp->rotations[4 * gn + 3];
            nx.o = kp->opacities[gn];
        };
        if (REC && BWD) {
            const bool want = live && cnt > 0u;
            if (want) {
                nx.e = __builtin_nontemporal_load(rec_block + lane_);
                const float *cs = reinterpret_cast<const float *>(rec_block + kRecColourWord) + lane_;
                for (int ch = 0; ch < 3; ++ch) nx.c[ch] = __builtin_nontemporal_load(cs + ch * DST_WAVE);
            }
            fetch_geometry(want);
        } else if (AHEAD) {
            nx.e = buf.e[0];
            fetch_geometry(live && cnt > 0u);
        }
#pragma unroll 1
        for (int it = 0; it < kChunk; ++it) {
            const bool on = live && !stop && (uint32_t)it < cnt;
            if (wave_ballot(on) == 0ull) break;
            STAT(if (!BWD) { ws.steps++; ws.t_hb += __popcll(wave_ballot(on)); })
            // next entry in depth order (consumed slots need no reset: the buffer is rebuilt for every chunk)
            uint64_t e;
            Ahead cur = nx;
            const bool want_next = AHEAD && live && it + 1 < kChunk && (uint32_t)(it + 1) < cnt;
            if (REC && BWD) {
                e = cur.e;
                if (want_next) {
                    nx.e = __builtin_nontemporal_load(rec_block + (it + 1) * DST_WAVE + lane_);
                    // (the colour slot of an entry that was not composited holds whatever was there: never used)
                    const float *cs = reinterpret_cast<const float *>(rec_block + kRecColourWord) + (it + 1) * 3 * DST_WAVE + lane_;
                    for (int ch = 0; ch < 3; ++ch) nx.c[ch] = __builtin_nontemporal_load(cs + ch * DST_WAVE);
                }
            } else {
                e = buf.e[0];
#pragma unroll
                for (int k = 0; k < kChunk - 1; ++k) buf.e[k] = buf.e[k + 1];
                if (AHEAD) {
                    nx.e = buf.e[0];
                    fetch_geometry(want_next);
                }
            }
            const float e_t = kb_t(e);
            const uint32_t e_i = kb_idx(e);
            HitData<AUXM> hit;
            if (REC && BWD) hit.fetch(fresh_params(), e_i, on);
            // ---- phase 1 (per lane): evaluate the entry, decide, composite ------------------------------
            bool did = false;          // this lane composited a hit in this iteration
            int g = 0;
            float Tp_hit = 1.f, alpha = 0.f, G = 0.f, w = 0.f, u = 0.f, v = 0.f, sx = 1.f, sy = 1.f, opac = 0.f;
            float nsign = 1.f, q0 = 1.f, q1 = 0.f, q2 = 0.f, q3 = 0.f, dpt_hit = 0.f;
            F3 xyz = f3(0, 0, 0), mean = f3(0, 0, 0), normal = f3(0, 0, 1);
            F3 R[3] = {f3(1, 0, 0), f3(0, 1, 0), f3(0, 0, 1)};
            float col[3] = {0.f, 0.f, 0.f};
            bool neg[3] = {false, false, false};
            const float *sh = nullptr;
            do {
                const const_params kp = fresh_params();
                if (!on) break;
                g = (int)(e_i >> 1);
                if (g == last_g) break;
                dpt = e_t + pay_dpt;
                xyz = f3(ro.x + dpt * rd.x, ro.y + dpt * rd.y, ro.z + dpt * rd.z);
                if (PACK) {
                    R[0] = f3(cur.w[0].x, cur.w[0].y, cur.w[0].z);
                    R[1] = f3(cur.w[1].x, cur.w[1].y, cur.w[1].z);
                    R[2] = f3(cur.w[2].x, cur.w[2].y, cur.w[2].z);
                    opac = cur.w[2].w;
                    sx = cur.w[3].x;
                    sy = cur.w[3].y;
                } else if (AHEAD) {
                    mean = f3(cur.m[0], cur.m[1], cur.m[2]);
                    sx = cur.s[0]; sy = cur.s[1];
                    q0 = cur.q[0]; q1 = cur.q[1]; q2 = cur.q[2]; q3 = cur.q[3];
                } else {
                    mean = ld3(kp->means3D + 3 * (size_t)g);
                    sx = kp->scales[2 * (size_t)g];
                    sy = kp->scales[2 * (size_t)g + 1];
                    const float *qp = kp->rotations + 4 * (size_t)g;
                    q0 = qp[0]; q1 = qp[1]; q2 = qp[2]; q3 = qp[3];
                }
                if (!PACK) quat_rows(q0, q1, q2, q3, R);
                const float tx = PACK ? cur.w[0].w : -dot(R[0], mean), ty = PACK ? cur.w[1].w : -dot(R[1], mean);
                const float ux = R[0].x * xyz.x + R[0].y * xyz.y + R[0].z * xyz.z + tx;
                const float uy = R[1].x * xyz.x + R[1].y * xyz.y + R[1].z * xyz.z + ty;
                u = PACK ? div_by(ux, sx, cur.w[3].z) : ux / sx;
                v = PACK ? div_by(uy, sy, cur.w[3].w) : uy / sy;
                float rho = u * u + v * v;
                if (PACK && !(rho == rho)) {   // out of div_by's range, or no number anyway
                    u = ux / sx;
                    v = uy / sy;
                    rho = u * u + v * v;
                }
                n_proc++;
                normal = R[2];
                const float cosv = -(rd.x * normal.x + rd.y * normal.y + rd.z * normal.z);
                if (cosv == 0.f) break;
                nsign = cosv > 0.f ? 1.0f : -1.0f;
                normal = cosv > 0.f ? normal : -normal;
                if (dpt < min_depth) break;
                const float power = -0.5f * rho;
                if (power > 0.0f) break;
                if (!PACK) opac = AHEAD ? cur.o : kp->opacities[g];
                G = exp_det(power);
                alpha = opac * G;
                alpha = (alpha < 0.99f) ? alpha : 0.99f;
                if (alpha < 1.0f / 255.0f) break;
                Tn = Tp * (1 - alpha);
                if (Tn < kTmin) { stop = true; break; }
                contrib++;
                if (contrib > kMaxContrib) { stop = true; break; }
                last_g = g;
                w = alpha * Tp;
                if (REC && BWD) {   // as the forward trace evaluated it
#pragma unroll
                    for (int ch = 0; ch < 3; ++ch) {
                        col[ch] = cur.c[ch];
                        // -0: clamped (a colour evaluated from SH is never negative; given colours may be)
                        neg[ch] = kp->colors_precomp == nullptr && (__float_as_uint(col[ch]) >> 31) != 0u;
                    }
                } else if (kp->colors_precomp == nullptr) {
                    sh = kp->shs + (size_t)g * kp->M * 3;
                    // (the binary16 source lives in the forward kernels that carry the rarely used options; a backward
                    // trace is given the widened values as shs)
                    const F3 c = (!BWD && DET && (kp->flags & DST_FLAG_SH_HALF)) ? sh_color_half(p, g, rd, neg)
                                                                              : sh_color(kp->D, ShF32{sh}, rd, neg);
                    col[0] = c.x; col[1] = c.y; col[2] = c.z;
                } else {
                    col[0] = kp->colors_precomp[3 * (size_t)g];
                    col[1] = kp->colors_precomp[3 * (size_t)g + 1];
                    col[2] = kp->colors_precomp[3 * (size_t)g + 2];
                }
                if (REC && !BWD && rec_colours != nullptr) {
                    float *cs = rec_colours + it * 3 * DST_WAVE + lane_;
#pragma unroll
                    for (int ch = 0; ch < 3; ++ch) __builtin_nontemporal_store(neg[ch] ? -0.0f : col[ch], cs + ch * DST_WAVE);
                }
                run.C[0] += w * col[0];
                run.C[1] += w * col[1];
                run.C[2] += w * col[2];
                if (kp->others_precomp != nullptr) {
#pragma unroll
                    for (int ch = 0; ch < AUXM; ++ch)
                        if (ch < kp->aux) run.O[ch] += w * ((REC && BWD) ? hit.others[ch] : kp->others_precomp[(size_t)kp->aux * g + ch]);
                }
                if (!BWD && DET && (kp->flags & DST_FLAG_DISTORTION)) {
                    // depth distortion of 2DGS with its running moments (x = distortion, y = M1, z = M2); the
                    // reference declares the three and leaves the computation open (forward.cu:286)
                    const float A_before = 1 - Tp;
                    const float m = kFar / (kFar - kNear) * (1 - kNear / dpt);
                    dist_acc.x += (m * m * A_before + dist_acc.z - 2 * m * dist_acc.y) * w;
                    dist_acc.y += m * w;
                    dist_acc.z += m * m * w;
                }
                run.D += w * dpt;
                run.N[0] += w * normal.x;
                run.N[1] += w * normal.y;
                run.N[2] += w * normal.z;
                n_con++;
                here++;
                did = true;
                Tp_hit = Tp;
                dpt_hit = dpt;
                Tp = Tn;
            } while (false);
            if (REC && BWD) fetch_geometry(want_next);
            const const_params kp = fresh_params();
            if (!BWD && kp->training && kp->a_weights != nullptr) {
                if (!MIXED && !DET) wet_add(tab_keys, tab_rows, kp->a_weights, did, (uint32_t)g, w);   // the wave's LDS table
                else wave_add_grouped(kp->a_weights, (DET && (kp->flags & DST_FLAG_DETERMINISTIC)) ? kp->det_workspace : nullptr, did,
                                      (uint32_t)g, w);
            }
            // ---- phase 2 (whole wave, backward only): gradients of the hits composited above -----------
            if (BWD && wave_ballot(did) != 0ull) {
                GradSink<AUXM, DET> sink;
                sink.rows = tab_rows;
                sink.stage = stage;
                sink.did = did;
                sink.g = (uint32_t)g;
                STAT(unsigned long long d0 = __builtin_readcyclecounter();)
                if (!KEEP_BASIS && p.colors_precomp == nullptr) sh_operand<GradSink<AUXM, DET>::stride>(stage, p.D, rd, basis);
                sink.plan(tab_keys);
                STAT(last_sh.t0 = __builtin_readcyclecounter();)
                if (!REC) hit.fetch(fresh_params(), did ? e_i : 0u, true);
                STAT(unsigned long long d1 = __builtin_readcyclecounter(); ws.t_plan += d1 - d0; ws.steps++;
                     ws.leaf_any += __popcll(wave_ballot(did));)
                hit_backward<AUXM>(fresh_params(), in, run, did ? g : 0, e_i, Tp_hit, alpha, G, w, dpt_hit, xyz, R, u, v, sx, sy, mean,
                                   q0, q1, q2, q3, opac, nsign, normal, col, neg, ro, rd, g_ro, g_rd, sink, basis, did, last_sh, hit);
                STAT(ws.t_hb += __builtin_readcyclecounter() - d1;)
            }
        }
        STAT(ws.t_comp += __builtin_readcyclecounter() - c1;)
        if (live) {
            bool fin = (Tn < kTmin) || (cnt < (uint32_t)kChunk) || (contrib > kMaxContrib);
            const float next_dpt = (float)((double)dpt + kStepEps);
            if (!(next_dpt > pay_dpt) && here == 0) fin = true;   // the reference would never leave this state
            if (fin) {
                live = false;
            } else {
                pay_dpt = next_dpt;
                ot = f3(ro.x + pay_dpt * rd.x, ro.y + pay_dpt * rd.y, ro.z + pay_dpt * rd.z);
            }
        }
        } while (false);
        if (BWD) {
            __syncthreads();   // every wave's additions of this round are in the table
            if (tab_keys[RowLayout<AUXM>::rows] > (uint32_t)(DST_TABLE_FLUSH_NUM * RowLayout<AUXM>::rows / 8)) {
                table_flush<AUXM, DET>(p, tab_keys, tab_rows);
                __syncthreads();
                table_clear_keys<AUXM, DET>(tab_keys);   // the barrier at the top of the next round publishes it
            }
        }
    }
    if (REC && !BWD && rec_chunks != 0u && __lane_id() == 0u)   // the replay's cost of this wave and bounce, for its launcher
        rv.dir[bounce] = (rv.dir[bounce] & kRecDirBlockMask) | (min(rec_chunks, 63u) << kRecDirBlockBits);
    STAT(if (BWD) { ws.nodes += last_sh.t_alg; ws.leaves += last_sh.t_sh; })
    if (BWD && p.colors_precomp == nullptr && last_sh.any)
        g_rd = sh_direction_gradient(p.D, ShF32{p.shs + (size_t)last_sh.g * p.M * 3}, rd, last_sh.gc);
    run.T = Tp;
    return false;
}

__device__ __forceinline__ F3 dnormvdv(F3 v, F3 dv) {
    float sum2 = v.x * v.x + v.y * v.y + v.z * v.z;
    float inv = 1.0f / __builtin_sqrtf(sum2 * sum2 * sum2);
    return f3(((+sum2 - v.x * v.x) * dv.x - v.y * v.x * dv.y - v.z * v.x * dv.z) * inv,
              (-v.x * v.y * dv.x + (sum2 - v.y * v.y) * dv.y - v.z * v.y * dv.z) * inv,
              (-v.x * v.z * dv.x - v.y * v.z * dv.y + (sum2 - v.z * v.z) * dv.z) * inv);
}
__device__ __forceinline__ F3 ddotndndn(F3 n, F3 d, F3 g) {
    float nd = dot(n, d);
    return f3(g.x * (nd + d.x * n.x) + g.y * d.x * n.y + g.z * d.x * n.z,
              g.x * d.y * n.x + g.y * (nd + d.y * n.y) + g.z * d.y * n.z,
              g.x * d.z * n.x + g.y * d.z * n.y + g.z * (nd + d.z * n.z));
}
__device__ __forceinline__ F3 ddotndndd(F3 n, F3 g) {
    return f3(g.x * n.x * n.x + g.y * n.x * n.y + g.z * n.x * n.z, g.x * n.y * n.x + g.y * n.y * n.y + g.z * n.y * n.z,
              g.x * n.z * n.x + g.y * n.z * n.y + g.z * n.z * n.z);
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// Position j in the dispatch order of an image grid -> block (bx, by): column strips `strip` blocks wide, row by row
// inside a strip (strip 0 or a ray list: row-major).  See trace_body for why.
__device__ __forceinline__ void block_of_position(uint32_t j, uint32_t btiles_x, uint32_t rows, uint32_t strip_width,
                                                  bool image, uint32_t &bx, uint32_t &by) {
    bx = j % btiles_x;
    by = j / btiles_x;
    if (strip_width != 0u && image) {
        const uint32_t per_strip = strip_width * rows, strip = j / per_strip, r = j % per_strip;
        if (strip * strip_width < btiles_x) {   // (positions past the grid keep the row-major numbers: their blocks leave)
            const uint32_t w = min(strip_width, btiles_x - strip * strip_width);
            bx = strip * strip_width + r % w;
            by = r / w;
        }
    }
}

// Order of the blocks of a replaying backward trace: longest first.  The forward trace left in the record's directory
// how many chunks every wave stored (what its replay costs); a block takes as long as the longest of its four waves
// (they take their chunks in step).  With the long blocks first, the chip runs out of work with short blocks, not
// with one long block per CU still going.  One workgroup: a counting sort over 64 cost classes, positions taken
// 1024 at a time so that blocks of equal cost keep their neighbourhood.
__global__ __launch_bounds__(1024) void k_block_order(const uint32_t *__restrict__ dir, uint32_t slots, uint32_t btiles_x,
                                                     uint32_t rows, uint32_t strip_width, int image, uint32_t n_blocks,
                                                     uint32_t *__restrict__ order) {
    __shared__ uint32_t s_count[64], s_base[64];
    auto cost_class = [&](uint32_t j) -> uint32_t {   // 0 = the most expensive
        uint32_t bx, by;
        block_of_position(j, btiles_x, rows, strip_width, image != 0, bx, by);
        if (by >= rows) return 63u;
        const uint32_t *d = dir + (size_t)(by * btiles_x + bx) * kWavesPerBlock * slots;
        uint32_t worst = 0u;
        for (uint32_t w = 0; w < (uint32_t)kWavesPerBlock; ++w) {
            uint32_t sum = 0u;
            for (uint32_t k = 0; k < slots; ++k) sum += d[w * slots + k] >> kRecDirBlockBits;
            worst = max(worst, sum);
        }
        return 63u - min(worst, 63u);
    };
    constexpr uint32_t kKept = 32768;   // classes of the first pass kept in LDS for the second (grids up to this size)
    __shared__ uint8_t s_class[kKept];
    if (threadIdx.x < 64) s_count[threadIdx.x] = 0u;
    __syncthreads();
    for (uint32_t j = threadIdx.x; j < n_blocks; j += blockDim.x) {
        const uint32_t c = cost_class(j);
        if (j < kKept) s_class[j] = (uint8_t)c;
        atomicAdd(&s_count[c], 1u);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t run = 0u;
        for (int c = 0; c < 64; ++c) {
            s_base[c] = run;
            run += s_count[c];
        }
    }
    __syncthreads();
    for (uint32_t base = 0; base < n_blocks; base += blockDim.x) {   // in order, 1024 positions at a time
        const uint32_t j = base + threadIdx.x;
        if (j < n_blocks) order[atomicAdd(&s_base[j < kKept ? (uint32_t)s_class[j] : cost_class(j)], 1u)] = j;
        __syncthreads();
    }
}

// Order of the blocks of a forward trace: those that look long first, so that no tile of a millisecond begins when the chip
// is about to run dry.  What a block will cost is guessed from how many leaf groups lie in the way of its rays, from the
// boxes alone: a wave walks down for sixty-four of its 256 rays (the outermost among them) as the tiles' waves will, without
// quads, windows or distances.  A guess that is off costs time and nothing else.  (It goes with the time of the block's longest
// tile at 0.75 to 0.9 on the scenes measured; of an 800x800 sphere's 10,000 tiles the last to begin ran from 0.6 to 1.75 ms.)
constexpr uint32_t kCostMax = 2047u;   // leaf groups counted; a wave stops there
__device__ __forceinline__ uint32_t block_cost(const DstParams &p, const DstAccelView &acc, uint32_t block, uint32_t btiles_x, lds_u32 area) {
    const uint32_t lane = __lane_id(), bx = block % btiles_x, by = block / btiles_x;
    const uint32_t px = 16u * bx + (lane & 7u) * 15u / 7u, py = 16u * by + (lane >> 3) * 15u / 7u;
    const bool inside = px < (uint32_t)p.W && py < (uint32_t)p.H;
    const size_t r = inside ? (size_t)py * p.W + px : 0;
    const F3 o = ld3(p.ray_o + 3 * r), d = ld3(p.ray_d + 3 * r);
    const float dmax = __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(d.x), __builtin_fabsf(d.y)), __builtin_fabsf(d.z));
    const bool usable = inside && (__builtin_fabsf(o.x) + __builtin_fabsf(o.y)) + __builtin_fabsf(o.z) < INFINITY && dmax > 0.f &&
                        (__builtin_fabsf(d.x) + __builtin_fabsf(d.y)) + __builtin_fabsf(d.z) < INFINITY;
    const uint64_t todo = wave_ballot(usable);
    uint32_t count = 0u;
    if (todo != 0ull && !(acc.root & DST_LEAF_BIT)) {
        const int lead = __builtin_ctzll(todo);
        const float lx = lane_value(d.x, lead), ly = lane_value(d.y, lead), lz = lane_value(d.z, lead);
        const float ax_ = __builtin_fabsf(lx), ay_ = __builtin_fabsf(ly), az_ = __builtin_fabsf(lz);
        const uint32_t ax = (ax_ >= ay_ && ax_ >= az_) ? 0u : (ay_ >= az_ ? 1u : 2u);
        const float sg = (ax == 0u ? lx : (ax == 1u ? ly : lz)) > 0.f ? 1.0f : -1.0f;
        const bool mine = usable && dmax <= kBwMaxSlope * (sg * axis_of(d, ax));   // (rays apart from the first: not looked at)
        const BundleLds lds = {area};
        (void)bundle_begin(lds.base, ax, sg, o, d, mine, __uint_as_float(acc.bounds->scale));
        count = bundle_count({acc.leaves, acc.wide, acc.n_leaves, acc.root}, lds, kCostMax);
    }
    return count;
}
// Counting sort by that guess, in one workgroup; blocks of equal cost keep their neighbourhood, 1024 at a time.
__global__ __launch_bounds__(1024) void k_cost_order(const uint32_t *__restrict__ cost, uint32_t n_blocks, uint32_t *__restrict__ order) {
    constexpr uint32_t kClasses = 128u;
    __shared__ uint32_t s_count[kClasses], s_base[kClasses];
    auto cost_class = [&](uint32_t j) { return kClasses - 1u - min(cost[j] / ((kCostMax + 1u) / kClasses), kClasses - 1u); };   // 0: the longest
    if (threadIdx.x < kClasses) s_count[threadIdx.x] = 0u;
    __syncthreads();
    for (uint32_t j = threadIdx.x; j < n_blocks; j += blockDim.x) atomicAdd(&s_count[cost_class(j)], 1u);
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t run = 0u;
        for (uint32_t c = 0; c < kClasses; ++c) {
            s_base[c] = run;
            run += s_count[c];
        }
    }
    __syncthreads();
    for (uint32_t base = 0; base < n_blocks; base += blockDim.x) {
        const uint32_t j = base + threadIdx.x;
        if (j < n_blocks) order[atomicAdd(&s_base[cost_class(j)], 1u)] = j;
        __syncthreads();
    }
}

// Tile hand-over (forward).  A bundle walk lists and tests what any of its 64 rays may need, one candidate after the
// other.  Over geometry much finer than the ray spacing (a dense cloud of surfels far smaller than a pixel) that is the
// whole content of the tile's frustum, wanted by one ray at best, and a single wave walks for milliseconds while the chip
// idles (150,000 quads of 2 mm in a ball of 12 cm, 64x64 pixels: 29.9 ms; handed over 2.8).  So the first walk of a tile
// may take `hand_arg` steps (nodes and candidates) and no more: a wave that runs into that limit has
// written nothing yet, puts its tile on the context's list and leaves, and a second, small launch right behind
// (kernels with the per-lane walk, hand_arg = 0: the takers) traces the listed tiles with every ray walking on its
// own - the same buffer content, so the same results bit for bit.  List: word 0 = tiles listed by this trace, word 1 =
// takers that have read their entry (the last one empties the list for the next trace: nothing on the host changes
// from call to call, so a captured launch pair can be replayed), word 2 = tiles handed over since the context was
// made, word 3 = not the list's: sums of the deterministic mode found out of range (its closing kernels count there),
// entries ((by * btiles_x + bx) * 4 + wave) from word 4.  A wave that finds the list full starts again without a limit.
constexpr uint32_t kHandHeader = kDstHandoverHeader, kHandCap = kDstHandoverCap;
// Ray lists that are traced in an order of their own: by tiles (contexts that hand tiles over, the backward trace without a
// record) from kOrderMinRays on, by rows from kOrderMinByRows on, where it pays (k_list_look, which has the figures).  A record
// that turned out too small is traced again by tiles: in the rows' order from kOrderManyRays on.  (In the rays' order / in the
// rows', us a training step: pixels of one camera, shuffled, 65,536 6381 / 6511 in a room of a million, 5188 / 6276 at a
// sphere of 100,000, 131,072 8636 / 8016 and 6305 / 6427, 262,144 16,472 / 13,022 and 12,479 / 8731; unrelated rays, 131,072
// 2282 / 2614 in a room of 300,000, 262,144 13,531 / 12,925 in one of a million.)
constexpr uint32_t kOrderMinRays = 2048, kOrderMinByRows = 65536, kOrderManyRays = 262144;

template <bool BWD, int AUXM, bool REC, bool MIXED, bool DET, bool HAND, bool PACK>
__device__ __forceinline__ void trace_body(const DstParams &p, const DstAccelView &acc, int tw_log2, int th_log2,
                                           uint32_t tiles_x, uint32_t tiles_y, uint32_t btiles_x,
                                           const uint32_t *ray_order, uint32_t strip_width,
                                           const uint32_t *__restrict__ block_order, uint32_t *handover,
                                           uint32_t hand_arg) {
    // a block = 2x2 wave tiles (16x16 pixels for the usual 8x8 tile): neighbouring rays share surfels, which
    // is what the block's gradient table and the caches live on
    constexpr int kTableRows = RowLayout<AUXM>::rows;
    __shared__ __attribute__((aligned(16))) uint32_t s_keys[BWD ? kTableRows + 1 : 1];   // + the count of claimed rows
    constexpr int kTableWords = RowLayout<AUXM>::words;
    __shared__ double s_rows[BWD ? kTableWords : 1];
    constexpr int kStageWords = RowLayout<AUXM>::stage;
    __shared__ float s_stage[BWD ? kWavesPerBlock * kStageWords : 1];
    uint32_t *tab_keys = s_keys;
    double *tab_rows = s_rows;
    // forward of an image at depth 0: the wave's table of blending weights (wet_add; in the kernels that carry the
    // per-lane walk it measured no gain and would take the LDS to the limit of 16 waves per CU)
    constexpr bool WET = !BWD && !MIXED && !DET;
    __shared__ uint32_t s_wet_keys[WET ? kFwdWavesPerBlock * kWetSlots : 1];
    __shared__ double s_wet_vals[WET ? kFwdWavesPerBlock * kWetSlots : 1];
    uint32_t *const wet_keys = s_wet_keys + (WET ? (threadIdx.x / DST_WAVE) * kWetSlots : 0);
    double *const wet_vals = s_wet_vals + (WET ? (threadIdx.x / DST_WAVE) * kWetSlots : 0);
    if (WET) {   // (a wave's LDS accesses keep their order: no barrier between this and the first use)
        for (int e = threadIdx.x % DST_WAVE; e < kWetSlots; e += DST_WAVE) {
            wet_keys[e] = 0xFFFFFFFFu;
            wet_vals[e] = 0.0;
        }
    }
    // Backward with a hit record: the launcher starts the replaying kernel and the re-tracing kernel one after
    // the other, and word 0 of the record (blocks the forward trace asked for) decides on the device which of
    // the two does the work: the host never has to wait for the forward trace to learn whether its record is complete.
    if (BWD && p.hit_record != nullptr) {
        const bool complete = p.hit_record[0] <= (uint64_t)p.hit_record_blocks;
        if (REC != complete || (REC && (uint32_t)p.hit_record[2] != 0u)) return;
        if (!REC && (uint32_t)p.hit_record[2] != 0u && (uint32_t)p.W < kOrderManyRays) ray_order = nullptr;   // (written by rows)
    }
    if (BWD) {
        table_clear_keys<AUXM, DET>(s_keys);
        for (int k = threadIdx.x; k < kTableWords; k += kWavesPerBlock * DST_WAVE) s_rows[k] = 0.0;
        __syncthreads();
    }
    // Backward: a block is the four waves of a 16x16 pixel tile (they share the gradient table).  Forward: the
    // waves share nothing, so each is a workgroup of its own and takes a free wave slot as soon as there is
    // one; workgroups x, x+8, x+16, x+24 (same XCD under round-robin dispatch) are the four waves of a tile.
    uint32_t bid = blockIdx.x, wv = threadIdx.x / DST_WAVE;
    if (!BWD && kFwdWavesPerBlock == 1) {
        bid = (blockIdx.x >> 5) * 8u + (blockIdx.x & 7u);
        wv = (blockIdx.x >> 3) & 3u;
    }
    // Image grids are walked in column strips eight blocks wide, row by row inside a strip.  Workgroups go to the
    // eight XCDs in turn, so in a full strip XCD q works its way down column q: the tiles an XCD has in flight are
    // vertical neighbours and meet the same BVH nodes in that XCD's own L2 (row-major order over a 120-block-wide image
    // gives an XCD blocks eight columns apart).  The last strip may be narrower; its blocks are spread over all XCDs
    // like the others.  The launcher chooses the width, and has the figures (launch()).
    // the longest blocks first (replay: k_block_order; forward: k_cost_order)
    if (block_order != nullptr) bid = bid < btiles_x * ((tiles_y + 1u) / 2u) ? block_order[bid] : bid;
    uint32_t bx, by;
    static_assert(!HAND || (!BWD && kFwdWavesPerBlock == 1), "tiles are handed over by forward kernels of one wave per workgroup");
    const bool taker = HAND && MIXED && handover != nullptr && hand_arg == 0u;
    block_of_position(bid, btiles_x, (tiles_y + 1u) / 2u, strip_width, th_log2 != 0, bx, by);
    if constexpr (HAND) {
        if (taker) {   // the tile comes from the list, not from the workgroup's number
            const uint32_t n = min(handover[0], gridDim.x);
            const uint32_t id = handover[kHandHeader + min(blockIdx.x, kHandCap - 1u)];
            wv = id & 3u;
            bx = (id >> 2) % btiles_x;
            by = (id >> 2) / btiles_x;
            // Every taker has read the count and its entry before it is counted itself (the fence keeps the reads in front
            // of the ticket), and no wave writes the list while takers run: the last one counted empties it.
            __threadfence();
            if (threadIdx.x == 0u) {
                const uint32_t ticket = atomicAdd(&handover[1], 1u);
                if (ticket == gridDim.x - 1u) {
                    handover[2] += n;
                    handover[1] = 0u;
                    handover[0] = 0u;
                }
            }
            if (blockIdx.x >= n) return;
        }
    }
    const bool flat = th_log2 == 0;   // a ray list: tiles of 1x64 rays, a block = four consecutive tiles
    if (flat ? by >= 1u : 2u * by >= tiles_y) return;   // padding of the forward grid (whole blocks)
    RecView rv = {nullptr, nullptr, nullptr, 0u};
    if (REC) {
        const uint32_t n_waves = btiles_x * ((tiles_y + 1u) / 2u) * kWavesPerBlock, slots_ = (uint32_t)p.mtd_alloc + 1u;
        rv.base = p.hit_record;
        rv.dir = reinterpret_cast<uint32_t *>(p.hit_record + 3) + (size_t)((by * btiles_x + bx) * kWavesPerBlock + wv) * slots_;
        rv.blocks = p.hit_record + record_header_words((uint64_t)p.H * p.W, th_log2, slots_, n_waves);
        rv.capacity = p.hit_record_blocks;
    }
    const uint32_t ty = flat ? 0u : 2u * by + (wv >> 1), tx = flat ? 4u * bx + wv : 2u * bx + (wv & 1u);
    const bool wave_on = ty < tiles_y && tx < tiles_x;
    if (!BWD && !wave_on) return;   // the backward kernel keeps every wave for the block-wide flush below
    const uint32_t lane = threadIdx.x % DST_WAVE;
    const uint32_t py = (ty << th_log2) + (lane >> tw_log2);
    const uint32_t px = (tx << tw_log2) + (lane & ((1u << tw_log2) - 1u));
    const bool inside = wave_on && py < (uint32_t)p.H && px < (uint32_t)p.W;
    // ray lists are traced in a coherent order (see k_ray_keys): position in that order -> ray number
    const size_t pos = inside ? ((size_t)py * p.W + px) : 0;
    // (forward: ray lists always run the MIXED kernels, so the image kernels need not look at the order)
    const size_t r = ((MIXED || BWD) && ray_order != nullptr && inside) ? (size_t)min(ray_order[pos], (uint32_t)p.W - 1u) : pos;
    const float max_abs = __uint_as_float(acc.bounds->scale);   // the size origins are compared with (rays_run_together)
    const int MID = 14 + p.aux, AUXO = 11, RGBO = 11 + p.aux;
    const int slots = p.mtd_alloc + 1, mtd = p.max_trace_depth;
    float *mid = p.mid_val + (size_t)slots * MID * r;
    const F3 ray_o = ld3(p.ray_o + 3 * r), ray_d = ld3(p.ray_d + 3 * r);
    uint32_t n_proc = 0, n_con = 0;
#ifdef DST_STATS
    WaveStats ws = {0, 0, 0, 0, 0, 0, 0, 0, 0};
#define WS_ARG , ws
#else
#define WS_ARG
#endif
    BounceAcc<AUXM> run;
    BounceIn<AUXM> in;
    F3 g_ro = f3(0, 0, 0), g_rd = f3(0, 0, 0);

    if (!BWD) {
        // reference forward.cu:318-424
        float out_rgb[3] = {0.f, 0.f, 0.f};
        F3 ot = ray_o, dt = ray_d;
        float s_prod = 1.0f;
        bool on = inside;
        uint32_t first_walk = (HAND && handover != nullptr) ? hand_arg : 0u;
        // (kernels without the per-lane walk trace the first bounce; k_row_fwd goes on from there)
        const int last = MIXED ? mtd : 0;
        for (int i = 0; i <= last; ++i) {
            const float min_depth = (i == 0) ? (p.start_from_first ? kNear : 0.0f) : kStartOffset;
            F3 dist_acc = f3(0, 0, 0);
            const bool gave_up = walk_bounce<false, AUXM, REC, MIXED, DET, HAND, PACK>(p, acc, max_abs, on, ot, dt, min_depth, run, in, g_ro, g_rd, n_proc, n_con, WET ? wet_keys : nullptr, WET ? wet_vals : nullptr, nullptr, rv, i, dist_acc, taker ? kWalkPerLane : (i == 0 ? first_walk : 0u) WS_ARG);
            if constexpr (HAND) if (gave_up) {   // (bounce 0, before anything was written; no else below)
                uint32_t slot = 0u;
                if (lane == 0u) slot = atomicAdd(&handover[0], 1u);
                slot = __builtin_amdgcn_readfirstlane(slot);
                if (slot < kHandCap) {
                    if (lane == 0u) handover[kHandHeader + slot] = ((by * btiles_x + bx) << 2) | wv;
                    return;
                }
                first_walk = 0u;   // the list is full: this wave keeps its tile
                --i;
                continue;
            }
            if (on) {
                run.C[0] += run.T * p.background[0];
                run.C[1] += run.T * p.background[1];
                run.C[2] += run.T * p.background[2];
                const float A = 1 - run.T;
                const F3 E = f3(ot.x + run.D * dt.x, ot.y + run.D * dt.y, ot.z + run.D * dt.z);
                if (i == 0) {
                    p.out_dpt[r] = run.D;
                    p.out_acc[r] = A;
                    p.out_norm[3 * r + 0] = run.N[0];
                    p.out_norm[3 * r + 1] = run.N[1];
                    p.out_norm[3 * r + 2] = run.N[2];
                    if (p.dist_channels == 1) {   // zeros unless DST_FLAG_DISTORTION (as the reference)
                        p.out_dist[r] = dist_acc.x;
                    } else {
                        p.out_dist[3 * r + 0] = dist_acc.x;
                        p.out_dist[3 * r + 1] = dist_acc.y;
                        p.out_dist[3 * r + 2] = dist_acc.z;
                    }
#pragma unroll
                    for (int ch = 0; ch < AUXM; ++ch)
                        if (ch < p.aux) p.out_aux[(size_t)p.aux * r + ch] = run.O[ch];
                }
                const float f_this = (i == mtd) ? 1.0f : 1 - run.O[0];
                out_rgb[0] += run.C[0] * f_this * s_prod;
                out_rgb[1] += run.C[1] * f_this * s_prod;
                out_rgb[2] += run.C[2] * f_this * s_prod;
                s_prod *= run.O[0];
                float *m = mid + (size_t)i * MID;
                m[0] = ot.x; m[1] = ot.y; m[2] = ot.z;
                m[3] = dt.x; m[4] = dt.y; m[5] = dt.z;
                m[6] = run.D;
                m[7] = A;
                m[8] = run.N[0]; m[9] = run.N[1]; m[10] = run.N[2];
#pragma unroll
                for (int ch = 0; ch < AUXM; ++ch)
                    if (ch < p.aux) m[AUXO + ch] = run.O[ch];
                m[RGBO + 0] = run.C[0];
                m[RGBO + 1] = run.C[1];
                m[RGBO + 2] = run.C[2];
                const F3 N = f3(run.N[0], run.N[1], run.N[2]);
                const float nl = length(N);
                if (nl == 0.0f || run.O[0] <= p.specular_threshold) {
                    on = false;
                    // slots of the bounces never traced read as zeros
                    for (int k = (i + 1) * MID; k < slots * MID; ++k) mid[k] = 0.f;
                } else {
                    const F3 n = N / nl;
                    dt = dt - 2 * dot(n, dt) * n;
                    ot = E + kStartOffset * dt;
                }
            }
        }
        if (inside) {
            if (on && last == mtd)
                for (int k = (mtd + 1) * MID; k < slots * MID; ++k) mid[k] = 0.f;
            p.out_rgb[3 * r + 0] = out_rgb[0];
            p.out_rgb[3 * r + 1] = out_rgb[1];
            p.out_rgb[3 * r + 2] = out_rgb[2];
        }
        if (WET && p.training && p.a_weights != nullptr) {   // the wave's blending weights: one addition per surfel
            for (int e = (int)lane; e < kWetSlots; e += DST_WAVE) {
                const uint32_t k = wet_keys[e];
                const float v = (float)wet_vals[e];
                if (k != 0xFFFFFFFFu && v != 0.f) aadd(p.a_weights + k, v);
            }
        }
        if (p.counters != nullptr) {
            uint32_t a = wave_sum(n_proc), b = wave_sum(n_con);
            if (lane == 0) {
                atomicAdd(p.counters + 0, (unsigned long long)a);
                atomicAdd(p.counters + 1, (unsigned long long)b);
#ifdef DST_STATS   // development build only: counters must then hold 8 entries
                atomicAdd(p.counters + 2, ws.nodes);
                atomicAdd(p.counters + 3, ws.leaves);
                atomicAdd(p.counters + 4, ws.t_trav);
                atomicAdd(p.counters + 5, ws.t_comp);
                atomicAdd(p.counters + 6, ws.chunks);
                atomicAdd(p.counters + 7, ws.leaf_any);
                atomicAdd(p.counters + 8, ws.t_plan);   // exact quad tests run (forward only)
                atomicAdd(p.counters + 9, ws.steps);    // compositing iterations of the wave
                atomicAdd(p.counters + 10, ws.t_hb);    // lanes with an entry, summed over those iterations
#endif
            }
        }
    } else {
        // reference backward.cu:658-853
        float C_prev[3], c_prev[3] = {0.f, 0.f, 0.f}, g_out_rgb[3];
        for (int ch = 0; ch < 3; ++ch) {
            C_prev[ch] = p.out_rgb[3 * r + ch];
            g_out_rgb[ch] = p.dL_drgb[3 * r + ch];
        }
        float s_prod = 1.0f;
        for (int i = 0; i < mtd; ++i) {
            for (int ch = 0; ch < 3; ++ch) {
                float c_curr = mid[ch + RGBO + i * MID];
                C_prev[ch] = C_prev[ch] + s_prod * (c_prev[ch] - c_curr);
                c_prev[ch] = c_curr;
            }
            s_prod *= mid[AUXO + i * MID];
        }
        for (int i = mtd; i >= 0; --i) {
            const float *m = mid + (size_t)i * MID;
            const F3 ot = ld3(m), dt = ld3(m + 3);
            const float s_prev = (i > 0) ? mid[AUXO + (i - 1) * MID] : 1.0f;
            const bool on = inside && !(length(dt) == 0.0f || s_prev <= p.specular_threshold);
            if (on) {
                for (int ch = 0; ch < 3; ++ch) in.rgb[ch] = m[RGBO + ch];
                in.dpt = m[6];
                in.acc = m[7];
                in.nrm[0] = m[8]; in.nrm[1] = m[9]; in.nrm[2] = m[10];
#pragma unroll
                for (int ch = 0; ch < AUXM; ++ch) {
                    in.aux[ch] = (ch < p.aux) ? m[AUXO + ch] : 0.f;
                    in.g_aux[ch] = 0.f;
                }
                in.g_dpt = 0.f;
                in.g_acc = 0.f;
                in.g_nrm[0] = in.g_nrm[1] = in.g_nrm[2] = 0.f;
                const float f_this = (i == mtd) ? 1.0f : 1 - in.aux[0];
                for (int ch = 0; ch < 3; ++ch) in.g_rgb[ch] = g_out_rgb[ch] * f_this * s_prod;
                s_prod /= s_prev;
                if (i != mtd) {
                    for (int ch = 0; ch < 3; ++ch) {
                        in.g_aux[0] += g_out_rgb[ch] * (C_prev[ch] / in.aux[0]);
                        c_prev[ch] = (i > 0) ? mid[ch + RGBO + (i - 1) * MID] : 0.0f;
                        C_prev[ch] = C_prev[ch] - s_prod * (c_prev[ch] - in.rgb[ch]);
                    }
                    const F3 nrm = f3(in.nrm[0], in.nrm[1], in.nrm[2]);
                    const float nl = length(nrm);
                    if (nl != 0.f) {
                        g_rd = g_rd + g_ro * (float)kStepEps;
                        const F3 n = nrm / nl;
                        in.g_dpt += g_ro.x * dt.x + g_ro.y * dt.y + g_ro.z * dt.z;
                        const F3 gn = dnormvdv(nrm, ddotndndn(n, dt, g_rd * -2.0f));
                        in.g_nrm[0] += gn.x;
                        in.g_nrm[1] += gn.y;
                        in.g_nrm[2] += gn.z;
                        g_rd = g_ro * in.dpt + g_rd + ddotndndd(n, g_rd * -2.0f);
                    }
                }
                if (i == 0) {
                    in.g_dpt += p.dL_ddpt[r];
                    in.g_acc += p.dL_dacc[r];
                    in.g_nrm[0] += p.dL_dnorm[3 * r + 0];
                    in.g_nrm[1] += p.dL_dnorm[3 * r + 1];
                    in.g_nrm[2] += p.dL_dnorm[3 * r + 2];
#pragma unroll
                    for (int ch = 0; ch < AUXM; ++ch)
                        if (ch < p.aux) in.g_aux[ch] += p.dL_daux[(size_t)p.aux * r + ch];
                }
            }
            const float min_depth = (i == 0) ? (p.start_from_first ? kNear : 0.0f) : kStartOffset;
            F3 no_dist = f3(0, 0, 0);
            (void)walk_bounce<true, AUXM, REC, MIXED, DET, false, false>(p, acc, max_abs, on, ot, dt, min_depth, run, in, g_ro, g_rd, n_proc, n_con, tab_keys, tab_rows, s_stage + wv * kStageWords, rv, i, no_dist, 0u WS_ARG);
        }
#ifdef DST_STATS   // development build only: counters must then hold 11 entries
        if (p.counters != nullptr && lane == 0) {
            atomicAdd(p.counters + 2, ws.steps);
            atomicAdd(p.counters + 3, ws.t_plan);
            atomicAdd(p.counters + 4, ws.t_trav);
            atomicAdd(p.counters + 5, ws.t_comp);
            atomicAdd(p.counters + 6, ws.chunks);
            atomicAdd(p.counters + 7, ws.t_hb);
            atomicAdd(p.counters + 8, ws.nodes);
            atomicAdd(p.counters + 9, ws.leaves);
            atomicAdd(p.counters + 10, ws.leaf_any);
        }
#endif
        if (inside) {
            p.dL_dray_o[3 * r + 0] = g_ro.x; p.dL_dray_o[3 * r + 1] = g_ro.y; p.dL_dray_o[3 * r + 2] = g_ro.z;
            p.dL_dray_d[3 * r + 0] = g_rd.x; p.dL_dray_d[3 * r + 1] = g_rd.y; p.dL_dray_d[3 * r + 2] = g_rd.z;
        }
        __syncthreads();
        table_flush<AUXM, DET>(p, s_keys, s_rows);
    }
}

// Occupancy the register allocator is told to aim for, waves per SIMD: enough in flight to cover the fetches, few enough
// for the working set to stay in registers.  1080p room, evaluated, at 2 / 3 / 4 forward waves: 5.09 / 3.81 / 5.23 ms,
// 800x800 sphere 2.16 / 1.85 / 2.12.  The kernels with the per-lane walk: see there.  Backward, training steps at 2 / 3
// waves (a table of 117 / 64 rows): room 10.7 / 12.7 ms, sphere 3.70 / 4.68, 233x417 room in fixed point 0.56 / 0.68.
#ifndef DST_FWD_WAVES
#define DST_FWD_WAVES 3
#endif
#ifndef DST_MIXED_WAVES
#define DST_MIXED_WAVES 4
#endif
// EXTRAS: the rarely used forward options (DstParams.flags: fixed-point blending weights, distortion output) live in
// a kernel of their own, so that the usual one does not carry their registers.
template <int AUXM, bool REC, bool MIXED, bool EXTRAS>
__global__ __launch_bounds__(kFwdWavesPerBlock *DST_WAVE) __attribute__((amdgpu_waves_per_eu(MIXED ? DST_MIXED_WAVES : DST_FWD_WAVES, MIXED ? DST_MIXED_WAVES : DST_FWD_WAVES)))
void k_trace_fwd(const DstParams p, const DstAccelView acc, int tw_log2, int th_log2, uint32_t tiles_x,
                 uint32_t tiles_y, uint32_t btiles_x, const uint32_t *ray_order, uint32_t strip_width, uint32_t *handover,
                 uint32_t hand_arg) {
    trace_body<false, AUXM, REC, MIXED, EXTRAS, kFwdWavesPerBlock == 1, false>(p, acc, tw_log2, th_log2, tiles_x, tiles_y, btiles_x, ray_order, strip_width, nullptr, handover, hand_arg);
}
// The forward kernel of image grids at depth 0 without the tile hand-over: what scenes without many small quads are
// traced with (the hand-over's counting and its few extra live values cost the walk 9 % on the 1080p room and 16 % on the
// 800x800 sphere, whether a tile is ever handed over or not: 3.80 -> 4.13 ms, 1.84 -> 2.13).
template <int AUXM, bool REC, bool PACK>
__global__ __launch_bounds__(kFwdWavesPerBlock *DST_WAVE) __attribute__((amdgpu_waves_per_eu(DST_FWD_WAVES, DST_FWD_WAVES)))
void k_trace_fwd_plain(const DstParams p, const DstAccelView acc, int tw_log2, int th_log2, uint32_t tiles_x,
                       uint32_t tiles_y, uint32_t btiles_x, const uint32_t *ray_order, uint32_t strip_width,
                       const uint32_t *block_order) {
    trace_body<false, AUXM, REC, false, false, false, PACK>(p, acc, tw_log2, th_log2, tiles_x, tiles_y, btiles_x, ray_order, strip_width, block_order, nullptr, 0u);
}
template <int AUXM, bool REC, bool MIXED, bool DET>
__global__ __launch_bounds__(kWavesPerBlock *DST_WAVE) __attribute__((amdgpu_waves_per_eu(DST_BWD_WAVES, DST_BWD_WAVES)))
void k_trace_bwd(const DstParams p, const DstAccelView acc, int tw_log2, int th_log2, uint32_t tiles_x,
                 uint32_t tiles_y, uint32_t btiles_x, const uint32_t *ray_order, uint32_t strip_width,
                 const uint32_t *block_order) {
    trace_body<true, AUXM, REC, MIXED, DET, false, false>(p, acc, tw_log2, th_log2, tiles_x, tiles_y, btiles_x, ray_order, strip_width, block_order, nullptr, 0u);
}

// Surfel record of surfel g: 40 bytes in, 64 out.
__device__ __forceinline__ void surfel_record(const DstParams &p, uint32_t g) {
    const F3 mean = ld3(p.means3D + 3 * (size_t)g);
    const float sx = p.scales[2 * (size_t)g], sy = p.scales[2 * (size_t)g + 1];
    const float *qp = p.rotations + 4 * (size_t)g;
    F3 R[3];
    quat_rows(qp[0], qp[1], qp[2], qp[3], R);
    auto inverse = [](float s) {   // (div_by's range)
        const float m = __builtin_fabsf(s);
        return m >= 0x1p-40f && m <= 0x1p40f ? 1.0f / s : __builtin_nanf("");
    };
    v4f *out = reinterpret_cast<v4f *>(reinterpret_cast<DstSurfel *>(p.scratch) + g);
    out[0] = v4f{R[0].x, R[0].y, R[0].z, -dot(R[0], mean)};
    out[1] = v4f{R[1].x, R[1].y, R[1].z, -dot(R[1], mean)};
    out[2] = v4f{R[2].x, R[2].y, R[2].z, p.opacities[g]};
    out[3] = v4f{sx, sy, inverse(sx), inverse(sy)};
}
// What a forward trace prepares, in one launch: the blocks' costs (a wave each, first, as they take longest) and the surfels'
// records (a thread each).
constexpr uint32_t kPrepareWaves = 4u;
__global__ __launch_bounds__(kPrepareWaves *DST_WAVE) void k_prepare(const DstParams p, const DstAccelView acc, uint32_t btiles_x, uint32_t *cost,
                                                                     uint32_t n_blocks) {
    __shared__ uint32_t s_lds[kPrepareWaves * (kBwStateWords + kBwStack)];
    const uint32_t of_cost = (n_blocks + kPrepareWaves - 1u) / kPrepareWaves;
    if (blockIdx.x < of_cost) {
        const uint32_t wave = uni(threadIdx.x / DST_WAVE), block = blockIdx.x * kPrepareWaves + wave;
        if (block >= n_blocks) return;
        const uint32_t count = block_cost(p, acc, block, btiles_x, (lds_u32)s_lds + wave * (kBwStateWords + kBwStack));
        if (__lane_id() == 0u) cost[block] = count;
    } else {
        const uint32_t g = (blockIdx.x - of_cost) * kPrepareWaves * DST_WAVE + threadIdx.x;
        if (g < (uint32_t)p.P) surfel_record(p, g);
    }
}

#include "row.inc"

// Closing kernel of a backward trace: the per-surfel sums (gradient rows, or the deterministic mode's fixed point) to the
// caller's tensors.  A workgroup takes kCloseSurfels surfels through LDS: rows in as they lie, tensors out as
// they lie, 16 bytes a lane for the SH gradient.  Bound by memory.  With p.grad_touched it writes the tensors (a caller
// has nothing to fill), reads the marked surfels' rows alone (a view meets a third of a room's surfels, a LiDAR frame a
// tenth of its scene's) and clears what it read, so that the rows stay zero between calls; without, it adds to them.
// (2M surfels, 4 auxiliary channels: rows filled 0.1 ms + tensors filled 0.1 ms + closing 0.24 ms before.)
// (A workgroup for every 64 surfels, and all it reads asked for at once: one that goes on to the next 64 waits for its stores,
// which memory counts with its loads.  8192 workgroups that go on / one for each:
// 2M surfels, 4 channels 181 / 127 us, 1M, 2 channels 84 / 66, 500,000, 8 channels 101 / 64.)
constexpr uint32_t kCloseSurfels = 64, kCloseThreads = 256;
template <int AUXM, bool DET>
__global__ __launch_bounds__(kCloseThreads) void k_close_gradients(const DstParams p, uint32_t *out_of_range) {
    constexpr uint32_t cols = RowLayout<AUXM>::cols, stride = cols | 1u;
    static_assert(kCloseSurfels == DST_WAVE && kColAux == DST_WAVE, "a bit per surfel, a lane per column");
    constexpr uint32_t kWaves = kCloseThreads / DST_WAVE, kMain = kCloseSurfels / kWaves, kAux = (kCloseSurfels * AUXM + kCloseThreads - 1u) / kCloseThreads;
    __shared__ float s_rows[kCloseSurfels * stride];
    __shared__ uint64_t s_on;   // whose rows are read
    const bool writes = p.grad_touched != nullptr, aux_rows = p.others_precomp != nullptr;
    const uint32_t tid = threadIdx.x, P = (uint32_t)p.P;
    const uint32_t base = blockIdx.x * kCloseSurfels, n = min(kCloseSurfels, P - base);
    if (tid < DST_WAVE) {
        const bool on = tid < n && (!writes || p.grad_touched[base + tid] != 0u);
        const uint64_t mask = wave_ballot(on);
        if (writes && on) p.grad_touched[base + tid] = 0u;
        if (tid == 0u) s_on = mask;
    }
    __syncthreads();
    const uint64_t on = s_on;
    const bool any = on != 0ull;
    if (any) {
        // a wave's rows, sixteen of 64 columns, and a thread's share of the auxiliary columns behind them: all asked for at once
        typedef typename std::conditional<DET, long long, float>::type Sum;
        Sum *const sums = DET ? (Sum *)p.det_workspace : (Sum *)p.grad_rows;
        Sum *const from = sums + (size_t)base * kColAux, *const from_aux = sums + (size_t)P * kColAux + (size_t)base * AUXM;
        const uint32_t wave = uni(tid / DST_WAVE), lane = tid % DST_WAVE;
        Sum main[kMain], aux[kAux];
        auto has = [&](uint32_t row) { return ((on >> row) & 1ull) != 0ull; };
#pragma unroll
        for (uint32_t j = 0; j < kMain; ++j) {
            const uint32_t row = wave + kWaves * j;
            main[j] = 0;
            if (has(row)) main[j] = from[row * DST_WAVE + lane];
        }
#pragma unroll
        for (uint32_t j = 0; j < kAux; ++j) {
            const uint32_t k = tid + j * kCloseThreads;
            aux[j] = 0;
            if (aux_rows && k < kCloseSurfels * AUXM && has(k / AUXM)) aux[j] = from_aux[k];
        }
        // `sum` of column `col`; the row is left empty
        auto take = [&](Sum sum, Sum *at, uint32_t col) {
            if (sum == 0) return 0.f;
            if (writes) *at = 0;
            if constexpr (DET) {
                if (det_out_of_range(sum)) atomicAdd(out_of_range, 1u);
                return from_fixed(sum, det_shift((int)col));
            } else {
                return sum;
            }
        };
#pragma unroll
        for (uint32_t j = 0; j < kMain; ++j) {
            const uint32_t row = wave + kWaves * j;
            s_rows[row * stride + lane] = take(main[j], from + row * DST_WAVE + lane, lane);
        }
#pragma unroll
        for (uint32_t j = 0; j < kAux; ++j) {
            const uint32_t k = tid + j * kCloseThreads;
            if (aux_rows && k < kCloseSurfels * AUXM) s_rows[(k / AUXM) * stride + kColAux + k % AUXM] = take(aux[j], from_aux + k, kColAux + k % AUXM);
        }
        __syncthreads();
    }
    auto put = [&](float *dst, float v) {
        if (writes) *dst = v;
        else if (v != 0.f) *dst += v;
    };
    // `width` columns from `col0` on of every surfel to the tensor `dst` (width, .)
    auto emit = [&](float *dst, uint32_t width, uint32_t col0) {
        if (dst == nullptr || (!any && !writes)) return;
        for (uint32_t e = tid; e < n * width; e += kCloseThreads)
            put(dst + (size_t)base * width + e, any ? s_rows[(e / width) * stride + col0 + e % width] : 0.f);
    };
    emit(p.dL_dcolors, 3u, kColColor);
    emit(p.dL_dopacities, 1u, kColOpac);
    emit(p.dL_dscales, 2u, kColScale);
    emit(p.dL_drotations, 4u, kColRot);
    emit(p.dL_dmeans3D, 3u, kColMean);
    emit(p.dL_dgrads3D, 3u, kColGrad);
    if (aux_rows) emit(p.dL_dothers, (uint32_t)p.aux, kColAux);
    else if (writes && p.dL_dothers != nullptr)   // nothing was given: zeros
        for (uint32_t e = tid; e < n * (uint32_t)p.aux; e += kCloseThreads) p.dL_dothers[(size_t)base * p.aux + e] = 0.f;
    if (p.colors_precomp == nullptr && p.dL_dshs != nullptr && (any || writes)) {
        const uint32_t width = 3u * (uint32_t)p.M;
        float *const dst = p.dL_dshs + (size_t)base * width;
        // element r of a surfel is coefficient r / 3, channel r % 3 (coefficients past the sixteenth have no gradient)
        auto of = [&](uint32_t row, uint32_t r) { return any && r < 48u ? s_rows[row * stride + kColSh + 16u * (r % 3u) + r / 3u] : 0.f; };
        if (writes && width == 48u && (reinterpret_cast<uintptr_t>(p.dL_dshs) & 15u) == 0u) {
            for (uint32_t e = tid; e < n * 12u; e += kCloseThreads) {
                const uint32_t row = e / 12u, r = 4u * (e - row * 12u);
                reinterpret_cast<float4 *>(dst)[e] = make_float4(of(row, r), of(row, r + 1u), of(row, r + 2u), of(row, r + 3u));
            }
        } else {
            for (uint32_t e = tid; e < n * width; e += kCloseThreads) {
                const uint32_t row = e / width;
                put(dst + e, of(row, e - row * width));
            }
        }
    }
}
__global__ void k_det_finish_weights(const DstParams p, uint32_t *out_of_range) {
    for (int g = blockIdx.x * blockDim.x + threadIdx.x; g < p.P; g += gridDim.x * blockDim.x) {
        const long long q = (long long)p.det_workspace[g];
        if (q != 0) p.a_weights[g] += from_fixed(q, kDetShiftOther);
        if (det_out_of_range(q)) atomicAdd(out_of_range, 1u);
    }
}

// Direction of a ray as a Morton code of its octahedral map (2 x 8 bits); 0 for one that has none (NaN, zero).
__device__ __forceinline__ uint32_t direction_code(const float *d) {
    const float l1 = fabsf(d[0]) + fabsf(d[1]) + fabsf(d[2]);
    if (!(l1 > 0.f && l1 < INFINITY)) return 0u;
    float u = d[0] / l1, v = d[1] / l1;
    if (d[2] < 0.f) {   // fold the lower hemisphere over the square's corners
        const float fu = (1.f - fabsf(v)) * (u >= 0.f ? 1.f : -1.f), fv = (1.f - fabsf(u)) * (v >= 0.f ? 1.f : -1.f);
        u = fu;
        v = fv;
    }
    uint32_t qu = (uint32_t)fminf(fmaxf((u * 0.5f + 0.5f) * 256.f, 0.f), 255.f);
    uint32_t qv = (uint32_t)fminf(fmaxf((v * 0.5f + 0.5f) * 256.f, 0.f), 255.f);
    auto spread8 = [](uint32_t x) {
        x = (x | (x << 4)) & 0x0F0Fu;
        x = (x | (x << 2)) & 0x3333u;
        x = (x | (x << 1)) & 0x5555u;
        return x;
    };
    return (spread8(qu) << 1) | spread8(qv);
}
// Cell of an origin on a grid of 2^(3 LOG2) cells over the scene; outside (and NaN): the nearest one.
template <int LOG2>
__device__ __forceinline__ uint32_t origin_cell(const float *o, const DstBounds *bounds) {
    const float ext = __uint_as_float(bounds->scale), half = 0.5f * (float)(1 << LOG2);
    const float inv = ext > 0.f ? half / ext : 0.f;
    uint32_t cell = 0u;
#pragma unroll
    for (int a = 0; a < 3; ++a) cell = (cell << LOG2) | (uint32_t)fminf(fmaxf(o[a] * inv + half, 0.f), 2.f * half - 1.f);   // NaN -> 0
    return cell;
}

// Sort key of a ray of a ray list, so that the 64 rays of a wave run side by side: the cell of the origin on a
// 32^3 grid over the scene (15 bits), then the direction's code.
__global__ void k_ray_keys(const float *__restrict__ ray_o, const float *__restrict__ ray_d, const DstBounds *bounds,
                           uint32_t *__restrict__ keys, uint32_t *__restrict__ vals, uint32_t n) {
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    keys[r] = (origin_cell<5>(ray_o + 3 * (size_t)r, bounds) << 16) | direction_code(ray_d + 3 * (size_t)r);
    vals[r] = r;
}

// Order of a list traced by rows, in the call's scratch memory and in three launches: is the list in order as it comes
// (k_list_look), how many rays have each key (k_list_count, whose last workgroup makes of these where the keys' rays begin), the
// order (k_list_place).  The keys' sixteen bits go to what tells the rays apart: as many as it takes to tell the cells of
// an 8^3 grid that origins lie in, the rest to the direction.  A camera's rays have all sixteen for it.  Rays of one key
// follow in no order.  A list that comes in order (neighbours with nearly the same ray: a sensor's frame, rows of an image) keeps it,
// and rays from more than kListPlaces cells are unrelated and gain only by the number: from kOrderManyRays on.
// Bound by latency: 6 us to look, 28 to count 131,072 rays, 5 to place them; 13 in all for a list that keeps its order.
// As the rays come / like this, us evaluated and us a training step:
//   pixels of one camera, shuffled: room of a million surfels, 32,768 835 / 709 and 1454 / 1180, 65,536 1315 / 1084 and 2421 /
//   1755, 131,072 2293 / 1862 and 4350 / 3028; of 300,000, 32,768 179 / 218 and 430 / 430, 131,072 482 / 558 and 1116 / 1022;
//   sphere of 100,000, 65,536 616 / 417 and 1167 / 900, 131,072 1005 / 662 and 1963 / 1469
//   of 32 cameras, shuffled: room of a million, 65,536 876 / 740 and 1646 / 1426, 131,072 1531 / 1177 and 2772 / 2281
//   unrelated rays, sorted all the same: room of a million, 131,072 1261 / 1286 and 2392 / 2390, 262,144 2254 / 2160 and 4252 / 4086
//   a sensor's frame in order, sorted all the same: 131,072 of two million surfels 148 / 266 and 567 / 677; kept 167 and 587
// (A list of fewer than 65,536 rays loses by it in as many scenes as it gains.)
// Where quads cover the scene a few times at most (DstBounds::layers), a list of fewer than 262,144 rays that is only evaluated
// is not looked at.  As the rays come / like this, us evaluated, pixels of one camera, shuffled: room of 50,000 (1.4 layers), 65,536
// 97 / 118, 131,072 162 / 192, of 100,000 (2.9) 108 / 123 and 189 / 207, of 150,000 (4.3) 150 / 159 and 266 / 257, sphere of 30,000
// (6.1) 125 / 109 and 279 / 203; frames of a sensor, shuffled, 131,072 of 600,000 surfels (0.8) 211 / 196, of two million
// (2.5) 460 / 391, 65,536 62 / 90 and 90 / 104; 131,072 in order 165 / 174 and 331 / 339.  Training steps gain there too: 271 / 270
// and 467 / 462, 300 / 286 and 534 / 515, 620 / 518, 1324 / 1027, and lose in order 493 / 500 and 950 / 955.
constexpr uint32_t kListKeys = 65536u, kListCells = 512u, kListLooks = kListCells, kListThreads = 1024u, kListPlaces = 128u;
struct ListHead {
    uint32_t sorts;                // 0: as the rays come
    uint32_t direction_bits;
    uint32_t finished;             // workgroups that have counted their rays
    uint32_t pad[29];
    uint32_t place[kListCells];    // of a cell: its number among those where rays begin
    uint32_t start[kListKeys];     // rays of a key, then the place of its first
};
__global__ __launch_bounds__(kListLooks) void k_list_look(const float *__restrict__ ray_o, const float *__restrict__ ray_d, const DstBounds *bounds,
                                                            ListHead *__restrict__ head, uint32_t n) {
    if (blockIdx.x != 0u) {
        head->start[(blockIdx.x - 1u) * kListLooks + threadIdx.x] = 0u;
        return;
    }
    // places all over the list, one in every stretch of it, and at each a ray and the next one.  (Not at even distances: of an
    // image that is some power of two wide, row after row, every other one would be the end of a row.)
    __shared__ uint32_t s_cells[kListCells / 32u], s_alike;
    const uint32_t tid = threadIdx.x, within = (tid * 2654435769u) >> 16;   // in its stretch, in 1 / 65536
    const uint32_t at = (uint32_t)((((uint64_t)tid << 16) | within) * (n - 1u) / (kListLooks << 16));
    if (tid < kListCells / 32u) s_cells[tid] = 0u;
    if (tid == 0u) s_alike = 0u;
    const float *o = ray_o + 3 * (size_t)at, *d = ray_d + 3 * (size_t)at;   // (the next ray's lie behind them)
    const uint32_t cell = origin_cell<3>(o, bounds);
    const F3 d0 = ld3(d), d1 = ld3(d + 3), c = cross(d0, d1);
    const float off = fmaxf(fmaxf(fabsf(o[3] - o[0]), fabsf(o[4] - o[1])), fabsf(o[5] - o[2]));
    // a sixteenth of a radian, and of the scene's size
    const bool alike = dot(c, c) <= (1.f / 256.f) * (dot(d0, d0) * dot(d1, d1)) && dot(d0, d1) > 0.f && off <= (1.f / 16.f) * __uint_as_float(bounds->scale);
    const uint64_t wave_alike = wave_ballot(alike);
    __syncthreads();
    atomicOr(&s_cells[cell / 32u], 1u << (cell % 32u));
    if (__lane_id() == 0u) atomicAdd(&s_alike, (uint32_t)__popcll(wave_alike));
    __syncthreads();
    const uint32_t n_alike = s_alike;
    uint32_t before = 0u, all = 0u;
    for (uint32_t w = 0u; w < kListCells / 32u; ++w) {
        if (w < tid / 32u) before += (uint32_t)__popc(s_cells[w]);
        all += (uint32_t)__popc(s_cells[w]);
    }
    const uint32_t bits = all <= 1u ? 0u : 32u - (uint32_t)__clz(all - 1u);
    const uint32_t mine = s_cells[tid / 32u], bit = 1u << (tid % 32u);
    // (a cell that no ray looked at begins in: with one of the others)
    head->place[tid] = (mine & bit) != 0u ? before + (uint32_t)__popc(mine & (bit - 1u)) : tid & ((1u << bits) - 1u);
    if (tid == 0u) {
        head->sorts = n_alike < kListLooks / 4u * 3u && (all <= kListPlaces || n >= kOrderManyRays) ? 1u : 0u;
        head->direction_bits = 16u - bits;
        head->finished = 0u;
    }
}
__global__ __launch_bounds__(kListThreads) void k_list_count(const float *__restrict__ ray_o, const float *__restrict__ ray_d, const DstBounds *bounds,
                                                             ListHead *head, uint32_t *__restrict__ keys, uint32_t *__restrict__ ranks, uint32_t n) {
    if (head->sorts == 0u) return;
    __shared__ uint32_t s_last, s_sum[kListThreads / DST_WAVE];
    const uint32_t tid = threadIdx.x, r = blockIdx.x * kListThreads + tid, bits = head->direction_bits;
    if (r < n) {
        const uint32_t key = (head->place[origin_cell<3>(ray_o + 3 * (size_t)r, bounds)] << bits) | (direction_code(ray_d + 3 * (size_t)r) >> (16u - bits));
        keys[r] = key;
        ranks[r] = atomicAdd(&head->start[key], 1u);
    }
    __syncthreads();
    if (tid == 0u) {   // (one fence for the workgroup: one for every wave made this 60 us of 131,072 rays)
        __threadfence();
        s_last = atomicAdd(&head->finished, 1u) == gridDim.x - 1u ? 1u : 0u;
    }
    __syncthreads();
    if (s_last == 0u) return;
    __threadfence();
    // a wave's stretch of the keys, sixteen bytes a lane at a time
    constexpr uint32_t kSteps = kListKeys / (4u * kListThreads);
    const uint32_t lane = tid % DST_WAVE, wave = tid / DST_WAVE;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    u32x4 *const from = reinterpret_cast<u32x4 *>(head->start) + (size_t)wave * kSteps * DST_WAVE + lane;
    u32x4 count[kSteps];
    uint32_t upto[kSteps], sum = 0u;
#pragma unroll
    for (uint32_t k = 0; k < kSteps; ++k) count[k] = from[k * DST_WAVE];
#pragma unroll
    for (uint32_t k = 0; k < kSteps; ++k) {
        const uint32_t mine = (count[k].x + count[k].y) + (count[k].z + count[k].w);
        uint32_t run = mine;
#pragma unroll
        for (uint32_t off = 1u; off < (uint32_t)DST_WAVE; off <<= 1) {
            const uint32_t other = __shfl_up(run, off);
            if (lane >= off) run += other;
        }
        upto[k] = sum + run - mine;
        sum += __shfl(run, DST_WAVE - 1);
    }
    if (lane == 0u) s_sum[wave] = sum;
    __syncthreads();
    uint32_t base = 0u;
    for (uint32_t w = 0u; w < wave; ++w) base += s_sum[w];
#pragma unroll
    for (uint32_t k = 0; k < kSteps; ++k) {
        const uint32_t a = base + upto[k], b = a + count[k].x, c = b + count[k].y;
        from[k * DST_WAVE] = u32x4{a, b, c, c + count[k].z};
    }
}
// (head == nullptr: no scratch memory)
__global__ __launch_bounds__(kListThreads) void k_list_place(const ListHead *__restrict__ head, const uint32_t *__restrict__ keys, const uint32_t *__restrict__ ranks,
                                                             uint32_t *__restrict__ order, uint32_t n) {
    const uint32_t r = blockIdx.x * kListThreads + threadIdx.x;
    if (r >= n) return;
    order[head != nullptr && head->sorts != 0u ? head->start[keys[r]] + ranks[r] : r] = r;
}

__global__ void k_pack_half(const float *__restrict__ src, uint16_t *__restrict__ dst, uint64_t n) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        dst[i] = __builtin_bit_cast(uint16_t, (_Float16)src[i]);   // round to nearest even
}

struct TileGrid {
    int tw_log2, th_log2;
    uint32_t tiles_x, tiles_y, btiles_x, btiles_y;
};

// 8x8 pixel tiles per wave, 2x2 tiles per block.  A thin grid (H < 8: a (B,N,3) ray list) is one flat list of
// H*W rays in tiles of 1x64, traced in a coherent order of its own where that pays (k_ray_keys, k_list_look).
constexpr int kThinRows = 8;
TileGrid tile_grid(int H, int W) {
    TileGrid t;
    if (H < kThinRows) {
        W = H * W;
        H = 1;
    }
    t.th_log2 = 3;
    while (t.th_log2 > 0 && (1 << t.th_log2) > H) --t.th_log2;
    t.tw_log2 = 6 - t.th_log2;
    t.tiles_x = ((uint32_t)W + (1u << t.tw_log2) - 1) >> t.tw_log2;
    t.tiles_y = ((uint32_t)H + (1u << t.th_log2) - 1) >> t.th_log2;
    if (t.th_log2 == 0) {   // a list: a block is four consecutive tiles
        t.btiles_x = (t.tiles_x + 3) / 4;
        t.btiles_y = 1;
    } else {
        t.btiles_x = (t.tiles_x + 1) / 2;
        t.btiles_y = (t.tiles_y + 1) / 2;
    }
    return t;
}

// Tiles evaluate hits from the surfels' records with up to this many auxiliary channels.  (With eight, from the tensors / from
// records, us evaluated and recorded: 1080p room of a million 2549 / 2601 and 2970 / 2981, 1280x720 room of 300,000 582 / 591 and
// 710 / 716, 640x480 of 100,000 145 / 151 and 196 / 198, 800x800 sphere of 100,000 1347 / 1304 and 1519 / 1444.)
constexpr int kPackedAux = 4;

// `handover` / `hand_arg`: see trace_body (forward only; hand_arg steps = 0 launches the takers of the listed tiles).
template <bool BWD, bool REC>
void launch(const DstParams &p, const DstAccelView &acc, const TileGrid &t, const uint32_t *ray_order, hipStream_t stream,
            const uint32_t *block_order = nullptr, uint32_t *handover = nullptr, uint32_t hand_arg = 0u, bool first_bounce = false) {
    const uint32_t n_blocks = t.btiles_x * t.btiles_y;
    dim3 grid(n_blocks), block(kWavesPerBlock * DST_WAVE);
    const bool takers = !BWD && handover != nullptr && hand_arg == 0u;
    if (!BWD && kFwdWavesPerBlock == 1) {
        grid = dim3((n_blocks + 7u) / 8u * 32u);
        block = dim3(DST_WAVE);
        if (takers) grid = dim3(std::min<uint32_t>(n_blocks * (uint32_t)kWavesPerBlock, kHandCap));
    }
    // The per-lane walk is built into the kernels that meet waves of unrelated rays: reflection bounces and ray lists
    // (thin grids) of contexts that can hand tiles over, and of the backward trace without a record.
    // Order of the blocks of an image grid (trace_body): column strips put vertical neighbours on one XCD.  Evaluated,
    // strips of 8 / 16 blocks / row-major: 3.81 / 3.80 / 4.08 ms on 120 x 68 blocks (1080p, 1M surfels); strips of 8 /
    // row-major 1.87 / 1.85 ms on 50 x 50 blocks (a sphere in front of an empty background): with only two or three rounds
    // of workgroups on the chip the order decides more about the last round than about the caches.  Training steps with
    // strips of 8 / 16 / none in both directions: 10.74 / 10.66 / 10.99 ms and 3.70 / 3.67 / 3.67.
    uint32_t strip = 0u;
    if (t.th_log2 != 0) strip = BWD ? (uint32_t)DST_STRIP_BWD : (n_blocks >= kStripMinBlocks ? (uint32_t)DST_STRIP_FWD : 0u);
    const bool mixed = takers || (p.max_trace_depth > 0 && !first_bounce) || t.th_log2 < 3;   // first_bounce: forward, nothing beyond it
    const bool det = (p.flags & DST_FLAG_DETERMINISTIC) != 0u;
#define DST_LAUNCH_M(AUX, MIXED)                                                                                   \
    do {                                                                                                           \
        if (BWD && det)                                                                                            \
            hipLaunchKernelGGL((k_trace_bwd<AUX, REC, (MIXED) && !REC, true>), grid, block, 0, stream, p, acc,      \
                               t.tw_log2, t.th_log2, t.tiles_x, t.tiles_y, t.btiles_x, ray_order, strip, block_order);    \
        else if (BWD)                                                                                              \
            hipLaunchKernelGGL((k_trace_bwd<AUX, REC, (MIXED) && !REC, false>), grid, block, 0, stream, p, acc,     \
                               t.tw_log2, t.th_log2, t.tiles_x, t.tiles_y, t.btiles_x, ray_order, strip, block_order);    \
        else if (!(MIXED) && p.flags == 0u && handover == nullptr && p.scratch != nullptr && (AUX) <= kPackedAux)  \
            hipLaunchKernelGGL((k_trace_fwd_plain<AUX, REC, ((AUX) <= kPackedAux)>), grid, block, 0, stream, p, acc, t.tw_log2, \
                               t.th_log2, t.tiles_x, t.tiles_y, t.btiles_x, ray_order, strip, block_order);               \
        else if (!(MIXED) && p.flags == 0u && handover == nullptr)                                                 \
            hipLaunchKernelGGL((k_trace_fwd_plain<AUX, REC, false>), grid, block, 0, stream, p, acc, t.tw_log2,           \
                               t.th_log2, t.tiles_x, t.tiles_y, t.btiles_x, ray_order, strip, block_order);               \
        else if (p.flags != 0u)                                                                                    \
            hipLaunchKernelGGL((k_trace_fwd<AUX, REC, MIXED, true>), grid, block, 0, stream, p, acc, t.tw_log2,    \
                               t.th_log2, t.tiles_x, t.tiles_y, t.btiles_x, ray_order, strip, handover, hand_arg);        \
        else                                                                                                       \
            hipLaunchKernelGGL((k_trace_fwd<AUX, REC, MIXED, false>), grid, block, 0, stream, p, acc, t.tw_log2,   \
                               t.th_log2, t.tiles_x, t.tiles_y, t.btiles_x, ray_order, strip, handover, hand_arg);        \
    } while (0)
#define DST_LAUNCH(AUX)                                                                                            \
    do {                                                                                                           \
        if (mixed) DST_LAUNCH_M(AUX, true);                                                                        \
        else DST_LAUNCH_M(AUX, false);                                                                             \
    } while (0)
    if (p.aux <= 2) DST_LAUNCH(2);
    else if (p.aux <= 4) DST_LAUNCH(4);
    else DST_LAUNCH(8);
#undef DST_LAUNCH_M
#undef DST_LAUNCH
}

// How the rays of this grid are traced.  Tiles: a wave per 64 rays.  Rows (sixteen lanes per ray): lists, whose rays
// are unrelated, and images so small that waves of 64 rays leave most of the chip idle or end with a few long ones.
// TilesThenRows: images with reflections - the primary rays as tiles, the bounces beyond as rows.
// Up to 25,600 rays a record is written ray by ray.  Larger images' records have the tiles' layout, which rows can write as
// well (RowTiles), and which costs them some; images that are only evaluated need none.  Rows / tiles in us, evaluated:
// cube of 10,000 surfels 192x192 156 / 483, 320x320 277 / 430, 400x400 387 / 393; room of 200,000 101 / 381, 218 / 252,
// 327 / 222; sphere of 100,000 (whose limb makes tiles of a millisecond and more) 256 / 3753, 452 / 2357, 645 / 1881.
// Training steps: cube 192x192 772 / 1137, 256x256 859 / 1083, 320x320 953 / 1025; room 419 / 672, 500 / 571, 604 / 542;
// sphere 1007 / 4482, 1204 / 3991, 1465 / 3187.
#ifndef DST_ROW_REC_RAYS
#define DST_ROW_REC_RAYS 65536
#define DST_ROW_EVAL_RAYS 102400
#endif
constexpr uint64_t kRowRecordedRays = DST_ROW_REC_RAYS, kRowEvaluatedRays = DST_ROW_EVAL_RAYS;
enum class TraceBy { Tiles, Rows, TilesThenRows };
// An image by rows: four rays a wave, one to a row; the hardware hands the next four to whichever wave slot is free.
// Sixteen left one wave per SIMD on 128x128 rays (training step on the cube 804 -> 473 us with four) and let lists end with
// a few waves whose sixteen rays all run along the ground (131,072 lidar rays 3230 -> 2384).
RowGrid row_squares(const DstParams &p, RowGrid g) {
    g.batch_log2 = 2u;
    g.side_log2 = 1u;
    g.tiles_x = ((uint32_t)p.W + 1u) / 2u;
    g.tiles_y = ((uint32_t)p.H + 1u) / 2u;
    g.n_waves = g.tiles_x * g.tiles_y;
    return g;
}
TraceBy row_grid(const DstParams &p, const TileGrid &t, RowGrid &g) {
    const uint64_t rays = (uint64_t)p.H * p.W;
    g.record_header = record_header_words(rays, t.th_log2, (uint32_t)p.mtd_alloc + 1u, (uint64_t)t.btiles_x * t.btiles_y * kWavesPerBlock);
    if (!rows_may_trace(rays, t.th_log2)) {
        g.batch_log2 = 4u;
        g.side_log2 = 3u;
        g.tiles_x = t.btiles_x;
        g.tiles_y = t.btiles_y;
        g.n_waves = t.btiles_x * t.btiles_y * kWavesPerBlock;
        return p.max_trace_depth == 0 ? TraceBy::Tiles : TraceBy::TilesThenRows;
    }
    if (t.th_log2 == 0) {
        g.batch_log2 = 2u;
        g.side_log2 = 0u;
        g.tiles_x = g.n_waves = (uint32_t)((rays + 3u) / 4u);
        g.tiles_y = 0u;
    } else {
        g = row_squares(p, g);
    }
    return TraceBy::Rows;
}
template <bool REC, int KIND>
void launch_row_fwd(const DstParams &p, const DstAccelView &acc, const RowGrid &g, const uint32_t *ray_order, hipStream_t stream) {
    const dim3 grid(KIND != RowRays ? g.n_waves : (g.n_waves + 31u) / 32u * 32u), block(row_waves(KIND) * DST_WAVE);
#define DST_ROW(AUX)                                                                                                       \
    do {                                                                                                                   \
        if (p.flags != 0u) hipLaunchKernelGGL((k_row_fwd<AUX, REC, true, KIND, false>), grid, block, 0, stream, p, acc, g, ray_order); \
        else if (KIND == RowBeyond && p.scratch != nullptr) hipLaunchKernelGGL((k_row_fwd<AUX, REC, false, KIND, KIND == RowBeyond>), grid, block, 0, stream, p, acc, g, ray_order); \
        else hipLaunchKernelGGL((k_row_fwd<AUX, REC, false, KIND, false>), grid, block, 0, stream, p, acc, g, ray_order);  \
    } while (0)
    if (p.aux <= 2) DST_ROW(2);
    else if (p.aux <= 4) DST_ROW(4);
    else DST_ROW(8);
#undef DST_ROW
}
void launch_row_bwd(const DstParams &p, RowGrid g, const uint32_t *ray_order, hipStream_t stream) {
    // a workgroup takes sixteen rays: a square of an image, a stretch of a list
    g.batch_log2 = 4u;
    if (g.tiles_y == 0u) {
        g.n_waves = ((uint32_t)p.W + 15u) / 16u;
    } else {
        g.side_log2 = 2u;
        g.tiles_x = ((uint32_t)p.W + 3u) / 4u;
        g.n_waves = g.tiles_x * (((uint32_t)p.H + 3u) / 4u);
    }
    const dim3 grid(g.n_waves), block(kWavesPerBlock * DST_WAVE);
    const bool det = (p.flags & DST_FLAG_DETERMINISTIC) != 0u;
#define DST_ROW(AUX)                                                                                        \
    do {                                                                                                    \
        if (det) hipLaunchKernelGGL((k_row_bwd<AUX, true>), grid, block, 0, stream, p, g, ray_order);       \
        else hipLaunchKernelGGL((k_row_bwd<AUX, false>), grid, block, 0, stream, p, g, ray_order);          \
    } while (0)
    if (p.aux <= 2) DST_ROW(2);
    else if (p.aux <= 4) DST_ROW(4);
    else DST_ROW(8);
#undef DST_ROW
}

// What a forward trace keeps in its scratch memory.  Of a list: what its order is made with (k_list_look).  Of an image: the
// surfels' records, and behind them the guessed cost of every block and the order that follows from it.  Records are worth their
// pass where there are no more than four surfels to a ray (0.03 ns a surfel against 0.09 a ray of the 1080p room), the order on
// grids that are walked row by row, as the guess numbers their blocks (block_cost, block_of_position; larger grids are walked in
// strips, where it has not been tried.  3600 blocks, a 1280x720 room: of 300,000 surfels 504 / 503 us without and with, of a million
// 1903 / 1708), and a single launch in front of them more than pays for it only where tiles take long, which is where quads cover
// the scene many times over (DstBounds::layers).  Without / with, us: 800x800 sphere of 100,000 (20 layers) 1588 / 1124, 600x600 of
// 30,000 (6) 378 / 297, 500x500 of 20,000 (4) 204 / 218; room of a million (29) 640x360 1163 / 918, 960x540 1395 / 1175, of 200,000
// (6) 640x360 183 / 173, of 100,000 (3) 121 / 119, of 50,000 (1.4) 83 / 90, 480x270 63 / 75.  Records of that last room cost it 1 us.
constexpr uint64_t kOrderedBlocks = 4095u;
static_assert(kOrderedBlocks < kStripMinBlocks, "the guessed costs' blocks are numbered row by row, those of a launch in strips by strips");
constexpr float kOrderedLayers = 5.0f, kRecordedLayers = 2.0f;
struct ScratchLayout {
    uint64_t records, blocks, list;   // 0: none
    ScratchLayout(int32_t P, int32_t H, int32_t W) : records(0), blocks(0), list(0) {
        const uint64_t rays = (uint64_t)std::max(H, 0) * (uint64_t)std::max(W, 0);
        if (P > 0 && H < kThinRows && rays >= kOrderMinByRows) list = rays;
        if (P <= 0 || H < kThinRows || rays <= kRowRecordedRays) return;
        const TileGrid t = tile_grid(H, W);
        if (rays >= (uint64_t)P / 4u) records = (uint64_t)P;
        if ((uint64_t)t.btiles_x * t.btiles_y <= kOrderedBlocks) blocks = (uint64_t)t.btiles_x * t.btiles_y;
    }
    // Of these, what the kernels that trace this call read.
    ScratchLayout(const dst_ctx *ctx, const DstParams &p) : ScratchLayout(p.P, p.H, p.W) {
        const bool hands = kFwdWavesPerBlock == 1 && dst_handover_active(ctx);
        const bool by_rows = ctx->handover_mode != DST_HANDOVER_OFF && (uint64_t)p.H * p.W <= (p.hit_record != nullptr ? kRowRecordedRays : kRowEvaluatedRays);
        if (hands || (p.hit_record == nullptr && list < kOrderManyRays && ctx->layers < kOrderedLayers)) list = 0u;
        if (hands || by_rows || p.flags != 0u) records = blocks = 0u;
        if (ctx->layers < kOrderedLayers) blocks = 0u;   // (no number, of a scene on a line: many)
        if (ctx->layers < kRecordedLayers || (p.aux > kPackedAux && p.max_trace_depth == 0)) records = 0u;
    }
    uint64_t bytes() const {
        return list != 0u ? sizeof(ListHead) + 3u * sizeof(uint32_t) * list : sizeof(DstSurfel) * records + 2u * sizeof(uint32_t) * blocks;
    }
};
// The order of a list traced by rows: in `kept`, the record's room for it (from kOrderMinByRows rays on the backward trace counts
// on finding one there), or else in the scratch memory.  Without scratch memory as the rays come (nullptr: the same).
const uint32_t *order_list(const dst_ctx *ctx, const DstParams &p, uint32_t n, uint32_t *kept, hipStream_t stream) {
    ListHead *const head = ScratchLayout(ctx, p).list != 0u ? reinterpret_cast<ListHead *>(p.scratch) : nullptr;
    if (head == nullptr && kept == nullptr) return nullptr;
    const dim3 grid((n + kListThreads - 1u) / kListThreads), block(kListThreads);
    uint32_t *keys = nullptr, *ranks = nullptr, *order = kept;
    if (head != nullptr) {
        keys = reinterpret_cast<uint32_t *>(head + 1);
        ranks = keys + n;
        if (order == nullptr) order = ranks + n;
        hipLaunchKernelGGL(k_list_look, dim3(1u + kListKeys / kListLooks), dim3(kListLooks), 0, stream, p.ray_o, p.ray_d, ctx->bounds, head, n);
        hipLaunchKernelGGL(k_list_count, grid, block, 0, stream, p.ray_o, p.ray_d, ctx->bounds, head, keys, ranks, n);
    }
    hipLaunchKernelGGL(k_list_place, grid, block, 0, stream, head, keys, ranks, order, n);
    return order;
}
// Made where the kernels that read it are launched next, plain tiles and the rows beyond them.  Returns the order of the blocks
// (nullptr: as they lie), and takes from p.scratch what these kernels shall not look for.
const uint32_t *make_scratch(const dst_ctx *ctx, DstParams &p, const DstAccelView &acc, const TileGrid &t, hipStream_t stream) {
    if (p.scratch == nullptr) return nullptr;
    const ScratchLayout s(ctx, p);
    if (s.records == 0u && s.blocks == 0u) {
        p.scratch = nullptr;
        return nullptr;
    }
    uint32_t *const cost = reinterpret_cast<uint32_t *>(reinterpret_cast<DstSurfel *>(p.scratch) + s.records), *const order = cost + s.blocks;
    const uint32_t n_blocks = (uint32_t)s.blocks, threads = kPrepareWaves * DST_WAVE;
    const uint32_t grid = (n_blocks + kPrepareWaves - 1u) / kPrepareWaves + ((uint32_t)s.records + threads - 1u) / threads;
    hipLaunchKernelGGL(k_prepare, dim3(grid), dim3(threads), 0, stream, p, acc, t.btiles_x, cost, n_blocks);
    if (n_blocks != 0u) hipLaunchKernelGGL(k_cost_order, dim3(1), dim3(1024), 0, stream, cost, n_blocks, order);
    if (s.records == 0u) p.scratch = nullptr;
    return n_blocks != 0u ? order : nullptr;
}

void launch_close(const DstParams &p, uint32_t *out_of_range, hipStream_t stream) {
    const bool det = (p.flags & DST_FLAG_DETERMINISTIC) != 0u;
    if (!det && p.grad_rows == nullptr) return;   // the sums are in the caller's tensors already
    const dim3 grid(((uint32_t)p.P + kCloseSurfels - 1u) / kCloseSurfels), block(kCloseThreads);
#define DST_CLOSE(AUX)                                                                                              \
    do {                                                                                                            \
        if (det) hipLaunchKernelGGL((k_close_gradients<AUX, true>), grid, block, 0, stream, p, out_of_range);       \
        else hipLaunchKernelGGL((k_close_gradients<AUX, false>), grid, block, 0, stream, p, out_of_range);          \
    } while (0)
    if (p.aux <= 2) DST_CLOSE(2);
    else if (p.aux <= 4) DST_CLOSE(4);
    else DST_CLOSE(8);
#undef DST_CLOSE
}

}  // namespace

int dst_launch_pack_half(const float *src, uint16_t *dst, uint64_t n, hipStream_t stream) {
    const uint32_t blocks = (uint32_t)std::min<uint64_t>((n + 255u) / 256u, 4096u);
    hipLaunchKernelGGL(k_pack_half, dim3(blocks), dim3(256), 0, stream, src, dst, n);
    return hipGetLastError() == hipSuccess ? DST_OK : DST_E_DEVICE;
}

uint64_t dst_det_workspace_words(int32_t P, int32_t aux, int backward) {
    if (P <= 0 || aux < 1 || aux > DST_MAX_AUX) return 0;
    if (!backward) return (uint64_t)P;
    const int cols = aux <= 2 ? RowLayout<2>::cols : (aux <= 4 ? RowLayout<4>::cols : RowLayout<8>::cols);
    return (uint64_t)P * cols;
}

uint64_t dst_trace_scratch_bytes(int32_t P, int32_t H, int32_t W) { return ScratchLayout(P, H, W).bytes(); }
uint64_t dst_trace_scratch_needed(const dst_ctx *ctx, const DstParams *p) { return ctx != nullptr && p != nullptr ? ScratchLayout(ctx, *p).bytes() : 0u; }

uint64_t dst_hit_record_layout(int32_t H, int32_t W, int32_t mtd_alloc, uint32_t blocks, uint64_t *header_words,
                               uint32_t *n_waves) {
    if (H <= 0 || W <= 0 || mtd_alloc < 0) {
        if (header_words) *header_words = 0;
        if (n_waves) *n_waves = 0;
        return 0;
    }
    const TileGrid t = tile_grid(H, W);
    const uint64_t waves = (uint64_t)t.btiles_x * t.btiles_y * kWavesPerBlock;
    const uint64_t header = record_header_words((uint64_t)H * W, t.th_log2, (uint32_t)mtd_alloc + 1u, waves);
    if (header_words) *header_words = record_order_at((uint64_t)H * W, t.th_log2, (uint32_t)mtd_alloc + 1u, waves);
    if (n_waves) *n_waves = (uint32_t)waves;
    return header + (uint64_t)blocks * kRecBlockWords;
}

int dst_launch_trace(dst_ctx *ctx, const DstParams &p_in, bool backward, hipStream_t stream) {
    if (p_in.H <= 0 || p_in.W <= 0) {   // empty ray grid: nothing to do but to write gradients of zero where they are written
        if (backward && p_in.grad_touched != nullptr) {
            launch_close(p_in, ctx->handover + kDstHandoverOutOfRange, stream);
            DST_HIP(ctx, hipGetLastError());
        }
        return DST_OK;
    }
    DstParams p = p_in;
    if (!backward) {
        // Refits count the small quads too, on the device; the count comes over behind the first forward trace after
        // a refit (a 4-byte copy on this stream, nobody waits for it) and serves the traces after that one.
        if (ctx->bounds_host != nullptr && ctx->bounds != nullptr) {
            if (ctx->small_quads_asked) ctx->small_quads = *(volatile const uint32_t *)&ctx->bounds_host->small_quads;
            if (ctx->small_quads_refits != ctx->refits) {
                DST_HIP(ctx, hipMemcpyAsync(&ctx->bounds_host->small_quads, &ctx->bounds->small_quads, sizeof(uint32_t),
                                            hipMemcpyDeviceToHost, stream));
                ctx->small_quads_refits = ctx->refits;
                ctx->small_quads_asked = true;
            }
        }
    }
    const uint32_t *ray_order = nullptr, *row_order = nullptr;   // row_order: of a list traced by rows
    if (p.H < kThinRows) {
        // a ray list: flat, and (when it is long enough to matter: kOrderMinByRows) in an order that puts similar rays in one
        // wave.  The backward trace takes it from the record, and without a record makes its own (kOrderMinRays).
        if ((uint64_t)p.H * p.W > 0x7FFFFFFFull) return dst_fail(ctx, DST_E_INVALID, "ray grid too large");
        p.W = p.H * p.W;
        p.H = 1;
        const uint32_t n = (uint32_t)p.W;
        uint32_t *kept = nullptr;   // in the record, where the forward trace leaves it for the backward trace
        if (p.hit_record != nullptr) {
            const TileGrid t = tile_grid(1, p.W);
            kept = reinterpret_cast<uint32_t *>(p.hit_record + record_order_at(n, t.th_log2, (uint32_t)p.mtd_alloc + 1u, (uint64_t)t.btiles_x * t.btiles_y * kWavesPerBlock));
        }
        const bool by_rows = !backward && !(kFwdWavesPerBlock == 1 && dst_handover_active(ctx));
        if (backward && kept != nullptr) {   // (what the forward trace left there; nobody looks where it left nothing)
            if (n >= kOrderMinRays) ray_order = kept;
            if (n >= kOrderMinByRows) row_order = kept;
        } else if (by_rows) {
            if (n >= kOrderMinByRows) row_order = order_list(ctx, p, n, kept, stream);
        } else if (n >= kOrderMinRays) {
            if (n > ctx->ray_capacity) {
                for (int k = 0; k < 2; ++k) {
                    if (ctx->ray_keys[k]) (void)hipFree(ctx->ray_keys[k]);
                    if (ctx->ray_vals[k]) (void)hipFree(ctx->ray_vals[k]);
                    ctx->ray_keys[k] = ctx->ray_vals[k] = nullptr;
                }
                if (ctx->ray_hist) (void)hipFree(ctx->ray_hist);
                ctx->ray_hist = nullptr;
                ctx->ray_capacity = 0;
                for (int k = 0; k < 2; ++k) {
                    DST_HIP(ctx, hipMalloc((void **)&ctx->ray_keys[k], sizeof(uint32_t) * n));
                    DST_HIP(ctx, hipMalloc((void **)&ctx->ray_vals[k], sizeof(uint32_t) * n));
                }
                DST_HIP(ctx, hipMalloc((void **)&ctx->ray_hist, sizeof(uint32_t) * dst_sort_hist_elems(n)));
                ctx->ray_capacity = n;
            }
            uint32_t *vals[2] = {kept != nullptr ? kept : ctx->ray_vals[0], ctx->ray_vals[1]};
            hipLaunchKernelGGL(k_ray_keys, dim3((n + 255u) / 256u), dim3(256), 0, stream, p.ray_o, p.ray_d, ctx->bounds,
                               ctx->ray_keys[0], vals[0], n);
            dst_sort_pairs(ctx->ray_keys, vals, ctx->ray_hist, n, stream);
            ray_order = vals[0];
        }
    }
    const TileGrid t = tile_grid(p.H, p.W);
    if ((uint64_t)t.tiles_x * t.tiles_y > 0x3FFFFFFFull) return dst_fail(ctx, DST_E_INVALID, "ray grid too large");
    DstAccelView acc;
    acc.wide = ctx->wide;
    acc.leaves = ctx->leaves;
    acc.pre = ctx->pre;
    acc.bounds = ctx->bounds;
    acc.n_leaves = ctx->n_leaves;
    acc.root = dst_root_ref(ctx->n_leaves);
    const bool rec = p.hit_record != nullptr;
    const bool det = (p.flags & DST_FLAG_DETERMINISTIC) != 0u;
    uint32_t *const out_of_range = ctx->handover + kDstHandoverOutOfRange;   // (a spare word of the list's header)
    RowGrid rows;
    const TraceBy by = row_grid(p, t, rows);
    if (backward) {
        const uint32_t n_blocks = t.btiles_x * t.btiles_y;
        // the kernel that fits the record (complete, written ray by ray or wave by wave; incomplete) does the work
        if (rec && by == TraceBy::Rows) launch_row_bwd(p, rows, row_order, stream);
        if (rec && n_blocks < kOrderMinBlocks) {
            launch<true, true>(p, acc, t, ray_order, stream);
        } else if (rec) {
            // the replay takes its blocks longest first (the forward left every wave's chunk count in the record)
            if (n_blocks > ctx->block_order_capacity) {
                if (ctx->block_order) (void)hipFree(ctx->block_order);
                ctx->block_order = nullptr;
                ctx->block_order_capacity = 0;
                DST_HIP(ctx, hipMalloc((void **)&ctx->block_order, sizeof(uint32_t) * n_blocks));
                ctx->block_order_capacity = n_blocks;
            }
            const uint32_t strip = t.th_log2 != 0 ? (uint32_t)DST_STRIP_BWD : 0u;
            hipLaunchKernelGGL(k_block_order, dim3(1), dim3(1024), 0, stream,
                               reinterpret_cast<const uint32_t *>(p.hit_record + 3), (uint32_t)p.mtd_alloc + 1u, t.btiles_x,
                               t.btiles_y, strip, t.th_log2 != 0 ? 1 : 0, n_blocks, ctx->block_order);
            launch<true, true>(p, acc, t, ray_order, stream, ctx->block_order);   // does the work if the record is complete,
        }
        launch<true, false>(p, acc, t, ray_order, stream);           // else this one does (it returns at once otherwise)
        launch_close(p, out_of_range, stream);
    } else {
        const uint32_t steps = std::max<uint32_t>(ctx->handover_steps, 1u);
        // the second launch of each pair traces the tiles the first one handed over (usually none: it leaves at once)
        uint32_t *const list = (kFwdWavesPerBlock == 1 && dst_handover_active(ctx)) ? ctx->handover : nullptr;
        // A hand-over mode is about tiles, so contexts that can hand them over (list != nullptr) and, for images without
        // reflections, contexts told not to (DST_HANDOVER_OFF) trace by tiles: OFF against AUTO shows what the hand-over is
        // worth, tile by tile.  Rows need none and would be faster for all of these: the ball of small quads above, 64x64,
        // takes 29.9 ms with OFF, 2.8 with the hand-over and 0.24 by rows, a list of 20,000 rays there 813 and 290 us, a
        // 637x1013 room with one reflection 5.5 ms against 3.5.
        if (by == TraceBy::Rows && list == nullptr && (ctx->handover_mode != DST_HANDOVER_OFF || p.max_trace_depth > 0 || t.th_log2 < 3)) {
            if (rec) launch_row_fwd<true, RowRays>(p, acc, rows, row_order, stream);
            else launch_row_fwd<false, RowRays>(p, acc, rows, row_order, stream);
        } else if (by != TraceBy::Rows && list == nullptr && ctx->handover_mode != DST_HANDOVER_OFF &&
                   (uint64_t)p.H * p.W <= (rec ? kRowRecordedRays : kRowEvaluatedRays)) {
            if (rec) launch_row_fwd<true, RowTiles>(p, acc, rows, ray_order, stream);
            else launch_row_fwd<false, RowRays>(p, acc, row_squares(p, rows), ray_order, stream);
        } else if (by == TraceBy::TilesThenRows && list == nullptr) {
            const uint32_t *const order = make_scratch(ctx, p, acc, t, stream);
            if (rec) {
                launch<false, true>(p, acc, t, ray_order, stream, order, nullptr, 0u, true);
                launch_row_fwd<true, RowBeyond>(p, acc, rows, ray_order, stream);
            } else {
                launch<false, false>(p, acc, t, ray_order, stream, order, nullptr, 0u, true);
                launch_row_fwd<false, RowBeyond>(p, acc, rows, ray_order, stream);
            }
        } else
        for (int pass = 0; pass < (list != nullptr ? 2 : 1); ++pass) {
            const uint32_t arg = pass == 0 ? steps : 0u;
            const uint32_t *const order = list == nullptr && t.th_log2 == 3 ? make_scratch(ctx, p, acc, t, stream) : nullptr;
            if (rec) launch<false, true>(p, acc, t, ray_order, stream, order, list, arg);
            else launch<false, false>(p, acc, t, ray_order, stream, order, list, arg);
        }
        if (det && p.training && p.a_weights != nullptr)
            hipLaunchKernelGGL(k_det_finish_weights, dim3(1024), dim3(256), 0, stream, p, out_of_range);
        if (rec && p.hit_record_asked != nullptr)
            DST_HIP(ctx, hipMemcpyAsync(p.hit_record_asked, p.hit_record, sizeof(uint64_t), hipMemcpyDeviceToHost, stream));
    }
    DST_HIP(ctx, hipGetLastError());
    return DST_OK;
}
