// gfx950 kernels of the render path.
//
//   k_face      per face: MVP transform of the three corners, backface test,
//               lighting, frustum clipping (wave-cooperative Sutherland-Hodgman
//               with ballot/popcount compaction), perspective divide + screen
//               transform, full-screen bin test, raster set-up. One workgroup
//               = 256 faces = 1792 slots in draw order. The workgroup then
//               counts its tile references in LDS and adds them to the global
//               tile counts.
//   k_bin_scan  one workgroup per frame: tile counts -> tile-list offsets, and
//               the slabs of tiles whose lists are split.
//   k_bin_fill  per face workgroup: scatter slots into tile lists, with one
//               global atomic per distinct tile per workgroup.
//   k_raster    one workgroup per screen tile or part of a split tile's list:
//               triangles staged in LDS,
//               visibility with a 64-bit (depth, draw-sequence) max key in LDS,
//               one deferred shading pass and a single write of colour + depth.
//
// Every float32 expression keeps the reference's evaluation order; the build
// uses -ffp-contract=off and correctly rounded division/sqrt.
#pragma clang fp contract(off)


#include <algorithm>
#include <cstddef>
#include <cstring>

#include "gr_device.h"
#include "gr_launch.h"

namespace gr {

// ---------------------------------------------------------------------------
// Go conversion semantics
// ---------------------------------------------------------------------------

// int(float32) on amd64 (CVTTSS2SQ): truncation, NaN/out of range -> INT64_MIN.
__device__ __forceinline__ int64_t go_int(float x) {
    if (!(x >= -9223372036854775808.0f && x < 9223372036854775808.0f)) return INT64_MIN;
    if (x > -2147483648.0f && x < 2147483648.0f) return (int64_t)(int32_t)x;
    return (int64_t)x;
}

// uint8(float32): CVTTSS2SL then the low byte; NaN/out of int32 range -> 0.
// One compare: -2^31 itself converts to INT32_MIN, whose low byte is 0 too.
__device__ __forceinline__ uint32_t go_uint8(float x) {
    return __builtin_fabsf(x) < 2147483648.0f ? (uint32_t)(int32_t)x & 0xFFu : 0u;
}

__device__ __forceinline__ int64_t wadd(int64_t a, int64_t b) {
    return (int64_t)((uint64_t)a + (uint64_t)b);
}
__device__ __forceinline__ int64_t wsub(int64_t a, int64_t b) {
    return (int64_t)((uint64_t)a - (uint64_t)b);
}
__device__ __forceinline__ int64_t wmul(int64_t a, int64_t b) {
    return (int64_t)((uint64_t)a * (uint64_t)b);
}

// Lanes of the wave for which p holds, as the compare's own mask (__ballot makes an
// integer of p and compares that: two more vector instructions).
__device__ __forceinline__ uint64_t ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }

// Load and store of one value through a global-address-space pointer: the
// pointers of DevFrame and DevMesh are generic, and a generic (flat) access
// also counts against the LDS wait counter, so a later LDS wait would wait for
// it too.
template <typename T>
__device__ __forceinline__ T gld(const T* p) {
    return *(const __attribute__((address_space(1))) T*)p;
}
template <typename T>
__device__ __forceinline__ void gst(T* p, T v) {
    *(__attribute__((address_space(1))) T*)p = v;
}
// Load of a 16-byte-aligned record through a global-address-space pointer
// (global_load rather than flat, so LDS traffic is not waited on with it).
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
template <typename T>
__device__ __forceinline__ T gload(const T* p) {
    static_assert(sizeof(T) % 16 == 0 && alignof(T) >= 16, "16-byte records only");
    typedef const __attribute__((address_space(1))) u32x4* gptr;
    const gptr src = (gptr)p;
    u32x4 tmp[sizeof(T) / 16];
#pragma unroll
    for (int i = 0; i < (int)(sizeof(T) / 16); i++) tmp[i] = src[i];
    T out;
    __builtin_memcpy(&out, tmp, sizeof(T));
    return out;
}

// Store of a 16-byte-aligned record through a global-address-space pointer.
template <typename T>
__device__ __forceinline__ void gstore(T* p, const T& v) {
    static_assert(sizeof(T) % 16 == 0 && alignof(T) >= 16, "16-byte records only");
    typedef __attribute__((ext_vector_type(4))) uint32_t v4;
    typedef __attribute__((address_space(1))) v4* gptr;
    v4 tmp[sizeof(T) / 16];
    __builtin_memcpy(tmp, &v, sizeof(T));
    const gptr dst = (gptr)p;
#pragma unroll
    for (int i = 0; i < (int)(sizeof(T) / 16); i++) dst[i] = tmp[i];
}

// A*x + B*y + C in wrapping 32-bit arithmetic, for A, B, x, y that fit 24
// bits signed, as two multiply-adds (v_mad_i32_i24). The empty asm keeps the
// partial sum whole, so that the compiler does not turn the two products and
// two additions into two multiplies and a three-operand add.
__device__ __forceinline__ uint32_t edge24(int A, int x, int B, int y, uint32_t C) {
    uint32_t u = (uint32_t)__mul24(B, y) + C;
    asm("" : "+v"(u));
    return (uint32_t)__mul24(A, x) + u;
}

// ---------------------------------------------------------------------------
// Exact float32 division from a correctly rounded reciprocal
// ---------------------------------------------------------------------------

// |d| in [2^-40, 2^41): quotients a/d of numerators in [2^-70, 2^70] then keep
// every intermediate of div_rcp in the normal range.
__device__ __forceinline__ bool rcp_range(float d) {
    const uint32_t e = (__float_as_uint(d) >> 23) & 0xFFu;
    return e - (127u - 40u) <= 80u;
}

// RN(a / d) given y = RN(1 / d). q0 = RN(a*y) is within 1.5 ulp of a/d; one
// residual correction brings it within 1 ulp; with y the correctly rounded
// reciprocal and q within 1 ulp, the residual a - d*q is exact and
// RN(q + r*y) = RN(a/d) (Markstein, IBM J. Res. Dev. 34(1), 1990; the
// Handbook of Floating-Point Arithmetic states it for any precision p).
// Domain: d with rcp_range(d), a == +0 or 2^-70 <= |a| <= 2^70 (a == -0
// would come back as +0 for d > 0). For another y see rcp_step.
__device__ __forceinline__ float div_rcp(float a, float d, float y) {
    float q = a * y;
    float r = __builtin_fmaf(-d, q, a);
    q = __builtin_fmaf(r, y, q);
    r = __builtin_fmaf(-d, q, a);
    return __builtin_fmaf(r, y, q);
}

// A reciprocal of d for several quotients by the same divisor: the hardware's, and
// one Newton step. It need not be the correctly rounded one, which div_rcp's theorem
// asks for; that div_rcp(a, d, rcp_step(d)) is RN(a / d) all the same, for |d| in
// [2^-41, 2^42] and |a| in [2^-80, 2^86], is what gr_check_exact_division tests.
__device__ __forceinline__ float rcp_step(float d) {
    const float y = __builtin_amdgcn_rcpf(d);
    return __builtin_fmaf(__builtin_fmaf(-d, y, 1.0f), y, y);
}

// ---------------------------------------------------------------------------
// Vector helpers in reference order
// ---------------------------------------------------------------------------

// asm_purego.go:9-19 / matrix.go:167-173: ((m0*x + m1*y) + m2*z) + m3*w per row.
__device__ __forceinline__ float4 xform(const float* m, float x, float y, float z, float w) {
    float4 r;
    r.x = m[0] * x + m[1] * y + m[2] * z + m[3] * w;
    r.y = m[4] * x + m[5] * y + m[6] * z + m[7] * w;
    r.z = m[8] * x + m[9] * y + m[10] * z + m[11] * w;
    r.w = m[12] * x + m[13] * y + m[14] * z + m[15] * w;
    return r;
}

// vector.go:115-125 (Vec4.Length + Divide, W dropped by ToVec3), then the
// Lambert term of renderer.go:331 / 336-337.
__device__ __forceinline__ float lambert(float4 n, const float* light, float ambient,
                                         float diffuse) {
    float len = __builtin_sqrtf(n.x * n.x + n.y * n.y + n.z * n.z + n.w * n.w);
    float x = n.x / len, y = n.y / len, z = n.z / len;
    float d = x * light[0] + y * light[1] + z * light[2];
    return ambient + d * diffuse;
}

// Clip-space vertex with its attributes.
struct CV {
    float x, y, z, w, u, v, i;
};

// clipping.go:93-129 plane (point, normal) for index p in draw order
// Left, Right, Top, Bottom, Near, Far.
__device__ __forceinline__ void plane_of(int p, float zn, float zf, float4& P, float4& N) {
    switch (p) {
    case 0: P = make_float4(-1.f, 0.f, 0.f, 1.f); N = make_float4(1.f, 0.f, 0.f, 1.f); break;
    case 1: P = make_float4(1.f, 0.f, 0.f, 1.f); N = make_float4(-1.f, 0.f, 0.f, 1.f); break;
    case 2: P = make_float4(0.f, -1.f, 0.f, 1.f); N = make_float4(0.f, 1.f, 0.f, 1.f); break;
    case 3: P = make_float4(0.f, 1.f, 0.f, 1.f); N = make_float4(0.f, -1.f, 0.f, 1.f); break;
    case 4: P = make_float4(0.f, 0.f, zn, 1.f); N = make_float4(0.f, 0.f, -1.f, 0.f); break;
    default: P = make_float4(0.f, 0.f, zf, 1.f); N = make_float4(0.f, 0.f, 1.f, 0.f); break;
    }
}

// clipping.go:74-76: (q - P) . N <= 0
__device__ __forceinline__ bool inside(const float4& P, const float4& N, const CV& q) {
    float d = (q.x - P.x) * N.x + (q.y - P.y) * N.y + (q.z - P.z) * N.z + (q.w - P.w) * N.w;
    return d <= 0.f;
}

// clipping.go:79-86 with q0 = A, q1 = B, then lerp32 / lerpUV (clipping.go:156-165).
__device__ __forceinline__ CV intersect(const float4& P, const float4& N, const CV& A,
                                        const CV& B) {
    float ux = B.x - A.x, uy = B.y - A.y, uz = B.z - A.z, uw = B.w - A.w;
    float wx = A.x - P.x, wy = A.y - P.y, wz = A.z - P.z, ww = A.w - P.w;
    float d = N.x * ux + N.y * uy + N.z * uz + N.w * uw;
    float n = -(N.x * wx + N.y * wy + N.z * wz + N.w * ww);
    float f = n / d;
    CV r;
    r.x = A.x + ux * f;
    r.y = A.y + uy * f;
    r.z = A.z + uz * f;
    r.w = A.w + uw * f;
    r.i = A.i + (B.i - A.i) * f;
    r.u = A.u + (B.u - A.u) * f;
    r.v = A.v + (B.v - A.v) * f;
    return r;
}

// Inside bits of a vertex for the 6 planes (bit p = inside plane p).
__device__ __forceinline__ uint32_t inside_mask(const CV& q, float zn, float zf) {
    uint32_t m = 0;
#pragma unroll
    for (int p = 0; p < 6; p++) {
        float4 P, N;
        plane_of(p, zn, zf, P, N);
        m |= inside(P, N, q) ? (1u << p) : 0u;
    }
    return m;
}

// renderer.go:246-250 (clip space, before the divide).
__device__ __forceinline__ bool facing_camera(const float4& v0, const float4& v1,
                                              const float4& v2) {
    float ax = v1.x - v0.x, ay = v1.y - v0.y, az = v1.z - v0.z;
    float bx = v2.x - v0.x, by = v2.y - v0.y, bz = v2.z - v0.z;
    float nx = ay * bz - az * by;
    float ny = az * bx - ax * bz;
    float nz = ax * by - ay * bx;
    float d = nx * (0.f - v0.x) + ny * (0.f - v0.y) + nz * (0.f - v0.z);
    return d > 0.f;
}

// Units x, x + 8, x + 16, ... of a frame with n units run on XCD x.
__host__ __device__ __forceinline__ int xcd_count(int x, int n) {
    return n > x ? (n - x + 7) >> 3 : 0;
}

// Last index i in [0, n) with key[i] <= b (key[0] <= b, keys ascending), by the
// 64 lanes of a wave at once: one round trip to memory per factor of 64, where a
// binary search takes one per factor of 2 (9 for the 512 frames of a batch, on
// the path of every face block and every tile).
template <typename T>
__device__ __forceinline__ int wave_last_le(const T* key, int n, T b) {
    if (n == 1) return 0;
    const int lane = (int)(threadIdx.x & 63u);
    int lo = 0, len = n;
    while (len > 64) {
        const int step = (len + 63) >> 6;
        const bool le = lane * step < len && gld(&key[lo + lane * step]) <= b;
        const int k = __popcll(ballot(le)) - 1;
        lo += k * step;
        len = min(step, len - k * step);
    }
    const bool le = lane < len && gld(&key[lo + lane]) <= b;
    return lo + __popcll(ballot(le)) - 1;
}

// Workgroup h -> (frame, unit within the frame) in the XCD-aware order: the
// hardware places workgroup h on XCD h % 8, and XCD x takes units x, x + 8, ...
// of every frame, frame after frame, so a unit's inputs stay in one XCD's L2
// across the frames of a batch while neighbouring units (whose cost varies
// together) spread over all XCDs. Returns false for the padding workgroups.
__device__ __forceinline__ bool xcd_unit(const int* table, int nframes, int h, int& f,
                                         int& local) {
    const int x = h & 7, k = h >> 3;
    const int* P = table + x * (nframes + 1);
    if (k >= P[nframes]) return false;
    f = wave_last_le(P, nframes, k);
    local = x + 8 * (k - P[f]);
    return true;
}

__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// The wave's total of a per-lane count that only lane 0 holds in the common
// case (the raster's covered-fragment count is wave-uniform except on the
// int64 path): the full reduction runs only when another lane holds a count.
__device__ __forceinline__ unsigned long long wave_total(unsigned long long v, int lane) {
    if (ballot(v != 0ull && lane != 0) == 0ull)
        return __builtin_amdgcn_readfirstlane((unsigned)v) |
               ((unsigned long long)__builtin_amdgcn_readfirstlane((unsigned)(v >> 32)) << 32);
    return wave_sum_u64(v);
}

// Reduction of v over the wave's 64 lanes (all active) with an associative,
// commutative f of identity `none`, in vector instructions (data-parallel
// primitives: shifts within rows of 16, then row broadcasts), no LDS traffic.
// The result is wave-uniform.
template <typename F>
__device__ __forceinline__ uint32_t wave_reduce(uint32_t v, uint32_t none, F f) {
#define GR_DPP(ctrl, rows) \
    v = f(v, (uint32_t)__builtin_amdgcn_update_dpp((int)none, (int)v, ctrl, rows, 0xF, false))
    GR_DPP(0x111, 0xF);  // row_shr:1
    GR_DPP(0x112, 0xF);  // row_shr:2
    GR_DPP(0x114, 0xF);  // row_shr:4
    GR_DPP(0x118, 0xF);  // row_shr:8: lane 15 of each row holds its row
    GR_DPP(0x142, 0xA);  // row_bcast:15 into rows 1 and 3
    GR_DPP(0x143, 0xC);  // row_bcast:31 into rows 2 and 3
#undef GR_DPP
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// Inclusive sums over the lanes of the wave (all active), by the same steps.
__device__ __forceinline__ uint32_t wave_scan_u32(uint32_t v) {
#define GR_DPP(ctrl, rows) \
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, rows, 0xF, false)
    GR_DPP(0x111, 0xF);
    GR_DPP(0x112, 0xF);
    GR_DPP(0x114, 0xF);
    GR_DPP(0x118, 0xF);
    GR_DPP(0x142, 0xA);
    GR_DPP(0x143, 0xC);
#undef GR_DPP
    return v;
}
// The same in 64 bits, from the sums of the 16-bit halves.
__device__ __forceinline__ unsigned long long wave_scan_u64(uint32_t v) {
    return (unsigned long long)wave_scan_u32(v & 0xFFFFu) +
           ((unsigned long long)wave_scan_u32(v >> 16) << 16);
}

__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t v) {
    return wave_reduce(v, 0u, [](uint32_t a, uint32_t b) { return a + b; });
}

// Maximum of each 16-bit half, unsigned.
__device__ __forceinline__ uint32_t max_u16x2(uint32_t a, uint32_t b) {
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t,
                              __builtin_elementwise_max(__builtin_bit_cast(u16x2, a),
                                                        __builtin_bit_cast(u16x2, b)));
}
__device__ __forceinline__ uint32_t wave_max_u16x2(uint32_t v) {
    return wave_reduce(v, 0u, [](uint32_t a, uint32_t b) { return max_u16x2(a, b); });
}

__device__ __forceinline__ uint64_t lanemask_lt(int lane) { return (1ull << lane) - 1ull; }

__device__ __forceinline__ CV shfl_cv(const CV& a, int src) {
    CV r;
    r.x = __shfl(a.x, src, 64);
    r.y = __shfl(a.y, src, 64);
    r.z = __shfl(a.z, src, 64);
    r.w = __shfl(a.w, src, 64);
    r.u = __shfl(a.u, src, 64);
    r.v = __shfl(a.v, src, 64);
    r.i = __shfl(a.i, src, 64);
    return r;
}

// ---------------------------------------------------------------------------
// Wave-cooperative ClipTriangle (clipping.go:167-236)
// ---------------------------------------------------------------------------

// Every lane passes the same triangle (a, b, c). Per plane pass, lane k owns
// edge (k, (k+1) % n) of the polygon and contributes [X, A], [A], [X] or []
// exactly as the reference's loop body; ballots give each lane its output
// position. The polygon ping-pongs between buf0 and buf1 in LDS (one pair per
// wave) and ends in buf0 after the 6 passes. Returns the final vertex count
// (uniform), 0 when clipped away, -1 when a pass would exceed 9 vertices.
__device__ int wave_clip(CV* buf0, CV* buf1, const CV& a, const CV& b, const CV& c, float zn,
                         float zf, int lane) {
    if (lane == 0) buf0[0] = a;
    if (lane == 1) buf0[1] = b;
    if (lane == 2) buf0[2] = c;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    int n = 3;
    CV* in = buf0;
    CV* out = buf1;
    for (int p = 0; p < 6; p++) {
        float4 P, N;
        plane_of(p, zn, zf, P, N);
        const bool act = lane < n;
        const int ai = act ? (lane + 1 == n ? 0 : lane + 1) : 0;
        const CV A = in[ai];
        const CV B = in[act ? lane : 0];
        const bool ia = act && inside(P, N, A);
        const bool ib = act && inside(P, N, B);
        const bool one = ia || ib;     // at least one output vertex
        const bool two = ia && !ib;    // [X, A]
        const uint64_t b1 = ballot(one), b2 = ballot(two);
        const uint64_t lt = lanemask_lt(lane);
        const int pos = __popcll(b1 & lt) + __popcll(b2 & lt);
        const int m = __popcll(b1) + __popcll(b2);
        if (m > kMaxClip) return -1;
        if (m == 0) return 0;
        if (ia != ib) {
            CV X = intersect(P, N, A, B);
            out[pos] = X;
            if (two) out[pos + 1] = A;
        } else if (one) {
            out[pos] = A;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        n = m;
        CV* t = in;
        in = out;
        out = t;
    }
    return n;
}

// ---------------------------------------------------------------------------
// Per-lane clipping of a triangle that straddles one plane
// ---------------------------------------------------------------------------

__device__ __forceinline__ CV sel(bool c, const CV& a, const CV& b) {
    CV r;
    r.x = c ? a.x : b.x;
    r.y = c ? a.y : b.y;
    r.z = c ? a.z : b.z;
    r.w = c ? a.w : b.w;
    r.u = c ? a.u : b.u;
    r.v = c ? a.v : b.v;
    r.i = c ? a.i : b.i;
    return r;
}

// Append v at position m of q[0..3] with register selects (no dynamic index).
__device__ __forceinline__ void append4(CV q[4], int& m, const CV& v) {
#pragma unroll
    for (int k = 0; k < 4; k++) q[k] = sel(m == k, v, q[k]);
    m++;
}

// ClipTriangle for a triangle whose three vertices are inside the planes before
// p and straddle plane p (at least one vertex inside). Passes before p only
// rotate the triangle left by one (clipping.go:204-224 with every vertex
// inside), so plane p sees it rotated by p mod 3; the pass over p runs the
// reference's edge loop. Each later plane is then either passed by every
// vertex (a pure rotation), failed by every vertex (the reference returns 0 at
// that pass, clipping.go:227-229), or straddled: only the last case needs the
// full clipper. Returns -1 for it, 0 when clipped away, otherwise the vertex
// count (3 or 4) of the final polygon in q.
__device__ int clip_one_plane(int p, const CV& c0, const CV& c1, const CV& c2, float zn,
                              float zf, CV q[4]) {
    const int r = p % 3;
    const CV R0 = sel(r == 0, c0, sel(r == 1, c1, c2));
    const CV R1 = sel(r == 0, c1, sel(r == 1, c2, c0));
    const CV R2 = sel(r == 0, c2, sel(r == 1, c0, c1));
    float4 P, N;
    plane_of(p, zn, zf, P, N);
    const bool i0 = inside(P, N, R0), i1 = inside(P, N, R1), i2 = inside(P, N, R2);
    q[0] = q[1] = q[2] = q[3] = R0;
    int m = 0;
    // edges b = 0, 1, 2 with A = R[(b+1) % 3], B = R[b]
    const CV As[3] = {R1, R2, R0}, Bs[3] = {R0, R1, R2};
    const bool iA[3] = {i1, i2, i0}, iB[3] = {i0, i1, i2};
#pragma unroll
    for (int b = 0; b < 3; b++) {
        if (iA[b]) {
            if (!iB[b]) append4(q, m, intersect(P, N, As[b], Bs[b]));
            append4(q, m, As[b]);
        } else if (iB[b]) {
            append4(q, m, intersect(P, N, As[b], Bs[b]));
        }
    }
    int rot = 0;
#pragma unroll
    for (int pl = 0; pl < 6; pl++) {
        if (pl <= p) continue;
        float4 P2, N2;
        plane_of(pl, zn, zf, P2, N2);
        int nin = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) nin += (k < m && inside(P2, N2, q[k])) ? 1 : 0;
        if (nin == 0) return 0;
        if (nin != m) return -1;
        rot++;
    }
    // `rot` more left rotations of an m-gon.
    rot %= m;
    CV t[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        // t[k] = q[(k + rot) % m]
        const int s3 = (k + rot) % 3, s4 = (k + rot) % 4;
        const int s = m == 3 ? s3 : s4;
        t[k] = sel(s == 0, q[0], sel(s == 1, q[1], sel(s == 2, q[2], q[3])));
    }
#pragma unroll
    for (int k = 0; k < 4; k++) q[k] = t[k];
    return m;
}

// ---------------------------------------------------------------------------
// Triangle set-up
// ---------------------------------------------------------------------------

// Per-lane counters of k_face packed in one word (one register for the whole
// kernel): TPF references in bits 0-15, binned triangles 16-23, front faces
// 24-27, clip overflows 28-31. A lane owns kFacesPerLane faces in pass 1 (at
// most 4 front faces) and, over at most 4 rounds of pass 2, at most 4 clip
// overflows and ~40 triangles of at most 16 references each: below these
// widths, and a wave's sums of the 16-bit fields stay below 2^16.
struct FaceStats {
    uint32_t packed;
};

// Box words of a record that is not rasterised: first 1, last 0.
constexpr uint32_t kEmptyBox = 1u;

// ---------------------------------------------------------------------------
// Debug overlays (renderer.go:191-216): lines and 3x3 rects write colour only,
// after their triangle's face, in draw order. Each overlay pixel keeps the max
// of (slot + 1) << 1 | vertex; the raster's shading pass shows the overlay
// where it comes at or after the depth winner (within a triangle the vertex
// rects are drawn last).
// ---------------------------------------------------------------------------

constexpr uint32_t kEdgeColor = 0xFF000000u;    // {0,0,0,255} (renderer.go:19)
constexpr uint32_t kVertexColor = 0xFF00A1FFu;  // {255,161,0,255} (renderer.go:18)
constexpr uint32_t kWhite = 0xFFFFFFFFu;        // edges without faces (renderer.go:194)

// utils.go:11-21: minInt maps to maxInt.
__device__ __forceinline__ int64_t go_abs(int64_t v) {
    if (v < 0) v = wsub(0, v);
    if (v < 0) v = wsub(v, 1);
    return v;
}

// Key maximum through a global-address-space pointer (see gld).
__device__ __forceinline__ void ov_key(const DevFrame& fr, uint32_t idx, uint32_t code) {
    typedef __attribute__((address_space(1))) uint32_t* gptr;
    __hip_atomic_fetch_max((gptr)(fr.okey + idx), code, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// FrameBuffer.Pixel (rasterizer.go:25-30): only the flat index is checked.
__device__ __forceinline__ void ov_pixel(const DevFrame& fr, int64_t x, int64_t y, uint32_t code) {
    const int64_t idx = wadd(wmul(y, (int64_t)fr.W), x);
    if (idx > 0 && idx < (int64_t)fr.W * fr.H) ov_key(fr, (uint32_t)idx, code);
}

// The same for |x|, |y| <= 2^16: flat indexes fit int32 (W <= 2^14).
constexpr int64_t kNear = 1 << 16;
__device__ __forceinline__ void ov_pixel32(const DevFrame& fr, int x, int y, uint32_t code) {
    const int idx = y * fr.W + x;
    if ((uint32_t)(idx - 1) < (uint32_t)(fr.W * fr.H - 1)) ov_key(fr, (uint32_t)idx, code);
}
__device__ __forceinline__ bool near_origin(int64_t x, int64_t y) {
    return x >= -kNear && x <= kNear - 4 && y >= -kNear && y <= kNear - 4;
}

// FrameBuffer.Rect (rasterizer.go:54-63) with width = height = 3.
__device__ __forceinline__ void ov_rect(const DevFrame& fr, int64_t x, int64_t y, uint32_t code) {
    if (x >= fr.W || y >= fr.H) return;
    if (near_origin(x, y)) {
#pragma unroll
        for (int k = 0; k < 9; k++) ov_pixel32(fr, (int)x + k % 3, (int)y + k / 3, code);
        return;
    }
    for (int64_t py = y; py < wadd(y, 3); py = wadd(py, 1))
        for (int64_t px = x; px < wadd(x, 3); px = wadd(px, 1)) ov_pixel(fr, px, py, code);
}

// FrameBuffer.Line (rasterizer.go:65-79): a float32 DDA accumulated step by step.
// Returns false, drawing nothing, for a line longer than kMaxOverlayLine.
__device__ __forceinline__ bool ov_line(const DevFrame& fr, int64_t x0, int64_t y0, int64_t x1,
                                        int64_t y1, uint32_t code) {
    const int64_t dx = wsub(x1, x0), dy = wsub(y1, y0);
    const int64_t ax = go_abs(dx), ay = go_abs(dy);
    const int64_t side = ax > ay ? ax : ay;
    if (side > kMaxOverlayLine) {
        atomicOr(&fr.ctrl->unsupported, 1u);
        return false;
    }
    const float xs = (float)dx / (float)side, ys = (float)dy / (float)side;
    float cx = (float)x0, cy = (float)y0;
    if (near_origin(x0, y0) && near_origin(x1, y1)) {
        // At most 2^16 steps, each rounded by half a unit in the last place of a
        // number below 2^17 (2^-8): the positions drift by 257 pixels at most, so
        // int() is the 32-bit conversion and y * W + x, with W <= 2^14, stays
        // below 2^31 (one position if side is 0).
        for (int i = 0; i <= (int)side; i++) {
            ov_pixel32(fr, (int)cx, (int)cy, code);
            cx += xs;
            cy += ys;
        }
        return true;
    }
    for (int64_t i = 0; i <= side; i++) {
        ov_pixel(fr, go_int(cx), go_int(cy), code);
        cx += xs;
        cy += ys;
    }
    return true;
}

// Overlay k of a binned triangle (renderer.go:191-216): edges 0..2, the centroid's
// rect, the vertices' rects 4..6. Returns false if its line was too long to draw.
constexpr uint32_t kOverlays = 7;
__device__ __forceinline__ bool draw_overlay(const DevFrame& fr, const OverlayRec& o, uint32_t slot,
                                             uint32_t k) {
    const uint32_t code = (slot + 1u) << 1;
    auto pick = [&](const float v[3], uint32_t j) { return j == 0 ? v[0] : j == 1 ? v[1] : v[2]; };
    if (k < 3) {
        if (!(fr.flags & kShowEdges)) return true;
        const uint32_t b = k == 2 ? 0 : k + 1;
        return ov_line(fr, go_int(pick(o.sx, k)), go_int(pick(o.sy, k)), go_int(pick(o.sx, b)),
                       go_int(pick(o.sy, b)), code);
    }
    if (k == 3) {
        if (!(fr.flags & kShowEdges) || !(fr.flags & kShowFaces)) return true;
        const float mx = (o.sx[0] + o.sx[1] + o.sx[2]) / 3.0f;
        const float my = (o.sy[0] + o.sy[1] + o.sy[2]) / 3.0f;
        ov_rect(fr, wsub(go_int(mx), 1), wsub(go_int(my), 1), code);
        return true;
    }
    if (fr.flags & kShowVertices)
        ov_rect(fr, wsub(go_int(pick(o.sx, k - 4)), 1), wsub(go_int(pick(o.sy, k - 4)), 1),
                code | 1u);
    return true;
}

// Tile references of a face block's triangles, counted for the list scan. The
// device atomics of one cache line (32 tile counters) are served one every 12 ns,
// so references are counted in LDS and flushed with one global atomic per touched
// tile when the block ends. Frames of at most kTableTiles tiles (1920x1080 at
// 32x32: 2,040) have a counter per tile, added to without a returned value.
// Before, references were counted in global memory and through a table with
// returned exchanges: k_face 481 -> 278 us for 8 requests over 4M resident
// triangles, 327 -> 252 us for 64 mixed frames.
//
// Larger frames: one-tile rectangles, and for dense meshes (at least one face per
// 4 pixels of the projected bounding box) rectangles of up to 2x2 tiles, are
// counted in a table of (tile, count) entries; a tile that finds its entry held
// by another tile, and other rectangles, whose tiles see few references each,
// add to global memory.
constexpr int kTableTiles = 2048;
constexpr int kTileTable = 256;
constexpr uint32_t kNoTile = 0xFFFFFFFFu;
typedef __attribute__((address_space(3))) uint32_t lds_u32;
struct TileTally {
    lds_u32* tag;
    lds_u32* cnt;
    uint32_t* global;
    bool dense;
};

__device__ __forceinline__ void tally_tile(const TileTally& tally, uint32_t t) {
    const uint32_t h = t & (uint32_t)(kTileTable - 1);
    uint32_t old = kNoTile;  // the entry's previous tag when the exchange fails
    __hip_atomic_compare_exchange_strong(tally.tag + h, &old, t, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_WORKGROUP);
    if (old == kNoTile || old == t)
        __hip_atomic_fetch_add(tally.cnt + h, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else
        atomicAdd(&tally.global[t], 1u);
}

__device__ __forceinline__ void count_tiles(const DevFrame& fr, const TileTally& tally, int tx0,
                                            int tx1, int ty0, int ty1) {
    if (tx0 == tx1 && ty0 == ty1) {
        tally_tile(tally, (uint32_t)(fr.tile_begin + ty0 * fr.tiles_x + tx0));
        return;
    }
    const bool small = tally.dense && tx1 - tx0 <= 1 && ty1 - ty0 <= 1;
    for (int ty = ty0; ty <= ty1; ty++)
        for (int tx = tx0; tx <= tx1; tx++) {
            const uint32_t t = (uint32_t)(fr.tile_begin + ty * fr.tiles_x + tx);
            if (small)
                tally_tile(tally, t);
            else
                atomicAdd(&tally.global[t], 1u);
        }
}

// A record that is never rasterised: its box words, all that is read of it.
__device__ __forceinline__ void store_empty_box(const DevFrame& fr, uint32_t ri) {
    gstore(reinterpret_cast<uint4*>(&fr.rrec[ri]) + 2, make_uint4(kEmptyBox, kEmptyBox, 0u, 0u));
}

// Writes the set-up of one post-clip triangle into record ri (renderer.go:361-394
// then the per-triangle part of rasterizer.go:98-137). Returns the TPF
// references in the low 16 bits and 1 << 16 when the triangle was binned, and the
// record's box words (bx0 | bx1 << 16, by0 | by1 << 16).
//
// k_face is bound by the instructions it issues, and most of them are here. The
// common triangle (screen coordinates within +-16384) takes 32-bit integers, a
// reference grid read at once, and one branch for what is rare in its three
// vertices; with 64-bit coordinates, a loop over the grid and Go's NaN and
// signed-zero rules worked out per minimum, 64 of them took 3.5 us (k_face for 32
// frames of 200,000 triangles 120 -> 106 us, for one of 40,000 18.8 -> 15.1).
__device__ __forceinline__ uint32_t emit_triangle(const DevFrame& fr, const CV& a, const CV& b,
                                                  const CV& c, int tex, uint32_t ri, uint2& box) {
    const float zw[3] = {a.w, b.w, c.w}, zz[3] = {a.z, b.z, c.z};
    const float vx[3] = {a.x, b.x, c.x}, vy[3] = {a.y, b.y, c.y};
    float sx[3], sy[3], pz[3] = {0.f, 0.f, 0.f};
    // The screen x and y rows use z/w only through screen[2] and screen[6]: when
    // both are zero, z/w matters only by being infinite or NaN (0 * z/w), and the
    // sign of a zero term never changes what the rasteriser does with sx, sy
    // (int(), comparisons). w/w is 1 for finite nonzero w, else NaN.
    bool need_z = fr.screen[2] != 0.f || fr.screen[6] != 0.f;
#pragma unroll
    for (int j = 0; j < 3; j++)
        need_z = need_z || !(__builtin_isfinite(zz[j]) &&
                             __builtin_fabsf(zz[j]) < __builtin_fabsf(zw[j]) * 0x1p100f);
    if (need_z) {
#pragma unroll
        for (int j = 0; j < 3; j++) pz[j] = zz[j] / zw[j];
    }
#pragma unroll
    for (int j = 0; j < 3; j++) {
        const float w = zw[j];
        const float px = vx[j] / w, py = vy[j] / w;
        const float pw = __builtin_isfinite(w) && w != 0.f ? 1.0f : __builtin_nanf("");
        sx[j] = fr.screen[0] * px + fr.screen[1] * py + fr.screen[2] * pz[j] + fr.screen[3] * pw;
        sy[j] = fr.screen[4] * px + fr.screen[5] * py + fr.screen[6] * pz[j] + fr.screen[7] * pw;
    }
    // Go's min and max of the three: only compared below, where the sign of a
    // zero does not matter and a NaN (which wins in Go) fails every comparison.
    const bool okx = !(sx[0] != sx[0]) && !(sx[1] != sx[1]) && !(sx[2] != sx[2]);
    const bool oky = !(sy[0] != sy[0]) && !(sy[1] != sy[1]) && !(sy[2] != sy[2]);
    const float fminx = __builtin_fminf(__builtin_fminf(sx[0], sx[1]), sx[2]);
    const float fmaxx = __builtin_fmaxf(__builtin_fmaxf(sx[0], sx[1]), sx[2]);
    const float fminy = __builtin_fminf(__builtin_fminf(sy[0], sy[1]), sy[2]);
    const float fmaxy = __builtin_fmaxf(__builtin_fmaxf(sy[0], sy[1]), sy[2]);
    // renderer.go:226-244 against the reference TPF grid. Its tiles are a
    // product grid (x bounds from tile % n, y bounds from tile / n,
    // renderer.go:61-67), so the overlapping tiles are the overlapping columns
    // times the overlapping rows (the bounds past a smaller grid are NaN).
    uint32_t cols = 0, rows = 0;
#pragma unroll
    for (int g = 0; g < 4; g++) {
        cols += (uint32_t)(fmaxx >= fr.ref_cols[g][0] && fminx <= fr.ref_cols[g][1]);
        rows += (uint32_t)(fmaxy >= fr.ref_rows[g][0] && fminy <= fr.ref_rows[g][1]);
    }
    const uint32_t tpf = okx && oky ? cols * rows : 0u;
    const bool binned = okx && oky && fmaxx >= 0.f && fminx <= (float)fr.W && fmaxy >= 0.f &&
                        fminy <= (float)fr.H;
    if (fr.orec) {
        // Screen positions for the overlay pass (binned triangles only draw them).
        OverlayRec o;
#pragma unroll
        for (int j = 0; j < 3; j++) {
            o.sx[j] = sx[j];
            o.sy[j] = sy[j];
        }
        o.binned = binned ? 1u : 0u;
        o.pad = 0;
        gstore(&fr.orec[ri], o);
    }
    box = make_uint2(kEmptyBox, kEmptyBox);
    if (binned && (fr.flags & kShowFaces)) {
        RasterRec rr;
        // Edge functions f_e(x,y) = A*x + B*y + C (rasterizer.go:107-117) with the
        // top-left adjustment folded into C (rasterizer.go:120-129). The pixel
        // sum fx12 + fx20 + fx01 is the sum of the C's (the A and B terms
        // cancel).
        constexpr int i0[3] = {0, 1, 2}, i1[3] = {1, 2, 0};
        int x0, x1, y0, y1;  // rasterizer.go:99-104 with tile (0,0)-(W,H) of the sequential renderer
        const float far = __builtin_fmaxf(
            __builtin_fmaxf(__builtin_fabsf(fminx), __builtin_fabsf(fmaxx)),
            __builtin_fmaxf(__builtin_fabsf(fminy), __builtin_fabsf(fmaxy)));
        const bool fast = far < (float)(kFastCoord + 1);
        if (fast) {
            // |x|, |y| <= 2^14: 24-bit products, and every value (the sum of
            // the three C's included) fits int32.
            int32_t X[3], Y[3], csum = 0;
#pragma unroll
            for (int j = 0; j < 3; j++) {
                X[j] = (int32_t)sx[j];
                Y[j] = (int32_t)sy[j];
            }
            x0 = max(min(min(X[0], X[1]), X[2]), 0);
            x1 = min(max(max(X[0], X[1]), X[2]), fr.W - 1);
            y0 = max(min(min(Y[0], Y[1]), Y[2]), 0);
            y1 = min(max(max(Y[0], Y[1]), Y[2]), fr.H - 1);
#pragma unroll
            for (int e = 0; e < 3; e++) {
                const int p = i0[e], q = i1[e];
                const int32_t A = Y[p] - Y[q], B = X[q] - X[p];
                int32_t C = __mul24(X[p], Y[q]) - __mul24(X[q], Y[p]);
                C -= (int32_t)!(B > 0 || (B == 0 && A > 0));
                rr.e[3 * e + 0] = A;
                rr.e[3 * e + 1] = B;
                rr.e[3 * e + 2] = C;
                csum += C;
            }
            rr.sf = (float)csum;
            rr.wide = 0;
            // A box of at most 2x2 pixels none of which passes the edge
            // test (the raster's, rasterizer.go:147) yields no fragment: it
            // stays out of the tile lists. Dense meshes far from the camera
            // emit mostly such sub-pixel triangles.
            if (x1 - x0 <= 1 && y1 - y0 <= 1) {
                int32_t any = 0;
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const int32_t x = min(x0 + (k & 1), x1), y = min(y0 + (k >> 1), y1);
                    const int32_t f0 = (int32_t)edge24(rr.e[0], x, rr.e[1], y, rr.e[2]);
                    const int32_t f1 = (int32_t)edge24(rr.e[3], x, rr.e[4], y, rr.e[5]);
                    const int32_t f2 = (int32_t)edge24(rr.e[6], x, rr.e[7], y, rr.e[8]);
                    any |= f0 & f1 & f2;
                }
                if (any >= 0) x1 = x0 - 1;
            }
        } else {
            // Wrapping int64 arithmetic as the reference's int.
            int64_t ix[3], iy[3];
#pragma unroll
            for (int j = 0; j < 3; j++) {
                ix[j] = go_int(sx[j]);
                iy[j] = go_int(sy[j]);
            }
            const int64_t mnx = max(min(min(ix[0], ix[1]), ix[2]), (int64_t)0);
            const int64_t mxx = min(max(max(ix[0], ix[1]), ix[2]), (int64_t)fr.W - 1);
            const int64_t mny = max(min(min(iy[0], iy[1]), iy[2]), (int64_t)0);
            const int64_t mxy = min(max(max(iy[0], iy[1]), iy[2]), (int64_t)fr.H - 1);
            const bool some = mnx <= mxx && mny <= mxy;
            x0 = some ? (int)mnx : 1;
            x1 = some ? (int)mxx : 0;
            y0 = (int)mny;
            y1 = (int)mxy;
            int64_t csum = 0;
            uint32_t adj = 0;
#pragma unroll
            for (int e = 0; e < 3; e++) {
                const int p = i0[e], q = i1[e];
                const int64_t A = wsub(iy[p], iy[q]);
                const int64_t B = wsub(ix[q], ix[p]);
                int64_t C = wsub(wmul(ix[p], iy[q]), wmul(ix[q], iy[p]));
                if (!(B > 0 || (B == 0 && A > 0))) {
                    C = wsub(C, 1);
                    adj |= 1u << e;
                }
                csum = wadd(csum, C);
            }
#pragma unroll
            for (int e = 0; e < 9; e++) rr.e[e] = 0;
            rr.sf = (float)csum;
            rr.wide = 1;
            WideRec wr;
#pragma unroll
            for (int j = 0; j < 3; j++) {
                wr.x[j] = ix[j];
                wr.y[j] = iy[j];
            }
            wr.adj = adj;
            wr.pad[0] = wr.pad[1] = wr.pad[2] = 0;
            if (some) gstore(&fr.wrec[ri], wr);
        }
        if (x0 <= x1 && y0 <= y1) {
            rr.bx0 = (int16_t)x0;
            rr.bx1 = (int16_t)x1;
            rr.by0 = (int16_t)y0;
            rr.by1 = (int16_t)y1;
            box = make_uint2((uint32_t)x0 | (uint32_t)x1 << 16, (uint32_t)y0 | (uint32_t)y1 << 16);
            rr.z0 = zw[0];
            rr.z1 = zw[1];
            rr.z2 = zw[2];
            rr.rsf = rr.rz0 = rr.rz1 = rr.rz2 = 0.f;
            // The divisions only the raster stage needs are done here, where the
            // triangle is in registers: in k_bin_fill they cost reading 64 and
            // writing 48 bytes of every record again (8 requests over 4M resident
            // triangles: k_bin_fill 177 -> 121 us, k_face unchanged; 32 frames of
            // 200,000: 50 -> 44 and 116 -> 122 us).
            //
            // The reciprocals of the divisors for the exact quotient path, whose
            // numerators are nonzero int32 edge values and barycentrics with
            // |alpha|, |beta| >= 2^-41 and gamma = +0 or |gamma| >= 2^-64 (left 0,
            // i.e. IEEE division, for int64 triangles and divisors outside
            // rcp_range).
            if (!rr.wide && rcp_range(rr.sf) && rcp_range(rr.z0) && rcp_range(rr.z1) &&
                rcp_range(rr.z2)) {
                rr.rsf = 1.0f / rr.sf;
                rr.rz0 = 1.0f / rr.z0;
                rr.rz1 = 1.0f / rr.z1;
                rr.rz2 = 1.0f / rr.z2;
            }
            ShadeRec sr;
            // rasterizer.go:132-137
            sr.uz[0] = a.u / rr.z0;
            sr.vz[0] = a.v / rr.z0;
            sr.uz[1] = b.u / rr.z1;
            sr.vz[1] = b.v / rr.z1;
            sr.uz[2] = c.u / rr.z2;
            sr.vz[2] = c.v / rr.z2;
            sr.in[0] = a.i;
            sr.in[1] = b.i;
            sr.in[2] = c.i;
            sr.tex = tex;
            sr.sf = rr.sf;
            sr.rsf = rr.wide ? kShadeWide : __float_as_uint(rr.rsf);
            gstore(&fr.srec[ri], sr);
            gstore(&fr.rrec[ri], rr);
        }
    }
    if (box.x == kEmptyBox) store_empty_box(fr, ri);
    return tpf | (binned ? 1u << 16 : 0u);
}

// A slot that holds no triangle (record ri): an empty box, never binned.
__device__ __forceinline__ void empty_record(const DevFrame& fr, uint32_t ri) {
    store_empty_box(fr, ri);
    if (fr.orec) {
        OverlayRec o = {};
        gstore(&fr.orec[ri], o);
    }
}

// Record of offset `off` of face block gb (of the batch) whose overflow
// records start at ovf.
__device__ __forceinline__ uint32_t block_rec(uint32_t gb, uint32_t ovf, uint32_t off) {
    return off < (uint32_t)kRecsPerBlock ? gb * (uint32_t)kRecsPerBlock + off
                                         : ovf + (off - (uint32_t)kRecsPerBlock);
}

// Record of slot `slot` of a frame (the block's overflow start is read only
// past its own range).
__device__ __forceinline__ uint32_t rec_index(const DevFrame& fr, uint32_t slot) {
    const uint32_t blk = slot / (uint32_t)kSlotsPerWg, off = slot % (uint32_t)kSlotsPerWg;
    // blk is below 2^32 / kSlotsPerWg: a 24-bit product.
    return off < (uint32_t)kRecsPerBlock
               ? __umul24(blk, (uint32_t)kRecsPerBlock) +
                     (uint32_t)fr.face_block_begin * (uint32_t)kRecsPerBlock + off
               : gld(&fr.blocks[blk].ovf) + (off - (uint32_t)kRecsPerBlock);
}

// General faces clipped per round by one wave; each fills kMaxFan lanes.
constexpr int kStage = 64 / kMaxFan;

__device__ __forceinline__ void add_emit(FaceStats& st, uint32_t e) {
    st.packed += (e & 0xFFFFu) + ((e >> 16) << 16);
}

// ---------------------------------------------------------------------------
// Workgroup tile binning helpers
// ---------------------------------------------------------------------------

constexpr int kLdsTiles = 1024;  // LDS tile counters per workgroup
// One wave per k_bin_fill workgroup: a face block emits a few dozen triangles
// in typical frames, and the workgroup's time is its chain of dependent memory
// round trips, so more resident workgroups per CU is what makes it faster.
constexpr int kFillThreads = 64;

struct TileRect {
    int tx0, tx1, ty0, ty1;
};

// Tile range of a raster record's box (empty: tx0 > tx1), from the record's
// piece 2 (bx0 | bx1 << 16, by0 | by1 << 16, wide, A01).
__device__ __forceinline__ TileRect box_tiles(uint32_t bx, uint32_t by, int twl, int thl) {
    const int bx0 = (int)(int16_t)(bx & 0xFFFFu), bx1 = (int)(int16_t)(bx >> 16);
    const int by0 = (int)(int16_t)(by & 0xFFFFu), by1 = (int)(int16_t)(by >> 16);
    TileRect t;
    if (bx0 > bx1) {
        t.tx0 = 1;
        t.tx1 = 0;
        t.ty0 = 1;
        t.ty1 = 0;
    } else {
        t.tx0 = bx0 >> twl;
        t.tx1 = bx1 >> twl;
        t.ty0 = by0 >> thl;
        t.ty1 = by1 >> thl;
    }
    return t;
}

// fn(x, y) for every point of a (wave-uniform) rectangle, by the lanes of one
// wave: a power of two of lanes per row.
template <typename F>
__device__ __forceinline__ void wave_rect(int x0, int y0, int x1, int y1, int lane, F fn) {
    const int l2 = min(x1 == x0 ? 0 : 32 - __builtin_clz((uint32_t)(x1 - x0)), 6);
    for (int y = y0 + (lane >> l2); y <= y1; y += 64 >> l2)
        for (int x = x0 + (lane & ((1 << l2) - 1)); x <= x1; x += 1 << l2) fn(x, y);
}

__device__ __forceinline__ TileRect rec_tiles(const RasterRec* r, int twl, int thl) {
    const uint4 p2 = gload(reinterpret_cast<const uint4*>(r) + 2);
    return box_tiles(p2.x, p2.y, twl, thl);
}

// ---------------------------------------------------------------------------
// k_face
// ---------------------------------------------------------------------------

// Clip-space corner k of a face: MVP * (x, y, z, w) (renderer.go:303-304,318-320).
__device__ __forceinline__ float4 corner(const DevObject& o, int v) {
    const float* p = o.m.pos + 3 * (size_t)v;
    float w = o.m.pw ? gld(&o.m.pw[v]) : 1.0f;
    return xform(o.mvp, gld(p), gld(p + 1), gld(p + 2), w);
}

// Gouraud intensity of normal n: World * normal, 4-D normalise (renderer.go:308-310,328-333).
__device__ __forceinline__ float normal_intensity(const DevObject& o, const DevFrame& fr, int n) {
    const float* q = o.m.nrm + 3 * (size_t)n;
    float w = o.m.nw ? gld(&o.m.nw[n]) : 1.0f;
    return lambert(xform(o.world, gld(q), gld(q + 1), gld(q + 2), w), fr.light, fr.ambient,
                   fr.diffuse);
}

// LDS writes of one wave made visible to the wave's other lanes.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One face block (kFacesPerWg faces of one object) per workgroup of NW waves.
//
// NW = 1, kFacesPerLane faces per lane: a block's few survivors keep one wave
// busy through the long per-survivor chain of pass 2 (dependent loads, lighting,
// clipping, set-up), so no sibling waves wait at barriers holding registers, and
// every resident wave works. The form for launches that fill the chip.
//
// NW = 4, a face per lane: pass 1 is a quarter as long and pass 2 one round
// instead of up to four, for launches whose blocks leave most of the chip idle
// (see launch_face).
__device__ __forceinline__ int sgpr(int v) { return __builtin_amdgcn_readfirstlane(v); }

template <int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(4))) void k_face(
    const DevObject* __restrict__ objs, const DevFrame* __restrict__ frames,
    uint32_t* __restrict__ tile_counts, FaceBlock* __restrict__ blocks, int twl, int thl,
    const int* __restrict__ xcd_face, const int* __restrict__ obj_first, int nframes,
    uint32_t* __restrict__ rec_pool, uint32_t npools, uint32_t pool_recs, uint32_t ovf_begin,
    DevControl* __restrict__ ctrl, uint32_t* __restrict__ frame_overflow) {
    constexpr int kFacesPerLane = kFacesPerWg / (64 * NW);
    static_assert(kFacesPerWg == 64 * NW * kFacesPerLane, "whole faces per lane");
    // What a wave keeps to itself.
    struct WaveLds {
        uint32_t sface[64 * kFacesPerLane];  // survivors in face order: offset | clip plane << 8
        CV poly[2][kMaxClip];
        CV stage[kStage][kMaxClip];          // clipped polygons of general faces
        int stage_k[kStage], stage_tex[kStage];
        int stage_off[kStage];               // the face's first offset in the block
    };
    __shared__ WaveLds lds_wave[NW];
    __shared__ uint32_t lds_sum[4][NW];  // per-wave terms of the block's sums
    __shared__ uint32_t lds_claim[2];    // the block's claim of overflow records
    // The tile counters (see kTableTiles): 16 bits a tile, or the entry table.
    // A block counts at most kSlotsPerWg references per tile.
    __shared__ uint4 lds_tiles[kTableTiles / 8];
    static_assert(2 * kTileTable * 4 <= sizeof(lds_tiles) && kSlotsPerWg < 65536, "tile counters");

    int bf, blocal;
    if (!xcd_unit(xcd_face, nframes, (int)blockIdx.x, bf, blocal)) return;
    const int lane = (int)threadIdx.x & 63, wave = NW > 1 ? sgpr((int)threadIdx.x >> 6) : 0;
    WaveLds& W = lds_wave[wave];
    auto block_sync = [&] {
        if constexpr (NW > 1)
            __syncthreads();
        else
            wave_sync();
    };
    // Sum of the waves' v (wave-uniform) before this one's; all of them in total.
    // Each k is used once.
    auto wave_prefix = [&](int k, uint32_t v, uint32_t& total) -> uint32_t {
        total = v;
        if constexpr (NW == 1) return 0u;
        if (lane == 0) lds_sum[k][wave] = v;
        __syncthreads();
        uint32_t before = 0u;
        total = 0u;
        for (int w = 0; w < NW; w++) {
            const uint32_t t = (uint32_t)sgpr((int)lds_sum[k][w]);
            before += w < wave ? t : 0u;
            total += t;
        }
        return before;
    };
    // Search only this frame's objects.
    const int b = frames[bf].face_block_begin + blocal;
    const int ob0 = frames[bf].obj_begin;
    const int oi = ob0 + wave_last_le(obj_first + ob0, frames[bf].obj_count, b);
    const DevObject& o = objs[oi];
    const DevMesh& m = o.m;
    const DevFrame& fr = frames[bf];
    lds_u32* const counters = (lds_u32*)lds_tiles;
    const TileTally tally{counters, counters + kTileTable, tile_counts, o.dense != 0};
    const int ntiles = fr.tiles_x * fr.tiles_y;
    const bool table = ntiles <= kTableTiles;  // wave-uniform
    const int groups = table ? (ntiles + 7) >> 3 : 2 * kTileTable / 4;  // uint4 pieces in use
    for (int i = (int)threadIdx.x; i < groups; i += 64 * NW) {
        const uint32_t v = !table && i < kTileTable / 4 ? kNoTile : 0u;
        lds_tiles[i] = make_uint4(v, v, v, v);
    }
    block_sync();
    // Counts the tiles of the lanes' boxes; every lane of the wave calls it. A box
    // of many tiles is counted by the whole wave.
    auto count = [&](const uint2& box) {
        const TileRect t = box_tiles(box.x, box.y, twl, thl);
        if (!table) {
            if (t.tx0 <= t.tx1) count_tiles(fr, tally, t.tx0, t.tx1, t.ty0, t.ty1);
            return;
        }
        auto add = [&](uint32_t i) {
            __hip_atomic_fetch_add(counters + (i >> 1), 1u << (16u * (i & 1u)), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
        };
        const int w = t.tx1 - t.tx0 + 1, n = w * (t.ty1 - t.ty0 + 1);
        constexpr int kLaneTiles = 16;
        if (w > 0 && n <= kLaneTiles)
            for (int ty = t.ty0; ty <= t.ty1; ty++)
                for (int tx = t.tx0; tx <= t.tx1; tx++) add((uint32_t)(ty * fr.tiles_x + tx));
        for (uint64_t big = ballot(w > 0 && n > kLaneTiles); big; big &= big - 1) {
            const int L = __builtin_ctzll(big);
            wave_rect(__builtin_amdgcn_readlane(t.tx0, L), __builtin_amdgcn_readlane(t.ty0, L),
                      __builtin_amdgcn_readlane(t.tx1, L), __builtin_amdgcn_readlane(t.ty1, L),
                      lane, [&](int tx, int ty) { add((uint32_t)(ty * fr.tiles_x + tx)); });
        }
    };
    const int wg_in_obj = b - o.face_block;
    const uint32_t flags = fr.flags;
    const int vis = o.vis;  // BoxVisibility, per object on the host

    FaceStats st = {0u};

    // Pass 1, faces lane, lane + 64, ... of the block: clip-space corners,
    // backface test and plane classification. The survivors (front faces the
    // clipper does not reject outright) are compacted in face order into LDS,
    // so the lighting, clipping and set-up below run on dense lanes.
    int nsurv = 0;      // wave-uniform
    uint32_t nrec = 0;  // records the survivors can need: 1, or kMaxFan when clipped
    if (vis != kBoxOutside) {
        // All the lane's vertex indices, then all its corners, are loaded
        // before any is used: lanes past the mesh's last face read its last
        // face (in bounds) and are not counted.
        const int fo0 = wave * 64 * kFacesPerLane + lane;  // the lane's first face of the block
        const int face0 = wg_in_obj * kFacesPerWg + fo0;
        int iv[kFacesPerLane][3];
#pragma unroll
        for (int k = 0; k < kFacesPerLane; k++) {
            const int face = min(face0 + 64 * k, m.F - 1);
            iv[k][0] = gld(&m.vi[3 * face + 0]);
            iv[k][1] = gld(&m.vi[3 * face + 1]);
            iv[k][2] = gld(&m.vi[3 * face + 2]);
        }
        float4 cv[kFacesPerLane][3];
#pragma unroll
        for (int k = 0; k < kFacesPerLane; k++)
#pragma unroll
            for (int c = 0; c < 3; c++) cv[k][c] = corner(o, iv[k][c]);
#pragma unroll
        for (int k = 0; k < kFacesPerLane; k++) {
            const int fo = k * 64 + fo0;  // face offset in the block
            const float4 v0 = cv[k][0], v1 = cv[k][1], v2 = cv[k][2];
            bool survivor = false;
            int p = 6;
            if (face0 + 64 * k < m.F &&
                (!(flags & kBackfaceCulling) || facing_camera(v0, v1, v2))) {
                st.packed += 1u << 24;
                uint32_t m0 = 0x3Fu, m1 = 0x3Fu, m2 = 0x3Fu;
                if ((flags & kFrustumClipping) && vis != kBoxInside) {
                    m0 = inside_mask(CV{v0.x, v0.y, v0.z, v0.w, 0.f, 0.f, 0.f}, fr.znear, fr.zfar);
                    m1 = inside_mask(CV{v1.x, v1.y, v1.z, v1.w, 0.f, 0.f, 0.f}, fr.znear, fr.zfar);
                    m2 = inside_mask(CV{v2.x, v2.y, v2.z, v2.w, 0.f, 0.f, 0.f}, fr.znear, fr.zfar);
                }
                const uint32_t all_in = m0 & m1 & m2;
                // First plane not passed by every vertex (6 if none). Earlier
                // planes leave the triangle untouched; when this one rejects
                // every vertex the pass yields an empty polygon.
                p = __builtin_ctz(~all_in | 0x40u);
                survivor = !(p < 6 && !(((m0 | m1 | m2) >> p) & 1u));
            }
            const uint64_t sm = ballot(survivor);
            if (survivor)
                W.sface[nsurv + __popcll(sm & lanemask_lt(lane))] = (uint32_t)fo | ((uint32_t)p << 8);
            nsurv += __popcll(sm);
            nrec += (uint32_t)__popcll(sm) + (kMaxFan - 1) * (uint32_t)__popcll(ballot(survivor && p < 6));
        }
    }
    wave_sync();

    // Records beyond the block's own range (sized for the largest fan of every
    // clipped survivor): a contiguous range of its overflow pool, claimed now.
    // Past the pool's end the block draws nothing and the batch reports an
    // overflow with a capacity that gives every pool this much (the caller
    // grows the capacity and draws it again); its frame is marked so that its
    // raster draws the background only.
    uint32_t ovf = 0u;  // block-uniform
    uint32_t nrec_block;
    (void)wave_prefix(0, nrec, nrec_block);
    if (nrec_block > (uint32_t)kRecsPerBlock) {
        const uint32_t extra = nrec_block - (uint32_t)kRecsPerBlock;
        const uint32_t pool = (uint32_t)b % npools;
        if (threadIdx.x == 0) {
            const uint32_t r = atomicAdd(&rec_pool[pool * kPoolStride], extra);
            const unsigned long long end = (unsigned long long)r + extra;
            lds_claim[0] = r;
            lds_claim[1] = end > pool_recs;
            if (end > pool_recs) {
                atomicMax(&ctrl->refs_needed, end * npools * kOvfRefs);
                atomicOr(&ctrl->overflow, 1u);
                atomicOr(&frame_overflow[bf], 1u);
            }
        }
        block_sync();
        if (sgpr((int)lds_claim[1]))
            nsurv = 0;
        else
            ovf = ovf_begin + pool * pool_recs + (uint32_t)sgpr((int)lds_claim[0]);
    }

    // Pass 2, survivor r0 + lane, 64 a round: lighting, texture coordinates,
    // clipping. 0: nothing, 1: emit the triangle as is, 2: full clipper in the
    // wave, 3: one-plane polygon. q[0..nq-1] holds the polygon to emit (the
    // triangle itself for modes 1 and 2), so only one set of corners stays
    // live across the emits.
    uint32_t run = 0;  // slots of the earlier rounds, or of the block (wave-uniform)
    for (int r0 = 0; r0 < (NW > 1 ? 1 : nsurv); r0 += 64) {
        int mode = 0;
        int n = 0;
        CV q[4];
        int nq = 0;
        int tex = -1;
        if (r0 + lane < nsurv) {
            CV c0, c1, c2;
            const uint32_t e = W.sface[r0 + lane];
            const int sf = wg_in_obj * kFacesPerWg + (int)(e & 0xFFu);
            const int sp = (int)(e >> 8);
            const int i0 = gld(&m.vi[3 * sf + 0]), i1 = gld(&m.vi[3 * sf + 1]),
                      i2 = gld(&m.vi[3 * sf + 2]);
            // The corners again (the same arithmetic as pass 1).
            const float4 w0 = corner(o, i0), w1 = corner(o, i1), w2 = corner(o, i2);
            c0 = CV{w0.x, w0.y, w0.z, w0.w, 0.f, 0.f, 0.f};
            c1 = CV{w1.x, w1.y, w1.z, w1.w, 0.f, 0.f, 0.f};
            c2 = CV{w2.x, w2.y, w2.z, w2.w, 0.f, 0.f, 0.f};
            float in0, in1, in2;
            if (flags & kLighting) {
                if (o.gouraud) {
                    int n0 = i0, n1 = i1, n2 = i2;
                    if (m.ni) {
                        n0 = gld(&m.ni[3 * sf + 0]);
                        n1 = gld(&m.ni[3 * sf + 1]);
                        n2 = gld(&m.ni[3 * sf + 2]);
                    }
                    in0 = normal_intensity(o, fr, n0);
                    in1 = normal_intensity(o, fr, n1);
                    in2 = normal_intensity(o, fr, n2);
                } else {
                    const float* f = m.fn + 4 * (size_t)sf;
                    float4 t = xform(o.world, gld(f), gld(f + 1), gld(f + 2), gld(f + 3));
                    in0 = in1 = in2 = lambert(t, fr.light, fr.ambient, fr.diffuse);
                }
            } else {
                in0 = in1 = in2 = fr.ambient;
            }
            c0.i = in0;
            c1.i = in1;
            c2.i = in2;
            if (m.uv_vert) {
                c0.u = gld(&m.uv_vert[2 * i0]);
                c0.v = gld(&m.uv_vert[2 * i0 + 1]);
                c1.u = gld(&m.uv_vert[2 * i1]);
                c1.v = gld(&m.uv_vert[2 * i1 + 1]);
                c2.u = gld(&m.uv_vert[2 * i2]);
                c2.v = gld(&m.uv_vert[2 * i2 + 1]);
            } else if (m.uv_face) {
                const float* uv = m.uv_face + 6 * (size_t)sf;
                c0.u = gld(uv);
                c0.v = gld(uv + 1);
                c1.u = gld(uv + 2);
                c1.v = gld(uv + 3);
                c2.u = gld(uv + 4);
                c2.v = gld(uv + 5);
            }
            if (flags & kShowTextures) tex = m.face_tex ? gld(&m.face_tex[sf]) : m.mesh_tex;
            if (sp == 6) {
                // Every pass only rotates the triangle; after 6 passes it is
                // unchanged (clipping.go:199-232); no clipping: as is.
                mode = 1;
                n = 1;
                nq = 3;
                q[0] = c0;
                q[1] = c1;
                q[2] = c2;
            } else {
                nq = clip_one_plane(sp, c0, c1, c2, fr.znear, fr.zfar, q);
                if (nq > 0) {
                    mode = 3;
                    n = nq - 2;
                } else if (nq < 0) {
                    nq = 0;
                    mode = 2;  // counted below, one face at a time
                    q[0] = c0;
                    q[1] = c1;
                    q[2] = c2;
                }
            }
        }

        // Faces for the full clipper reserve the largest fan (kMaxFan slots):
        // the slots their polygon leaves unused get empty records, which are
        // never binned, so slots stay in draw order and each face is clipped
        // once. The prefix of the fan sizes (0, 1, 2 or kMaxFan) in face order
        // is counted from three ballots.
        if (mode == 2) n = kMaxFan;
        const uint64_t b1 = ballot(n == 1), b2 = ballot(n == 2), b7 = ballot(n == kMaxFan);
        const uint64_t lt = lanemask_lt(lane);
        // The lane's slots start at offset off of the block's.
        uint32_t total;
        const uint32_t before = wave_prefix(
            1, (uint32_t)(__popcll(b1) + 2 * __popcll(b2) + kMaxFan * __popcll(b7)), total);
        const uint32_t off = run + before + (uint32_t)(__popcll(b1 & lt) + 2 * __popcll(b2 & lt) +
                                                       kMaxFan * __popcll(b7 & lt));
        run += total;
        // Fan of q (Polygon.Triangulate, clipping.go:44-62): (P0, P1, P2),
        // then (P0, P2, P3) for a quad.
        bool emit = mode == 1 || mode == 3;
#pragma unroll 1
        for (uint32_t t = 0;; t++) {
            uint2 box = make_uint2(kEmptyBox, kEmptyBox);
            if (emit)
                add_emit(st, emit_triangle(fr, q[0], q[1], q[2], tex, block_rec(b, ovf, off + t),
                                           box));
            count(box);
            emit = mode == 3 && nq == 4;
            if (t == 1 || !ballot(emit)) break;
            if (emit) {
                q[1] = q[2];
                q[2] = q[3];
            }
        }

        // General faces, kStage at a time: the wave clips each one into its
        // stage (clipping.go:167-236), then one lane per fan slot emits the
        // triangle (P0, P_t+1, P_t+2) of Polygon.Triangulate
        // (clipping.go:44-62) or an empty record.
        CV* buf0 = W.poly[0];
        CV* buf1 = W.poly[1];
        for (uint64_t gen = ballot(mode == 2); gen;) {
            int nst = 0;
            for (; gen && nst < kStage; gen &= gen - 1, nst++) {
                const int L = __builtin_ctzll(gen);
                const CV a = shfl_cv(q[0], L), bb = shfl_cv(q[1], L), c = shfl_cv(q[2], L);
                const int texL = __shfl(tex, L, 64);
                const int sL = __shfl((int)off, L, 64);
                const int k = wave_clip(buf0, buf1, a, bb, c, fr.znear, fr.zfar, lane);
                if (k < 0 && lane == L) st.packed += 1u << 28;
                if (lane < k) W.stage[nst][lane] = buf0[lane];
                if (lane == 0) {
                    W.stage_k[nst] = k;
                    W.stage_tex[nst] = texL;
                    W.stage_off[nst] = sL;
                }
                wave_sync();
            }
            const int r = lane / kMaxFan, t = lane - r * kMaxFan;
            uint2 box = make_uint2(kEmptyBox, kEmptyBox);
            if (r < nst) {
                const int k = W.stage_k[r];
                const uint32_t ri = block_rec(b, ovf, (uint32_t)W.stage_off[r] + (uint32_t)t);
                const CV* P = W.stage[r];
                if (t < k - 2)
                    add_emit(st, emit_triangle(fr, P[0], P[t + 1], P[t + 2], W.stage_tex[r],
                                               ri, box));
                else
                    empty_record(fr, ri);
            }
            count(box);
            wave_sync();
        }
    }

    // The block's slots, first overflow record and counters (two wave sums of
    // 16-bit fields: TPF references | binned triangles, front faces | clip
    // overflows) in one store; k_bin_scan sums the counters of a frame's blocks.
    // (Added to the frame's counters, one cache line, the blocks queue up: 47 us
    // for the 3,900 blocks of a million faces.)
    {
        const uint32_t w0 = wave_sum_u32((st.packed & 0xFFFFu) | (((st.packed >> 16) & 0xFFu) << 16));
        const uint32_t w1 = wave_sum_u32(((st.packed >> 24) & 0xFu) | ((st.packed >> 28) << 16));
        uint32_t c0, c1;
        (void)wave_prefix(2, w0, c0);
        (void)wave_prefix(3, w1, c1);
        if (threadIdx.x == 0)
            gstore(&blocks[b], FaceBlock{run | (c1 & 0xFFFFu) << 11 | (c1 >> 16) << 20, ovf, c0,
                                         (uint32_t)bf});
    }
    // Every count is in the table (the sums' barriers order the waves): flush it.
    wave_sync();
    if (!table) {
        for (int i = (int)threadIdx.x; i < kTileTable; i += 64 * NW) {
            const uint32_t v = counters[kTileTable + i];
            if (v) atomicAdd(&tile_counts[counters[i]], v);
        }
        return;
    }
    for (int i = (int)threadIdx.x; i < groups; i += 64 * NW) {
        const uint4 v = lds_tiles[i];
        if (!(v.x | v.y | v.z | v.w)) continue;
        uint32_t* dst = tile_counts + fr.tile_begin + 8 * i;
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (w[k] & 0xFFFFu) atomicAdd(dst + 2 * k, w[k] & 0xFFFFu);
            if (w[k] >> 16) atomicAdd(dst + 2 * k + 1, w[k] >> 16);
        }
    }
}

// ---------------------------------------------------------------------------
// k_overlay: debug overlays of every binned triangle (frames that ask for them)
// ---------------------------------------------------------------------------

// One overlay per lane, kind by kind, so that a wave's lanes walk alike; gridDim.y
// workgroups share a face block. With a lane per triangle, its three lines and four
// rects one after the other in 64-bit coordinates, most lanes of a block idled: 59
// us for 20,000 faces at 1280x720, against 32.
__global__ __launch_bounds__(256) void k_overlay(const DevFrame* __restrict__ frames,
                                                 const FaceBlock* __restrict__ blocks,
                                                 unsigned long long* __restrict__ stats) {
    const int b = blockIdx.x;
    const FaceBlock fb = gload(&blocks[b]);
    const DevFrame& fr = frames[fb.frame];
    if (!fr.orec) return;
    const uint32_t cnt = fb.slots(), ovf = fb.ovf;
    const uint32_t blk = (uint32_t)(b - fr.face_block_begin);  // in the frame
    const uint32_t slot0 = blk * kSlotsPerWg;
    for (uint32_t w = blockIdx.y * 256u + threadIdx.x; w < kOverlays * cnt; w += gridDim.y * 256u) {
        const uint32_t k = w / cnt, i = w - k * cnt;
        const OverlayRec rec = gload(&fr.orec[block_rec(b, ovf, i)]);
        // A frame with a line too long is counted on its own, besides the
        // batch's control word, so a caller can tell which frames failed.
        if (rec.binned && !draw_overlay(fr, rec, slot0 + i, k))
            atomicAdd(&stats[fb.frame * kNumStats + kStatLongLines], 1ull);
    }
}

// ---------------------------------------------------------------------------
// k_decorate: the end of Draw outside demo mode (renderer.go:476-480)
// ---------------------------------------------------------------------------

// FrameBuffer.Pixel (rasterizer.go:25-30) straight into the colour buffer:
// only the flat index is checked, so an x beyond a row wraps into the next.
__device__ __forceinline__ void fb_pixel(const DevFrame& fr, int64_t x, int64_t y, uint32_t c) {
    const int64_t idx = wadd(wmul(y, fr.W), x);
    if (idx > 0 && idx < (int64_t)fr.W * fr.H) ((uint32_t*)fr.rgba)[idx] = c;
}

// FrameBuffer.Line (rasterizer.go:65-79) along one axis, a pixel per lane. The
// float32 DDA steps by exactly -1, 0 or 1 on whole coordinates below 2^24, so
// its position after i steps is the start plus i steps, in any order.
__device__ __forceinline__ void fb_axis_line(const DevFrame& fr, int x0, int y0, int x1, int y1,
                                             uint32_t c, int lane) {
    const int sx = (x1 > x0) - (x1 < x0), sy = (y1 > y0) - (y1 < y0);
    const int side = max(abs(x1 - x0), abs(y1 - y0));
    for (int i = lane; i <= side; i += 64) fb_pixel(fr, x0 + i * sx, y0 + i * sy, c);
}

// One workgroup per frame: the reference tiles' borders (drawTilesBoundaries,
// renderer.go:422-434), a wave per line, in red; then the crosshair
// (CrossHair, rasterizer.go:209-217) in yellow. Colour only, after the frame.
// A frame has 64 lines of up to a quarter of its side: walked by one lane each
// they are one serial chain of stores (207 us at 1280x720); 16 waves write them
// 64 pixels at a time (debug frames of 20k triangles in flight: 135 -> 71 us).
constexpr int kDecorateThreads = 1024;
__global__ __launch_bounds__(kDecorateThreads) void k_decorate(
    const DevFrame* __restrict__ frames) {
    const DevFrame& fr = frames[blockIdx.x];
    if (!(fr.flags & (kShowTileBounds | kShowCrosshair))) return;  // uniform per block
    const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
    if (fr.flags & kShowTileBounds) {
        constexpr uint32_t kRed = 0xFF0000FFu;  // {255, 0, 0, 255}
        for (int l = wave; l < 4 * fr.ref_tiles; l += kDecorateThreads / 64) {
            // Tile bounds are whole numbers within the frame (at most 16384).
            const int ng = fr.ref_tiles == 16 ? 4 : 1, t = l >> 2;
            const float *cx = fr.ref_cols[t % ng], *cy = fr.ref_rows[t / ng];
            const int sx = (int)cx[0], sy = (int)cy[0], ex = (int)cx[1], ey = (int)cy[1];
            switch (l & 3) {
            case 0: fb_axis_line(fr, sx, sy, ex, sy, kRed, lane); break;
            case 1: fb_axis_line(fr, ex, sy, ex, ey, kRed, lane); break;
            case 2: fb_axis_line(fr, ex, ey, sx, ey, kRed, lane); break;
            default: fb_axis_line(fr, sx, ey, sx, sy, kRed, lane); break;
            }
        }
    }
    __syncthreads();  // the crosshair is drawn over the borders
    if ((fr.flags & kShowCrosshair) && wave < 4) {
        constexpr uint32_t kYellow = 0xFF00FFFFu;  // {255, 255, 0, 255}
        constexpr int size = 5, offset = 3;
        const int x = fr.W / 2, y = fr.H / 2;
        switch (wave) {
        case 0: fb_axis_line(fr, x - size, y, x - offset, y, kYellow, lane); break;
        case 1: fb_axis_line(fr, x + offset, y, x + size, y, kYellow, lane); break;
        case 2: fb_axis_line(fr, x, y - size, x, y - offset, kYellow, lane); break;
        default: fb_axis_line(fr, x, y + offset, x, y + size, kYellow, lane); break;
        }
    }
}

// FrameBuffer.Fog (rasterizer.go:185-207) with blendRGBA's
// uint8(float32(a)*(1-f) + float32(b)*f) per channel.
__global__ __launch_bounds__(256) void k_fog(uint32_t* __restrict__ rgba,
                                             const float* __restrict__ depth, uint64_t n,
                                             float fog_start, float fog_end, uint32_t color) {
    for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * 256u) {
        const float d = depth[i];
        if (d >= fog_start) continue;
        if (d <= fog_end) {
            rgba[i] = color;
            continue;
        }
        const float f = 1 - ((fog_end - d) / (fog_end - fog_start));
        const uint32_t p = rgba[i];
        uint32_t out = 0;
        for (int k = 0; k < 4; k++) {
            const float a = (float)((p >> (8 * k)) & 0xFFu), b = (float)((color >> (8 * k)) & 0xFFu);
            const float u = a * (1 - f);
            const float v = b * f;
            out |= (go_uint8(u + v) & 0xFFu) << (8 * k);
        }
        rgba[i] = out;
    }
}

// ---------------------------------------------------------------------------
// k_bin_scan: tile counts -> list offsets, one workgroup per frame
// ---------------------------------------------------------------------------

// A kernel of its own: a last-block scan inside k_face would need a device-scope
// release in every face workgroup, which on a multi-XCD part writes back and
// invalidates L2 each time.
//
// A tile whose list is longer than part_refs and than one share of the launch's
// entries over the raster workgroups that the chip holds (or than split_refs,
// whatever the share) is split over several raster workgroups: it takes a slab
// (depth keys of its pixels), and its entries a range [split_first[slab], + count)
// of the split tiles' entries put end to end (split_tile[slab] = the tile). One
// counter hands out both, so the ranges ascend with the slabs. With no slab left
// the tile stays whole (slower, same result).
//
// Lists up to a share end with the others anyway, and their parts cost a merge: 200,000
// small triangles all over 2560x1440, k_raster 67 us with every list over 64 split, 46
// so (20,000 of 60 pixels at 3840x2160 in 64x64 tiles 141 | 118). With two shares
// instead of one, 500,000 faces in the middle of 1920x1080 take 114 us for 91.
constexpr int kScanThreads = 1024;
__global__ __launch_bounds__(kScanThreads) void k_bin_scan(
    const DevFrame* __restrict__ frames, int nframes, uint32_t* __restrict__ tile_counts,
    uint32_t* __restrict__ tile_offsets, uint32_t* __restrict__ tile_cursor,
    uint32_t* __restrict__ frame_overflow, unsigned long long* __restrict__ stats,
    DevBatchCounters* __restrict__ counters, DevControl* __restrict__ ctrl,
    unsigned long long refs_capacity, uint32_t* __restrict__ tile_slab,
    uint32_t* __restrict__ split_first, uint32_t* __restrict__ split_tile, uint32_t max_slabs,
    uint32_t part_refs, uint32_t split_refs, uint32_t* __restrict__ rec_pool,
    const FaceBlock* __restrict__ blocks, int total_tiles, float inv_held) {
    constexpr int NW = kScanThreads / 64;
    __shared__ unsigned long long wsum[NW], wsplit[NW];
    __shared__ uint32_t wstat[NW][4];
    __shared__ unsigned long long base_s, split_s;
    __shared__ uint32_t longest_s;  // the longest list left whole
    const int f = blockIdx.x;
    const DevFrame& fr = frames[f];
    const int ntiles = fr.tiles_x * fr.tiles_y;
    uint32_t* cnt = tile_counts + fr.tile_begin;
    const int lane = threadIdx.x & 63, wave = sgpr(threadIdx.x >> 6);

    // The first tiles of the thread stay in registers from the totals to the
    // offsets (2,048 tiles in all); later ones are read again.
    constexpr int kKeep = 2;
    uint32_t v0[kKeep];
#pragma unroll
    for (int k = 0; k < kKeep; k++) {
        const int i = (int)threadIdx.x + k * kScanThreads;
        v0[k] = i < ntiles ? gld(&cnt[i]) : 0u;
    }
    // The launch's references (in 32 bits: with more it overflows), where parts are
    // smaller than split_refs (launches of few tiles). A frame that overflowed may be
    // clearing its own counts: its batch is drawn again.
    const bool shared = nframes > 1 && part_refs < split_refs;  // at most kAllTiles tiles
    constexpr int kAllTiles = 4 * kScanThreads;
    uint4 all4 = make_uint4(0u, 0u, 0u, 0u);
    uint32_t all1 = 0u;
    if (shared) {
        const int quads = min(total_tiles, kAllTiles) >> 2, i = 4 * quads + (int)threadIdx.x;
        if ((int)threadIdx.x < quads)
            all4 = gload(reinterpret_cast<const uint4*>(tile_counts) + threadIdx.x);
        if (threadIdx.x < 3 && i < min(total_tiles, kAllTiles)) all1 = gld(&tile_counts[i]);
    }

    // k_face is done with the record pools: their total to the batch counters,
    // and the counters back to zero for the next draw.
    static_assert(kRecPools % 64 == 0 && kRecPools <= kScanThreads,
                  "whole waves read the pool counters");
    if (f == 0 && threadIdx.x < kRecPools) {
        uint32_t* pc = &rec_pool[threadIdx.x * kPoolStride];
        const uint32_t v = *pc;
        *pc = 0u;
        const unsigned long long t = wave_sum_u64(v);
        if (lane == 0) atomicAdd(&counters->recs_used, t);
    }

    // The counters of the frame's face blocks: TPF references, binned
    // triangles, front faces, clip overflows, 65536 blocks a round at most, so
    // that a wave's sums of 16-bit fields fit 32 bits.
    unsigned long long bt = 0;  // lanes 0..3 of wave 1: the totals
    for (int r0 = 0; r0 < fr.face_blocks; r0 += 65536) {
        uint32_t bs[4] = {0, 0, 0, 0};
        const int end = min(fr.face_blocks, r0 + 65536);
        for (int i = r0 + (int)threadIdx.x; i < end; i += kScanThreads) {
            const FaceBlock fb = gload(&blocks[fr.face_block_begin + i]);
            bs[0] += fb.c0 & 0xFFFFu;
            bs[1] += fb.c0 >> 16;
            bs[2] += (fb.c >> 11) & 511u;
            bs[3] += fb.c >> 20;
        }
#pragma unroll
        for (int k = 0; k < 4; k++) bs[k] = wave_sum_u32(bs[k]);
        if (r0) __syncthreads();  // the last round's terms are read
        if (lane < 4) wstat[wave][lane] = lane == 0 ? bs[0] : lane == 1 ? bs[1] : lane == 2 ? bs[2] : bs[3];
        __syncthreads();
        if (wave == 1 && lane < 4)
            for (int w = 0; w < NW; w++) bt += wstat[w][lane];
    }
    if (wave == 1 && lane < 4) {
        const int idx[4] = {kStatTpf, kStatTriangles, kStatFront, kStatClipOverflow};
        stats[f * kNumStats + idx[lane]] = bt;
    }

    // The frame's references, and its range of the lists.
    unsigned long long local = 0;
#pragma unroll
    for (int k = 0; k < kKeep; k++) local += v0[k];
    for (int i = (int)threadIdx.x + kKeep * kScanThreads; i < ntiles; i += kScanThreads)
        local += gld(&cnt[i]);
    local = wave_sum_u64(local);
    if (lane == 0) wsum[wave] = local;
    if (shared) {
        const uint32_t all = wave_sum_u32(all4.x + all4.y + all4.z + all4.w + all1);
        if (lane == 0) wsplit[wave] = all;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long tot = 0;
        for (int w = 0; w < NW; w++) tot += wsum[w];
        uint32_t all = (uint32_t)tot;
        if (shared) {
            all = 0u;
            for (int w = 0; w < NW; w++) all += (uint32_t)wsplit[w];
        }
        longest_s = min(split_refs, max(part_refs, (uint32_t)((float)all * inv_held)));
        // One frame starts at 0, without waiting for the counter.
        unsigned long long base = 0;
        if (nframes > 1) base = atomicAdd(&counters->refs_used, tot);
        stats[f * kNumStats + kStatRefs] = tot;
        if (base + tot > refs_capacity) {
            frame_overflow[f] = 1u;
            atomicOr(&ctrl->overflow, 1u);
            atomicMax(&ctrl->refs_needed, base + tot);
        }
        base_s = base;
    }
    __syncthreads();
    const bool over = frame_overflow[f] != 0u;
    const uint32_t longest = longest_s;
    unsigned long long run = base_s;
    for (int c = 0; c < ntiles; c += kScanThreads) {
        const int i = c + (int)threadIdx.x;
        uint32_t v;
        if (c == 0)
            v = v0[0];
        else if (c == kScanThreads)
            v = v0[1];
        else
            v = i < ntiles ? gld(&cnt[i]) : 0u;
        const bool split = !over && v > longest;
        if (v > part_refs && !split) tile_slab[fr.tile_begin + i] = kNoSlab;
        const uint64_t sm = ballot(split);
        const unsigned long long x = wave_scan_u64(v);
        const uint32_t sv = split ? v : 0u;
        const uint32_t xi = sm ? wave_scan_u32(sv) : 0u;
        if (c) __syncthreads();  // the last round's terms are read
        if (lane == 63) {
            wsum[wave] = x;
            wsplit[wave] = (unsigned long long)__popcll(sm) << 32 | xi;
        }
        __syncthreads();
        unsigned long long wbase = 0, ctot = 0, sbase = 0, stot = 0;
        for (int w = 0; w < NW; w++) {
            if (w < wave) {
                wbase += wsum[w];
                sbase += wsplit[w];
            }
            ctot += wsum[w];
            stot += wsplit[w];
        }
        if (i < ntiles) {
            const uint32_t offv = (uint32_t)(run + wbase + x - v);
            tile_offsets[fr.tile_begin + i] = offv;
            tile_cursor[fr.tile_begin + i] = offv;
            if (over) cnt[i] = 0u;  // overflowed frame: raster draws background only
        }
        if (stot) {  // the same in every thread
            if (threadIdx.x == 0) split_s = atomicAdd(&counters->split, stot);
            __syncthreads();
            sbase += split_s;
            const uint32_t slab = (uint32_t)(sbase >> 32) + (uint32_t)__popcll(sm & lanemask_lt(lane));
            if (split) {
                const uint32_t tile = (uint32_t)(fr.tile_begin + i);
                if (slab <= max_slabs) split_first[slab] = (uint32_t)sbase + xi - sv;
                if (slab < max_slabs) split_tile[slab] = tile;
                tile_slab[tile] = slab < max_slabs ? slab : kNoSlab;
            }
            const uint64_t cm = ballot(split && slab < max_slabs && v > split_refs);
            if (cm && lane == 0)
                atomicAdd(&stats[f * kNumStats + kStatSplit], (unsigned long long)__popcll(cm));
        }
        run += ctot;
    }
}

// ---------------------------------------------------------------------------
// k_bin_fill
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(kFillThreads) void k_bin_fill(const DevFrame* __restrict__ frames,
                                                  const FaceBlock* __restrict__ blocks,
                                                  const uint32_t* __restrict__ frame_overflow,
                                                  uint32_t* __restrict__ tile_cursor,
                                                  uint32_t* __restrict__ refs, int twl,
                                                  int thl) {
    __shared__ uint32_t lcnt[kLdsTiles];
    const int b = blockIdx.x;
    const FaceBlock fb = gload(&blocks[b]);
    const uint32_t cnt = fb.slots(), ovf = fb.ovf;
    if (cnt == 0 || frame_overflow[fb.frame]) return;
    const DevFrame& fr = frames[fb.frame];
    // The block's slots start at slot0; its records are block_rec(b, ovf, i).
    const uint32_t blk = (uint32_t)(b - fr.face_block_begin);  // in the frame
    const uint32_t slot0 = blk * kSlotsPerWg;
    // Tile ranges of the block's first kFillKeep records stay in LDS (the records
    // are read once); later records, if any, are read again in each pass.
    constexpr uint32_t kFillKeep = 256;
    __shared__ uint2 lrange[kFillKeep];  // tx0 | tx1 << 16, ty0 | ty1 << 16
    uint32_t ux = 0u, uy = 0u;  // union: last + 1 | (0xFFFF - first) << 16
    for (uint32_t i = threadIdx.x; i < cnt; i += kFillThreads) {
        const uint32_t ri = block_rec(b, ovf, i);
        const TileRect t = rec_tiles(&fr.rrec[ri], twl, thl);
        if (i < kFillKeep)
            lrange[i] = make_uint2((uint32_t)t.tx0 | (uint32_t)t.tx1 << 16,
                                   (uint32_t)t.ty0 | (uint32_t)t.ty1 << 16);
        if (t.tx0 > t.tx1) continue;
        ux = max_u16x2(ux, (uint32_t)(t.tx1 + 1) | (uint32_t)(0xFFFF - t.tx0) << 16);
        uy = max_u16x2(uy, (uint32_t)(t.ty1 + 1) | (uint32_t)(0xFFFF - t.ty0) << 16);
    }
    // fn(t, i) for the tile range of every record i, 64 records at a time by all
    // lanes of the wave (empty past the last record).
    auto each_range = [&](auto&& fn) {
        for (uint32_t i0 = 0; i0 < cnt; i0 += kFillThreads) {
            const uint32_t i = i0 + threadIdx.x;
            TileRect t{1, 0, 1, 0};
            if (i < cnt) {
                if (i < kFillKeep) {
                    const uint2 v = lrange[i];
                    t = TileRect{(int)(v.x & 0xFFFFu), (int)(v.x >> 16), (int)(v.y & 0xFFFFu),
                                 (int)(v.y >> 16)};
                } else {
                    t = rec_tiles(&fr.rrec[block_rec(b, ovf, i)], twl, thl);
                }
            }
            fn(t, i);
        }
    };
    // The union of the ranges, in vector instructions (LDS minima and maxima of
    // one address by 64 lanes take the lanes one by one: 8 of the 20 us of a
    // block with many triangles).
    ux = wave_max_u16x2(ux);
    uy = wave_max_u16x2(uy);
    const int rx0 = 0xFFFF - (int)(ux >> 16), rx1 = (int)(ux & 0xFFFFu) - 1;
    const int ry0 = 0xFFFF - (int)(uy >> 16), ry1 = (int)(uy & 0xFFFFu) - 1;
    if (rx1 < 0) return;
    // fn(tx, ty, i) for every reference of record i to a tile of [x0, x1] x [y0, y1]:
    // each box by its record's lane, or the boxes of many tiles one after the other
    // by the whole wave where that takes fewer steps (a step here is one box, plus
    // one per 64 tiles). One lane walking the 2,040 tiles of a full-screen triangle
    // kept its workgroup 300 us after all others were done; but where most lanes
    // have such a box, the lanes are the faster side: 2,000 triangles of some 190
    // tiles at 1280x720 90 us, 209 with every box over 16 tiles placed by the wave.
    auto each_ref = [&](int x0, int y0, int x1, int y1, auto&& fn) {
        each_range([&](const TileRect& t, uint32_t i) {
            const int bx0 = max(t.tx0, x0), bx1 = min(t.tx1, x1);
            const int by0 = max(t.ty0, y0), by1 = min(t.ty1, y1);
            const int m = max(bx1 - bx0 + 1, 0) * max(by1 - by0 + 1, 0);
            constexpr int kLaneTiles = 16;
            uint64_t big = ballot(m > kLaneTiles);
            if (big) {
                const uint32_t most = wave_reduce((uint32_t)m, 0u, [](uint32_t a, uint32_t b) {
                    return a > b ? a : b;
                });
                if ((uint32_t)__popcll(big) * (3u + (most >> 6)) >= most) big = 0ull;
            }
            if (m > 0 && (m <= kLaneTiles || !big))
                for (int ty = by0; ty <= by1; ty++)
                    for (int tx = bx0; tx <= bx1; tx++) fn(tx, ty, i);
            for (; big; big &= big - 1) {
                const int L = __builtin_ctzll(big);
                const uint32_t bi = (uint32_t)__builtin_amdgcn_readlane((int)i, L);
                wave_rect(__builtin_amdgcn_readlane(bx0, L), __builtin_amdgcn_readlane(by0, L),
                          __builtin_amdgcn_readlane(bx1, L), __builtin_amdgcn_readlane(by1, L),
                          (int)threadIdx.x, [&](int tx, int ty) { fn(tx, ty, bi); });
            }
        });
    };
    // The union in windows of at most kLdsTiles tiles.
    const int ww = min(rx1 - rx0 + 1, kLdsTiles), wh = min(ry1 - ry0 + 1, kLdsTiles / ww);
    const uint32_t windows = (uint32_t)((rx1 - rx0) / ww + 1) * (uint32_t)((ry1 - ry0) / wh + 1);
    bool sparse = false;
    if (windows > 1u) {
        // Triangles scattered over a large frame: one global atomic per reference,
        // where that is less than the windows cost. A lane's atomics in a row take
        // some 0.4 us each; a window some 8 us, and 0.06 for every step of those rows
        // that falls into it (about half do). Many atomics queue up at the cache
        // lines of the frame's tiles, so the more face blocks, the fewer references.
        // us by windows | by references, 32x32 tiles but where stated: 20,000
        // triangles of 8 pixels at 3840x2160 90 | 14, at 7680x4320 238 | 14, of 60
        // pixels 154 | 49 and 437 | 49; 200,000 of 30 pixels at 1920x1080 78 | 176,
        // at 2560x1440 83 | 111, at 3840x2160 137 | 60; 2,000 of 150 pixels at
        // 1920x1080 87 | 152, at 3840x2160 304 | 154; 20,000 of 60 pixels at 1280x720
        // in 8x8 tiles 498 | 351; a sphere of 212 faces at 1920x1080 43 | 77.
        uint32_t row = 0u, nrefs = 0u;  // atomics in a row; references
        each_range([&](const TileRect& t, uint32_t) {
            const uint32_t m = (uint32_t)((t.tx1 - t.tx0 + 1) * (t.ty1 - t.ty0 + 1));
            row += wave_reduce(m, 0u, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
            nrefs += m;
        });
        nrefs = wave_sum_u32(nrefs);
        const uint32_t most = min(8192u, 300000u / (uint32_t)max(fr.face_blocks, 1));
        sparse = nrefs < max(64u, most) * (windows - 1u) &&
                 0.4f * (float)row < (float)windows * (8.f + 0.06f * (float)row);
    }
    if (sparse) {
        each_ref(rx0, ry0, rx1, ry1, [&](int tx, int ty, uint32_t i) {
            refs[atomicAdd(&tile_cursor[fr.tile_begin + ty * fr.tiles_x + tx], 1u)] = slot0 + i;
        });
        return;
    }
    for (int wy = ry0; wy <= ry1; wy += wh)
        for (int wx = rx0; wx <= rx1; wx += ww) {
            const int xe = min(wx + ww - 1, rx1), ye = min(wy + wh - 1, ry1);
            const int n = ww * (ye - wy + 1);
            for (int k = threadIdx.x; k < n; k += kFillThreads) lcnt[k] = 0u;
            __syncthreads();
            each_ref(wx, wy, xe, ye, [&](int tx, int ty, uint32_t) {
                atomicAdd(&lcnt[(ty - wy) * ww + tx - wx], 1u);
            });
            __syncthreads();
            // One global reservation per touched tile; lcnt becomes the write
            // cursor.
            for (int k = threadIdx.x; k < n; k += kFillThreads) {
                const uint32_t v = lcnt[k];
                if (v)
                    lcnt[k] = atomicAdd(
                        &tile_cursor[fr.tile_begin + (wy + k / ww) * fr.tiles_x + wx + k % ww], v);
            }
            __syncthreads();
            each_ref(wx, wy, xe, ye, [&](int tx, int ty, uint32_t i) {
                refs[atomicAdd(&lcnt[(ty - wy) * ww + tx - wx], 1u)] = slot0 + i;
            });
            __syncthreads();
        }
}

// ---------------------------------------------------------------------------
// k_raster
// ---------------------------------------------------------------------------

// Key ordering: reference pixels keep the LAST fragment whose depth equals the
// maximum depth of all fragments >= -1 (rasterizer.go:156 with the >= test
// and z cleared to -1, rasterizer.go:37). Max over (depth, draw sequence) with
// -0 folded into +0 (they compare equal in the reference) selects it.
__device__ __forceinline__ unsigned long long depth_key(float z, uint32_t seq) {
    uint32_t b = __float_as_uint(z);
    if (b == 0x80000000u) b = 0u;
    uint32_t ord = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
    return ((unsigned long long)ord << 32) | seq;
}

constexpr unsigned long long kBackgroundKey = 0x407FFFFFull << 32;  // depth -1, seq 0

// Barycentrics and the reciprocal depth of one inside pixel (rasterizer.go:149-153)
// from its edge values f12, f20: d = (sf, z0, z1, z2), rc = their reciprocals
// or zeros (IEEE division path).
struct Bary {
    float alpha, beta, gamma, zrec;
};

// The reciprocal path of bary(), for a triangle whose reciprocals are set.
__device__ __forceinline__ Bary bary_rcp(float f12f, float f20f, const float4& d,
                                         const float4& rc) {
    Bary b;
    b.alpha = div_rcp(f12f, d.x, rc.x);
    b.beta = div_rcp(f20f, d.x, rc.x);
    b.gamma = 1.0f - b.alpha - b.beta;
    b.zrec = -(div_rcp(b.alpha, d.y, rc.y) + div_rcp(b.beta, d.z, rc.z) +
               div_rcp(b.gamma, d.w, rc.w));
    return b;
}

__device__ __forceinline__ Bary bary(float f12f, float f20f, const float4& d, const float4& rc) {
    Bary b;
    if (rc.x != 0.f) {
        b = bary_rcp(f12f, f20f, d, rc);
    } else {
        b.alpha = f12f / d.x;
        b.beta = f20f / d.x;
        b.gamma = 1.0f - b.alpha - b.beta;
        b.zrec = -(b.alpha / d.y + b.beta / d.z + b.gamma / d.w);
    }
    return b;
}

// Edge values f01, f12, f20 of pixel (x, y) of a triangle beyond the int32
// range, in wrapping int64 arithmetic (rasterizer.go:107-129).
__device__ __forceinline__ void wide_edges(const WideRec* wr, int x, int y, int64_t f[3]) {
    const int i0[3] = {0, 1, 2}, i1[3] = {1, 2, 0};
#pragma unroll
    for (int k = 0; k < 3; k++) {
        int p = i0[k], q = i1[k];
        int64_t A = wsub(wr->y[p], wr->y[q]);
        int64_t B = wsub(wr->x[q], wr->x[p]);
        int64_t C = wsub(wmul(wr->x[p], wr->y[q]), wmul(wr->x[q], wr->y[p]));
        if (wr->adj >> k & 1u) C = wsub(C, 1);
        f[k] = wadd(wadd(wmul(A, x), wmul(B, y)), C);
    }
}

// Low 32 bits of int(v) (CVTTSS2SQ).
__device__ __forceinline__ int32_t go_int_lo(float v) {
    if (__builtin_fabsf(v) < 2147483648.0f) return (int32_t)v;
    return (int32_t)go_int(v);
}

// int(v) % m, Go's truncated remainder, for 0 < m < 2^31.
__device__ __forceinline__ int32_t go_int_rem(float v, int32_t m) {
    if (__builtin_fabsf(v) < 2147483648.0f) return (int32_t)v % m;
    return (int32_t)(go_int(v) % (int64_t)m);
}

// texture.go:69-88. Textures hold at most 2^28 texels, so indexes fit int32.
__device__ __forceinline__ uint32_t sample(const DevTexture& t, float u, float v) {
    switch (t.type) {
    case 0:
        return t.color;
    case 2: {
        const int32_t x = go_int_lo((1 - u) * t.scale * t.wf) & (t.w - 1);
        const int32_t y = go_int_lo(v * t.scale * t.hf) & (t.h - 1);
        return gld(&t.texels[y * t.w + x]);
    }
    case 1: {
        const int32_t x = go_int_rem((1 - u) * t.scale * t.wf, t.w);
        const int32_t y = go_int_rem(v * t.scale * t.hf, t.h);
        int32_t idx = y * t.w + x;
        if (idx < 0) idx = 0;
        return gld(&t.texels[idx]);
    }
    default:
        return 0xFFFF00FFu;  // magenta {255,0,255,255}
    }
}

// |v| % m for |v| < 2^20, 0 < m < 2^31 and rm = RN(1 / m) or a neighbour, with v's
// sign: go_int_rem of such a v. The quotient's error is below 2^20 * 3 * 2^-24, so
// its floor is one off at most, and one of the two additions sets that right.
__device__ __forceinline__ int32_t rem_small(float v, uint32_t m, float rm) {
    const float a = __builtin_fabsf(v);
    // A quotient above 0 has m <= 2^20: a 24-bit product.
    uint32_t r = (uint32_t)a - (uint32_t)__umul24((uint32_t)(a * rm), m);
    r = min(r, r + m);
    r = min(r, r - m);
    return v < 0.f ? -(int32_t)r : (int32_t)r;
}

// sample() for a texture the wave shares, with its descriptor in scalar registers.
__device__ __forceinline__ uint32_t sample_shared(const DevTexture& t, float u, float v) {
    typedef const __attribute__((address_space(1))) char* gbytes;
    const float fx = (1 - u) * t.scale * t.wf, fy = v * t.scale * t.hf;
    if (t.type == 2) {
        // Sides are powers of two, at most 2^28 texels.
        const uint32_t x = (uint32_t)go_int_lo(fx) & (uint32_t)(t.w - 1);
        const uint32_t y = (uint32_t)go_int_lo(fy) & (uint32_t)(t.h - 1);
        const uint32_t at = ((y << __builtin_ctz((uint32_t)t.w)) + x) << 2;
        return *(const __attribute__((address_space(1))) uint32_t*)((gbytes)t.texels + at);
    }
    if (t.type == 1 &&
        ballot(!(__builtin_fabsf(fx) < 1048576.f && __builtin_fabsf(fy) < 1048576.f)) == 0ull) {
        const int32_t x = rem_small(fx, (uint32_t)t.w, __builtin_amdgcn_rcpf(t.wf));
        const int32_t y = rem_small(fy, (uint32_t)t.h, __builtin_amdgcn_rcpf(t.hf));
        const uint32_t at = (uint32_t)max(y * t.w + x, 0) << 2;
        return *(const __attribute__((address_space(1))) uint32_t*)((gbytes)t.texels + at);
    }
    return sample(t, u, v);
}

// rasterizer.go:81-88
__device__ __forceinline__ uint32_t color_intensity(uint32_t c, float k) {
    const float r = (float)(c & 0xFFu) * k, g = (float)((c >> 8) & 0xFFu) * k,
                b = (float)((c >> 16) & 0xFFu) * k;
    if (ballot(!(__builtin_fabsf(k) < 8388608.f)) == 0ull) {
        // Every product of the wave is within int32: the low bytes of the
        // conversions, put together by byte selects.
        const uint32_t rg = __builtin_amdgcn_perm((uint32_t)(int32_t)g, (uint32_t)(int32_t)r, 0x0C0C0400u);
        return rg | __builtin_amdgcn_perm(c, (uint32_t)(int32_t)b, 0x07000C0Cu);
    }
    return go_uint8(r) | (go_uint8(g) << 8) | (go_uint8(b) << 16) | (c & 0xFF000000u);
}

// The raster stage reads a staged RasterRec as five 16-byte pieces: divisors,
// reciprocals, then (box x, box y, wide, A01), (B01, C01, A12, B12),
// (C12, A20, B20, C20).
static_assert(offsetof(RasterRec, bx0) == 32 && offsetof(RasterRec, by0) == 36 &&
                  offsetof(RasterRec, wide) == 40 && offsetof(RasterRec, e) == 44 &&
                  sizeof(RasterRec) == 80,
              "raster records are staged as five uint4 pieces");


// Exact depth of `count` queued fragments of one wave (rasterizer.go:149-156),
// one per lane, and the (depth, sequence) max into the tile key.
template <int TW>
__device__ __forceinline__ void frag_depth(const uint32_t (*q)[128], uint32_t head,
                                           uint32_t count, const uint4* lrec,
                                           const uint32_t* lslot, unsigned long long* key,
                                           int lane) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if ((uint32_t)lane < count) {
        const uint32_t k = (head + (uint32_t)lane) & 127u;
        const uint32_t pk = q[0][k];
        const int32_t f12 = (int32_t)q[1][k], f20 = (int32_t)q[2][k];
        const uint32_t i = pk >> 12, px_idx = pk & 0xFFFu;
        const uint4 d = lrec[i * 5], rc = lrec[i * 5 + 1];
        const float4 df = make_float4(__uint_as_float(d.x), __uint_as_float(d.y),
                                      __uint_as_float(d.z), __uint_as_float(d.w));
        const float4 rf = make_float4(__uint_as_float(rc.x), __uint_as_float(rc.y),
                                      __uint_as_float(rc.z), __uint_as_float(rc.w));
        // Almost every triangle has reciprocals: when all of the wave's do, the
        // branch is taken once for the wave instead of per lane.
        const Bary b = ballot(rf.x == 0.f) == 0ull ? bary_rcp((float)f12, (float)f20, df, rf)
                                                      : bary((float)f12, (float)f20, df, rf);
        if (b.zrec >= -1.0f) atomicMax(&key[px_idx], depth_key(b.zrec, lslot[i] + 1u));
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDS of k_raster beyond the key array: 64 staged records (80 B) and slots,
// the per-wave fragment rings and the stats reduction.
constexpr int kRasterChunk = 64;
constexpr int kRasterLdsFixed = kRasterChunk * (80 + 4) + 4 * 3 * 128 * 4 + 4 * 2 * 8 + 16;
constexpr int kStartWords = kRasterChunk + 2;  // of a dense workgroup, 8 bytes each

// Waves per SIMD the tile's LDS allows (one wave per SIMD per workgroup), at
// most 8: the register budget follows from it (512 / waves VGPRs).
constexpr int raster_waves(int npx, bool dense = false) {
    const int lds = npx * 8 + kRasterLdsFixed + (dense ? kStartWords * 8 : 0);
    return (160 * 1024) / lds >= 8 ? 8 : (160 * 1024) / lds;
}

// Boxes walked by their pixels in dense lists, and how many of a chunk's 64 make
// it one. 8 requests of 500,000 faces, k_raster: 369 us with (64, 24), 382 (64, 40),
// 389 (32, 24), 406 (32, 40), 425 (16, 40), 436 with each box walked on its own.
constexpr uint32_t kSmallBox = 64;
constexpr int kSmallBoxes = 24;
static_assert(kRasterChunk * kSmallBox <= 64 * kRasterChunk, "a start word per 64 candidates");

// Walk form of a record for one tile (piece 2 of the staged record): the box
// clamped to the tile as one word (x0 - X0 | y0 - Y0 << 6 | x1 - x0 << 12 |
// height << 18 | log2 lanes per row << 25 | wide << 28; height 0 when the box
// misses the tile) and, on the int32 path, the three edge values at the
// clamped box's corner (x0, y0), A*x0 + B*y0 + C (rasterizer.go:107-129 at the
// first pixel of the walk). Inputs are the record's pieces 2..4: box x, box y,
// wide, A01 | B01, C01, A12, B12 | C12, A20, B20, C20.
constexpr uint32_t kWalkWide = 1u << 28;
template <int TW, int TH>
__device__ __forceinline__ uint4 walk_form(const uint4& w2, const uint4& w3, const uint4& w4,
                                           int X0, int Y0) {
    const int x0 = max((int)(int16_t)(w2.x & 0xFFFFu), X0);
    const int x1 = min((int)(int16_t)(w2.x >> 16), X0 + TW - 1);
    const int y0 = max((int)(int16_t)(w2.y & 0xFFFFu), Y0);
    const int y1 = min((int)(int16_t)(w2.y >> 16), Y0 + TH - 1);
    if (x1 < x0 || y1 < y0) return make_uint4(0u, 0u, 0u, 0u);
    const int bw = x1 - x0 + 1;
    int l2 = bw <= 1 ? 0 : 32 - __builtin_clz((uint32_t)(bw - 1));
    if (l2 > 6) l2 = 6;
    uint32_t info = (uint32_t)(x0 - X0) | (uint32_t)(y0 - Y0) << 6 | (uint32_t)(x1 - x0) << 12 |
                    (uint32_t)(y1 - y0 + 1) << 18 | (uint32_t)l2 << 25;
    if (w2.z) return make_uint4(info | kWalkWide, 0u, 0u, 0u);
    // |A|, |B| <= 2^15 and |x|, |y| < 2^14 on the int32 path: exact 24-bit
    // products, and the sums fit int32.
    const int f0 = __mul24((int)w2.w, x0) + __mul24((int)w3.x, y0) + (int)w3.y;
    const int f1 = __mul24((int)w3.z, x0) + __mul24((int)w3.w, y0) + (int)w4.x;
    const int f2 = __mul24((int)w4.y, x0) + __mul24((int)w4.z, y0) + (int)w4.w;
    return make_uint4(info, (uint32_t)f0, (uint32_t)f1, (uint32_t)f2);
}

// Resolves n tile-list entries (slots) into the tile's depth keys: the
// visibility part of rasterizer.go:139-156 for every listed triangle. Returns
// this lane's share of the covered-fragment count (summed over the wave).
//
// Each record's box is walked by a wave, 64 pixels a step: right where boxes are
// large. Dense lists hold boxes of a few pixels, which leave most lanes idle
// (some 30 vector instructions for 1 to 5 pixels). DENSE puts the pixels of a
// chunk's small boxes end to end and tests 64 of them a step, whichever records
// they are of: 8 requests of 500,000 faces, k_raster 430 -> 360 us. Its registers
// and set-up cost sparse lists 4% (32 frames of 200,000 triangles 295 -> 307 us,
// 1,000,000 faces of instances in one frame 36.5 -> 38.2), so it is a variant.
// Lanes by record, or four lanes a record, were slower: the largest box of the
// wave sets the steps.
template <int TW, int TH, bool DENSE>
__device__ __forceinline__ unsigned long long raster_list(
    const DevFrame& fr, int X0, int Y0, const uint32_t* __restrict__ list, uint32_t cnt,
    unsigned long long* key, uint4* lrec, uint32_t* lslot, uint32_t (*q)[128],
    unsigned long long* starts, int lane, int wave) {
    constexpr int CHUNK = kRasterChunk;  // triangles staged in LDS at a time
    static_assert(TW * TH <= 4096 && CHUNK <= (1 << 20),
                  "fragment codes hold the pixel index in 12 bits");
    static_assert(TW <= 64 && TH <= 64, "a clamped box fits one column block of lanes");
    unsigned long long covered_lane = 0;  // wide path, per lane
    uint32_t covered_wave = 0;            // int32 path, wave-uniform
    for (uint32_t base = 0; base < cnt; base += CHUNK) {
        const uint32_t n = min(cnt - base, (uint32_t)CHUNK);
        // Stage the chunk: slots (one coalesced read), then the raster records,
        // all loads of the chunk in flight together. Waves 1 and 2 copy the
        // divisors and reciprocals (pieces 0 and 1) of record t; wave 0 reads
        // the box and edge coefficients of record t and writes their walk
        // form in place of pieces 2..4 (once per record, a lane each, rather
        // than once per record in every wave's scalar unit).
        __syncthreads();
        if (threadIdx.x < n) lslot[threadIdx.x] = list[base + threadIdx.x];
        if (DENSE && wave == 3) starts[lane] = 0ull;
        __syncthreads();
        {
            const uint32_t t = threadIdx.x & 63u;
            if (wave < 3 && t < n) {
                const uint4* src = reinterpret_cast<const uint4*>(&fr.rrec[rec_index(fr, lslot[t])]);
                if (wave > 0) {
                    lrec[t * 5 + wave - 1] = gload(src + wave - 1);
                } else {
                    const uint4 w2 = gload(src + 2), w3 = gload(src + 3), w4 = gload(src + 4);
                    lrec[t * 5 + 2] = walk_form<TW, TH>(w2, w3, w4, X0, Y0);
                    lrec[t * 5 + 3] = make_uint4(w2.w, w3.z, w4.y, w3.x);  // A01 A12 A20 B01
                    if (DENSE) {
                        *reinterpret_cast<uint2*>(&lrec[t * 5 + 4]) = make_uint2(w3.w, w4.z);
                    } else {
                        lrec[t * 5 + 4] = make_uint4(w3.w, w4.z, 0u, 0u);  // B12 B20
                    }
                }
            }
            if (DENSE && wave == 0) {
                // Small boxes: their first candidates, and a bit at each in
                // starts; a box walked on its own has one candidate, of width 0.
                const uint32_t info = t < n ? lrec[t * 5 + 2].x : 0u;
                const uint32_t bw = ((info >> 12) & 63u) + 1u;
                const uint32_t area = bw * ((info >> 18) & 127u);
                uint64_t small = ballot(area != 0u && area <= kSmallBox && !(info & kWalkWide));
                uint32_t end = 0u;
                if (__popcll(small) >= kSmallBoxes) {
                    const bool sm = (small >> lane) & 1u;
                    const uint32_t cand = t < n ? (sm ? area : 1u) : 0u;
                    end = wave_scan_u32(cand);
                    if (t < n) {
                        const uint32_t at = end - cand;
                        const uint32_t px = ((info >> 6) & 63u) * (uint32_t)TW + (info & 63u);
                        // First candidate | first pixel << 16, 2^16 / width (from
                        // above, exact for 64 pixels) | width << 20.
                        *(reinterpret_cast<uint2*>(&lrec[t * 5 + 4]) + 1) = make_uint2(
                            at | px << 16,
                            ((uint32_t)(65536.f * __builtin_amdgcn_rcpf((float)bw)) + 1u) |
                                (sm ? bw << 20 : 0u));
                        atomicOr(reinterpret_cast<uint32_t*>(starts) + (at >> 5), 1u << (at & 31u));
                    }
                } else {
                    small = 0ull;
                }
                const uint64_t own = ballot(area != 0u) & ~small;
                if (lane == 63) {
                    starts[kRasterChunk] = own;
                    starts[kRasterChunk + 1] = end;
                }
            }
        }
        __syncthreads();
        // Lanes with all < 0 hold an inside fragment (every edge value < 0,
        // rasterizer.go:147, and the pixel inside the box); they go to the wave's
        // LDS ring by ballot, and every 64 queued fragments get their exact depth
        // on a full wave.
        uint32_t qhead = 0, qtail = 0;  // wave-uniform ring positions
        auto step = [&](int all, int g1, int g2, uint32_t pk) {
            const uint64_t mask = ballot(all < 0);
            if (mask) {
                if (all < 0) {
                    const uint32_t k =
                        __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                                  __builtin_amdgcn_mbcnt_lo((uint32_t)mask, qtail)) &
                        127u;
                    q[0][k] = pk;
                    q[1][k] = (uint32_t)g1;
                    q[2][k] = (uint32_t)g2;
                }
                const uint32_t m = (uint32_t)__popcll(mask);
                qtail += m;
                covered_wave += m;
                if (qtail - qhead >= 64u) {
                    frag_depth<TW>(q, qhead, 64u, lrec, lslot, key, lane);
                    qhead += 64u;
                }
            }
        };
        uint64_t own = 0;  // DENSE: the wave's records still to be walked
        if (DENSE) {
            const uint32_t total = (uint32_t)sgpr((int)(uint32_t)starts[kRasterChunk + 1]);
            const uint32_t first = (uint32_t)lane < n ? lrec[lane * 5 + 4].z & 0xFFFFu : ~0u;
            for (uint32_t b = (uint32_t)wave * 64u; b < total; b += 256u) {
                // A candidate's record: the last with a start at or before it.
                const unsigned long long sv = starts[b >> 6];
                const uint64_t m = ((uint64_t)(uint32_t)sgpr((int)(sv >> 32)) << 32 |
                                    (uint32_t)sgpr((int)(uint32_t)sv)) >> 1;
                const uint32_t r0 = (uint32_t)__popcll(ballot(first <= b)) - 1u;
                const uint32_t i = __builtin_amdgcn_mbcnt_hi(
                    (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, r0));
                const uint4 w2 = lrec[i * 5 + 2], w3 = lrec[i * 5 + 3], w4 = lrec[i * 5 + 4];
                const uint32_t c = b + (uint32_t)lane, p = c - (w4.z & 0xFFFFu);
                const uint32_t y = __umul24(p, w4.w & 0xFFFFFu) >> 16;
                const uint32_t x = p - __umul24(y, w4.w >> 20);
                const int g0 = (int)edge24((int)w3.x, (int)x, (int)w3.w, (int)y, w2.y);
                const int g1 = (int)edge24((int)w3.y, (int)x, (int)w4.x, (int)y, w2.z);
                const int g2 = (int)edge24((int)w3.z, (int)x, (int)w4.y, (int)y, w2.w);
                const int in = c < total && (w4.w >> 20) != 0u ? -1 : 0;
                step(g0 & g1 & g2 & in, g1, g2, (i << 12) + (w4.z >> 16) + y * (uint32_t)TW + x);
            }
            const unsigned long long ov = starts[kRasterChunk];
            own = ((uint64_t)(uint32_t)sgpr((int)(ov >> 32)) << 32 |
                   (uint32_t)sgpr((int)(uint32_t)ov)) &
                  (0x1111111111111111ull << wave);
        }
        // Per wave, one triangle at a time: lanes cover an lpr x (64/lpr) pixel
        // block of its clamped box, stepping the int32 edge values by additions
        // (rasterizer.go:139-183 walks them the same way).
        for (uint32_t i = wave; DENSE ? own != 0 : i < n; i += 4) {
            if (DENSE) {
                i = (uint32_t)__builtin_ctzll(own);
                own &= own - 1;
            }
            // The walk form of the record (see walk_form): the box word moves
            // to a scalar register, the coefficients stay in vector registers
            // (the same value in every lane).
            const uint4 w2 = lrec[i * 5 + 2], w3 = lrec[i * 5 + 3], w4 = lrec[i * 5 + 4];
            const uint32_t info = (uint32_t)sgpr((int)w2.x);
            const int bh = (int)((info >> 18) & 127u);
            if (bh == 0) continue;  // the box misses the tile
            const int ox = (int)(info & 63u), oy = (int)((info >> 6) & 63u);
            const int dxm = (int)((info >> 12) & 63u), l2 = (int)((info >> 25) & 7u);
            const int x0 = X0 + ox, x1 = x0 + dxm, y0 = Y0 + oy, y1 = y0 + bh - 1;
            const int lpr = 1 << l2, rows = 64 >> l2;
            const int lx = lane & (lpr - 1), ly = lane >> l2;
            if (info & kWalkWide) {
                // Coordinates beyond the int32 range: direct int64 evaluation.
                const uint32_t slot = (uint32_t)sgpr((int)lslot[i]);
                const WideRec* wr = &fr.wrec[rec_index(fr, slot)];
                const uint4 d4 = lrec[i * 5], r4 = lrec[i * 5 + 1];
                const float4 rp[2] = {
                    make_float4(__uint_as_float(d4.x), __uint_as_float(d4.y),
                                __uint_as_float(d4.z), __uint_as_float(d4.w)),
                    make_float4(__uint_as_float(r4.x), __uint_as_float(r4.y),
                                __uint_as_float(r4.z), __uint_as_float(r4.w))};
                for (int yb = y0; yb <= y1; yb += rows) {
                    const int y = yb + ly;
                    for (int xb = x0; xb <= x1; xb += lpr) {
                        const int x = xb + lx;
                        if (y > y1 || x > x1) continue;
                        int64_t f[3];
                        wide_edges(wr, x, y, f);
                        if (!(f[0] < 0 && f[1] < 0 && f[2] < 0)) continue;
                        covered_lane++;
                        const Bary b = bary((float)f[1], (float)f[2], rp[0], rp[1]);
                        if (b.zrec >= -1.0f)
                            atomicMax(&key[(y - Y0) * TW + (x - X0)],
                                      depth_key(b.zrec, slot + 1u));
                    }
                }
                continue;
            }
            // Edge values of the lane's pixel: the value at the clamped box's
            // corner (x0, y0) plus A*lx + B*ly; |A|, |B| <= 2^15 and lx, ly
            // < 64 on this path, so the 24-bit products are exact and every
            // edge value fits int32 (|x|, |y| < 2^14).
            const int A0 = (int)w3.x, A1 = (int)w3.y, A2 = (int)w3.z;
            const int B0 = (int)w3.w, B1 = (int)w4.x, B2 = (int)w4.y;
            int f0 = (int)edge24(A0, lx, B0, ly, w2.y);
            int f1 = (int)edge24(A1, lx, B1, ly, w2.z);
            int f2 = (int)edge24(A2, lx, B2, ly, w2.w);
            const int sy0 = (int)((uint32_t)B0 << (6 - l2));  // B * rows
            const int sy1 = (int)((uint32_t)B1 << (6 - l2));
            const int sy2 = (int)((uint32_t)B2 << (6 - l2));
            // Fragment code: list index << 12 | the pixel's index in the tile
            // (y * TW + x, below 4096 for every tile size), exact in every lane
            // that enqueues (its pixel lies inside the tile).
            const uint32_t prow = (i << 12) + (uint32_t)(oy * TW + ox) + (uint32_t)(ly * TW + lx);
            // The box is at most TW <= 64 pixels wide, so one column block of
            // lanes covers it: a flat loop over row blocks. The lane's column
            // is inside the box iff gx < 0; only the last block can hold rows
            // beyond it.
            const int gx = lx - dxm - 1;
            const int nfull = bh >> (6 - l2);  // blocks of `rows` whole rows
            uint32_t pk = prow;
            for (int sb = 0; sb < nfull; sb++) {
                step(f0 & f1 & f2 & gx, f1, f2, pk);
                f0 += sy0;
                f1 += sy1;
                f2 += sy2;
                pk += (uint32_t)rows * (uint32_t)TW;
            }
            const int rest = bh - (nfull << (6 - l2));
            if (rest > 0) {
                const int gy = ly - rest;  // negative iff the lane's row is inside
                step(f0 & f1 & f2 & gx & gy, f1, f2, pk);
            }
        }
        while (qtail != qhead) {
            const uint32_t cnt_q = min(qtail - qhead, 64u);
            frag_depth<TW>(q, qhead, cnt_q, lrec, lslot, key, lane);
            qhead += cnt_q;
        }
    }
    return covered_lane + (lane == 0 ? (unsigned long long)covered_wave : 0ull);
}

// Deferred shading of the winning fragment of each pixel of the tile, one
// write per pixel. Returns the wave's count of shaded pixels.
//
// Where frames are many k_raster is bound by its instructions (512 frames of
// 1280x720: vector issue in 74% of its cycles, pairs counted once, at 7.5 of 8
// waves), so a pixel's are kept few: one
// reciprocal for u and v, indices of a shared texture by shift or by a reciprocal
// of its side, colour bytes put together by byte selects, 32-bit offsets, and the
// dot grid by one product. 32 frames of 200,000 triangles: k_raster 301 -> 294 us;
// 64 mixed frames: 516 -> 505.
template <int TW, int TH>
__device__ __forceinline__ unsigned long long shade_tile(const DevFrame& fr, int X0, int Y0,
                                                         const unsigned long long* key,
                                                         const DevTexture* __restrict__ textures) {
    constexpr int NPX = TW * TH;
    static_assert(256 % TW == 0, "a thread keeps its column");
    const uint32_t dot_color = fr.dot_color, clear_color = fr.clear_color;
    const int x = X0 + (int)(threadIdx.x % TW);
    int y = Y0 + (int)(threadIdx.x / TW);
    // DotGrid (rasterizer.go:46-52): x, y in {step, 2*step, ...}, the multiples of
    // step but 0. n is one iff n * (dot_inv + 1) mod 2^32 <= dot_inv, dot_inv =
    // floor((2^32 - 1) / step), for the n < 2^14 of a frame (with n = k * step + r
    // and step * (dot_inv + 1) = 2^32 + e, 0 <= e < step, the product is
    // k * e + r * (dot_inv + 1), and k * e <= n < dot_inv; a step above n has
    // k = 0); dot_inv 0, of no grid, takes 0 alone.
    const uint32_t dot_inv = fr.dot_inv;
    const bool dot_x = x != 0 && (uint32_t)x * (dot_inv + 1u) <= dot_inv;
    uint32_t dot_y = (uint32_t)y * (dot_inv + 1u);
    uint32_t at = ((uint32_t)y * (uint32_t)fr.W + (uint32_t)x) << 2;  // below 2^30
    typedef __attribute__((address_space(1))) char* gbytes;
    uint32_t shaded = 0;  // wave-uniform
    for (int i = threadIdx.x; i < NPX; i += 256, y += 256 / TW, dot_y += (256 / TW) * (dot_inv + 1u),
             at += (uint32_t)fr.W * (uint32_t)(256 / TW * 4)) {
        const bool inframe = x < fr.W && y < fr.H;
        const unsigned long long k = key[i];
        const uint32_t seq = (uint32_t)k;
        shaded += (uint32_t)__popcll(ballot(inframe && seq != 0u));
        if (!inframe) continue;
        uint32_t color;
        float depth;
        if (seq == 0u) {
            color = dot_x && y != 0 && dot_y <= dot_inv ? dot_color : clear_color;
            depth = -1.0f;
        } else {
            const uint32_t ri = rec_index(fr, seq - 1u);
            // The shading record and pieces 3 and 4 of the raster record (B01,
            // C01, A12, B12 | C12, A20, B20, C20), in one round trip.
            const uint4* rq = reinterpret_cast<const uint4*>(&fr.rrec[ri]);
            const ShadeRec s = gload(&fr.srec[ri]);
            const uint4 e3 = gload(rq + 3), e4 = gload(rq + 4);
            // The int32 edge values are formed before the wide test; a wide
            // record replaces them (its int32 values are never used, and the
            // sums wrap as unsigned).
            float f12f = (float)(int32_t)edge24((int)e3.z, x, (int)e3.w, y, e4.x);
            float f20f = (float)(int32_t)edge24((int)e4.y, x, (int)e4.z, y, e4.w);
            // The key holds zRec's bits (with -0 folded into +0): only a zero
            // zRec is recomputed; alpha and beta are as in bary().
            const uint32_t ord = (uint32_t)(k >> 32);
            const float zkey = __uint_as_float((ord & 0x80000000u) ? (ord & 0x7FFFFFFFu) : ~ord);
            // rsf is 0 or kShadeWide (IEEE division) unless the raster record
            // holds reciprocals.
            const bool common = __builtin_fabsf(zkey) >= 0x1p-41f && __builtin_fabsf(zkey) <= 0x1p42f &&
                                s.rsf != 0u && s.rsf != kShadeWide;
            const bool fast = ballot(!common) == 0ull;
            Bary b;
            if (fast) {
                // Every pixel of the wave: int32 edge values, reciprocals, and
                // zRec from the key (one branch for the wave, not per lane).
                const float rsf = __uint_as_float(s.rsf);
                b.alpha = div_rcp(f12f, s.sf, rsf);
                b.beta = div_rcp(f20f, s.sf, rsf);
                b.gamma = 1.0f - b.alpha - b.beta;
                b.zrec = zkey;
            } else {
                if (s.rsf == kShadeWide) {
                    int64_t f[3];
                    wide_edges(&fr.wrec[ri], x, y, f);
                    f12f = (float)f[1];
                    f20f = (float)f[2];
                }
                if (zkey != 0.0f) {
                    const float rsf = __uint_as_float(s.rsf);
                    if (s.rsf != 0u && s.rsf != kShadeWide) {
                        b.alpha = div_rcp(f12f, s.sf, rsf);
                        b.beta = div_rcp(f20f, s.sf, rsf);
                    } else {
                        b.alpha = f12f / s.sf;
                        b.beta = f20f / s.sf;
                    }
                    b.gamma = 1.0f - b.alpha - b.beta;
                    b.zrec = zkey;
                } else {
                    const float4 d = gload(reinterpret_cast<const float4*>(rq)),
                                 rc = gload(reinterpret_cast<const float4*>(rq) + 1);
                    b = bary(f12f, f20f, d, rc);
                }
            }
            // rasterizer.go:158-170
            const float un = b.alpha * s.uz[0] + b.beta * s.uz[1] + b.gamma * s.uz[2];
            const float vn = b.alpha * s.vz[0] + b.beta * s.vz[1] + b.gamma * s.vz[2];
            const float inten = b.alpha * s.in[0] + b.beta * s.in[1] + b.gamma * s.in[2];
            uint32_t c;
            const int tex0 = sgpr(s.tex);
            if (ballot(s.tex != tex0) == 0ull) {
                // One texture (or none) for the wave's pixels: its descriptor
                // is read once, with scalar loads.
                if (tex0 < 0) {
                    c = fr.face_color;
                } else {
                    static_assert(sizeof(DevTexture) == 40, "ten words");
                    typedef const __attribute__((address_space(4))) uint32_t* cword;
                    const cword src = (cword)(textures + tex0);
                    uint32_t w[10];
#pragma unroll
                    for (int k = 0; k < 10; k++) w[k] = src[k];
                    DevTexture t;
                    __builtin_memcpy(&t, w, sizeof(DevTexture));
                    float u, v;
                    if (fast && __builtin_fabsf(t.scale) >= 0x1p-40f && __builtin_fabsf(t.scale) <= 0x1p10f) {
                        // Both quotients from one reciprocal (rcp_step), for
                        // |numerator| in [2^-80, 2^86] the exact ones. Below,
                        // |u| < 2^-38: 1 - u is 1, and v * scale * h is under 1
                        // either way. Above, a quotient is the same one, or at
                        // least 2^127, infinite or a NaN, and so past int64 once
                        // scaled, in both ways.
                        const float y = rcp_step(b.zrec);
                        u = div_rcp(un, b.zrec, y);
                        v = div_rcp(vn, b.zrec, y);
                    } else {
                        u = un / b.zrec;
                        v = vn / b.zrec;
                    }
                    c = sample_shared(t, u, v);
                }
            } else {
                c = s.tex < 0 ? fr.face_color : sample(textures[s.tex], un / b.zrec, vn / b.zrec);
            }
            color = color_intensity(c, inten);
            depth = b.zrec;
        }
        if (fr.okey) {
            // Overlay keys are zero between draws: each pixel's is read once.
            uint32_t* const o = fr.okey + (at >> 2);
            const uint32_t ok = gld(o);
            if (ok) {
                gst(o, 0u);
                if ((ok >> 1) >= seq)
                    color = (ok & 1u) ? kVertexColor : ((fr.flags & kShowFaces) ? kEdgeColor : kWhite);
            }
        }
        *(__attribute__((address_space(1))) uint32_t*)((gbytes)fr.rgba + at) = color;
        *(__attribute__((address_space(1))) float*)((gbytes)fr.depth + at) = depth;
    }
    return shaded;
}

// LDS of one raster workgroup.
template <int TW, int TH, bool DENSE>
struct RasterLds {
    unsigned long long key[TW * TH];
    uint4 lrec[kRasterChunk * 5];  // the staged raster records
    uint32_t lslot[kRasterChunk];
    uint32_t qbuf[4][3][128];      // per-wave ring: pixel, f12, f20
    unsigned long long red[4][2];  // per wave: covered fragments, shaded pixels
    uint32_t last;                 // the workgroup shades a split tile
    // Per 64 candidates of a dense chunk, which start a record; then the records
    // walked on their own, and the number of candidates.
    unsigned long long starts[DENSE ? kStartWords : 1];
};

// Entries of the batch's split tiles (k_bin_scan) and the size of their parts:
// part_refs, or what `extra` workgroups need to take one part each. Entries past
// the last slab are of tiles left whole.
struct SplitLists {
    uint32_t n_slabs, entries, part;
};
__device__ __forceinline__ SplitLists split_lists(const DevBatchCounters* counters,
                                                  const uint32_t* split_first, uint32_t max_slabs,
                                                  uint32_t part_refs, uint32_t extra) {
    const unsigned long long split = counters->split;
    const uint32_t n = (uint32_t)(split >> 32);
    SplitLists s;
    s.n_slabs = min(n, max_slabs);
    s.entries = n > max_slabs ? split_first[max_slabs] : (uint32_t)split;
    s.part = max(part_refs, s.entries / max(extra, 1u) + 1u);
    return s;
}

// One part of a tile's list, resolved into LDS keys, and the tile shaded where the
// part is all of it.
//
// The split tiles' entries, put end to end, are cut at every multiple of s.part and
// at the tiles' ends: item k >= 0 is the part that starts at entry k * s.part, and
// the tile's own workgroup (item < 0, tile g) takes its first entries, up to the
// first such multiple. So every workgroup has one part, whatever the lists' lengths.
// The parts of a tile merge their keys into its slab with a 64-bit max (the (depth,
// sequence) resolve does not depend on order); the workgroup that merges last takes
// them back, leaves the slab and its counter cleared for the next draw, and shades.
// No part waits for another. Every thread of the workgroup calls it.
template <int TW, int TH, bool DENSE>
__device__ __forceinline__ void raster_part(
    const DevFrame* __restrict__ frames, const int* __restrict__ tile_first, int nframes,
    uint32_t* __restrict__ tile_counts, const uint32_t* __restrict__ tile_offsets,
    const uint32_t* __restrict__ tile_slab, const uint32_t* __restrict__ refs,
    const DevTexture* __restrict__ textures, unsigned long long* __restrict__ stats,
    const uint32_t* __restrict__ split_first, const uint32_t* __restrict__ split_tile,
    unsigned long long* __restrict__ slabs, uint32_t* __restrict__ slab_done, uint32_t part_refs,
    const DevBatchCounters* __restrict__ counters, uint32_t max_slabs, uint32_t extra, int g,
    int item, RasterLds<TW, TH, DENSE>& L, int lane, int wave) {
    constexpr int NPX = TW * TH;
    // Only parts of split tiles look at the split lists: in every workgroup, their
    // counter ahead of everything else and the values held past it took frames of
    // 129,600 empty 8x8 tiles from 89 to 126 us and 8,160 tiles of large triangles
    // from 194 to 226.
    SplitLists s{0u, 0u, 1u};
    uint32_t slab_i = kNoSlab, first = 0u, pos = 0u;
    if (item >= 0) {
        s = split_lists(counters, split_first, max_slabs, part_refs, extra);
        const unsigned long long at = (unsigned long long)item * s.part;
        if (at >= s.entries) return;
        pos = (uint32_t)at;
        slab_i = (uint32_t)wave_last_le(split_first, (int)s.n_slabs, pos);
        first = (uint32_t)sgpr((int)split_first[slab_i]);
        if (pos == first) return;  // the tile's own workgroup starts there
        g = sgpr((int)split_tile[slab_i]);
    }
    const uint32_t cnt_v = tile_counts[g], off = tile_offsets[g];
    const int fi = wave_last_le(tile_first, nframes, g);
    const DevFrame& fr = frames[fi];
    const int t = g - fr.tile_begin;
    const int X0 = (t % fr.tiles_x) * TW, Y0 = (t / fr.tiles_x) * TH;
    for (int i = threadIdx.x; i < NPX; i += 256) L.key[i] = kBackgroundKey;
    const uint32_t cnt = (uint32_t)sgpr((int)cnt_v);
    if (item < 0 && cnt > part_refs) {
        slab_i = (uint32_t)sgpr((int)tile_slab[g]);
        if (slab_i != kNoSlab) {
            s = split_lists(counters, split_first, max_slabs, part_refs, extra);
            pos = first = (uint32_t)sgpr((int)split_first[slab_i]);
        }
    }
    // Parts of the tile, and this one's entries [beg, beg + n).
    uint32_t beg = 0u, n = cnt, parts = 1u;
    if (slab_i != kNoSlab) {
        parts += (first + cnt - 1u) / s.part - first / s.part;
        beg = pos - first;
        n = min(cnt - beg, s.part - pos % s.part);
    }

    // raster_list's first barrier orders the initialisation before its use.
    const unsigned long long covered =
        raster_list<TW, TH, DENSE>(fr, X0, Y0, refs + off + beg, n, L.key, L.lrec, L.lslot,
                            L.qbuf[wave], L.starts, lane, wave);
    __syncthreads();
    bool shade = true;
    if (parts > 1u) {
        unsigned long long* slab = slabs + (size_t)slab_i * NPX;
        for (int i = threadIdx.x; i < NPX; i += 256) {
            const unsigned long long k = L.key[i];
            if ((uint32_t)k != 0u) atomicMax(&slab[i], k);
        }
        // Device-scope atomics are performed at memory, and counted as complete
        // only then: every wave's merges are in the slab before its workgroup
        // counts itself done. This rests on gfx950, not on the memory model, which
        // promises an order between the relaxed atomics of the slab and of its
        // counter only with a release and an acquire. (Those write back and
        // invalidate the XCD's L2 in every part: 458 -> 1,220 us for 8 dense
        // requests.)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0)
            L.last = __hip_atomic_fetch_add(&slab_done[slab_i], 1u, __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT) == parts - 1u;
        __syncthreads();
        shade = sgpr((int)L.last) != 0;
        if (shade) {
            // Read at memory too (past this XCD's caches).
            for (int i = threadIdx.x; i < NPX; i += 256) {
                const unsigned long long k =
                    __hip_atomic_load(&slab[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                L.key[i] = k ? k : kBackgroundKey;
                slab[i] = 0ull;
            }
            if (threadIdx.x == 0) slab_done[slab_i] = 0u;
            __syncthreads();
        }
    }
    unsigned long long shaded = 0;
    if (shade) {
        // Tile counts are zero between draws: the face stage of the next draw
        // accumulates into them again.
        if (threadIdx.x == 0 && cnt) tile_counts[g] = 0u;
        shaded = shade_tile<TW, TH>(fr, X0, Y0, L.key, textures);
    }
    const unsigned long long cov = wave_total(covered, lane);
    if (lane == 0) {
        L.red[wave][0] = cov;
        L.red[wave][1] = shaded;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        const unsigned long long sum = L.red[0][threadIdx.x] + L.red[1][threadIdx.x] +
                                       L.red[2][threadIdx.x] + L.red[3][threadIdx.x];
        if (sum)
            atomicAdd(&stats[fi * kNumStats + (threadIdx.x ? kStatShaded : kStatCovered)], sum);
    }
}

// XCD-aware tile order. Workgroup h runs on XCD h mod 8; each XCD takes runs
// of kTileRun consecutive tiles (runs x, x + 8, x + 16, ... for XCD x), so
// neighbouring tiles, which share triangle records, read them through one L2.
constexpr int kTileRun = 128;
__device__ __forceinline__ int xcd_tile(int h) {
    const int x = h & 7, j = h >> 3;
    return ((j / kTileRun) * 8 + x) * kTileRun + j % kTileRun;
}

// `extra` workgroups (a multiple of 8) for the later parts of split tiles, one item
// each, then one per screen tile (total_tiles rounded up to whole runs of all XCDs;
// workgroups past the last tile or item return at once). One item each, not a loop:
// what it keeps in scalar registers across items spills (k_raster 295 -> 325 us for
// 32 frames of 200,000 triangles). Parts in a kernel of their own ahead of the tiles'
// took 13 us more for a single frame and 75 of 533 us for 8 dense requests.
template <int TW, int TH, bool DENSE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(raster_waves(TW * TH, DENSE))))
void k_raster(
    const DevFrame* __restrict__ frames, const int* __restrict__ tile_first, int nframes,
    int total_tiles, uint32_t* __restrict__ tile_counts,
    const uint32_t* __restrict__ tile_offsets, const uint32_t* __restrict__ tile_slab,
    const uint32_t* __restrict__ refs, const DevTexture* __restrict__ textures,
    unsigned long long* __restrict__ stats, const DevBatchCounters* __restrict__ counters,
    const uint32_t* __restrict__ split_first, const uint32_t* __restrict__ split_tile,
    unsigned long long* __restrict__ slabs, uint32_t* __restrict__ slab_done, uint32_t max_slabs,
    uint32_t part_refs, int extra) {
    __shared__ RasterLds<TW, TH, DENSE> L;
    const int lane = threadIdx.x & 63, wave = sgpr(threadIdx.x >> 6);
    const int it = (int)blockIdx.x < extra ? (int)blockIdx.x : -1;
    const int g = it < 0 ? xcd_tile((int)blockIdx.x - extra) : 0;
    if (g >= total_tiles) return;
    raster_part<TW, TH, DENSE>(frames, tile_first, nframes, tile_counts, tile_offsets, tile_slab, refs,
                        textures, stats, split_first, split_tile, slabs, slab_done, part_refs,
                        counters, max_slabs, (uint32_t)extra, g, it, L, lane, wave);
}

// Persistent form: a fixed grid (every CU at the raster's occupancy) in which
// workgroup w takes w, w + grid, w + 2 * grid, ... of the items and then the tiles.
template <int TW, int TH>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(raster_waves(TW * TH))))
void k_raster_persistent(
    const DevFrame* __restrict__ frames, const int* __restrict__ tile_first, int nframes,
    int total_tiles, uint32_t* __restrict__ tile_counts,
    const uint32_t* __restrict__ tile_offsets, const uint32_t* __restrict__ tile_slab,
    const uint32_t* __restrict__ refs, const DevTexture* __restrict__ textures,
    unsigned long long* __restrict__ stats, const DevBatchCounters* __restrict__ counters,
    const uint32_t* __restrict__ split_first, const uint32_t* __restrict__ split_tile,
    unsigned long long* __restrict__ slabs, uint32_t* __restrict__ slab_done, uint32_t max_slabs,
    uint32_t part_refs, int extra) {
    __shared__ RasterLds<TW, TH, false> L;
    const int lane = threadIdx.x & 63, wave = sgpr(threadIdx.x >> 6);
    for (int j = (int)blockIdx.x; j < extra + total_tiles; j += (int)gridDim.x) {
        raster_part<TW, TH, false>(frames, tile_first, nframes, tile_counts, tile_offsets, tile_slab,
                            refs, textures, stats, split_first, split_tile, slabs, slab_done,
                            part_refs, counters, max_slabs, (uint32_t)extra,
                            j < extra ? 0 : j - extra, j < extra ? j : -1, L, lane, wave);
        // The LDS state is rewritten by the next tile.
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Mesh set-up: face normals as NewMesh computes them (mesh.go:53-60)
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(256) void k_face_normals(const float* __restrict__ pos,
                                                      const int32_t* __restrict__ vi, int F,
                                                      float* __restrict__ fn) {
    int f = blockIdx.x * 256 + threadIdx.x;
    if (f >= F) return;
    const float* a = pos + 3 * (size_t)vi[3 * f];
    const float* b = pos + 3 * (size_t)vi[3 * f + 1];
    const float* c = pos + 3 * (size_t)vi[3 * f + 2];
    float ax = b[0] - a[0], ay = b[1] - a[1], az = b[2] - a[2];
    float bx = c[0] - a[0], by = c[1] - a[1], bz = c[2] - a[2];
    float nx = ay * bz - az * by;
    float ny = az * bx - ax * bz;
    float nz = ax * by - ay * bx;
    float len = __builtin_sqrtf(nx * nx + ny * ny + nz * nz);
    fn[4 * (size_t)f + 0] = nx / len;
    fn[4 * (size_t)f + 1] = ny / len;
    fn[4 * (size_t)f + 2] = nz / len;
    fn[4 * (size_t)f + 3] = 1.0f;
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------

void launch_face_normals(const float* pos, const int32_t* vi, int F, float* fn, hipStream_t s) {
    if (F <= 0) return;
    hipLaunchKernelGGL(k_face_normals, dim3((F + 255) / 256), dim3(256), 0, s, pos, vi, F, fn);
}

int raster_workgroups(int npx) { return 256 * raster_waves(npx); }

constexpr int kWideFaceBlocks = 4096, kWideFaceBlocksPast = 384;
void launch_face(const LaunchParams& p, hipStream_t s) {
    if (p.face_blocks == 0) return;
    // Four waves a block for launches that leave the chip part idle, one past
    // that, whose waves do not wait for each other. The chip holds 4,096 waves (4
    // on each of 1,024 SIMDs). us with one | four waves: 2 blocks 27.5 | 19.6,
    // 20 18.8 | 12.1, 157 29.5 | 18.8, 782 33.7 | 30.6, 4,000 57 | 50, 20,000
    // 254 | 262, 25,000 119 | 266, 38,000 279 | 458.
    // In frames past the tile table (kTableTiles) a dense mesh is bound by the
    // atomics of its tiles, which more waves at once only queue up longer (a sphere
    // in the middle of 2560x1440: 200 blocks 42 | 41, 391 73 | 79, 586 100 | 125,
    // 1,953 357 | 471); where it is not, four waves gain a few us, and a frame
    // among others nothing, from 200 blocks on.
    auto launch = [&](auto kernel, int threads) {
        hipLaunchKernelGGL(kernel, dim3(p.face_grid), dim3(threads), 0, s, p.objs, p.frames,
                           p.tile_counts, p.blocks, p.tw_log2, p.th_log2, p.xcd_face,
                           p.obj_first, p.nframes, p.rec_pool, p.rec_pools, p.pool_recs,
                           p.ovf_begin, p.ctrl, p.frame_overflow);
    };
    if (p.face_blocks <= (p.frame_tiles <= kTableTiles ? kWideFaceBlocks : kWideFaceBlocksPast))
        launch(k_face<4>, 256);
    else
        launch(k_face<1>, 64);
}

void xcd_tables(const int* n, int nframes, int* table, int* grid) {
    int longest = 0;
    for (int x = 0; x < 8; x++) {
        int* P = table + x * (nframes + 1);
        P[0] = 0;
        for (int f = 0; f < nframes; f++)
            P[f + 1] = P[f] + xcd_count(x, n[f]);
        longest = std::max(longest, P[nframes]);
    }
    *grid = 8 * longest;
}

void launch_decorate(const LaunchParams& p, hipStream_t s) {
    if (p.nframes == 0) return;
    hipLaunchKernelGGL(k_decorate, dim3(p.nframes), dim3(kDecorateThreads), 0, s, p.frames);
}

void launch_fog(void* rgba, const void* depth, uint64_t n, float fog_start, float fog_end,
                uint32_t color, hipStream_t s) {
    if (n == 0) return;
    const uint64_t blocks = std::min<uint64_t>((n + 255) / 256, 4096);
    hipLaunchKernelGGL(k_fog, dim3((unsigned)blocks), dim3(256), 0, s, (uint32_t*)rgba,
                       (const float*)depth, n, fog_start, fog_end, color);
}

void launch_overlay(const LaunchParams& p, hipStream_t s) {
    if (p.face_blocks == 0) return;
    // Enough workgroups to fill the chip where the blocks alone do not.
    const unsigned share = p.face_blocks >= 2048 ? 1u : 8u;
    hipLaunchKernelGGL(k_overlay, dim3(p.face_blocks, share), dim3(256), 0, s, p.frames,
                       p.blocks, p.stats);
}

void launch_bin_scan(const LaunchParams& p, hipStream_t s) {
    hipLaunchKernelGGL(k_bin_scan, dim3(p.nframes), dim3(kScanThreads), 0, s, p.frames, p.nframes,
                       p.tile_counts, p.tile_offsets, p.tile_cursor, p.frame_overflow, p.stats,
                       p.counters, p.ctrl, p.refs_capacity, p.tile_slab, p.split_first,
                       p.split_tile, p.max_slabs, p.part_refs, p.split_refs, p.rec_pool, p.blocks,
                       p.total_tiles, 1.0f / raster_workgroups(1 << (p.tw_log2 + p.th_log2)));
}

void launch_bin_fill(const LaunchParams& p, hipStream_t s) {
    if (p.face_blocks == 0) return;
    hipLaunchKernelGGL(k_bin_fill, dim3(p.face_blocks), dim3(kFillThreads), 0, s, p.frames,
                       p.blocks, p.frame_overflow, p.tile_cursor, p.refs,
                       p.tw_log2, p.th_log2);
}

// Self-check of div_rcp against IEEE division: pair i is drawn from SplitMix64(seed
// + i) in four families over the documented domain (|d| in [2^-40, 2^41),
// |a| in [2^-70, 2^70] or +0): random floats; quotients next to a rounding
// midpoint; divisors with extreme mantissas (all ones, powers of two); integer
// numerators over integer divisors as the raster stage divides them. Each pair is
// then taken once more for the quotients of a shared reciprocal (rcp_step), with
// exponents over its own domain, the ends included.
__device__ __forceinline__ uint64_t splitmix64(uint64_t x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

__device__ __forceinline__ float make_float(uint32_t sign, int exp, uint32_t mant) {
    return __uint_as_float((sign << 31) | ((uint32_t)(exp + 127) << 23) | (mant & 0x7FFFFFu));
}

__global__ __launch_bounds__(256) void k_check_div(uint64_t n, uint64_t seed,
                                                   unsigned long long* mismatches,
                                                   float* first_bad) {
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * 256) {
        const uint64_t r0 = splitmix64(seed + 2 * i), r1 = splitmix64(seed + 2 * i + 1);
        const int fam = (int)(i & 3);
        float a, d;
        const int ed = (int)(r0 % 81) - 40;
        if (fam == 0) {
            d = make_float((uint32_t)(r0 >> 63), ed, (uint32_t)(r0 >> 8));
            const int ea = (int)(r1 % 141) - 70;
            a = ((r1 >> 40) & 255) == 0 ? 0.0f
                                        : make_float((uint32_t)(r1 >> 63), ea, (uint32_t)(r1 >> 8));
        } else if (fam == 1) {
            // a = RN(d * m) with m = a float plus half an ulp: a/d lies next to m.
            d = make_float((uint32_t)(r0 >> 63), ed, (uint32_t)(r0 >> 8));
            const int em = (int)(r1 % 61) - 30;
            const double m = (double)make_float(0, em, (uint32_t)(r1 >> 8)) +
                             ldexp(1.0, em - 24) * ((r1 >> 62) & 1 ? 1.0 : -1.0);
            a = (float)((double)d * m);
            if (__builtin_fabsf(a) < 0x1p-70f || __builtin_fabsf(a) > 0x1p70f) a = 1.0f;
        } else if (fam == 2) {
            const uint32_t mant = (r0 >> 40) & 1 ? 0x7FFFFFu : ((r0 >> 41) & 1 ? 0u : 1u);
            d = make_float((uint32_t)(r0 >> 63), ed, mant);
            const int ea = (int)(r1 % 141) - 70;
            a = make_float((uint32_t)(r1 >> 63), ea, (uint32_t)(r1 >> 8));
        } else {
            d = (float)(int32_t)(((r0 >> 16) & 0x7FFFFFFFu) | 1u) * ((r0 >> 63) ? -1.0f : 1.0f);
            a = (float)(int32_t)(((r1 >> 16) & 0x7FFFFFFFu) | 1u) * ((r1 >> 63) ? -1.0f : 1.0f);
            if (((r1 >> 8) & 3) == 0) a = (float)(int32_t)((r1 >> 20) & 0xFFF) + 1.0f;
        }
        auto check = [&](float num, float div, float y) {
            const float want = num / div;
            const float got = div_rcp(num, div, y);
            if (__float_as_uint(want) != __float_as_uint(got) &&
                atomicAdd(mismatches, 1ull) == 0ull) {
                first_bad[0] = num;
                first_bad[1] = div;
                first_bad[2] = want;
                first_bad[3] = got;
            }
        };
        check(a, d, 1.0f / d);
        // z of the pair's significand in [2^-41, 2^42]; a of its own in [2^-80, 2^86]
        // (the next to a midpoint: the product with z of a float plus half an ulp).
        const uint64_t r2 = splitmix64(r0 ^ r1);
        const int ez = (int)(r2 % 84) - 41, ea = (int)((r2 >> 8) % 167) - 80;
        const float z = make_float((uint32_t)(r2 >> 63), ez, ez == 42 ? 0u : __float_as_uint(d));
        float num = make_float((uint32_t)(r2 >> 62) & 1u, ea, ea == 86 ? 0u : __float_as_uint(a));
        if (fam == 1) {
            const int em = (int)((r2 >> 16) % 101) - 50;
            num = (float)((double)z * ((double)make_float(0, em, (uint32_t)(r2 >> 24)) +
                                       ldexp(1.0, em - 24)));
            if (__builtin_fabsf(num) < 0x1p-80f || __builtin_fabsf(num) > 0x1p86f) num = 1.0f;
        }
        check(num, z, rcp_step(z));
    }
}

void launch_check_div(uint64_t n, uint64_t seed, unsigned long long* mismatches, float* first_bad,
                      hipStream_t s) {
    const uint64_t blocks = std::min<uint64_t>((n + 255) / 256, 16384);
    if (blocks)
        hipLaunchKernelGGL(k_check_div, dim3((unsigned)blocks), dim3(256), 0, s, n, seed,
                           mismatches, first_bad);
}

// Plain device-to-device copy: 16-byte vector copies when both pointers and the
// size allow it, else bytes. Also the known-size kernel that HBM counters are
// calibrated against.
__global__ __launch_bounds__(256) void k_copy16(const uint4* __restrict__ src,
                                                uint4* __restrict__ dst, size_t n) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        dst[i] = src[i];
}

__global__ __launch_bounds__(256) void k_copy8(const uint8_t* __restrict__ src,
                                               uint8_t* __restrict__ dst, size_t n) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        dst[i] = src[i];
}

void launch_copy(void* dst, const void* src, size_t bytes, hipStream_t s) {
    if (bytes == 0) return;
    const bool vec = ((uintptr_t)dst % 16 == 0) && ((uintptr_t)src % 16 == 0) && bytes % 16 == 0;
    const size_t n = vec ? bytes / 16 : bytes;
    const size_t blocks = std::min<size_t>((n + 255) / 256, 8192);
    if (vec)
        hipLaunchKernelGGL(k_copy16, dim3((unsigned)blocks), dim3(256), 0, s,
                           (const uint4*)src, (uint4*)dst, n);
    else
        hipLaunchKernelGGL(k_copy8, dim3((unsigned)blocks), dim3(256), 0, s,
                           (const uint8_t*)src, (uint8_t*)dst, n);
}

// Fills n 32-bit words with v: the zeroing of tile counters, slabs and control
// words (a kernel rather than hipMemsetAsync, so that the launch sequence of a
// batch can be captured in a graph).
__global__ __launch_bounds__(256) void k_fill32(uint32_t* __restrict__ p, uint32_t v, size_t n) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        p[i] = v;
}

void launch_fill32(uint32_t* p, uint32_t v, size_t n, hipStream_t s) {
    if (n == 0) return;
    const size_t blocks = std::min<size_t>((n + 255) / 256, 4096);
    hipLaunchKernelGGL(k_fill32, dim3((unsigned)blocks), dim3(256), 0, s, p, v, n);
}

// Order-independent 64-bit digest of n words: the sum over i of a mix of
// (word i, i), accumulated into *out (so one digest covers several buffers).
__global__ __launch_bounds__(256) void k_checksum(const uint32_t* __restrict__ p, size_t n,
                                                  unsigned long long* __restrict__ out) {
    unsigned long long acc = 0;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        unsigned long long x = ((unsigned long long)p[i] << 32) ^ (unsigned long long)i;
        x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
        x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
        acc += x ^ (x >> 31);
    }
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if ((threadIdx.x & 63) == 0 && acc) atomicAdd(out, acc);
}

void launch_checksum(const void* p, size_t words, unsigned long long* out, hipStream_t s) {
    if (words == 0) return;
    const size_t blocks = std::min<size_t>((words + 255) / 256, 2048);
    hipLaunchKernelGGL(k_checksum, dim3((unsigned)blocks), dim3(256), 0, s, (const uint32_t*)p,
                       words, out);
}

// Writes the words carried by the kernel's arguments to their two places and
// clears the zero ranges: host data reaches device memory without a host buffer
// that must outlive the call, and without an allocation.
__global__ __launch_bounds__(256) void k_put(PutChunk c) {
    const uint32_t t = blockIdx.x * 256u + threadIdx.x, step = gridDim.x * 256u;
    for (uint32_t i = t; i < c.n[0] + c.n[1]; i += step)
        (i < c.n[0] ? c.dst[0][i] : c.dst[1][i - c.n[0]]) = c.w[i];
#pragma unroll
    for (int k = 0; k < 3; k++)
        for (size_t i = t; i < c.zero_n[k]; i += step) c.zero[k][i] = make_uint4(0u, 0u, 0u, 0u);
}

void launch_put(const PutSpan put[2], const ZeroSpan zero[3], hipStream_t s) {
    // The first launch clears; as many follow as the words need.
    size_t done[2] = {0, 0};
    size_t most = 0;
    for (int k = 0; k < 3; k++) most = std::max(most, zero[k].bytes / 16);
    for (bool first = true;; first = false) {
        PutChunk c;
        std::memset(&c, 0, sizeof c);
        size_t room = kPutWords, at = 0;
        for (int k = 0; k < 2; k++) {
            const size_t words = (put[k].bytes + 3) / 4;
            const size_t n = std::min(room, words - done[k]);
            const size_t b0 = done[k] * 4;
            c.dst[k] = (uint32_t*)put[k].dst + done[k];
            c.n[k] = (uint32_t)n;
            if (n)
                std::memcpy(c.w + at, (const char*)put[k].src + b0,
                            std::min(n * 4, put[k].bytes - b0));
            done[k] += n;
            room -= n;
            at += n;
        }
        if (!first && at == 0) return;
        size_t blocks = 1;
        if (first) {
            for (int k = 0; k < 3; k++) {
                c.zero[k] = (uint4*)zero[k].p;
                c.zero_n[k] = zero[k].bytes / 16;
            }
            blocks = std::min<size_t>(std::max<size_t>(1, (most + 255) / 256), 1024);
        }
        hipLaunchKernelGGL(k_put, dim3((unsigned)blocks), dim3(256), 0, s, c);
    }
}

template <int TW, int TH>
static void raster_t(const LaunchParams& p, hipStream_t s) {
    // Workgroups for split tiles' parts: four times what fills every CU at the
    // raster's occupancy, so that the parts of a dense batch end close together
    // (8 dense requests, 7,560 tiles, before the dense form: 628 us with one time,
    // 481 with two, 423 with four, 425 with eight); fewer for a small batch (one frame: 256, 1,024 and
    // 2,048 alike), and one time for a batch whose tiles alone fill the chip over
    // and over (64 mixed frames: one, two, four and eight times alike; they return
    // at once where nothing is split, 2,048 in 1 of 300 us, 8,192 in 4).
    const int fill = raster_workgroups(TW * TH);
    const int most = p.total_tiles > 8 * fill ? fill : 4 * fill;
    const int extra =
        p.max_slabs ? (std::min(most, std::max(1024, p.total_tiles)) + 7) / 8 * 8 : 0;
    if (p.raster_persistent) {
        hipLaunchKernelGGL((k_raster_persistent<TW, TH>), dim3(std::min(p.total_tiles, fill)),
                           dim3(256), 0, s, p.frames, p.tile_first, p.nframes,
                           p.total_tiles, p.tile_counts, p.tile_offsets, p.tile_slab, p.refs,
                           p.textures, p.stats, p.counters, p.split_first, p.split_tile, p.slabs,
                           p.slab_done, p.max_slabs, p.part_refs, extra);
        return;
    }
    constexpr int kRound = 8 * kTileRun;
    const int tiles = (p.total_tiles + kRound - 1) / kRound * kRound;
    hipLaunchKernelGGL((p.dense ? k_raster<TW, TH, true> : k_raster<TW, TH, false>),
                       dim3(tiles + extra), dim3(256), 0, s, p.frames, p.tile_first, p.nframes,
                       p.total_tiles, p.tile_counts, p.tile_offsets, p.tile_slab, p.refs, p.textures,
                       p.stats, p.counters, p.split_first, p.split_tile, p.slabs, p.slab_done,
                       p.max_slabs, p.part_refs, extra);
}

bool launch_raster(const LaunchParams& p, hipStream_t s) {
    if (p.total_tiles == 0) return true;
#define GR_RASTER_CASE(W, H)                \
    if (p.tw_log2 == W && p.th_log2 == H) { \
        raster_t<(1 << W), (1 << H)>(p, s); \
        return true;                        \
    }
    GR_RASTER_CASE(3, 3) GR_RASTER_CASE(3, 4) GR_RASTER_CASE(3, 5) GR_RASTER_CASE(3, 6)
    GR_RASTER_CASE(4, 3) GR_RASTER_CASE(4, 4) GR_RASTER_CASE(4, 5) GR_RASTER_CASE(4, 6)
    GR_RASTER_CASE(5, 3) GR_RASTER_CASE(5, 4) GR_RASTER_CASE(5, 5) GR_RASTER_CASE(5, 6)
    GR_RASTER_CASE(6, 3) GR_RASTER_CASE(6, 4) GR_RASTER_CASE(6, 5) GR_RASTER_CASE(6, 6)
#undef GR_RASTER_CASE
    return false;
}

}  // namespace gr
