// diff.hip — the differentiable shading pass of libprh: forward and adjoint
// of the deferred Blinn-Phong shading at fixed visibility.
//
// polyred has no derivative path; this extends its shading model
// (shader/blinn_cpu.go:24-106, the sums before Round) with real-valued
// parameters:
//   albedo     per transformed vertex, interpolated perspective-correctly as
//              drawClipped interpolates the vertex colour (render/raster.go:
//              500-507); it stands where FragmentShader reads the uniform
//              texture colour (ambient and diffuse terms);
//   normal     per transformed vertex, unit(sum bc_k N_k) as drawClipped's
//              normal (render/raster.go:509-511);
//   Kd, Ks     per material (RGB, the 0..255 scale of BlinnPhong.Diffuse and
//              .Specular), shininess per material;
//   position and intensity of every light.
// A pixel's geometry is rebuilt from its visibility key as k_shade does (a
// clipped piece takes its parent triangle); the world position, view vector
// and light colours are fixed.  The loss is sum over shaded pixels and RGB of
// (lin - target)^2.  Light gradients and the loss are accumulated in each
// thread's registers over all its tiles, material gradients in per-lane LDS
// bins, vertex gradients in a
// workgroup's LDS table.
//
// Shadows enter at fixed visibility, as the reference applies them after the
// shading (render/raster.go:339-347): the pixel's sums are scaled by
// 2^-count, count the lights for which shadingVisibility reported true in the
// frame that fixed the visibility.  A view's pixel state is either rebuilt
// from the visibility buffer at every launch or read from a stored G-buffer.
#include "kernels.hpp"
#include "roots.hpp"

#include <algorithm>
#include <type_traits>

using namespace gm;

namespace prh {

namespace {

struct F3 {
    float x, y, z;
};
__device__ __forceinline__ F3 f3(float x, float y, float z) { return F3{x, y, z}; }
__device__ __forceinline__ F3 operator+(F3 a, F3 b) { return f3(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ __forceinline__ F3 operator-(F3 a, F3 b) { return f3(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ F3 operator*(float s, F3 a) { return f3(s * a.x, s * a.y, s * a.z); }
// This pass has no bit-exact counterpart in the reference, so it may fuse
// (the file is compiled with -ffp-contract=off for gomath.hpp's sake).
__device__ __forceinline__ float fma1(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ F3 fma3(float s, F3 a, F3 c) { return f3(fma1(s, a.x, c.x), fma1(s, a.y, c.y), fma1(s, a.z, c.z)); }
__device__ __forceinline__ float dot(F3 a, F3 b) { return fma1(a.x, b.x, fma1(a.y, b.y, a.z * b.z)); }
__device__ __forceinline__ F3 ld3(const float* p) { return f3(p[0], p[1], p[2]); }
__device__ __forceinline__ F3 xyz(float4 a) { return f3(a.x, a.y, a.z); }
// 1 / x and x / y by the steps of roots.hpp, and 1 / sqrt(x) within 0.51 ulp from
// the hardware estimate (1 ulp) and one Newton step, with the residual 1 - x r^2
// to both halves of x r: a third of the instructions of the compiler's
// expansions (1 / sqrtf(x) rounds twice).  They hold for 2^-100 <= |x| < 2^100; `off` collects
// the inputs outside, and a pixel that had one is computed again with SAFE,
// the library's.
template <bool SAFE>
struct Ops {
    uint32_t off = 0;
    __device__ __forceinline__ void note(float x) {
        if (!SAFE) off = max(off, (__float_as_uint(x) & 0x7fffffffu) - 0x0d800000u);
    }
    __device__ __forceinline__ bool bad() const { return !SAFE && off >= 0x64000000u; }
    __device__ __forceinline__ float rsqrt(float x) {
        if (SAFE) return 1.0f / __builtin_sqrtf(x);
        note(x);
        const float r = __builtin_amdgcn_rsqf(x);
        const float h = x * r, hl = fma1(x, r, -h);
        const float e = fma1(-hl, r, fma1(-h, r, 1.0f));
        return fma1(0.5f * r, e, r);
    }
    __device__ __forceinline__ float rcp(float x) {
        if (SAFE) return 1.0f / x;
        note(x);
        return rcp_exact(x);
    }
    // x / y with r = rcp(y)
    __device__ __forceinline__ float quot(float x, float y, float r) {
        if (SAFE) return x / y;
        return quot_exact(x, y, r);
    }
};
// x / 255: a product with the rounded 1 / 255 alone would scale every colour
// by 1 + 6e-8, a bias the sums over pixels do not average out.  For the same
// reason it divides a pixel's products and never a material's colour, whose
// rounding all of its pixels would share (the loss's relative error at 800x600
// 7.8e-8 that way, 1.2e-8 this).
__device__ __forceinline__ float div255(float x) {
    constexpr float hi = (float)(1.0 / 255.0), lo = (float)(1.0 / 255.0 - (double)hi);
    return fma1(x, hi, x * lo);
}
// x^y and log2(x) for x in [0, 1] (x = 0: log2 is not used), within 0.57 and
// 0.51 ulp for x in (0, 1] and y in [2^-8, 2048] (the library's powf is within
// 1 ulp, and its logf came on top): log2 of the mantissa from the atanh
// series, 2^f from the exponential series, their leading terms in double and
// the rest, which is at most 2^-12 of log2 and 2^-3 of 2^f, in float32.  (All
// of them in double took 20 more instructions and 44 registers of constants.)
// Other y take the library.
__device__ __forceinline__ float pow_log2(float x, float y, float& lg) {
    lg = 0.0f;
    if (x == 0.0f && y > 0.0f) return 0.0f;
    if (!(x > 0.0f && y >= 0.00390625f && y <= 2048.0f)) {
        lg = __builtin_log2f(x);
        return __builtin_powf(x, y);
    }
    constexpr double LN2 = 0.69314718055994531;
    float mf = __builtin_amdgcn_frexp_mantf(x);  // [1/2, 1)
    int e = __builtin_amdgcn_frexp_expf(x);
    const bool low = mf < 0.70710678f;
    mf = low ? mf + mf : mf;
    e -= low ? 1 : 0;
    // log2(m) = (2 / ln 2) atanh(s), s = (m - 1) / (m + 1), s^2 < 0.0295
    const double m = mf, d = m + 1.0;
    double r = __builtin_amdgcn_rcp(d);  // 2^-23, squared by the step
    r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
    const double sv = (m - 1.0) * r, s2 = sv * sv;
    const float t2 = (float)s2;
    float q = (float)(2 / (13 * LN2));
    q = fma1(q, t2, (float)(2 / (11 * LN2)));
    q = fma1(q, t2, (float)(2 / (9 * LN2)));
    q = fma1(q, t2, (float)(2 / (7 * LN2)));
    q = fma1(q, t2, (float)(2 / (5 * LN2)));
    const double u = __builtin_fma(__builtin_fma((double)q, s2, 2 / (3 * LN2)), s2, 2 / LN2);
    const double l = __builtin_fma(sv, u, (double)e);
    lg = (float)l;
    const double t = (double)y * l;
    if (t < -160.0) return 0.0f;  // below half the smallest float32
    const double k = __builtin_rint(t), f = t - k;
    // 2^f = 1 + f (ln 2 + f (ln2^2 / 2! + ...))
    const float g = (float)f;
    float p = 1.32154867901e-6f;
    p = fma1(p, g, 1.52527338041e-5f);
    p = fma1(p, g, 1.54035303934e-4f);
    p = fma1(p, g, 1.33335581464e-3f);
    p = fma1(p, g, 9.61812910763e-3f);
    p = fma1(p, g, 5.55041086648e-2f);
    p = fma1(p, g, 0.2402265069591f);
    return (float)__builtin_ldexp(__builtin_fma(f, LN2 + (double)(p * g), 1.0), (int)k);
}

// Sum over the wave, in lane 63: DPP adds over each row of 16 lanes, then
// row 0 and 2 into 1 and 3, then rows 0-1 into 2-3 (no LDS traffic, which a
// shuffle's ds_bpermute costs per step).
__device__ __forceinline__ float wave_sum63(float v) {
    auto step = [](float a, auto ctrl, auto rows) {
        return a + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(a), decltype(ctrl)::value,
                                                              decltype(rows)::value, 0xf, false));
    };
    using std::integral_constant;
    v = step(v, integral_constant<int, 0x111>{}, integral_constant<int, 0xf>{});
    v = step(v, integral_constant<int, 0x112>{}, integral_constant<int, 0xf>{});
    v = step(v, integral_constant<int, 0x114>{}, integral_constant<int, 0xf>{});
    v = step(v, integral_constant<int, 0x118>{}, integral_constant<int, 0xf>{});
    v = step(v, integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{});
    v = step(v, integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{});
    return v;
}
__device__ __forceinline__ double wsum(double v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// Memory no one writes while the kernel runs, read at one address by every
// lane: through the constant address space, so the loads are scalar ones.
template <class T>
using Const = const __attribute__((address_space(4))) T;
template <class T>
__device__ __forceinline__ Const<T>* konst(const T* p) {
    return (Const<T>*)p;
}

// What one pixel needs for the shading and its adjoint.
struct DPix {
    int mat, vid[3];
    float w[3], bc[3];  // perspective weights (albedo) and barycentrics (normal)
    F3 a, n, x, V;
    float rn;  // 1 / |sum bc_k N_k|
    float sw;  // shadow scale 2^-count
    bool flat;
};

// A pixel's triangle record (the setup's: transformed vertices and flat
// material; w < 0: nothing to differentiate), or the first plane of the stored
// G-buffer, whose last word is the material too.
template <class B>
__device__ __forceinline__ int4 pixel_rec(const B& b, size_t at) {
    if (b.gbuf) return *reinterpret_cast<const int4*>(b.gbuf + at);
    const uint64_t key = b.vis[at];
    return key == VIS_EMPTY ? make_int4(0, 0, 0, -1) : b.tri_rec[(uint32_t)key >> 3];
}

// G-buffer planes: (x, material), (n, shadow scale), (V, 0), (albedo, 0).
__device__ __forceinline__ DPix stored_pixel(const float4* gbuf, size_t P, size_t at, const int4& rec) {
    DPix p;
    const float4 g1 = gbuf[P + at], g2 = gbuf[2 * P + at], g3 = gbuf[3 * P + at];
    p.mat = rec.w;
    p.x = f3(__int_as_float(rec.x), __int_as_float(rec.y), __int_as_float(rec.z));
    p.n = xyz(g1), p.sw = g1.w, p.V = xyz(g2), p.a = xyz(g3);
    p.rn = 1.0f, p.flat = true;  // no normal gradient from a stored pixel
    for (int k = 0; k < 3; k++) p.vid[k] = 0, p.w[k] = p.bc[k] = 0.0f;
    return p;
}

// The per-vertex inputs of a pixel's triangle, all loaded at once.
struct DTri {
    float4 P[3];
    F3 A[3], N[3], M[3];
    bool flat;
    int count;
};
template <class B>
__device__ __forceinline__ DTri load_tri(const DevScene& s, const B& b, size_t at, const int4& rec) {
    DTri t;
    const int vid[3] = {rec.x, rec.y, rec.z};
    for (int k = 0; k < 3; k++) {
        t.P[k] = b.tv_scr[vid[k]];
        t.M[k] = xyz(b.tv_wp[vid[k]]);
        t.N[k] = b.normal ? ld3(b.normal + 3 * (size_t)vid[k]) : xyz(b.tv_nor[vid[k]]);
        t.A[k] = ld3(b.albedo + 3 * (size_t)vid[k]);
    }
    t.flat = s.mats[rec.w].flat_shading != 0;
    t.count = b.shadow_count ? (int)b.shadow_count[at] : 0;
    return t;
}
template <bool SAFE>
__device__ __forceinline__ DPix diff_pixel(Ops<SAFE>& op, const DTri& t, const int4& rec, bool perspect, F3 cam, int x,
                                           int y) {
    DPix p;
    p.mat = rec.w;
    p.vid[0] = rec.x, p.vid[1] = rec.y, p.vid[2] = rec.z;
    // The geometry is the forward pass's, to the bit: barycentrics at the pixel
    // centre from its rounded areas (a needle's are far below the products
    // they are the differences of, so better ones would be other ones: 1e-4 of
    // its colour), perspective weights, world position.
    const float4(&P)[3] = t.P;
    const TriSetup ts = tri_setup(P[0].x, P[0].y, P[1].x, P[1].y, P[2].x, P[2].y);
    float area[3];
    tri_areas(ts, (float)x + 0.5f, (float)y + 0.5f, area);
    const float rs = op.rcp(ts.sabc);
    for (int k = 0; k < 3; k++) p.bc[k] = op.quot(area[k], ts.sabc, rs);
    const float wc[3] = {P[0].w * p.bc[0], P[1].w * p.bc[1], P[2].w * p.bc[2]};
    const float norm = perspect ? op.rcp(wc[0] + wc[1] + wc[2]) : 1.0f;
    F3 nraw = f3(0, 0, 0);
    p.a = f3(0, 0, 0), p.x = f3(0, 0, 0);
    for (int k = 0; k < 3; k++) {
        p.w[k] = wc[k] * norm;
        p.a = fma3(p.w[k], t.A[k], p.a);
        nraw = fma3(p.bc[k], t.N[k], nraw);
        p.x = p.x + p.bc[k] * t.M[k];
    }
    p.flat = t.flat;
    if (p.flat) {  // the face normal: fixed
        const F3 e1 = t.M[1] - t.M[0], e2 = t.M[2] - t.M[0];
        nraw = f3(e1.y * e2.z - e1.z * e2.y, e1.z * e2.x - e1.x * e2.z, e1.x * e2.y - e1.y * e2.x);
    }
    p.rn = op.rsqrt(dot(nraw, nraw));
    p.n = p.rn * nraw;
    const F3 vv = cam - p.x;
    p.V = op.rsqrt(dot(vv, vv)) * vv;
    p.sw = __builtin_ldexpf(1.0f, -t.count);
    return p;
}

}  // namespace

// A workgroup's accumulators in LDS, flushed to the global gradients once,
// after its last pixels.
//
// Materials: every lane adds its 7 values (dKd, dKs, dshininess) to its own
// copy, lane & (copies - 1), of its material's bins with LDS atomics: with 32
// copies (up to 18 materials) no two lanes of a half-wave share a bank or an
// address, and the wave does no reduction at all (one reduction of 7 values
// per distinct material, by shuffles, was a quarter of the adjoint).  More
// materials take fewer copies; above DIFF_MAT_SLOTS / 7 of them the bins of the
// materials the workgroup meets are found by open addressing (DIFF_MAT_KEYS of
// them, their keys in the rest of the array), and only one that finds no bin in
// DIFF_MAT_PROBES goes to memory; kernels of their own (FOUND), as the search's
// registers cost the others 1 to 4 %.  (All lanes adding to memory took 6.5 ms a
// step of 8 views with 700 materials; 0.09 now, 0.06 with 8.)
constexpr int DIFF_MAT_SLOTS = 4096, DIFF_MAT_KEYS = 512, DIFF_MAT_PROBES = 8;
static_assert(8 * DIFF_MAT_KEYS <= DIFF_MAT_SLOTS, "seven values and a key a bin");
struct DiffAcc {
    float mat[DIFF_MAT_SLOTS];
    float light[4 * DIFF_MAX_LIGHTS];
    double loss;
};
__host__ __device__ __forceinline__ int mat_copies(int n_mats) {  // 0: found bins
    int c = 32;
    while (c > 0 && 7 * n_mats * c > DIFF_MAT_SLOTS) c >>= 1;
    return c;
}

// The bin of material `mat` among the found ones (a bin's value j is at
// mat[j * DIFF_MAT_KEYS + bin]), or -1.
__device__ __forceinline__ int32_t* mat_keys(DiffAcc& a) {  // material + 1, 0: free
    return reinterpret_cast<int32_t*>(a.mat + 7 * DIFF_MAT_KEYS);
}
__device__ __forceinline__ int mat_bin(DiffAcc& a, int mat) {
    int32_t* keys = mat_keys(a);
    int h = mat & (DIFF_MAT_KEYS - 1);
    for (int probe = 0; probe < DIFF_MAT_PROBES; probe++, h = (h + 1) & (DIFF_MAT_KEYS - 1)) {
        int32_t k = keys[h];
        if (k == 0) {
            k = atomicCAS(&keys[h], 0, mat + 1);
            if (k == 0) k = mat + 1;
        }
        if (k == mat + 1) return h;
    }
    return -1;
}
template <bool FOUND>
__device__ __forceinline__ void acc_clear(DiffAcc& a, int n_mats, int copies) {
    const int used = FOUND ? 8 * DIFF_MAT_KEYS : 7 * n_mats * copies;
    for (int i = threadIdx.x; i < used; i += blockDim.x) a.mat[i] = 0.0f;  // (a free key's bits too)
    if (threadIdx.x < 4 * DIFF_MAX_LIGHTS) a.light[threadIdx.x] = 0.0f;
    if (threadIdx.x == 0) a.loss = 0.0;
    __syncthreads();
}

// After the workgroup's last pixels: every wanted, nonzero sum to its gradient.
// Each workgroup adds to one of the DIFF_REPS replicas of these gradients and
// of the loss (its XCD's, as the dispatcher deals them): 1024 workgroups adding
// to the same five cache lines took 25 us of a launch, an eighth of them 4.
template <bool FOUND, class B>
__device__ __forceinline__ void acc_flush(const DevScene& s, const B& b, DiffAcc& a, int copies) {
    __syncthreads();
    const size_t rep = b.reps > 1 ? blockIdx.x % DIFF_REPS : 0, ro = rep * b.rep_stride;
    const uint32_t want = b.want;
    for (int i = threadIdx.x; i < 4 * s.n_lights; i += blockDim.x) {
        const float v = a.light[i];
        const bool pos = (i & 3) < 3;
        if (v != 0.0f && (want & (pos ? DIFF_LIGHT_POS : DIFF_LIGHT_INT)))
            atomicAdd((pos ? &b.g_lpos[3 * (i >> 2) + (i & 3)] : &b.g_lint[i >> 2]) + ro, v);
    }
    auto material = [&](int m, int j, float v) {
        if (v != 0.0f && (want & (j < 3 ? DIFF_KD : j < 6 ? DIFF_KS : DIFF_SHININESS)))
            atomicAdd((j < 3 ? &b.g_kd[3 * (size_t)m + j] : (j < 6 ? &b.g_ks[3 * (size_t)m + j - 3] : &b.g_shin[m])) + ro, v);
    };
    if constexpr (FOUND) {
        for (int i = threadIdx.x; i < 7 * DIFF_MAT_KEYS; i += blockDim.x) {
            const int k = mat_keys(a)[i & (DIFF_MAT_KEYS - 1)];
            if (k != 0) material(k - 1, i / DIFF_MAT_KEYS, a.mat[i]);
        }
    } else {
        for (int i = threadIdx.x; i < 7 * s.n_materials; i += blockDim.x) {
            float v = 0.0f;
            for (int k = 0; k < copies; k++) v += a.mat[i * copies + ((k + i) & (copies - 1))];  // (banks rotated)
            const int m = i / 7;
            material(m, i - 7 * m, v);
        }
    }
    if (threadIdx.x == 0 && a.loss != 0.0) atomicAdd(b.loss + rep, a.loss);
}

// The vertices' albedo and normal gradients, summed in LDS by vertex (open
// addressing) before they go to memory: of 256 pixels a vertex's triangles
// cover tens, so they send one atomic per vertex and value instead of one per
// pixel, corner and value (a wave reduction per distinct triangle and value, by
// shuffles, was most of the adjoint where vertices are wanted).  A vertex that
// finds no slot in DIFF_VTX_PROBES goes to memory directly.  A triangle that holds
// DIFF_VTX_LANES lanes of a wave or more is summed over the wave first, and the
// table goes to memory only once it holds DIFF_VTX_FULL vertices (or at the
// end): lanes that add to one address take their turns, in LDS as in memory
// (one plane of two triangles across 2048x2048: 1.19 ms by shuffles, 2.75
// without either, 0.40 now; across 512x512 0.097, 0.203, 0.097; of two thousand
// there 0.070, 0.075, 0.053; the 100 thousand of 104 spheres 0.132, 0.059, 0.058).
// From 16 or 32 lanes on instead, a plane of 32 thousand takes 0.077 against
// 0.061; from 4 the same.
constexpr int DIFF_VTX_SLOTS = 512, DIFF_VTX_PROBES = 8, DIFF_VTX_LANES = 8, DIFF_VTX_FULL = 128;
struct VtxAcc {
    int32_t key[DIFF_VTX_SLOTS];  // vertex + 1, 0: free
    float g[6][DIFF_VTX_SLOTS];   // albedo, normal
    int32_t used;                 // slots taken
};
// One pixel's share: corner k's albedo gets w[k] gA, its normal bc[k] gN.
struct VtxGrad {
    int vid[3];  // vid[0] < 0: no pixel
    float w[3], bc[3];
    F3 gA, gN;
};
struct NoVtxAcc {};
struct NoVtxGrad {};
__device__ __forceinline__ void vtx_clear(NoVtxAcc&) {}
__device__ __forceinline__ void vtx_clear(VtxAcc& t) {
    for (int i = threadIdx.x; i < DIFF_VTX_SLOTS; i += blockDim.x) {
        t.key[i] = 0;
        for (int j = 0; j < 6; j++) t.g[j][i] = 0.0f;
    }
    if (threadIdx.x == 0) t.used = 0;
    __syncthreads();
}
template <class B>
__device__ __forceinline__ void vtx_add(VtxAcc& t, const B& b, int vid, const float (&g)[6]) {
    const uint32_t want = b.want;
    uint32_t h = ((uint32_t)vid * 2654435761u) >> 23;  // 9 bits
    for (int probe = 0; probe < DIFF_VTX_PROBES; probe++, h = (h + 1) & (DIFF_VTX_SLOTS - 1)) {
        int32_t k = t.key[h];
        if (k == 0) {
            k = atomicCAS(&t.key[h], 0, vid + 1);
            if (k == 0) k = vid + 1, atomicAdd(&t.used, 1);
        }
        if (k == vid + 1) {
            for (int j = 0; j < 6; j++) atomicAdd(&t.g[j][h], g[j]);
            return;
        }
    }
    for (int j = 0; j < 3; j++) {
        if (want & DIFF_ALBEDO) atomicAdd(&b.g_albedo[3 * (size_t)vid + j], g[j]);
        if (want & DIFF_NORMAL) atomicAdd(&b.g_normal[3 * (size_t)vid + j], g[3 + j]);
    }
}
// A wave's pixels into the table (every lane of the wave takes part).
template <class B>
__device__ __forceinline__ void vtx_wave(VtxAcc& t, const B& b, const VtxGrad& v) {
    const int lane = threadIdx.x & 63;
    bool left = v.vid[0] >= 0;
    uint64_t pending = __ballot(left);
    for (int round = 0; round < 64 / DIFF_VTX_LANES && __popcll(pending) >= DIFF_VTX_LANES; round++) {
        const int l = __builtin_ctzll(pending);
        int id[3];
        for (int k = 0; k < 3; k++) id[k] = __builtin_amdgcn_readlane(v.vid[k], l);
        const bool same = left && v.vid[0] == id[0] && v.vid[1] == id[1] && v.vid[2] == id[2];
        const uint64_t m = __ballot(same);
        pending &= ~m;
        if (__popcll(m) < DIFF_VTX_LANES) continue;
        for (int k = 0; k < 3; k++) {
            const float w = v.w[k], bc = v.bc[k];
            const float g[6] = {wave_sum63(same ? w * v.gA.x : 0.0f),  wave_sum63(same ? w * v.gA.y : 0.0f),
                                wave_sum63(same ? w * v.gA.z : 0.0f),  wave_sum63(same ? bc * v.gN.x : 0.0f),
                                wave_sum63(same ? bc * v.gN.y : 0.0f), wave_sum63(same ? bc * v.gN.z : 0.0f)};
            if (lane == 63) vtx_add(t, b, id[k], g);
        }
        left = left && !same;
    }
    if (left) {
        for (int k = 0; k < 3; k++) {
            const float g[6] = {v.w[k] * v.gA.x,  v.w[k] * v.gA.y,  v.w[k] * v.gA.z,
                                v.bc[k] * v.gN.x, v.bc[k] * v.gN.y, v.bc[k] * v.gN.z};
            vtx_add(t, b, v.vid[k], g);
        }
    }
}
// The sums to memory, the table empty for the next pixels.  Four lanes a slot, a
// vertex's three values in one instruction: their line takes one turn, not
// three, where every workgroup adds to the same few vertices.
template <class B>
__device__ __forceinline__ void vtx_flush(VtxAcc& t, const B& b) {
    __syncthreads();
    const uint32_t want = b.want;
    for (int i = threadIdx.x; i < 4 * DIFF_VTX_SLOTS; i += blockDim.x) {
        const int h = i >> 2, j = i & 3;
        const int32_t k = t.key[h];
        if (k == 0 || j == 3) continue;
        const size_t o = 3 * (size_t)(k - 1) + j;
        const float a = t.g[j][h], n = t.g[3 + j][h];
        t.g[j][h] = t.g[3 + j][h] = 0.0f;
        if (a != 0.0f && (want & DIFF_ALBEDO)) atomicAdd(&b.g_albedo[o], a);
        if (n != 0.0f && (want & DIFF_NORMAL)) atomicAdd(&b.g_normal[o], n);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < DIFF_VTX_SLOTS; i += blockDim.x) t.key[i] = 0;
    if (threadIdx.x == 0) t.used = 0;
    __syncthreads();
}

// The lights, uniform: loaded once, before the first tile.
struct LightC {
    F3 p;  // position, or (directional) the direction towards the light
    float i;
    F3 color;
    int32_t kind;
};
template <int NLMAX, class B>
__device__ __forceinline__ void load_lights(const DevScene& s, const B& b, LightC (&l)[NLMAX]) {
    Const<DevLight>* lights = konst(s.lights);
    Const<float>*lpos = konst(b.light_pos), *lint = konst(b.light_int);
#pragma unroll
    for (int i = 0; i < NLMAX; i++) {
        if (i < s.n_lights) {
            l[i].kind = lights[i].kind;
            l[i].p = l[i].kind == 0 ? f3(lpos[3 * i], lpos[3 * i + 1], lpos[3 * i + 2])
                                    : f3(-lights[i].dir[0], -lights[i].dir[1], -lights[i].dir[2]);
            l[i].i = lint[i];
            l[i].color = f3(lights[i].color[0], lights[i].color[1], lights[i].color[2]);
        }
    }
}
// What the adjoint keeps of a light's terms from the forward sums: the roots
// and the power.  The vectors and products are a dozen instructions away, and
// with them kept as well (5 more registers a light) a SIMD held 3 waves, not
// 5, of which most wait for memory.
struct DLight {
    float r, rh, Ls, lg;
};
struct DVecs {
    F3 L, h;
    float nL, nH;
};
__device__ __forceinline__ DVecs light_vecs(const LightC& l, const DPix& p, float r, float rh) {
    DVecs v;
    v.L = l.p;
    if (l.kind == 0) v.L = r * (l.p - p.x);
    v.h = v.L + p.V;
    v.nL = dot(p.n, v.L);
    v.nH = rh * dot(p.n, v.h);
    return v;
}
__device__ __forceinline__ float clamp01(float x) { return fminf(fmaxf(x, 0.0f), 1.0f); }
template <int NLMAX, bool SAFE>
__device__ __forceinline__ void light_sums(Ops<SAFE>& op, const LightC (&lc)[NLMAX], int NL, const DPix& p, float shin,
                                           DLight (&t)[NLMAX], float& sLd, F3& sLs) {
    sLd = 0.0f, sLs = f3(0, 0, 0);
#pragma unroll
    for (int li = 0; li < NLMAX; li++) {
        if (li < NL) {
            DLight& q = t[li];
            q.r = 1.0f;
            if (lc[li].kind == 0) {
                const F3 d = lc[li].p - p.x;
                q.r = op.rsqrt(dot(d, d));
            }
            const DVecs v = light_vecs(lc[li], p, q.r, 1.0f);
            const float I = lc[li].i * q.r;
            q.rh = op.rsqrt(dot(v.h, v.h));
            q.Ls = pow_log2(clamp01(q.rh * v.nH), shin, q.lg);
            sLd = fma1(clamp01(v.nL), I, sLd);
            sLs = fma3(q.Ls * I, lc[li].color, sLs);
        }
    }
}
// A thread's own sums over its pixels: the lights' gradients (4 each) and the
// loss, reduced over the wave once, after the last (a reduction of 4 values
// per light per 64 pixels, by shuffles, was over a third of the adjoint).
template <int NLMAX>
struct ThreadAcc {
    float light[4 * NLMAX];
    double loss;
};

// The forward of one pixel: its state, the lights' terms and the linear colour.
template <int NLMAX>
struct DFwd {
    DPix p;
    DLight t[NLMAX];
    float sLd;
    F3 sLs, kd, ks, lin;
};
// NLMAX: at least s.n_lights.
template <int NLMAX, class V, class B>
__device__ __forceinline__ DFwd<NLMAX> diff_forward(const DevScene& s, const V& v, const B& b,
                                                    const LightC (&lc)[NLMAX], int x, int y, size_t o, const int4& rec) {
    const int NL = s.n_lights, mat = rec.w;
    const F3 cam = f3(v.cam[0], v.cam[1], v.cam[2]);
    const bool perspect = v.perspect != 0;
    DFwd<NLMAX> f;
    Ops<false> op;
    const F3 kd = ld3(b.kd + 3 * (size_t)mat), ks = ld3(b.ks + 3 * (size_t)mat);
    const float shin = b.shininess[mat];
    if (b.gbuf) f.p = stored_pixel(b.gbuf, (size_t)v.W * v.H, o, rec);
    else f.p = diff_pixel(op, load_tri(s, b, o, rec), rec, perspect, cam, x, y);
    light_sums(op, lc, NL, f.p, shin, f.t, f.sLd, f.sLs);
    if (op.bad()) {  // (vectors of no, tiny or overflowing length)
        Ops<true> safe;
        if (!b.gbuf) f.p = diff_pixel(safe, load_tri(s, b, o, rec), rec, perspect, cam, x, y);
        light_sums(safe, lc, NL, f.p, shin, f.t, f.sLd, f.sLs);
    }
    const float amb = b.ambient;
    f.kd = kd, f.ks = ks;
    // (the ambient term by its own product with the albedo: added to the diffuse
    // factor, which is a multiple of a far larger unit, it would always be
    // rounded by the same amount)
    auto channel = [&](float a, float d, float sp, float sl) {
        return f.p.sw * fma1(amb, a, div255(fma1(d * f.sLd, a, sp * sl)));
    };
    f.lin = f3(channel(f.p.a.x, kd.x, ks.x, f.sLs.x), channel(f.p.a.y, kd.y, ks.y, f.sLs.y),
               channel(f.p.a.z, kd.z, ks.z, f.sLs.z));
    return f;
}

// Its adjoint, into the accumulators.  VTX: albedo or normal gradients are
// wanted.
template <int NLMAX, bool VTX, bool FOUND, class B, class T>
__device__ __forceinline__ void diff_adjoint(const DFwd<NLMAX>& f, const DevScene& s, const B& b,
                                             const LightC (&lc)[NLMAX], F3 tg, DiffAcc& acc, int copies,
                                             ThreadAcc<NLMAX>& mine, T& out) {
    const int NL = s.n_lights, mat = f.p.mat;
    const DPix& p = f.p;
    const DLight(&t)[NLMAX] = f.t;
    const float shin = b.shininess[mat];
    const F3 e = f.lin - tg;
    mine.loss += (double)e.x * (double)e.x + (double)e.y * (double)e.y + (double)e.z * (double)e.z;
    const F3 gl = (2.0f * p.sw) * e;  // through the fixed shadow scale
    const F3 ga = f3(gl.x * p.a.x, gl.y * p.a.y, gl.z * p.a.z);
    const F3 gk = f3(div255(gl.x * f.ks.x), div255(gl.y * f.ks.y), div255(gl.z * f.ks.z));
    const float gD = div255(dot(ga, f.kd));  // dloss / d(sum Ld I)
    float gshin = 0.0f;
    F3 gn = f3(0, 0, 0);
#pragma unroll
    for (int li = 0; li < NLMAX; li++) {
        if (li < NL) {
            const DLight& q = t[li];
            const DVecs u = light_vecs(lc[li], p, q.r, q.rh);
            const float I = lc[li].i * q.r;
            const float gS = dot(gk, lc[li].color);
            const float gI = fma1(gD, clamp01(u.nL), gS * q.Ls);
            const float gLd = u.nL > 0.0f && u.nL < 1.0f ? gD * I : 0.0f;
            // d(nH^s)/dnH = s Ls / nH (below 2^-100 it is taken as 0)
            const bool in = u.nH > 0x1p-100f && u.nH < 1.0f;
            const float nH = in ? u.nH : 1.0f, z = in ? gS * I * q.Ls : 0.0f;
            // (outside, the logarithm may be infinite: of 0, at a shininess of 0)
            gshin = fma1(z, in ? q.lg : 0.0f, gshin);
            Ops<false> unused;
            const float gLs = z * shin * unused.rcp(nH);
            if (VTX) gn = fma3(gLd, u.L, fma3(gLs * q.rh, u.h, gn));
            if (lc[li].kind == 0) {
                // through H = h / |h| (u.g of the unit vector's pullback is gLs nH), then L = d / |d|
                // and I = i0 / |d|
                const float sH = gLs * q.rh;
                const F3 gL = fma3(gLd, p.n, sH * (p.n - (u.nH * q.rh) * u.h));
                const F3 gd = q.r * fma3(-fma1(gI, I, dot(u.L, gL)), u.L, gL);
                mine.light[4 * li] += gd.x, mine.light[4 * li + 1] += gd.y, mine.light[4 * li + 2] += gd.z;
                mine.light[4 * li + 3] = fma1(gI, q.r, mine.light[4 * li + 3]);
            } else {
                mine.light[4 * li + 3] += gI;
            }
        }
    }
    gshin *= 0.69314718056f;  // log2 -> log
    if (b.want & (DIFF_KD | DIFF_KS | DIFF_SHININESS)) {
        const float d = div255(f.sLd);
        const float gm_[7] = {ga.x * d, ga.y * d, ga.z * d, gl.x * div255(f.sLs.x), gl.y * div255(f.sLs.y),
                              gl.z * div255(f.sLs.z), gshin};
        if constexpr (!FOUND) {
            float* bin = acc.mat + 7 * mat * copies + (threadIdx.x & (copies - 1));
            for (int j = 0; j < 7; j++) atomicAdd(bin + j * copies, gm_[j]);
        } else if (const int bin = mat_bin(acc, mat); bin >= 0) {
            for (int j = 0; j < 7; j++) atomicAdd(&acc.mat[j * DIFF_MAT_KEYS + bin], gm_[j]);
        } else {
            for (int j = 0; j < 3; j++) {
                atomicAdd(&b.g_kd[3 * (size_t)mat + j], gm_[j]);
                atomicAdd(&b.g_ks[3 * (size_t)mat + j], gm_[3 + j]);
            }
            atomicAdd(&b.g_shin[mat], gm_[6]);
        }
    }
    if constexpr (VTX) {  // (a stored G-buffer keeps no vertices: the host refuses that combination)
        const F3 gA = f3(gl.x * (b.ambient + div255(f.kd.x * f.sLd)), gl.y * (b.ambient + div255(f.kd.y * f.sLd)),
                         gl.z * (b.ambient + div255(f.kd.z * f.sLd)));
        F3 gN = f3(0, 0, 0);
        if (!p.flat) gN = p.rn * fma3(-dot(p.n, gn), p.n, gn);
        out.gA = gA, out.gN = gN;
        for (int k = 0; k < 3; k++) out.vid[k] = p.vid[k], out.w[k] = p.w[k], out.bc[k] = p.bc[k];
    }
}

template <int NLMAX>
__device__ __forceinline__ void thread_acc_clear(ThreadAcc<NLMAX>& mine) {
    for (int j = 0; j < 4 * NLMAX; j++) mine.light[j] = 0.0f;
    mine.loss = 0.0;
}
// Every thread's sums into the workgroup's.
template <int NLMAX>
__device__ __forceinline__ void thread_acc_reduce(const ThreadAcc<NLMAX>& mine, int n_lights, DiffAcc& acc) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < 4 * NLMAX; j++) {
        if (j < 4 * n_lights) {
            const float v = wave_sum63(mine.light[j]);
            if (lane == 63) atomicAdd(&acc.light[j], v);
        }
    }
    const double l = wsum(mine.loss);
    if (lane == 0) atomicAdd(&acc.loss, l);
}

// ---- forward: every pixel of a view, a 16x16 tile a workgroup (four 8x8 waves)
template <int NLMAX, class V, class B>
__device__ __forceinline__ void forward_tile(const DevScene& s, const V& v, const B& b, int tile) {
    const int W = v.W, H = v.H, tiles_x = v.tiles_x;
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
    const int x = (tile % tiles_x) * TILE + (wv & 1) * 8 + (lane & 7);
    const int y = (tile / tiles_x) * TILE + (wv >> 1) * 8 + (lane >> 3);
    if (x >= W || y >= H) return;
    const size_t o = (size_t)y * W + x;
    const int4 rec = pixel_rec(b, o);
    float* out = b.linear + 3 * o;
    if (rec.w < 0) {
        out[0] = out[1] = out[2] = __builtin_nanf("");
        return;
    }
    LightC lc[NLMAX];
    load_lights(s, b, lc);
    const F3 lin = diff_forward(s, v, b, lc, x, y, o, rec).lin;
    out[0] = lin.x, out[1] = lin.y, out[2] = lin.z;
}
template <int NLMAX>
__global__ __launch_bounds__(256) void k_diff_forward(DevScene s, ViewConsts v, DiffBuffers b) {
    forward_tile<NLMAX>(s, v, b, blockIdx.x);
}

// Many views of one scene in one launch: view i owns the workgroups
// [block0, block0 + nblocks), block0 ascending and a multiple of 8 (so a
// view's tiles keep the XCD spread of its own launch).
__device__ __forceinline__ int view_at(Const<DiffView>* tab, int n, int32_t DiffView::*start, int b) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (tab[mid].*start <= b) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}
template <int NLMAX>
__global__ __launch_bounds__(256) void k_diff_forward_views(DevScene s, const DiffView* __restrict__ views, int32_t n) {
    Const<DiffView>* tab = konst(views);
    const int i = view_at(tab, n, &DiffView::block0, blockIdx.x);
    forward_tile<NLMAX>(s, tab[i].v, tab[i].b, blockIdx.x - tab[i].block0);
}

// ---- adjoint: the pixels there is something to differentiate at
//
// The visibility is fixed, so the adjoint runs over a list of the views'
// shaded pixels: its waves are full where a tile's are not (half of a view's
// 8x8 blocks are empty, and the others 80 % covered), and the waves share the
// list evenly where tiles shared unevenly (strided over 1024 workgroups, the
// covered ones left the average workgroup done at 3/4 of the launch).
//
// k_diff_list makes it, a strip of DIFF_STRIP tiles a workgroup: the strip's
// shaded pixels (x | y << 16), by 8x8 block, go to the strip's own part of
// the view's list (the count of its pixels before it in strip order: P words in
// all), and chunks of up to 64 of them, {start, count | view << 7}, to the
// table all views share, placed by one atomic a strip.  It reads 8 bytes of
// key and 16 of record a pixel, once per call (a fit's steps share it).
constexpr int DIFF_STRIP = 4;
__global__ __launch_bounds__(256) void k_diff_list(const DiffView* __restrict__ views, int32_t n, DiffView one,
                                                   uint2* __restrict__ chunks, int32_t* __restrict__ count) {
    __shared__ int32_t s_cnt[DIFF_STRIP * 4 + 1], s_base;
    const int vi = views ? view_at(konst(views), n, &DiffView::strip0, blockIdx.x) : 0;
    const DiffView& w = views ? views[vi] : one;
    const int strip = blockIdx.x - (views ? w.strip0 : 0);
    const int W = w.v.W, H = w.v.H, per_row = (w.v.tiles_x + DIFF_STRIP - 1) / DIFF_STRIP;
    const int ty = strip / per_row, tx0 = (strip % per_row) * DIFF_STRIP;
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
    const int y = ty * TILE + (wv >> 1) * 8 + (lane >> 3);
    const int rows = min(TILE, H - ty * TILE);
    uint32_t* list = w.b.list + (size_t)ty * TILE * W + (size_t)tx0 * TILE * rows;
    uint64_t bal[DIFF_STRIP];
    int x[DIFF_STRIP], mat[DIFF_STRIP];
#pragma unroll
    for (int k = 0; k < DIFF_STRIP; k++) {
        x[k] = (tx0 + k) * TILE + (wv & 1) * 8 + (lane & 7);
        mat[k] = x[k] < W && y < H ? pixel_rec(w.b, (size_t)y * W + x[k]).w : -1;
    }
#pragma unroll
    for (int k = 0; k < DIFF_STRIP; k++) {
        bal[k] = __ballot(mat[k] >= 0);
        if (lane == 0) s_cnt[4 * k + wv] = __popcll(bal[k]);
    }
    __syncthreads();
    if (wv == 0) {  // exclusive scan: the blocks' order
        constexpr int NB = DIFF_STRIP * 4;
        const int c = lane < NB ? s_cnt[lane] : 0;
        int incl = c;
        for (int off = 1; off < NB; off <<= 1) {
            const int u = __shfl_up(incl, off);
            if (lane >= off) incl += u;
        }
        if (lane < NB) s_cnt[lane] = incl - c;
        if (lane == NB - 1) {
            s_cnt[NB] = incl;
            s_base = incl ? atomicAdd(count, (incl + 63) >> 6) : 0;
        }
    }
    __syncthreads();
    const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
    for (int k = 0; k < DIFF_STRIP; k++)
        if (mat[k] >= 0) list[s_cnt[4 * k + wv] + __popcll(bal[k] & below)] = (uint32_t)x[k] | ((uint32_t)y << 16);
    const int total = s_cnt[DIFF_STRIP * 4];
    const uint32_t start = (uint32_t)(list - w.b.list);
    if (64 * tid < total)
        chunks[s_base + tid] = make_uint2(start + 64 * tid, (uint32_t)min(64, total - 64 * tid) | ((uint32_t)vi << 7));
}

template <bool VTX>
struct VtxOf {
    using acc = NoVtxAcc;
    using grad = NoVtxGrad;
};
template <>
struct VtxOf<true> {
    using acc = VtxAcc;
    using grad = VtxGrad;
};
// A workgroup takes four consecutive chunks (a wave each: neighbouring
// pixels, which share vertices) at a time.  Each XCD has an eighth of the list
// to itself and its workgroups (every eighth of the grid) walk it side by
// side, so that the lines its chunks gather, some 20 KB of vertices each, come
// from its own L2: strided over the whole list instead, every XCD fetched every
// part of the scene.  Each
// chunk's pixels are loaded two rounds ahead, their keys one, and their
// triangles' records half a round, so a round waits for its vertices only.
//
// What bounds it: VALU issue, 64 % of it busy at the 4 waves a SIMD that 128
// registers leave (with 5, spilling, 9.9 ms; with 3, 9.6).  A wave's pixels
// take about 1000 instructions with 4 lights.  32 views of 256^2 to 1024^2 (8.4
// M shaded pixels): 1184 -> 369 us a step; 6 views of 200^2 to 500^2 from the
// stored G-buffer 94 -> 37 us; one of 512^2 with the vertices' gradients 130 ->
// 55 us, its list included.
template <int NLMAX, bool VTX, bool FOUND, class B, class F>
__device__ __forceinline__ void adjoint_chunks(const DevScene& s, const B& b0, const uint2* __restrict__ chunks,
                                               int n_chunks, F&& view) {
    __shared__ DiffAcc acc;
    __shared__ typename VtxOf<VTX>::acc vtx;
    // this XCD's groups of four chunks, [gb, ge), and the workgroup's stride
    const int groups = (n_chunks + 3) >> 2, xcd = blockIdx.x & 7, per = (int)(gridDim.x >> 3);
    const int gb = (int)((int64_t)groups * xcd >> 3), ge = (int)((int64_t)groups * (xcd + 1) >> 3);
    const int g0 = gb + (int)(blockIdx.x >> 3);
    if (g0 >= ge) return;
    const int copies = mat_copies(s.n_materials), lane = threadIdx.x & 63;
    ThreadAcc<NLMAX> mine;
    thread_acc_clear(mine);
    acc_clear<FOUND>(acc, s.n_materials, copies);
    vtx_clear(vtx);
    LightC lc[NLMAX];
    load_lights(s, b0, lc);
    Const<uint2>* tab = konst(chunks);
    const int end = min(n_chunks, 4 * ge), stride = 4 * per;
    // chunk c's pixel of this lane (~0: none) and its view
    auto pixel = [&](int c, uint32_t& px, int& vi) {
        px = ~0u, vi = 0;
        if (c >= end) return;
        const uint32_t start = tab[c].x, n = tab[c].y;
        vi = (int)(n >> 7);
        if (lane < (int)(n & 127u)) px = view(vi).b.list[start + lane];
    };
    auto at = [](uint32_t px, int W) { return (size_t)(px >> 16) * W + (px & 0xffffu); };
    auto key = [&](uint32_t px, int vi) -> uint32_t {  // (a listed pixel's key is never empty)
        const auto& w = view(vi);
        return px == ~0u || w.b.gbuf ? 0u : *reinterpret_cast<const uint32_t*>(w.b.vis + at(px, w.v.W));
    };
    auto record = [&](uint32_t px, int vi, uint32_t k) {
        const auto& w = view(vi);
        int4 r = make_int4(0, 0, 0, -1);
        if (px != ~0u) r = w.b.gbuf ? *reinterpret_cast<const int4*>(w.b.gbuf + at(px, w.v.W)) : w.b.tri_rec[k >> 3];
        return r;
    };
    const int c0 = 4 * g0 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint32_t px0, px1, px2;
    int v0, v1, v2;
    pixel(c0, px0, v0);
    pixel(c0 + stride, px1, v1);
    int4 rec = record(px0, v0, key(px0, v0));
    for (int g = g0, c = c0; g < ge; g += per, c += stride) {
        const uint32_t k1 = key(px1, v1);
        pixel(c + 2 * stride, px2, v2);
        const auto& w = view(v0);
        int4 rec1 = make_int4(0, 0, 0, -1);
        typename VtxOf<VTX>::grad vg{};
        if constexpr (VTX) vg.vid[0] = -1;
        if (px0 != ~0u) {
            const int x = (int)(px0 & 0xffffu), y = (int)(px0 >> 16);
            const size_t o = at(px0, w.v.W);
            const F3 tg = ld3(w.b.target + 3 * o);
            const DFwd<NLMAX> f = diff_forward(s, w.v, w.b, lc, x, y, o, rec);
            diff_adjoint<NLMAX, VTX, FOUND>(f, s, w.b, lc, tg, acc, copies, mine, vg);
        }
        rec1 = record(px1, v1, k1);
        if constexpr (VTX) {
            vtx_wave(vtx, b0, vg);
            // (one answer for the workgroup: what a wave reads here another may be adding to)
            if (__syncthreads_or(vtx.used >= DIFF_VTX_FULL)) vtx_flush(vtx, b0);
        }
        px0 = px1, v0 = v1, px1 = px2, v1 = v2, rec = rec1;
    }
    if constexpr (VTX) vtx_flush(vtx, b0);
    thread_acc_reduce(mine, s.n_lights, acc);
    acc_flush<FOUND>(s, b0, acc, copies);
}

// waves a SIMD holds: the registers bound them
constexpr int adjoint_waves(int nlmax) { return nlmax > 4 ? 3 : 4; }
template <int NLMAX, bool VTX, bool FOUND>
__global__ __launch_bounds__(256, adjoint_waves(NLMAX)) void k_adjoint(DevScene s, DiffView w,
                                                                    const uint2* __restrict__ chunks,
                                                                    const int32_t* __restrict__ count) {
    adjoint_chunks<NLMAX, VTX, FOUND>(s, w.b, chunks, *count, [&](int) -> const DiffView& { return w; });
}
// Many views of one scene: their parameters, gradients and loss are the same.
// `step` (may be null): a fit's step counter, advanced by one.
template <int NLMAX, bool VTX, bool FOUND>
__global__ __launch_bounds__(256, adjoint_waves(NLMAX)) void k_adjoint_views(DevScene s,
                                                                          const DiffView* __restrict__ views,
                                                                          const uint2* __restrict__ chunks,
                                                                          const int32_t* __restrict__ count,
                                                                          int32_t* step) {
    if (step && blockIdx.x == 0 && threadIdx.x == 0) *step += 1;  // (k_adam reads it)
    Const<DiffView>* tab = konst(views);
    adjoint_chunks<NLMAX, VTX, FOUND>(s, tab[0].b, chunks, *count, [&](int i) -> Const<DiffView>& { return tab[i]; });
}

// Zeroes an adjoint's gradients, its loss and its count of chunks.
__global__ __launch_bounds__(256) void k_diff_clear(float* __restrict__ grad, size_t n, double* __restrict__ loss,
                                                    int32_t* count) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) grad[i] = 0.0f;
    if (blockIdx.x == 0 && threadIdx.x < DIFF_REPS) loss[threadIdx.x] = 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) *count = 0;
}

// A fit's start: the parameters kept as the base, the Adam state and what the
// steps accumulate at zero (one kernel in place of a copy and five fills).
__global__ __launch_bounds__(256) void k_fit_start(const float* __restrict__ par, float* __restrict__ base,
                                                   float* __restrict__ theta, float* __restrict__ m,
                                                   float* __restrict__ v, size_t n, float* __restrict__ grad,
                                                   size_t n_grad, double* __restrict__ loss, int32_t* count,
                                                   int32_t* step) {
    const size_t i0 = blockIdx.x * (size_t)blockDim.x + threadIdx.x, stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = i0; i < n; i += stride) base[i] = par[i], theta[i] = m[i] = v[i] = 0.0f;
    for (size_t i = i0; i < n_grad; i += stride) grad[i] = 0.0f;
    if (i0 < DIFF_REPS) loss[i0] = 0.0;
    if (i0 == 0) *count = 0, *step = 0;
}

__global__ __launch_bounds__(256) void k_diff_gbuffer(DevScene s, ViewConsts v, DiffBuffers b, float4* __restrict__ g) {
    const size_t P = (size_t)v.W * v.H;
    const size_t o = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (o >= P) return;
    const int x = (int)(o % (size_t)v.W), y = (int)(o / (size_t)v.W);
    const int4 rec = pixel_rec(b, o);
    if (rec.w < 0) {
        g[o] = make_float4(0.0f, 0.0f, 0.0f, __int_as_float(-1));
        return;
    }
    const DTri tri = load_tri(s, b, o, rec);
    const F3 cam = f3(v.cam[0], v.cam[1], v.cam[2]);
    Ops<false> op;
    DPix p = diff_pixel(op, tri, rec, v.perspect != 0, cam, x, y);
    if (op.bad()) {
        Ops<true> safe;
        p = diff_pixel(safe, tri, rec, v.perspect != 0, cam, x, y);
    }
    g[o] = make_float4(p.x.x, p.x.y, p.x.z, __int_as_float(p.mat));
    g[P + o] = make_float4(p.n.x, p.n.y, p.n.z, p.sw);
    g[2 * P + o] = make_float4(p.V.x, p.V.y, p.V.z, 0.0f);
    g[3 * P + o] = make_float4(p.a.x, p.a.y, p.a.z, 0.0f);
}

// Adam on the listed parameters, one a thread.  The step counter was advanced
// by this step's adjoint (k_adjoint_views); each listed gradient is zeroed here
// once read, and the loss by workgroup 0 once kept (the loss is that of the
// parameters before this step), so a step is these two launches with no
// clearing pass.  Memory: 40 bytes a parameter.  One workgroup for every
// parameter took 238 us with 87 k of them (the vertex colours of 60 spheres);
// a grid of them 5 us.
__global__ __launch_bounds__(256) void k_adam(float* __restrict__ par, float* __restrict__ grad,
                                              const float* __restrict__ base, float* __restrict__ theta,
                                              float* __restrict__ m, float* __restrict__ v,
                                              const int32_t* __restrict__ idx, const float* __restrict__ lower,
                                              AdamConsts a, const int32_t* __restrict__ step, double* loss,
                                              double* hist) {
    const int t = *step;
    const float c1 = (float)(1.0 - pow64((double)a.beta1, (double)t));
    const float c2 = (float)(1.0 - pow64((double)a.beta2, (double)t));
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < a.n) {
        const int i = idx[k];
        const float b0 = base[i];
        float gi = grad[i];
        grad[i] = 0.0f;
        if (i >= a.rep_from) {
            for (int r = 1; r < a.reps; r++) {
                gi += grad[i + r * (size_t)a.rep_stride];
                grad[i + r * (size_t)a.rep_stride] = 0.0f;
            }
        }
        const float g = gi * b0;  // d loss / d theta for p = base * (1 + theta)
        const float mk = a.beta1 * m[k] + (1.0f - a.beta1) * g;
        const float vk = a.beta2 * v[k] + (1.0f - a.beta2) * (g * g);
        m[k] = mk, v[k] = vk;
        float th = theta[k] - a.lr * (mk / c1) / (__builtin_sqrtf(vk / c2) + a.eps);
        float pv = b0 * (1.0f + th);
        if (pv < lower[k]) {
            pv = lower[k];
            if (b0 != 0.0f) th = pv / b0 - 1.0f;
        }
        theta[k] = th, par[i] = pv;
    }
    if (k == 0) {
        double l = 0.0;
        for (int r = 0; r < DIFF_REPS; r++) l += loss[r], loss[r] = 0.0;
        if (t <= a.hist_cap) hist[t - 1] = l;
    }
}

static int n_strips(const ViewConsts& v) { return ((v.tiles_x + DIFF_STRIP - 1) / DIFF_STRIP) * v.tiles_y; }
int32_t diff_blocks(const ViewConsts& v) { return ((v.tiles_x * v.tiles_y + 7) / 8) * 8; }
int32_t diff_strips(const ViewConsts& v) { return n_strips(v); }
// A strip's pixels make at most one chunk more than a 64th of them.
size_t diff_chunks(const ViewConsts& v) { return (size_t)n_strips(v) * (DIFF_STRIP * 4 + 1); }

void launch_diff_forward(hipStream_t st, const DevScene& s, const ViewConsts& v, const DiffBuffers& b) {
    const int n = v.tiles_x * v.tiles_y;
    if (n <= 0) return;
    if (s.n_lights <= 4) hipLaunchKernelGGL(k_diff_forward<4>, dim3(n), dim3(256), 0, st, s, v, b);
    else hipLaunchKernelGGL(k_diff_forward<8>, dim3(n), dim3(256), 0, st, s, v, b);
}
void launch_diff_forward_views(hipStream_t st, const DevScene& s, const DiffView* views, int32_t n, int32_t blocks) {
    if (n <= 0 || blocks <= 0) return;
    if (s.n_lights <= 4) hipLaunchKernelGGL(k_diff_forward_views<4>, dim3(blocks), dim3(256), 0, st, s, views, n);
    else hipLaunchKernelGGL(k_diff_forward_views<8>, dim3(blocks), dim3(256), 0, st, s, views, n);
}
void launch_diff_clear(hipStream_t st, float* grad, size_t n, double* loss, int32_t* count) {
    const unsigned grid = (unsigned)std::min<size_t>((n + 255) / 256 + 1, 1024);
    hipLaunchKernelGGL(k_diff_clear, dim3(grid), dim3(256), 0, st, grad, n, loss, count);
}
void launch_fit_start(hipStream_t st, const float* par, float* base, float* theta, float* m, float* v, size_t n,
                      float* grad, size_t n_grad, double* loss, int32_t* count, int32_t* step) {
    const unsigned grid = (unsigned)std::min<size_t>((std::max(n, n_grad) + 255) / 256 + 1, 1024);
    hipLaunchKernelGGL(k_fit_start, dim3(grid), dim3(256), 0, st, par, base, theta, m, v, n, grad, n_grad, loss, count,
                       step);
}
void launch_diff_list(hipStream_t st, const DiffView& w, uint2* chunks, int32_t* count) {
    const int n = n_strips(w.v);
    if (n > 0) hipLaunchKernelGGL(k_diff_list, dim3(n), dim3(256), 0, st, (const DiffView*)nullptr, 1, w, chunks, count);
}
void launch_diff_list_views(hipStream_t st, const DiffView* views, int32_t n, int32_t strips, uint2* chunks,
                            int32_t* count) {
    if (n > 0 && strips > 0)
        hipLaunchKernelGGL(k_diff_list, dim3(strips), dim3(256), 0, st, views, n, DiffView{}, chunks, count);
}
// The adjoint's workgroups: at most 4 per CU (its 4 waves a SIMD), so that each
// keeps its sums over many chunks and the flushes, atomics to the same few
// lines, stay few; of a small view one per four chunks it may have.
static unsigned adjoint_grid(size_t max_chunks) { return (unsigned)std::min<size_t>((max_chunks + 31) / 32 * 8 + 8, 1024); }
// The kernel for a scene's lights and materials: pick(NLMAX, VTX, FOUND).
template <class F>
static auto adjoint_variant(const DevScene& s, bool vtx, F&& pick) {
    using std::integral_constant;
    auto by_found = [&](auto nl, auto v) {
        return mat_copies(s.n_materials) == 0 ? pick(nl, v, std::true_type{}) : pick(nl, v, std::false_type{});
    };
    auto by_vtx = [&](auto nl) { return vtx ? by_found(nl, std::true_type{}) : by_found(nl, std::false_type{}); };
    return s.n_lights <= 4 ? by_vtx(integral_constant<int, 4>{}) : by_vtx(integral_constant<int, 8>{});
}
void launch_adjoint(hipStream_t st, const DevScene& s, const DiffView& w, const uint2* chunks, const int32_t* count) {
    const dim3 grid(adjoint_grid((size_t)w.v.W * w.v.H / 64 + n_strips(w.v)));
    const bool vtx = (w.b.want & (DIFF_ALBEDO | DIFF_NORMAL)) != 0 && !w.b.gbuf;
    const auto k = adjoint_variant(s, vtx, [](auto nl, auto v, auto found) {
        return k_adjoint<decltype(nl)::value, decltype(v)::value, decltype(found)::value>;
    });
    hipLaunchKernelGGL(k, grid, dim3(256), 0, st, s, w, chunks, count);
}
void launch_adjoint_views(hipStream_t st, const DevScene& s, const DiffView* views, size_t max_chunks,
                          const uint2* chunks, const int32_t* count, bool vertices, int32_t* step) {
    const dim3 grid(adjoint_grid(max_chunks));
    const auto k = adjoint_variant(s, vertices, [](auto nl, auto v, auto found) {
        return k_adjoint_views<decltype(nl)::value, decltype(v)::value, decltype(found)::value>;
    });
    hipLaunchKernelGGL(k, grid, dim3(256), 0, st, s, views, chunks, count, step);
}

void launch_diff_store_gbuffer(hipStream_t st, const DevScene& s, const ViewConsts& v, const DiffBuffers& b,
                               float4* gbuf) {
    const size_t P = (size_t)v.W * v.H;
    if (P) hipLaunchKernelGGL(k_diff_gbuffer, dim3((unsigned)((P + 255) / 256)), dim3(256), 0, st, s, v, b, gbuf);
}

void launch_adam(hipStream_t st, float* par, float* grad, const float* base, float* theta, float* m, float* v,
                 const int32_t* idx, const float* lower, AdamConsts a, const int32_t* step, double* loss,
                 double* hist) {
    const unsigned grid = a.n > 256 ? (unsigned)((a.n + 255) / 256) : 1u;
    hipLaunchKernelGGL(k_adam, dim3(grid), dim3(256), 0, st, par, grad, base, theta, m, v, idx, lower, a, step, loss,
                       hist);
}

}  // namespace prh
