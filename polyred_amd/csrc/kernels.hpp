// kernels.hpp — host-side launchers of libprh's gfx950 kernels.
#pragma once

#include "prh_internal.hpp"

namespace prh {

struct ShadeConsts {
    ViewConsts v;
    uint8_t gamma_lut[256];   // shader.GammaCorrection per 8-bit value
    uint32_t background;      // render.Background RGBA8
    int32_t shadow_map;       // render.ShadowMap
    int32_t gamma_correct;    // render.GammaCorrection
    int32_t n_lights;
    float ao_dir[16];         // material/ao.go:26 directions {cos, sin} x 8
    int32_t SW, SH;           // shadow map size
    gm::M4 svp;               // ViewportMatrix(SW, SH)
    int32_t shadow_sparse;    // the light views' last row is (0 0 0 1) and the light projections and svp
                              // have zeros everywhere but the diagonal and the last column
};

// A shadow-casting light's transforms for the shading's shadow test where
// they have the sparse shape (light view's last row (0 0 0 1), projection and
// map viewport diagonal plus last column): the coefficients that multiply a
// coordinate in an fma64 held as float64 (exact), so the test converts none
// of them, and the last-column terms it multiplies in float32 as float.
struct ShadowXf {
    double view[9];   // light view rows 0-2, columns 0-2
    double proj[3];   // light projection diagonal
    double svp[3];    // map viewport diagonal
    float view_c[3];  // light view column 3, rows 0-2
    float proj_c[3];
    float svp_c[3];
    float pad[3];
};

struct ShadeBuffers {
    const uint64_t* vis;
    const float* depth;
    const float4* tv_scr;
    const float4* tv_nor;
    const float4* tv_wp;
    const int4* tri_rec;       // per triangle: transformed vertices and flat material (k_tri_rec)
    const uint32_t* tv_col;    // per transformed vertex: colour
    const float2* tv_uv;       // and UV (scenes with textures)
    const ClipRec* clips;
    const int32_t* tri_clip_slot;
    const uint32_t* smaps;     // [slots][SH][SW] ordered depth bits
    const gm::M4* light_view;  // [n_lights]
    const gm::M4* light_proj;  // [n_lights]
    const ShadowXf* light_xf;  // [n_lights], read where ShadeConsts.shadow_sparse is set
    uint32_t* image;           // [H][W] RGBA8, top row first
    uint32_t* pregamma;        // optional [H][W] raster rows
    float* linear;             // optional [H][W][3]
    uint32_t* bg;              // [2] uncovered colour, pixel (0,0)'s colour
    float* bg_lin;             // [3]
    const PassCounters* cnt;   // the main view's, then the shadow passes': nothing is shaded after an overflow
    Counters* cnt_host;        // pinned host copy of both, written once they are final
    float* ao;                 // [H][W] AO factor of the pixels that need it
    int32_t* ao_xs;            // [H][W] per row, the columns of the pixels k_ao computes, left to right (k_resolve)
    int32_t* ao_cnt;           // [H] and their count
    float *ao_col, *ao_box;    // [(H+3)/4][W] and [(H+3)/4][(W+3)/4], the marches' depth bounds (k_ao_max)
    const float* ao_tab;       // AO march tables (tap offsets, diagonal distances)
    int32_t ao_fast;           // the tables hold for this frame size
    int32_t bg_inline;         // k_shade shades the uncovered pixels itself: no k_shade_bg ran
    float* depth_out;          // set: no k_resolve ran, and k_shade writes the depth
    uint32_t* col_pre;         // set: k_shade is the first half of a split shading (colour before AO)
    uint8_t* post_flag;        // and per pixel what the second half does: 0 colour as is, 1 with the AO
                               // factor, 2 uncovered (the uncovered colour)
};

// The differentiable shading pass (diff.hip): parameters, fixed inputs and
// gradient outputs, all in HBM.
constexpr int DIFF_MAX_LIGHTS = 8;
constexpr int DIFF_REPS = 8;
struct DiffBuffers {
    const uint64_t* vis;       // fixed visibility (the last frame)
    const int4* tri_rec;       // per triangle: transformed vertices and flat material (k_tri_rec)
    const float4* tv_scr;      // screen xy + recipw per transformed vertex
    const float4* tv_nor;      // n.Apply(Normal) per transformed vertex (the default normals)
    const float4* tv_wp;       // back-transformed position per transformed vertex
    const float* albedo;       // [Vt][3]
    const float* normal;       // [Vt][3], or null: tv_nor
    const float* kd;           // [M][3]
    const float* ks;           // [M][3]
    const float* shininess;    // [M]
    const float* light_pos;    // [L][3]
    const float* light_int;    // [L]
    float ambient;             // sum of the ambient intensities
    const uint8_t* shadow_count;  // [H][W] fixed shadow visibility: the shading is scaled by 2^-count; or null
    const float4* gbuf;        // [4][H][W] stored G-buffer (diff_store_gbuffer), or null: rebuilt from vis
    const float* target;       // [H][W][3] raster rows (adjoint)
    uint32_t* list;            // [H*W] the shaded pixels, x | y << 16, by strips (adjoint; launch_diff_list)
    float* linear;             // [H][W][3] raster rows (forward), NaN where not shaded
    float *g_albedo, *g_normal, *g_kd, *g_ks, *g_shin, *g_lpos, *g_lint;  // zeroed before the adjoint
    double* loss;              // [DIFF_REPS] summed by the reader
    uint32_t want;             // DIFF_* gradient groups to accumulate
    // replicas of g_kd .. g_lint, rep_stride floats apart, summed by the
    // reader: DIFF_REPS or 1
    int32_t reps, rep_stride;
};
// Gradient groups (the bits of prh.h's PRH_FIT_* flags).
constexpr uint32_t DIFF_ALBEDO = 1, DIFF_NORMAL = 2, DIFF_KD = 4, DIFF_KS = 8, DIFF_SHININESS = 16,
                   DIFF_LIGHT_POS = 32, DIFF_LIGHT_INT = 64, DIFF_ALL = 127;
// One view of a multi-view launch: its forward's workgroups are [block0,
// block0 + nblocks), its list's [strip0, ...).
struct DiffView {
    ViewConsts v;
    DiffBuffers b;
    int32_t block0, nblocks, strip0;
};
int32_t diff_blocks(const ViewConsts& v);
int32_t diff_strips(const ViewConsts& v);
size_t diff_chunks(const ViewConsts& v);  // entries of the chunk table a view may fill
void launch_diff_forward(hipStream_t st, const DevScene& s, const ViewConsts& v, const DiffBuffers& b);
void launch_diff_forward_views(hipStream_t st, const DevScene& s, const DiffView* views, int32_t n, int32_t blocks);
// The adjoint: the gradients (n floats), the loss and the count of chunks
// zeroed, the views' shaded pixels listed, then the adjoint over the list.
void launch_diff_clear(hipStream_t st, float* grad, size_t n, double* loss, int32_t* count);
void launch_fit_start(hipStream_t st, const float* par, float* base, float* theta, float* m, float* v, size_t n,
                      float* grad, size_t n_grad, double* loss, int32_t* count, int32_t* step);
void launch_diff_list(hipStream_t st, const DiffView& w, uint2* chunks, int32_t* count);
void launch_diff_list_views(hipStream_t st, const DiffView* views, int32_t n, int32_t strips, uint2* chunks,
                            int32_t* count);
void launch_adjoint(hipStream_t st, const DevScene& s, const DiffView& w, const uint2* chunks, const int32_t* count);
// vertices: the views want albedo or normal gradients (and store no
// G-buffer); step (may be null): a fit's step counter, advanced by the adjoint
void launch_adjoint_views(hipStream_t st, const DevScene& s, const DiffView* views, size_t max_chunks,
                          const uint2* chunks, const int32_t* count, bool vertices, int32_t* step);
// The stored G-buffer of one view (world position + material, normal +
// shadow scale, view vector, albedo: 4 float4 planes of H*W).
void launch_diff_store_gbuffer(hipStream_t st, const DevScene& s, const ViewConsts& v, const DiffBuffers& b,
                               float4* gbuf);
// Adam (Kingma & Ba 2015, Algorithm 1) on the parameters p = base * (1 + theta)
// listed in idx; t is the device step counter, loss the step's loss, kept
// in hist[t - 1].  Leaves the listed gradients and the loss at zero for the
// next step's adjoint.  Gradients from rep_from on have `reps` replicas,
// rep_stride apart.
struct AdamConsts {
    float lr, beta1, beta2, eps;
    int32_t n, hist_cap;
    int32_t reps, rep_from, rep_stride;
};
void launch_adam(hipStream_t st, float* par, float* grad, const float* base, float* theta, float* m, float* v,
                 const int32_t* idx, const float* lower, AdamConsts a, const int32_t* step, double* loss,
                 double* hist);

// Layout of the AO march tables, in float (4-byte) units.  Binade buckets are
// frexp exponents AO_EXP_MIN .. AO_EXP_MIN + AO_EXP_N - 1.
constexpr int AO_EXP_MIN = -10;
constexpr int AO_EXP_N = 24;
constexpr int AO_DIST_PER_DIR = AO_EXP_N * AO_EXP_N * 100;  // doubles
constexpr int AO_TAB_OFF = 0;           // float [8 directions][2][100 t]: fl(dir * t)
constexpr int AO_TAB_T64 = 8 * 200;     // double [100]: fl64(1 / t)
constexpr int AO_TAB_DIST = AO_TAB_T64 + 200;  // double [4 diagonals][AO_EXP_N][AO_EXP_N][100 t]: fl64(1 / distance)
// int32 [4 axis directions][4]: major axis (1 = x), sign of the major
// offset (+-1, exactly +-t), the smallest minor coordinate from which the
// minor offset never moves the tap off its row/column (INT32_MAX: none)
constexpr int AO_TAB_AXIS = AO_TAB_DIST + 2 * 4 * AO_DIST_PER_DIR;
constexpr int AO_TAB_SIZE = AO_TAB_AXIS + 16;
// k_ao's LDS window of a row for its x marches: a chunk of AO pixels
// spanning up to AO_WIN - 99 columns
constexpr int AO_WIN = 448;
// Third descriptor word of a raw (unstrided, untyped) buffer on gfx9 parts.
constexpr uint32_t BUF_DWORD3 = 0x00020000u;

// Where a kernel writes the device's clock as it starts or ends (null: not at
// all), for the passes' times.
struct Stamp {
    unsigned long long* start = nullptr;
    unsigned long long* end = nullptr;
};

// Host copies (k_push, k_pull): device memory src[0, n) to dst[off, off + n).
constexpr int PUSH_SEGS = 4, PUSH_CHUNKS = 32;
struct PushSeg {
    const uint8_t* src;
    uint32_t off, n;
};
struct PushArgs {
    PushSeg seg[PUSH_SEGS];
    int32_t n_segs;
    uint8_t* dst;  // page-locked host memory, as the device sees it
    uint32_t chunk;  // a multiple of 16
    int32_t n_chunks, sets;
    uint32_t* done;   // [PUSH_CHUNKS] zero before and after
    uint32_t* flags;  // [PUSH_CHUNKS] page-locked host memory
    uint32_t serial;
};
void launch_pull(hipStream_t st, uint8_t* dst, const uint8_t* src, size_t n);
void launch_push(hipStream_t st, PushArgs a);

void launch_fill_u32(hipStream_t st, uint32_t* p, size_t n, uint32_t v);
void launch_fill_u64(hipStream_t st, uint64_t* p, size_t n, uint64_t v);
void launch_frame_clear(hipStream_t st, uint32_t* cnt, int32_t n_cnt, uint64_t* vis, size_t n_vis, Stamp stamp);
// A frame's start: counters to zero, the visibility buffer emptied.  Each
// stream's first pass (the vertex passes) does its part before its own
// work, with k_frame_clear only where that pass has nothing to launch.
struct FrameClear {
    uint32_t* cnt;
    int32_t n_cnt;
    uint64_t* vis;
    size_t n_vis;
};
void launch_vertex_main(hipStream_t st, const DevScene& s, const gm::M4* trans, const gm::M4* normal,
                        const ViewConsts& vc, float4* tv_scr, float4* tv_nor, float4* tv_wp, uint32_t* tv_col,
                        float2* tv_uv, const FrameClear& clr, Stamp stamp);
void launch_vertex_shadow(hipStream_t st, const DevScene& s, const gm::M4* strans, const ShadowConsts& sc,
                          float3* ts, const FrameClear& clr, Stamp stamp);
// The setup's workgroups (each writes its unclipped primitives to
// blk_prims[its index]) and then the clipper's (blk_prims[setup_blocks +
// its index]: its pieces); blk_prims holds setup_blocks(n_tris) + CLIP_GRID.
constexpr int CLIP_GRID = 512;
int setup_blocks(int32_t n_tris);
int clip_grid(const Capacities& cap);
// blk_pairs (may be null): likewise the raster tiles the primitives left to the
// raster touch
void launch_setup_main(hipStream_t st, const DevScene& s, const ViewConsts& vc, const float4* tv_scr,
                       const float4* tv_nor, const JobQueues& jobs, ClipRec* clips, int32_t* tri_clip_slot,
                       ClipJob* clip_list, int32_t* blk_prims, int32_t* blk_pairs, Counters* cnt, Capacities cap,
                       unsigned long long* vis, int32_t draw_small, int32_t count_small, const int4* tri_rec,
                       Stamp stamp);
void launch_setup_shadow(hipStream_t st, const DevScene& s, const ShadowConsts& sc, const int4* tri_rec,
                         const float3* ts, const JobQueues& jobs, Counters* cnt, uint32_t* smaps);
// Each global triangle's record, fixed by the scene: its transformed
// vertices and its material in the flat table (-1: vertex colour, matAt's
// rule), or x = -1 when Triangle.IsValid is false.  Once per renderer.
void launch_tri_rec(hipStream_t st, const DevScene& s, int4* tri_rec);
// mode: 0 visibility, 1 visibility in exact order (NaN rule), 2 shadow maps;
// direct: the setup drew the triangles of at most so many centres
void launch_raster(hipStream_t st, int mode, int direct, int n_workgroups, const JobQueues& jobs, Counters* cnt,
                   const RasterTarget& rt, Stamp stamp);
void launch_resolve(hipStream_t st, bool exact, const RasterTarget& rt, Counters* cnt, float* depth, const DevScene& s,
                    int32_t* ao_xs, int32_t* ao_cnt, const int4* tri_rec, Stamp stamp);
void launch_ao(hipStream_t st, const DevScene& s, const ShadeConsts& c, const ShadeBuffers& b);
void launch_shade_bg(hipStream_t st, const DevScene& s, const ShadeConsts& c, const ShadeBuffers& b, Stamp stamp);
void launch_shade(hipStream_t st, const DevScene& s, const ShadeConsts& c, const ShadeBuffers& b, Stamp stamp);
// false (and nothing launched) without the colour before AO, the AO factors or the triangle records
bool launch_shade_post(hipStream_t st, const DevScene& s, const ShadeConsts& c, const ShadeBuffers& b, Stamp stamp);
void launch_shadow_count(hipStream_t st, const DevScene& s, const ShadeConsts& c, const ShadeBuffers& b,
                         uint8_t* out);

// Wide launches: many views' frames as one launch per stage (kernels.hip).
struct WideBatch;
WideBatch* wide_new();
void wide_free(WideBatch* w);
void wide_record(WideBatch* w);  // launch_* calls record into w (nullptr: launch again)
void wide_stage(int stage);      // the stage of the following launch_* calls
size_t wide_layout(WideBatch* w);  // device bytes of the argument arrays (0: unusable)
int wide_upload(const WideBatch* w, uint8_t* dev);
void wide_launch(const WideBatch* w, hipStream_t st, const uint8_t* dev);
// out[y][x] (out_rows x out_w) = 8-bit bilinear filter of row x of `in` at y
void launch_resize(hipStream_t st, const uint32_t* in, int32_t in_w, uint32_t* out, int32_t out_w, int32_t out_rows,
                   const int16_t* coeffs, const int32_t* start, int32_t fl, Stamp stamp = {});

}  // namespace prh
