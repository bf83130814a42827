// gs_internal.h -- host-side declarations shared by the C ABI layer, the
// kernel launchers and the C++ stage classes.  Not part of the public ABI.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstddef>
#include <cstdint>

#include "gs_hip.h"

namespace gsd { struct CamArgs; }
namespace gsr { struct RasterArgs; struct GradArgs; struct MultiRaster; struct MultiPix; struct MultiGrads; }
namespace gso { struct AdamArgs; struct AdamDev; }
namespace gsb { struct BinArgs; }

// Small fixed scratch owned by each context.
constexpr size_t GS_SMALL_BYTES = 4096;
constexpr size_t GS_SMALL_TOTAL64 = 0;    // uint64 pair total of the last scan
constexpr size_t GS_SMALL_OVERFLOW = 64;  // uint32 capacity-overflow flag

struct gs_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    void* ws = nullptr;  // pair-count-sized scratch (sorts, pair words)
    size_t ws_bytes = 0;
    void* ws2 = nullptr;  // Gaussian-count-sized scratch (depth order, ranked offsets)
    size_t ws2_bytes = 0;
    void* small = nullptr;
    bool capturing = false;
    int radix_bits = 8;
    int raster_batch = 256;
    int raster_bwd_batch = 256;
    // Knobs of earlier binning kernels (Gaussians per group, tiles per lane):
    // kept for stored tunings, without effect (the layout follows the sizes).
    int bin_chunk = 4096;
    int bin_tpl = 1;
    int persistent_per_cu = 6;  // batched raster: persistent groups per CU (0: one group per tile)
    int split_groups = 64;      // likewise: the forward no longer runs in two rounds
    void* coarse = nullptr;     // bin records of a binning whose first guess was too small
    size_t coarse_bytes = 0;
    gsb::BinArgs* bin = nullptr;  // the binning that gs_bin_prepare left for gs_bin_finish
    bool bin_pending = false;
    long long bin_pairs = 0;      // its pair count, once read back
};

int gs_set_error(int code, const char* fmt, ...);
int gs_hip_status(hipError_t e, const char* what);
int gs_ws_get(gs_ctx* c, size_t bytes, void** out);
int gs_ws2_get(gs_ctx* c, size_t bytes, void** out);
int gs_small_get(gs_ctx* c, void** out);
int check_cam_cfg(const gs_camera* cam, const gs_render_cfg* cfg);
int gs_tile_key_bits(int num_tiles);

extern "C" int gs_ctx_set_tuning(gs_ctx* c, int radix_bits, int raster_batch, int raster_bwd_batch);
extern "C" int gs_ctx_reserve(gs_ctx* c, size_t bytes);
extern "C" int gs_ctx_set_binning(gs_ctx* c, int gaussians_per_group, int tiles_per_lane);
// Direct-placement binning of one view.  Queues everything up to the pair
// count, with the current capacity for bin records; then, either
//  - host_counts (mapped, coherent pinned memory, device address) set: the
//    kernels write {pairs, records} there, ev_total is recorded after them,
//    and the caller compares both with the capacities before using results
//    (gs_bin_fits); or
//  - host_counts null: waits, grows the record buffer and repeats what needs it
//    if the records did not fit, and returns the count in *pairs.
int gs_bin_prepare(gs_ctx* c, int n, const gs_preprocessed* pre, int width, int height, long long* pairs,
                   unsigned long long* host_counts, hipEvent_t ev_total);
// Places the prepared pairs and writes the ranges; pairs past the capacity
// are dropped (overflow flag) and the ranges clamped to it.
int gs_bin_finish(gs_ctx* c, uint32_t* values, uint32_t capacity, uint32_t* ranges);
// The same two halves over prepared arguments (order, sizes, views, rectangles
// or means set; the workspace carved), for the eval_3D binning.
// guess: gs_bin_guess_bytes of workspace for the records.
int gs_bin_count(gs_ctx* c, gsb::BinArgs& a, void* guess, unsigned long long* pairs);
size_t gs_bin_guess_bytes(const gsb::BinArgs& a);
// Whether `records` bin records fit the context's buffer; grows it if not.
int gs_bin_fits(gs_ctx* c, const gsb::BinArgs& a, unsigned long long records, bool* fits);
extern "C" int gs_check_overflow(gs_ctx* c, int* overflowed);

// kernel launchers
hipError_t launch_preprocess_fwd(const gs_gaussians& G, const gsd::CamArgs& c, const gs_preprocessed& out, int deg,
                                 hipStream_t s);
hipError_t launch_activate(const gs_gaussians& G, float* pos, float* sc, float* rot, float* sh, float* op,
                           hipStream_t s);
hipError_t launch_preprocess_bwd(const gs_gaussians& G, const gsd::CamArgs& c, const int* radii,
                                 const gs_raster_grads& rg, const gs_param_grads& out, int accumulate, int sh_deg,
                                 hipStream_t s);
uint32_t scan_partials_needed(uint32_t n);
hipError_t launch_scan_tiles(const int* in, uint32_t n, uint32_t* out, unsigned long long* partial, uint32_t* total32,
                             unsigned long long* total64, hipStream_t s);
hipError_t launch_duplicate(int n, const float* means2D, const float* depths, const int* radii,
                            const uint32_t* offsets, int gx, int gy, uint64_t* keys, uint32_t* values,
                            uint32_t capacity, uint32_t* overflow, hipStream_t s);
size_t radix_workspace_bytes(uint32_t n, int radix_bits);
hipError_t launch_radix_sort(const uint64_t* keys_in, const uint32_t* vals_in, uint64_t* keys_out, uint32_t* vals_out,
                             uint32_t n, int key_bits, int radix_bits, void* workspace, hipStream_t s);
hipError_t launch_radix_sort_bits(const uint64_t* keys_in, const uint32_t* vals_in, uint64_t* keys_out,
                                  uint32_t* vals_out, uint32_t n, int begin_bit, int end_bit, int radix_bits,
                                  void* workspace, hipStream_t s, const uint32_t* n_dev);
hipError_t launch_tile_ranges(const uint64_t* keys_sorted, uint32_t n, uint32_t num_tiles, uint32_t* ranges,
                              hipStream_t s, const uint32_t* n_dev = nullptr);
hipError_t launch_depth_keys(int n, const float* depths, const int* radii, uint64_t* keys, uint32_t* idx,
                             hipStream_t s);
hipError_t launch_depth_words(int n, const float* depths, const int* radii, uint64_t* words, hipStream_t s,
                              const float* means2D = nullptr, int gx = 0, int gy = 0, uint32_t* rects = nullptr);
hipError_t launch_gather_tiles(int n, const uint32_t* order, const int* tiles, int* out, hipStream_t s);
hipError_t launch_duplicate_ranked(int n, const uint32_t* order, const float* means2D, const int* radii,
                                   const uint32_t* offsets, int gx, int gy, uint64_t* words, uint32_t capacity,
                                   uint32_t* overflow, hipStream_t s);
hipError_t launch_raster_fwd(const gsr::RasterArgs& a, int num_tiles, int batch, float* img, float* T_final,
                             int* n_contrib, uint32_t* last_contrib, hipStream_t s);
hipError_t launch_raster_bwd(const gsr::RasterArgs& a, int num_tiles, int batch, const float* T_final,
                             const uint32_t* last_contrib, const float* d_image, const gsr::GradArgs& g,
                             hipStream_t s);
int l1_partials_needed(uint32_t n);
hipError_t launch_l1(const float* r, const float* g, float* d, uint32_t n, double* partial, double* loss,
                     hipStream_t s);
hipError_t launch_adam(const gso::AdamArgs& a, hipStream_t s);
// One thread: *counter += 1 when *flag is nonzero (counts steps whose update a
// capacity overflow suppressed).
hipError_t launch_count_if(const uint32_t* flag, uint32_t* counter, hipStream_t s);
hipError_t launch_sgd(const gso::AdamArgs& a, hipStream_t s);
hipError_t launch_zero(void* ptr, size_t bytes, hipStream_t s);

// multi-view
hipError_t launch_preprocess_fwd_multi(const gs_gaussians& G, const gsd::CamArgs* cams_dev, int V,
                                       const gs_preprocessed& out, uint64_t* dkeys, uint32_t* didx, int index_shift, int deg,
                                       hipStream_t s, uint32_t* rects = nullptr);
hipError_t launch_preprocess_bwd_multi(const gs_gaussians& G, const gsd::CamArgs* cams_dev,
                                       const gsd::CamArgs* cam_val, int V, const int* radii, const gs_raster_grads& rg,
                                       const gs_param_grads& out, float* const adam_p[5], float* const adam_m[5],
                                       float* const adam_v[5], const gso::AdamDev* hp, const gso::AdamDev* hp_val,
                                       int sh_deg, hipStream_t s, const uint32_t* skip = nullptr);
hipError_t launch_gather_tiles_multi(uint32_t total, int N, const uint64_t* skeys, const uint32_t* sidx,
                                     const int* tiles, int* out, hipStream_t s);
hipError_t launch_duplicate_multi(uint32_t total, int N, const uint64_t* skeys, const uint32_t* sidx,
                                  const float* means2D, const int* radii, const uint32_t* offsets, const int4* views,
                                  uint64_t* words, uint32_t capacity, uint32_t* overflow, hipStream_t s);
// direct-placement binning (k_bin.hip); larger views use the word sort
constexpr int GS_BIN_MAX_TILES_XY = 255;  // tiles per row and per column (4080 pixels)
constexpr int GS_BIN_MAX_BINS = 1024;     // bins per view
int bin_side(int max_gx, int max_gy);     // tiles per bin side for views of at most this many tiles
int bin_count_of_view(int side, int gx, int gy);
size_t bin_record_bytes(const gsb::BinArgs& a);
void bin_layout(gsb::BinArgs& a);  // V, N, NB, total_tiles set: chunks, groups and table lengths
size_t bin_workspace_bytes(const gsb::BinArgs& a);
void bin_carve(gsb::BinArgs& a, void* workspace);
// Bin records, tile counts and their scan.  records (device or mapped host):
// the record count; total32 / total64 (optional): the pair count.  counted:
// repeat after the record buffer grew (the bins' starts are there already).
hipError_t launch_bin_lists(const gsb::BinArgs& a, hipStream_t s, unsigned long long* records, uint32_t* total32,
                            unsigned long long* total64, bool counted = false);
hipError_t launch_bin_place(const gsb::BinArgs& a, hipStream_t s);
hipError_t launch_bin_ranges(const gsb::BinArgs& a, uint32_t* ranges, hipStream_t s);
// total32 / total64 (optional, device): the sum of all n inputs
hipError_t launch_scan_u32_exclusive(const uint32_t* in, uint32_t n, uint32_t* out, unsigned long long* partial,
                                     hipStream_t s, uint32_t* total32 = nullptr, unsigned long long* total64 = nullptr);
hipError_t launch_tile_ranges_multi(const uint64_t* words, uint32_t n_cap, const uint32_t* n_dev, const int4* views,
                                    uint32_t* ranges, hipStream_t s);
hipError_t launch_raster_fwd_multi(const gsr::MultiRaster& m, const gsr::MultiPix& o, int batch,
                                   int persistent_groups, hipStream_t s);
hipError_t launch_raster_bwd_multi(const gsr::MultiRaster& m, const gsr::MultiPix& o, const gsr::MultiGrads& g,
                                   int batch, int persistent_groups, hipStream_t s);
// adaptive density control (k_density.hip)
hipError_t launch_density_accumulate(int n, const float* d_means2D, const int* radii, float* accum, float* denom,
                                     int* max_radii, hipStream_t s);
hipError_t launch_density_classify(int n, const float* accum, const float* denom, const float* log_scales,
                                   float threshold, float size_threshold, uint32_t* clone, uint32_t* split,
                                   hipStream_t s);
hipError_t launch_density_map(int n, const uint32_t* clone, const uint32_t* split, const uint32_t* rank_c,
                              const uint32_t* rank_s, uint32_t n_clone, uint32_t n_split, int2* map, hipStream_t s);
hipError_t launch_density_prune(int m1, int n, const int2* map, const float* log_scales, const float* opacity,
                                const int* max_radii, float scale_factor, float min_opacity, int max_screen_size,
                                float world_threshold, uint32_t* keep, hipStream_t s);
hipError_t launch_density_scatter(int m1, int max_coeffs, const int2* map, const uint32_t* keep, const uint32_t* slot,
                                  const float* const src[5], const float* noise, float scale_factor,
                                  float* const dst[5], hipStream_t s);
hipError_t launch_fill(int n, float v, float* out, hipStream_t s);
hipError_t launch_l1_multi(const float* r, const float* g, float* d, const int* pix_off_dev, int V, int nb,
                           double* partial, double* loss, hipStream_t s);
