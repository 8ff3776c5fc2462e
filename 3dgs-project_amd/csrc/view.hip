// One 3D view in three calls: the stages' entry points (preprocess, count, depth order | fill,
// forward blend | blend backward, preprocess backward) run in order over buffers that a caller
// allocates as two arenas, so that a host program pays for two allocations and three calls per
// view instead of about twenty of each. The stages and their checks are those of the entry points;
// what a later stage would refuse is refused before the first is enqueued.
#include "gs_host.h"

namespace gs {

static int64_t up256(int64_t v) { return (v + 255) & ~int64_t(255); }

// The regions of the state arena, in order (GS_VIEW_REC ...), and its size.
static int64_t state_layout(int64_t n, const CamK& k, int flags, int64_t* off) {
  const int64_t T = static_cast<int64_t>(k.tiles_x) * k.tiles_y, P = static_cast<int64_t>(k.width) * k.height;
  const bool bwd = (flags & GS_VIEW_BACKWARD) != 0, image = !(flags & GS_VIEW_NO_IMAGE);
  const int64_t bytes[GS_VIEW_STATE_REGIONS] = {64 * n,
                                                4 * n,
                                                4 * (n + 1),
                                                8 * T,
                                                4 * (T + 1),
                                                image ? 4 * P : 0,
                                                bwd ? 4 * P : 0,
                                                bwd ? 4 * T : 0};
  int64_t o = 0;
  for (int r = 0; r < GS_VIEW_STATE_REGIONS; ++r) {
    off[r] = o;
    o += up256(bytes[r]);
  }
  return o;
}

// The scratch of gs_view_begin: depth keys, wave counts, the depth ordering's workspace.
struct BeginScratch {
  int64_t dkeys, waves, prep, end;
};

static BeginScratch begin_scratch(int64_t n) {
  BeginScratch s;
  s.dkeys = 0;
  s.waves = up256(4 * n);
  s.prep = s.waves + up256(4 * ((n + 63) / 64));
  s.end = s.prep + up256(static_cast<int64_t>(gs_bin_prepare_workspace_size(n)));
  return s;
}

static int check_arena(const void* p, size_t have, int64_t need, const char* name) {
  GS_REQUIRE(p, GS_ERR_ARG, "null pointer argument (%s)", name);
  GS_REQUIRE(aligned(p, 256), GS_ERR_ALIGN, "the %s must be 256-byte aligned", name);
  GS_REQUIRE(have >= static_cast<size_t>(need), GS_ERR_WORKSPACE, "%s too small: need %lld bytes", name,
             static_cast<long long>(need));
  return GS_OK;
}

}  // namespace gs

using namespace gs;

extern "C" int gs_view_plan(int64_t n, const gs_camera* cam, int flags, int64_t* state_offsets, int64_t* sizes) {
  clear_error();
  if (int e = check_cam(cam)) return e;
  GS_REQUIRE(n >= 0 && n < (int64_t(1) << 32) && state_offsets && sizes, GS_ERR_ARG, "invalid view_plan arguments");
  sizes[0] = state_layout(n, make_cam(*cam), flags, state_offsets);
  sizes[1] = begin_scratch(n).end;
  sizes[2] = gs_bin_path(n, cam);
  return GS_OK;
}

extern "C" int gs_view_plan_count(int64_t n, int64_t m, const gs_camera* cam, int flags, int64_t* list_offsets,
                                  int64_t* sizes) {
  clear_error();
  if (int e = check_cam(cam)) return e;
  GS_REQUIRE(n >= 0 && m >= 0 && m < (int64_t(1) << 32) && list_offsets && sizes, GS_ERR_ARG,
             "invalid view_plan_count arguments (n=%lld, m=%lld)", static_cast<long long>(n), static_cast<long long>(m));
  const CamK k = make_cam(*cam);
  const bool bwd = (flags & GS_VIEW_BACKWARD) != 0;
  // >= sum over tiles of ceil(len / 32)
  const int64_t nb = bwd ? (m + (kBucket - 1) * (static_cast<int64_t>(k.tiles_x) * k.tiles_y)) / kBucket : 0;
  const int64_t bytes[GS_VIEW_LIST_REGIONS] = {4 * m, bwd ? 4 * nb : 0, bwd ? 4 * (kListHeader + nb) : 0,
                                               bwd ? 4096 * nb : 0, (flags & GS_VIEW_KEYS) ? 8 * m : 0};
  int64_t o = 0;
  for (int r = 0; r < GS_VIEW_LIST_REGIONS; ++r) {
    list_offsets[r] = o;
    o += up256(bytes[r]);
  }
  sizes[0] = o;
  sizes[1] = static_cast<int64_t>(gs_bin_fill_3d_workspace_size(n, m, cam));
  sizes[2] = nb;
  return GS_OK;
}

extern "C" int gs_view_begin(const float* means, const float* log_scales, const float* quats,
                             const float* opacity_logits, const float* sh, const float* sh_rest, int64_t n,
                             int sh_coeffs, int sh_degree, const gs_camera* cam, int flags, void* state,
                             size_t state_bytes, uint32_t* tiles_touched, void* scratch, size_t scratch_bytes,
                             void* stream) {
  clear_error();
  if (int e = check_cam(cam)) return e;
  GS_REQUIRE(n > 0 && n < (int64_t(1) << 32), GS_ERR_ARG, "invalid view_begin arguments");
  int64_t off[GS_VIEW_STATE_REGIONS];
  const int64_t need = state_layout(n, make_cam(*cam), flags, off);
  const BeginScratch s = begin_scratch(n);
  if (int e = check_arena(state, state_bytes, need, "state arena")) return e;
  if (int e = check_arena(scratch, scratch_bytes, s.end, "scratch")) return e;
  if (int e = check_count()) return e;
  char* st = static_cast<char*>(state);
  char* sc = static_cast<char*>(scratch);
  const auto u32 = [](char* p) { return reinterpret_cast<uint32_t*>(p); };
  float* rec = reinterpret_cast<float*>(st + off[GS_VIEW_REC]);
  if (int e = gs_preprocess_fwd(means, log_scales, quats, opacity_logits, sh, sh_rest, n, sh_coeffs, sh_degree, cam, rec,
                                tiles_touched, u32(sc + s.dkeys), u32(sc + s.waves), stream))
    return e;
  if (int e = gs_count_begin(u32(sc + s.waves), (n + 63) / 64, 0, stream)) return e;
  const int e = gs_bin_prepare_3d(rec, tiles_touched, u32(sc + s.dkeys), n, cam, u32(st + off[GS_VIEW_ORDER]),
                                  gs_bin_path(n, cam) == GS_BIN_PATH_SPANS ? nullptr : u32(st + off[GS_VIEW_OFFSETS]),
                                  sc + s.prep, static_cast<size_t>(s.end - s.prep), stream);
  if (e) {
    uint64_t m;
    gs_count_end(&m);  // the count is not left pending
    return e;
  }
  return GS_OK;
}

extern "C" int gs_view_finish(int64_t n, int64_t m, const gs_camera* cam, int flags, void* state, size_t state_bytes,
                              void* lists, size_t lists_bytes, uint32_t* bucket_offsets, void* workspace,
                              size_t workspace_bytes, const float* bg, float* image, float* alpha, float* clear,
                              int64_t clear_floats, void* stream) {
  clear_error();
  if (int e = check_cam(cam)) return e;
  GS_REQUIRE(!(flags & (GS_VIEW_NO_IMAGE | GS_VIEW_KEYS)), GS_ERR_ARG, "invalid view_finish arguments");
  int64_t so[GS_VIEW_STATE_REGIONS], lo[GS_VIEW_LIST_REGIONS], sizes[3];
  const CamK k = make_cam(*cam);
  if (int e = gs_view_plan_count(n, m, cam, flags, lo, sizes)) return e;
  if (int e = check_arena(state, state_bytes, state_layout(n, k, flags, so), "state arena")) return e;
  if (int e = check_arena(lists, lists_bytes, sizes[0], "list arena")) return e;
  // (the blend's own checks, made before the fill is enqueued)
  GS_REQUIRE(image, GS_ERR_ARG, "null pointer argument");
  GS_REQUIRE(clear_floats >= 0 && clear_floats % 4 == 0 && (clear || clear_floats == 0), GS_ERR_ARG,
             "clear must hold a multiple of 4 floats");
  GS_REQUIRE(aligned(clear, 16), GS_ERR_ALIGN, "clear must be 16-byte aligned");
  char* st = static_cast<char*>(state);
  char* li = static_cast<char*>(lists);
  const auto u32 = [](char* p) { return reinterpret_cast<uint32_t*>(p); };
  const bool bwd = (flags & GS_VIEW_BACKWARD) != 0;
  const float* rec = n ? reinterpret_cast<float*>(st + so[GS_VIEW_REC]) : nullptr;
  uint32_t* offsets = gs_bin_path(n, cam) == GS_BIN_PATH_SPANS ? nullptr : u32(st + so[GS_VIEW_OFFSETS]);
  uint32_t* point_list = m ? u32(li + lo[GS_VIEW_POINT_LIST]) : nullptr;
  uint32_t* ranges = u32(st + so[GS_VIEW_RANGES]);
  uint32_t* boff = bucket_offsets ? bucket_offsets : u32(st + so[GS_VIEW_BUCKET_OFFSETS]);
  uint32_t* blist = bwd ? u32(li + lo[GS_VIEW_BUCKET_LIST]) : nullptr;
  if (int e = gs_bin_fill_3d(rec, nullptr, u32(st + so[GS_VIEW_ORDER]), offsets, n, cam, m, nullptr, point_list, ranges,
                             boff, blist, workspace, workspace_bytes, stream))
    return e;
  return gs_blend_fwd_3d(rec, ranges, point_list, boff, k.width, k.height, bg, image,
                         reinterpret_cast<float*>(st + so[GS_VIEW_FINAL_T]), alpha,
                         bwd ? reinterpret_cast<int32_t*>(st + so[GS_VIEW_N_CONTRIB]) : nullptr,
                         bwd ? u32(st + so[GS_VIEW_TILE_MAX]) : nullptr,
                         bwd ? reinterpret_cast<float*>(li + lo[GS_VIEW_CKPT]) : nullptr, blist,
                         bwd && sizes[2] ? u32(li + lo[GS_VIEW_BUCKET_TO_TILE]) : nullptr, clear, clear_floats,
                         bwd ? GS_BLEND_LIST_CLEARED : 0, stream);
}

extern "C" int gs_view_backward(const float* means, const float* log_scales, const float* quats,
                                const float* opacity_logits, const float* sh, const float* sh_rest, int64_t n,
                                int sh_coeffs, int sh_degree, int64_t m, const gs_camera* cam, void* state,
                                size_t state_bytes, void* lists, size_t lists_bytes, const uint32_t* bucket_offsets,
                                const uint32_t* tiles_touched, const float* image, const float* grad_image,
                                const float* grad_alpha, float* grad2d, double* grad_conic64, int flags,
                                float* grad_means, float* grad_log_scales, float* grad_quats,
                                float* grad_opacity_logits, float* grad_sh, float* grad_sh_rest, void* stream) {
  clear_error();
  if (int e = check_cam(cam)) return e;
  if (int e = check_sh(sh_coeffs, sh_degree)) return e;
  int64_t so[GS_VIEW_STATE_REGIONS], lo[GS_VIEW_LIST_REGIONS], sizes[3];
  const CamK k = make_cam(*cam);
  if (int e = gs_view_plan_count(n, m, cam, GS_VIEW_BACKWARD, lo, sizes)) return e;
  if (int e = check_arena(state, state_bytes, state_layout(n, k, GS_VIEW_BACKWARD, so), "state arena")) return e;
  if (int e = check_arena(lists, lists_bytes, sizes[0], "list arena")) return e;
  // (the preprocess backward's own checks, made before the blend's is enqueued)
  GS_REQUIRE(n == 0 || (means && log_scales && quats && opacity_logits && sh && tiles_touched && grad2d && grad_means &&
                        grad_log_scales && grad_quats && grad_opacity_logits && grad_sh),
             GS_ERR_ARG, "null pointer argument");
  GS_REQUIRE(n == 0 || !sh_rest == !grad_sh_rest, GS_ERR_ARG, "sh_rest and grad_sh_rest go together");
  GS_REQUIRE(n == 0 || !(sh_rest && sh_coeffs == 1), GS_ERR_ARG, "sh_rest given for a DC-only model");
  GS_REQUIRE(n == 0 || (aligned(quats, 16) && aligned(grad_quats, 16)), GS_ERR_ALIGN,
             "quats and grad_quats must be 16-byte aligned");
  char* st = static_cast<char*>(state);
  char* li = static_cast<char*>(lists);
  const auto u32 = [](char* p) { return reinterpret_cast<uint32_t*>(p); };
  if (int e = gs_blend_bwd_3d(n ? reinterpret_cast<float*>(st + so[GS_VIEW_REC]) : nullptr, u32(st + so[GS_VIEW_RANGES]),
                              m ? u32(li + lo[GS_VIEW_POINT_LIST]) : nullptr,
                              bucket_offsets ? bucket_offsets : u32(st + so[GS_VIEW_BUCKET_OFFSETS]),
                              sizes[2] ? u32(li + lo[GS_VIEW_BUCKET_TO_TILE]) : nullptr, sizes[2], n, k.width, k.height,
                              image, grad_image, reinterpret_cast<float*>(st + so[GS_VIEW_FINAL_T]), grad_alpha,
                              reinterpret_cast<int32_t*>(st + so[GS_VIEW_N_CONTRIB]), u32(st + so[GS_VIEW_TILE_MAX]),
                              reinterpret_cast<float*>(li + lo[GS_VIEW_CKPT]), u32(li + lo[GS_VIEW_BUCKET_LIST]), grad2d,
                              grad_conic64, flags | GS_ACCUMULATE, nullptr, stream))
    return e;
  return gs_preprocess_bwd(means, log_scales, quats, opacity_logits, sh, sh_rest, n, sh_coeffs, sh_degree, cam,
                           tiles_touched, grad2d, grad_conic64, grad_means, grad_log_scales, grad_quats,
                           grad_opacity_logits, grad_sh, grad_sh_rest, stream);
}
