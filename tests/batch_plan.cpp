// Plans of batches and of a server's staging without a device, for tests/test_batch_plan.py (linked with
// libmlgi.so).
#include "../include/mlgi_scene.h"

#include "../many-lights-gi_amd/csrc/capi_internal.hpp"

// A batch of n frames of 96 x 64, vpl[i] VPLs and a side[i] atlas: what its
// plan says. The buffers are addresses that nothing reads.
extern "C" int plan_tiles(int n, const int* vpl, const int* side, uint64_t* bytes, int* max_side) {
  std::vector<mlgi_frame_desc> frames(n);
  char* at = (char*)((uintptr_t)1 << 20);
  auto take = [&](size_t b) {
    char* p = at;
    at += (b + 255) / 256 * 256;
    return p;
  };
  for (int i = 0; i < n; ++i) {
    mlgi_frame_desc& d = frames[i];
    d = mlgi_frame_desc{};
    mlgi_params_default(&d.params);
    d.params.atlas_side = side[i];
    d.params.pull_push_levels = 2;
    d.params.shuffle_lights = 0;  // its table lives on the device
    const size_t px = 96 * 64;
    d.rsm.width = d.rsm.height = 128;
    d.rsm.diffuse = d.rsm.face_normal = d.rsm.depth = (float*)take(1 << 20);
    d.gbuffer.width = d.image.width = 96;
    d.gbuffer.height = d.image.height = 64;
    d.gbuffer.depth = d.gbuffer.face_normal = (float*)take(px * 12);
    d.image.rgb = (float*)take(px * 12);
    d.vpls.records = (float*)take((size_t)vpl[i] * 128);
    d.vpls.count = vpl[i];
    d.atlas.texels = (uint32_t*)take((size_t)side[i] * side[i] * 4);
    d.ism.texels = (uint16_t*)take((size_t)side[i] * side[i] * 2);
    d.atlas.side = d.ism.side = side[i];
  }
  mlgi_context ctx;
  std::vector<mlgi::BatchFrame> table;
  mlgi_capi::BatchPlan plan;
  const int rc = mlgi_capi::batch_plan(&ctx, frames.data(), n, &table, &plan);
  *bytes = plan.tile_bytes;
  *max_side = plan.max_ism_side;
  return rc;
}

extern "C" size_t stage_slot(int slots, size_t largest, int max_batch) {
  return mlgi_capi::stage_slot_bytes(slots, largest, max_batch);
}

extern "C" int pp_group(int ism_side, int isms, int frames) {
  return mlgi::pullpush_group(ism_side, (uint64_t)isms * frames, isms);
}

extern "C" int streams(uint64_t bytes) { return mlgi::tiles_stream(bytes); }
