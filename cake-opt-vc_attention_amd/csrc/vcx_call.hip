// One attention call from Q/K/V to the output: grouping, preparation and the fused kernel from a
// single entry point on one workspace, so that a caller pays for one library call and two
// allocations instead of four and fifteen: at [1,2,2048,128], where a call's kernels take about 35
// us, the host's share went from 88 to 30 us.
#include "vcx_common.hpp"

namespace vcx {

size_t ws_prepare_v(int64_t BH, int64_t N, int64_t D);
size_t ws_group(int64_t BH, int64_t N, int64_t D, int clusters);
int prepare_together(const vcx_call& c, const int64_t* perm, void* q8, float* qs, void* k8, float* ks, uint8_t* v8,
                     float* vs, uint16_t* means, double* ksum, float* km, void* v_scratch, void* stream);

namespace {

struct CallWs {
  int8_t *q8, *k8;
  uint8_t* v8;
  float *qs, *ks, *vs;
  uint16_t* means;
  int64_t* perm;
  float* km;
  void *v_scratch, *group_scratch;
  size_t group_bytes, bytes;
};

bool groups(const vcx_call& c) { return c.smooth && c.perm == nullptr; }

// V scales per channel: without smoothing there are no others, whatever the option says.
bool channel_scales(const vcx_call& c) { return !c.smooth || c.channel_scale; }

// Two places serve twice, as the stages run one after another on the stream: the grouping's scratch
// lies over all that is written after it, and K's tile sums (8 bytes per channel and tile), which
// the Q launch reads last, over the V payload (128 bytes), which the launch after that writes.
CallWs call_ws(const vcx_call& c) {
  const int64_t BH = c.B * c.H, tq = cdiv(c.Nq, 64), tiles = cdiv(c.Nk, kTile);
  size_t off = 0;
  auto take = [&](size_t bytes) {
    char* p = static_cast<char*>(c.workspace) + off;
    off += (bytes + 255) & ~size_t(255);
    return p;
  };
  CallWs w{};
  if (groups(c)) w.perm = reinterpret_cast<int64_t*>(take(sizeof(int64_t) * BH * c.Nk));
  const size_t shared = off;
  w.q8 = reinterpret_cast<int8_t*>(take(BH * c.Nq * c.D));
  w.k8 = reinterpret_cast<int8_t*>(take(BH * c.Nk * c.D));
  w.v8 = reinterpret_cast<uint8_t*>(take(BH * c.D * tiles * kTile));
  w.qs = reinterpret_cast<float*>(take(sizeof(float) * BH * tq * (c.qk_fp8 ? 1 : 32)));
  w.ks = reinterpret_cast<float*>(take(sizeof(float) * BH * tiles * (c.qk_fp8 ? 1 : 4)));
  w.vs = reinterpret_cast<float*>(take(sizeof(float) * BH * c.D * (channel_scales(c) ? 1 : tiles)));
  if (c.smooth) w.means = reinterpret_cast<uint16_t*>(take(sizeof(uint16_t) * BH * tiles * c.D));
  w.km = reinterpret_cast<float*>(take(sizeof(float) * BH * c.D));
  w.v_scratch = take(ws_prepare_v(BH, c.Nk, c.D));
  if (groups(c)) {
    w.group_scratch = static_cast<char*>(c.workspace) + shared;
    w.group_bytes = ws_group(BH, c.Nk, c.D, static_cast<int>(c.clusters));
    off = std::max(off, shared + w.group_bytes);
  }
  w.bytes = off;
  return w;
}

int check_call(const vcx_call* c) {
  VCX_REQUIRE(c != nullptr, "call is null");
  VCX_REQUIRE(c->B >= 1 && c->H >= 1 && c->Nq >= 1 && c->Nk >= 1, "B, H, Nq, Nk must be positive");
  VCX_REQUIRE(c->D == 64 || c->D == 128, "D must be 64 or 128");
  VCX_REQUIRE(c->B <= 65535 && c->H <= 65535 && c->B * c->H <= 65535, "B*H exceeds 65535");
  VCX_REQUIRE(c->Nq < (int64_t(1) << 30) && c->Nk < (int64_t(1) << 30), "sequence too long");
  // the stages take these as int: nothing may be lost on the way
  VCX_REQUIRE(c->dtype == VCX_FLOAT16 || c->dtype == VCX_BFLOAT16, "dtype must be float16 or bfloat16");
  VCX_REQUIRE(c->expcast >= 0 && c->expcast <= 2, "expcast must be 0, 1 or 2");
  VCX_REQUIRE(!groups(*c) || (c->clusters >= 1 && c->clusters <= 256 && c->iterations >= 1 && c->iterations <= 100),
              "clusters must be in [1, 256] and iterations in [1, 100]");
  VCX_REQUIRE(!groups(*c) || c->group_mode == VCX_GROUP_AUTO || c->group_mode == VCX_GROUP_GENERAL,
              "mode must be VCX_GROUP_AUTO or VCX_GROUP_GENERAL");
  VCX_REQUIRE(!c->qk_fp8 || (!c->smooth && !c->rotate && c->perm == nullptr),
              "FP8 QK takes no V smoothing, rotation or permutation");
  return VCX_OK;
}

}  // namespace
}  // namespace vcx

using namespace vcx;

extern "C" int vcx_attention_call_bytes(const vcx_call* c, size_t* bytes) {
  VCX_REQUIRE(bytes != nullptr, "bytes is null");
  if (int rc = check_call(c)) return rc;
  *bytes = call_ws(*c).bytes;
  return VCX_OK;
}

extern "C" int vcx_attention_call(const vcx_call* c, void* stream) {
  if (int rc = check_call(c)) return rc;
  VCX_REQUIRE(c->workspace != nullptr && aligned(c->workspace, 256), "workspace must be non-null and 256-byte aligned");
  const CallWs w = call_ws(*c);
  VCX_REQUIRE(c->workspace_bytes >= 0 && static_cast<size_t>(c->workspace_bytes) >= w.bytes,
              "workspace too small: need %zu bytes", w.bytes);
  const int dtype = static_cast<int>(c->dtype);
  const int64_t* perm = c->perm;
  if (groups(*c)) {
    if (int rc = vcx_group_values(c->v, dtype, c->B, c->H, c->Nk, c->D, c->v_sb, c->v_sh, c->v_sn,
                                  static_cast<int>(c->clusters), static_cast<int>(c->iterations),
                                  static_cast<int>(c->group_mode), nullptr, w.perm, nullptr, nullptr, nullptr,
                                  w.group_scratch, w.group_bytes, stream))
      return rc;
    perm = w.perm;
  }
  double* ksum = reinterpret_cast<double*>(w.v8);
  if (int rc = prepare_together(*c, perm, w.q8, w.qs, w.k8, w.ks, w.v8, w.vs, w.means, ksum, w.km, w.v_scratch, stream))
    return rc;
  if (c->qk_fp8)
    return vcx_attention_fwd_fp8(reinterpret_cast<uint8_t*>(w.q8), reinterpret_cast<uint8_t*>(w.k8), w.v8, w.qs, w.ks,
                                 w.vs, c->B, c->H, c->Nq, c->Nk, c->D, static_cast<int>(c->expcast),
                                 static_cast<float>(c->sm_scale), dtype, c->out, c->o_sb, c->o_sh, c->o_sn, nullptr, 0,
                                 0, stream);
  return vcx_attention_fwd(w.q8, w.k8, w.v8, w.qs, w.ks, w.vs, w.means, c->B, c->H, c->Nq, c->Nk, c->D,
                           static_cast<int>(c->expcast), c->smooth != 0, channel_scales(*c),
                           static_cast<float>(c->sm_scale), dtype, c->out, c->o_sb, c->o_sh, c->o_sn, nullptr, 0, 0,
                           stream);
}
