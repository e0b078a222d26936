// Latent attention of whole prompts (include/vmi_hybrid.h: vmi_hy_latent_prompt): where an entry has no past, its keys and values are the step's own rows, and a head's
// 128 + 64 columns of key and 128 of value, made for all its tokens by one product, are a third of the 576 + 512 that the latent stands for.  csrc/hybrid_latent.hip walks
// the latents, as it must where they come from pages.
//
// A workgroup takes 64 query positions of one head and walks the keys up to its last position in tiles of 64, each through LDS once (requested one tile ahead into registers, two
// barriers a tile, so that three workgroups fit a compute unit).  A wave owns 16 queries for all of it: scores are formed transposed, S^T = K Q^T, so a lane keeps the scores of ONE
// query and its probabilities, as they lie, are the B operand of O^T = V^T P^T: the sum over keys may take them in any order, so k-index 8 kc + e of a step of 32 stands for
// key 4 kc + e (e < 4) and 16 + 4 kc + e - 4, and the V^T operand is read column-wise from LDS in that order.  Sums are a product with ones.  Scores, softmax and accumulators are
// fp32; a probability is rounded once to the element type and what is summed is what multiplies V.  The longest walks come first, over all heads.
//
// Bound by the vector unit's share of the softmax and the chain of a tile (1.4 us).  Attention, us, the latents walked -> here, rank 512: 16 heads, 4 prompts of up to 1024 tokens
// 117 -> 39, 1 of 500 28 + 12 (its splits added up) -> 16, 16 of up to 200 33 -> 15; 8 heads, 1 of 60 14.6 -> 5.8, 35 of up to 21 14.4 -> 5.7, 1 of 1024 45 + 12 -> 26; and one product of the latents
// with both up-projections stands for two by heads, of the same work (16 heads, 2773 rows 27 + 19 us).
// All kernels of a layer between its norms, latents / here, us, prompts only; 16 heads, dim + rot, rank, 1 x 60, 1 x 200, 16 x up to 200, 4 x up to 1024, 1 x 1024: 128 + 64, 512 52 / 44, 70 / 54, 124 / 92, 243 / 137, 153 / 90;
// 128 + 64, 64 46 / 43, 58 / 50, 94 / 88, 164 / 126, 110 / 87; 128 + 32, 64 45 / 42, 58 / 50, 93 / 86, 160 / 120, 106 / 86; 64 + 64, 64 44 / 39, 55 / 44, 86 / 76, 153 / 105, 105 / 75; 64 + 32, 64 44 / 39, 55 / 42, 84 / 72, 145 / 95,
// 103 / 70; so also where a latent row is no longer than a head's columns, as each of 16 ranks and heads measured is, and for prompts of any length: rank 512, 1 x 2 35.2 / 33.7, 1 x 8 42 / 35, 1 x 24 45 / 36, 6 x up to 20 64 / 53.
// Beside entries with a past, which keep the latents and their launches: 64 of those behind 1000 tokens and 1 x 100 111 / 101; 12 behind 300 and 1 x 8, 48, 100, 500 51 / 57, 64 / 68, 72 / 76, 111 / 110.
// Off 64 bits by as much, latents / here, eight draws each: 8 heads, 60 rows 0.00346 / 0.00350, 300 + 200 + 100 0.00355 / 0.00357, 600 0.00364 / 0.00363; 16 heads, 1024 0.00362 / 0.00360.
#include "hybrid_latent_prep.hpp"
#include "hybrid_linear.hpp"
#include "hybrid_softmax.hpp"

namespace vmi_hybrid {

constexpr int PQ = 64;   // queries of a workgroup, keys of a tile

struct LatentPrompt {
  const b16 *proj, *kv, *rows, *gate;
  b16* out;
  const int* tiles;   // [..][2]: entry, first position; NULL: the places of `entries` entries from entry0 on, the last of `places` first
  int64_t ldp, ldkv, ldr, ldg, ldo;
  int heads, rank, row0, tile0;   // kv and rows begin at token row0, a launch at tile tile0
  int places, entry0, entries, mixed;   // mixed: some of them have a past, and are others'
  float scale;
};

// DN + DR columns of a key, the last DR shared by the heads; VD of a value
template <int DN, int DR, int VD>
__global__ __launch_bounds__(256, 2) void latent_prompt_kernel(const LatentPrompt p, const vmi_hy_step s) {
  constexpr int DK = DN + DR, LDK = DK + 8, LDV = VD + 8, NK = DK / 32, NT = VD / 16;
  constexpr int UN = PQ * DN / 2048, UR = PQ * DR / 2048, UV = PQ * VD / 2048;   // units of eight columns a thread
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  b16* ks = reinterpret_cast<b16*>(smem);   // [64][LDK]
  b16* vs = ks + PQ * LDK;                  // [64][LDV]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), kc = lane >> 4, r16 = lane & 15;
  const int group = blockIdx.x / p.heads, h = blockIdx.x - group * p.heads, tile = p.tile0 + group, place = tile / p.entries;
  const int e = p.tiles ? p.tiles[2 * tile] : p.entry0 + tile - place * p.entries, q0 = p.tiles ? p.tiles[2 * tile + 1] : (p.places - 1 - place) * PQ;
  const int qs = s.q_start[e], len = s.q_len[e];
  if (p.mixed && s.ctx[e] != 0) return;
  if (q0 >= len) return;
  const int nkt = (min(len, q0 + PQ) + PQ - 1) / PQ;
  const b16* kv = p.kv + (int64_t)(qs - p.row0) * p.ldkv + h * (DN + VD);
  const b16* shared = p.rows + (int64_t)(qs - p.row0) * p.ldr + p.rank;
  const b16* qrow = p.proj + (int64_t)qs * p.ldp + h * DK;

  b16x8 kn[UN], kr[UR], vr[UV];
  auto load = [&](int kt) {   // (keys past the end repeat the last one: no lane-wise condition around a load)
    auto row = [&](int key) { return (int64_t)min(kt * PQ + key, len - 1); };
#pragma unroll
    for (int i = 0; i < UN; ++i) {
      const int u = tid + 256 * i;
      kn[i] = load8(kv + row(u / (DN / 8)) * p.ldkv + u % (DN / 8) * 8);
    }
#pragma unroll
    for (int i = 0; i < UR; ++i) {
      const int u = tid + 256 * i;
      kr[i] = load8(shared + row(u / (DR / 8)) * p.ldr + u % (DR / 8) * 8);
    }
#pragma unroll
    for (int i = 0; i < UV; ++i) {
      const int u = tid + 256 * i;
      vr[i] = load8(kv + row(u / (VD / 8)) * p.ldkv + DN + u % (VD / 8) * 8);
    }
  };
  load(0);
  const int w0 = q0 + wave * 16;   // this wave's first position
  b16x8 qf[NK];
#pragma unroll
  for (int k = 0; k < NK; ++k) qf[k] = load8(qrow + (int64_t)min(w0 + r16, len - 1) * p.ldp + 32 * k + 8 * kc);
  b16x8 ones;
#pragma unroll
  for (int i = 0; i < 8; ++i) ones[i] = (b16)1.f;
  f32x4 o[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) o[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float mrun = -1e30f, lrun = 0.f;
  const float sc2 = p.scale * 1.4426950408889634f;   // scores in units of log 2

  for (int kt = 0; kt < nkt; ++kt) {
    const int key0 = kt * PQ;
    if (kt > 0) __syncthreads();   // the tile before has been read
#pragma unroll
    for (int i = 0; i < UN; ++i) {
      const int u = tid + 256 * i;
      *reinterpret_cast<b16x8*>(ks + u / (DN / 8) * LDK + u % (DN / 8) * 8) = kn[i];
    }
#pragma unroll
    for (int i = 0; i < UR; ++i) {
      const int u = tid + 256 * i;
      *reinterpret_cast<b16x8*>(ks + u / (DR / 8) * LDK + DN + u % (DR / 8) * 8) = kr[i];
    }
#pragma unroll
    for (int i = 0; i < UV; ++i) {
      const int u = tid + 256 * i;
      *reinterpret_cast<b16x8*>(vs + u / (VD / 8) * LDV + u % (VD / 8) * 8) = vr[i];
    }
    if (kt + 1 < nkt) load(kt + 1);
    __syncthreads();
    if (w0 >= len || key0 > w0 + 15) continue;   // (wave-uniform: none of its queries exists, or sees the tile)
    f32x4 sc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      sc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < NK; ++k) mma(sc[j], load8(ks + (j * 16 + r16) * LDK + 32 * k + 8 * kc), qf[k]);
    }
    if (key0 + PQ - 1 > w0) {   // some query does not see every key
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (key0 + j * 16 + 4 * kc + r > w0 + r16) sc[j][r] = -INFINITY;
    }
    float mx = sc[0][0];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) mx = fmaxf(mx, sc[j][r]);
    auto more = [](float a, float b) { return fmaxf(a, b); };
    mx = fmaxf(mrun, sc2 * vmi_lanes::across32(vmi_lanes::across16(mx, more), more));
    const float alpha = exp2_hw(mrun - mx);
    mrun = mx;
    b16x8 pf[2];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) pf[j >> 1][(j & 1) * 4 + r] = (b16)exp2_hw(fmaf(sc[j][r], sc2, -mx));
    f32x4 sum{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 2; ++k) mma(sum, ones, pf[k]);
    lrun = fmaf(lrun, alpha, sum[0]);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) o[nt] *= alpha;
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const b16* a = vs + (32 * k + 4 * kc + (r16 >> 2)) * LDV + nt * 16 + 4 * (r16 & 3);
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)a);
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(a + 16 * LDV));
        mma(o[nt], __builtin_shufflevector(__builtin_bit_cast(b16x4, lo), __builtin_bit_cast(b16x4, hi), 0, 1, 2, 3, 4, 5, 6, 7), pf[k]);
      }
  }
  const int q = w0 + r16;
  if (q >= len) return;
  const float inv = sigmoid((float)p.gate[(int64_t)(qs + q) * p.ldg + h]) / lrun;
  b16* out = p.out + (int64_t)(qs + q) * p.ldo + h * VD + 4 * kc;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    b16x4 y;
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] = (b16)(o[nt][r] * inv);
    *reinterpret_cast<b16x4*>(out + nt * 16) = y;
  }
}

template <int DN, int DR>
static int launch_prompt(LatentPrompt p, int n_tiles, const vmi_hy_step& s, hipStream_t st) {
  auto* fn = latent_prompt_kernel<DN, DR, DN>;
  constexpr size_t lds = (size_t)PQ * (DN + DR + 8 + DN + 8) * 2;
  if (int rc = allow_lds(fn, lds, "vmi_hy_latent_prompt")) return rc;
  const int most = ((1 << 24) - 1) / p.heads;   // (a launch is of fewer than 2^32 work items)
  for (p.tile0 = 0; p.tile0 < n_tiles; p.tile0 += std::min(most, n_tiles - p.tile0)) {
    hipLaunchKernelGGL(fn, dim3((uint32_t)(p.heads * std::min(most, n_tiles - p.tile0))), dim3(256), lds, st, p, s);
    if (int rc = launched("vmi_hy_latent_prompt")) return rc;
  }
  return VMI_HY_OK;
}

}  // namespace vmi_hybrid

using namespace vmi_hybrid;

extern "C" {

int32_t vmi_hy_latent_prompt_fits(int32_t dim, int32_t rot, int32_t vdim, int32_t rank, int32_t rot_n, int32_t dtype) {
  return dtype == VMI_HY_BF16 && (dim == 64 || dim == 128) && vdim == dim && (rot == 32 || rot == 64) && rank > 0 && (rank & 63) == 0 && rot_n > 0 && (rot_n & 15) == 0 && rot_n <= rot;
}

static int run_prompt(const LatentPrompt& p, int dim, int rot, int64_t tiles, const vmi_hy_step& s, hipStream_t st, const char* who) {
  if (tiles <= 0 || tiles > INT32_MAX || p.heads <= 0 || p.heads > 65535 || !(p.scale > 0.f)) return fail(VMI_HY_E_ARG, who, "a size out of range");
  if (((p.ldp | p.ldkv) & 7) || (p.ldo & 3) || (((uintptr_t)p.proj | (uintptr_t)p.kv | (uintptr_t)p.rows) & 15) || ((uintptr_t)p.out & 7))
    return fail(VMI_HY_E_SHAPE, who, "needs rows aligned to 16 bytes");
  const int n = (int)tiles;
  if (dim == 128) return rot == 64 ? launch_prompt<128, 64>(p, n, s, st) : launch_prompt<128, 32>(p, n, s, st);
  return rot == 64 ? launch_prompt<64, 64>(p, n, s, st) : launch_prompt<64, 32>(p, n, s, st);
}
static const b16* rows_of(const void* p) { return static_cast<const b16*>(p); }

int vmi_hy_latent_prompt(const void* proj, int64_t ldp, const void* kv, int64_t ldkv, const void* rows, const void* gate, int64_t ldg, void* out, int64_t ldo, int32_t heads, int32_t dim,
                         int32_t rot, int32_t vdim, int32_t rank, int32_t max_len, float scale, int32_t dtype, int32_t device, const vmi_hy_step* s, void* stream) {
  static const char* who = "vmi_hy_latent_prompt";
  if (!proj || !kv || !rows || !gate || !out || !s || !s->q_start || !s->q_len || s->T <= 0 || s->B <= 0 || max_len <= 0) return fail(VMI_HY_E_ARG, who, "null pointer or a size out of range");
  if (!vmi_hy_latent_prompt_fits(dim, rot, vdim, rank, 16, dtype)) return fail(VMI_HY_E_SHAPE, who, "built for bfloat16 heads of 64 or 128 beside 32 or 64 rotated columns");
  DeviceScope dev(device);
  if (!dev.ok) return fail(VMI_HY_E_HIP, who, "hipSetDevice failed");
  const int places = (max_len - 1) / PQ + 1;
  const LatentPrompt p{rows_of(proj), rows_of(kv), rows_of(rows), rows_of(gate), static_cast<b16*>(out), nullptr, ldp, ldkv, rank + rot, ldg, ldo, heads, rank, 0, 0, places, 0, s->B, 0, scale};
  return run_prompt(p, dim, rot, (int64_t)places * s->B, *s, static_cast<hipStream_t>(stream), who);
}

int vmi_hy_latent_prompts(const vmi_hy_latent_prep_args* a, const vmi_hy_latent_attention_args* past, const void* w_uk, const void* w_uv, const void* w_kv, const void* gate, int64_t ldg,
                          void* out, int64_t ldo, void* rows, void* kv, const int32_t* tiles, int32_t n_tiles, int32_t max_len, const int32_t span[6], float scale,
                          const vmi_hy_step* s, void* stream) {
  static const char* who = "vmi_hy_latent_prompts";
  if (!a || !w_kv || !gate || !out || !kv || !span || !s || !s->q_start || !s->q_len || s->T <= 0 || s->B <= 0 || span[0] < 0 || span[1] <= span[0] || span[1] > s->T ||
      (tiles ? n_tiles <= 0 : (max_len <= 0 || span[4] < 0 || span[5] <= span[4] || span[5] > s->B)) || span[3] < 0 || (span[3] > 0 && !s->ctx))
    return fail(VMI_HY_E_ARG, who, "null pointer or a size out of range");
  const int first = span[0], n = span[1] - first, at = span[2], others = span[3] == 0 ? 0 : span[3] - at, heads = a->heads, dim = a->dim, rank = a->rank, row = rank + a->rot;
  if (others < 0 || at < 0 || span[3] > s->T || (others && (!past || !w_uk || !w_uv || !a->q || past->q != a->q || !past->out || past->heads != heads || past->rank != rank ||
                                                            past->rot != a->rot || past->dtype != a->dtype || past->device != a->device)))
    return fail(VMI_HY_E_ARG, who, "what the entries beside the prompts take does not fit");
  if (int rc = check_latent_prompt_prep(a, rows, first, others > 0, s, who)) return rc;
  DeviceScope dev(a->device);
  if (!dev.ok) return fail(VMI_HY_E_HIP, who, "hipSetDevice failed");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t ldkv = (int64_t)heads * 2 * dim;
  vmi_hy_linear_args l{};
  l.groups = heads, l.scale = 1.f, l.x_kind = VMI_HY_X_ROWS, l.epilogue = VMI_HY_E_STORE, l.dtype = a->dtype, l.device = a->device;
  if (others) {   // (their rows among the prompts' hold nothing, and give nothing: products are by rows)
    vmi_hy_linear_args uk = l, uv = l;
    uk.x = rows_of(a->proj) + at * a->ldp, uk.w = w_uk, uk.y = static_cast<b16*>(a->q) + (int64_t)at * heads * row, uk.ldx = a->ldp, uk.ldy = (int64_t)heads * row;
    uk.x_gstride = dim + a->rot, uk.y_gstride = row, uk.M = others, uk.N = rank, uk.K = dim;
    uv.x = static_cast<b16*>(past->out) + (int64_t)at * heads * rank, uv.w = w_uv, uv.y = static_cast<b16*>(out) + at * ldo, uv.ldx = (int64_t)heads * rank, uv.ldy = ldo;
    uv.x_gstride = rank, uv.y_gstride = dim, uv.M = others, uv.N = dim, uv.K = rank, uv.epilogue = VMI_HY_E_GATED, uv.gate = rows_of(gate) + at * ldg, uv.ldg = ldg;
    if (int rc = check_linear(&uk, who)) return rc;
    if (int rc = check_linear(&uv, who)) return rc;
    if (int rc = launch_latent_prompt_in(uk, *a, rows, first, others > 0, *s, st, who)) return rc;
    if (int rc = vmi_hy_latent_attention(past, s, st)) return rc;
    if (int rc = vmi_hy_linear(&uv, st)) return rc;
  } else if (int rc = launch_latent_prompt_prep(*a, rows, first, others > 0, *s, st, who)) {
    return rc;
  }
  l.x = rows, l.w = w_kv, l.y = kv, l.ldx = row, l.ldy = ldkv, l.M = n, l.N = (int)ldkv, l.K = rank, l.groups = 1;
  if (int rc = vmi_hy_product_tiles(&l, st)) return rc;
  const int places = tiles ? 0 : (max_len - 1) / PQ + 1, entries = tiles ? 1 : span[5] - span[4];
  const LatentPrompt p{rows_of(a->proj), rows_of(kv), rows_of(rows), rows_of(gate), static_cast<b16*>(out), tiles, a->ldp, ldkv, row, ldg, ldo, heads, rank, first, 0,
                       places, span[4], entries, !tiles && others, scale};
  return run_prompt(p, dim, a->rot, tiles ? n_tiles : (int64_t)places * entries, *s, st, who);
}

}  // extern "C"
